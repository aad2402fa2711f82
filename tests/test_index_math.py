"""Index arithmetic of the kernels and rules of launches (csrc/index_math.h) on the host, at
sizes that no test on a device reaches."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "gpu-rt_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def _run(tmp_path, body):
    """Compiles the body of a host main() against csrc/index_math.h; its output's words."""
    src, exe = tmp_path / "probe.cpp", tmp_path / "probe"
    src.write_text("#include <cstdio>\n#include <vector>\n#include \"index_math.h\"\nusing namespace gpurt_impl;\n"
                   "int main() {\n" + body + "\nreturn 0;\n}\n")
    subprocess.run([HIPCC, "--offload-host-only", "-x", "hip", "-std=c++17", "-O1", "-I", CSRC, str(src), "-o", str(exe)],
                   check=True, timeout=120)
    return subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=60).stdout.split()


def test_64_bit_keys_from_halves(tmp_path):
    """Halves from 2^31 on keep the other half as it is."""
    halves = [0, 1, 0x7FFFFFFF, 0x80000000, 0xFFFFFFFF]
    out = _run(tmp_path, "const unsigned v[] = {" + ", ".join("%du" % h for h in halves) + "};\n"
               "for (unsigned hi : v) for (unsigned lo : v)\n"
               "    printf(\"%llu\\n\", (unsigned long long)u64_of_halves((int)hi, (int)lo));")
    assert [int(x) for x in out] == [hi << 32 | lo for hi in halves for lo in halves]


def test_grid_stride_ends_at_every_32_bit_count(tmp_path):
    """Counts up to 2^32 - 1 with the step of the refit's vertex check (512 blocks of 256): each
    thread sees its indices once and stops."""
    step = 512 * 256
    cases = [(n, first) for n in (1, step, step + 1, 2**32 - step - 1, 2**32 - step, 2**32 - step + 1, 2**32 - 1)
             for first in (0, 1, step - 1)]
    out = _run(tmp_path, "const unsigned c[][2] = {" + ", ".join("{%du, %du}" % c for c in cases) + "};\n"
               "for (auto& k : c) {\n"
               "    unsigned long long seen = 0, last = 0;\n"
               "    grid_stride(k[0], k[1], %d, [&](unsigned i) { seen++; last = i; if (seen > 40000) throw 1; });\n"
               "    printf(\"%%llu %%llu\\n\", seen, last);\n}" % step)
    got = list(zip(map(int, out[::2]), map(int, out[1::2])))
    for (n, first), g in zip(cases, got):
        r = range(first, n, step)
        assert g == (len(r), r[-1] if len(r) else 0)


def test_mesh_of_a_key_in_few_steps(tmp_path):
    """The mesh that holds a batch-wide vertex, from any earlier mesh, with empty meshes
    between; and over 100,000 meshes in a logarithmic number of reads."""
    n_off = [[0, 5], [0, 0, 0, 3], [0, 2, 2, 2, 7, 7], [0, 1, 2, 3, 4, 5, 6, 7, 8, 9], [0, 4, 4, 4, 4, 4, 4, 4, 4, 6, 6, 9]]
    body = "std::vector<std::vector<uint64_t>> offs = {" + ", ".join(
        "{" + ", ".join(map(str, o)) + "}" for o in n_off) + "};\n"
    body += """for (auto& o : offs) {
        const uint32_t n = (uint32_t)o.size() - 1;
        for (uint64_t key = 0; key < o[n]; key++)
            for (uint32_t lo = 0; lo < n && o[lo] <= key; lo++) printf("%u\\n", last_from(o.data(), n, lo, key));
    }
    std::vector<uint64_t> big(100001, 1ull << 40);
    big[0] = 0;
    big[100000] = (1ull << 40) + 8;
    int reads = 0;
    struct Counted {
        const uint64_t* p;
        int* reads;
        uint64_t operator[](uint32_t i) const { return ++*reads, p[i]; }
    };
    printf("%u\\n", last_from(Counted{big.data(), &reads}, 100000, 0, (1ull << 40) + 3));
    printf("%d\\n", reads);
"""
    out = [int(x) for x in _run(tmp_path, body)]
    want = []
    for o in n_off:
        n = len(o) - 1
        for key in range(o[n]):
            m = max(k for k in range(n) if o[k] <= key)
            want += [m for lo in range(n) if o[lo] <= key]
    assert out[:-1] == want + [99999]
    assert out[-1] <= 2 * 17 + 1


def test_waves_of_closest_point_sets(tmp_path):
    """12 waves per CU only for small sets on oriented nodes: from 65,537 points of 256 CUs on,
    and on every other encoding, 16 (12 was up to a half slower there)."""
    n = [1, 65536, 65537, 131072, 196608, 200000, 262144, 262145, 1 << 40]
    out = _run(tmp_path, "for (bool o : {true, false}) for (size_t n : {" + ", ".join("%dull" % k for k in n) + "})\n"
               "    printf(\"%d\\n\", point_waves_per_cu(n, 256, o));")
    assert [int(x) for x in out] == [12 if k <= 65536 else 16 for k in n] + [16] * len(n)


def test_collapse_launches(tmp_path):
    """Launches per tree: the levels that trees of the size have and some, with room below the
    64 supported levels; binary trees of large meshes get more, most with treelets."""
    n = [1, 2, 5000, 65536, 65537, 1_000_000, 2_300_000, (1 << 28) - 9]
    out = _run(tmp_path, "for (unsigned n : {" + ", ".join("%du" % k for k in n) + "})\n"
               "    for (int w : {2, 4, 8}) for (bool t : {false, true}) printf(\"%d\\n\", collapse_launches(n, w, t));")
    got = {(k, w, t): int(out.pop(0)) for k in n for w in (2, 4, 8) for t in (0, 1)}
    assert max(got.values()) < 64 and min(got.values()) >= 2
    assert [got[k, 4, t] for k in (5000, 2_300_000) for t in (0, 1)] == [12, 12, 19, 19]
    assert [got[1_000_000, 2, t] for t in (0, 1)] == [30, 42]
    assert all(got[k, w, 0] == got[k, w, 1] for k in n for w in (2, 4, 8) if w > 2 or k <= 65536)


def test_vertex_sums_rule(tmp_path):
    """The default mode adds in the fixed order from 600,000 terms (200,000 queries) on, and from
    2^21 in a call recorded into a graph; the other modes always and never."""
    n = [0, 3, 3 * 199_999, 3 * 200_000, (1 << 21) - 1, 1 << 21, 1 << 33]
    out = _run(tmp_path, "for (int m : {GPURT_SUMS_AUTO, GPURT_SUMS_FIXED_ORDER, GPURT_SUMS_ATOMIC}) for (bool r : {false, true})\n"
               "    for (size_t n : {" + ", ".join("%dull" % k for k in n) + "}) printf(\"%d\\n\", fixed_order_rule(m, n, r));")
    want = [int(k >= lim) for lim in (600_000, 1 << 21) for k in n] + [1] * 14 + [0] * 14
    assert [int(x) for x in out] == want
