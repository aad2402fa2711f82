"""Index arithmetic of the kernels (csrc/index_math.h) on the host, at sizes that no test on
a device reaches."""
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
