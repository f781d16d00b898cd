"""Host programs made of the library's headers: what the kernels compute with
integers alone can be checked without a device."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def run(tmp_path, body, headers, *args):
    """compiles main() { body } against the library's headers and returns its output;
    a crash (a division by zero, say) or a nonzero exit fails the test"""
    src, exe = os.path.join(str(tmp_path), "check.hip"), os.path.join(str(tmp_path), "check")
    with open(src, "w") as f:
        f.write("#include <cstdio>\n#include <cstdlib>\n#include <vector>\n#include <algorithm>\n#include <cmath>\n"
                "#include <cstring>\n")
        f.writelines(f'#include "{h}"\n' for h in headers)
        f.write(body)
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    subprocess.run([hipcc, "--offload-host-only", "-O1", "-std=c++17", "-w", "-I", os.path.join(ROOT, "qcu_amd", "csrc"),
                    src, "-o", exe], check=True)
    r = subprocess.run([exe, *map(str, args)], capture_output=True, text=True)
    assert r.returncode == 0, f"exit {r.returncode}: {r.stdout}{r.stderr}"
    return r.stdout
