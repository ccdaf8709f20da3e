"""Launch bookkeeping on the CPU: kg_runtime.hip and kg_launch() built for the host
alone, against a HIP whose launches the test makes fail."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]

HIP = r'''
#include "%(csrc)s/kg_internal.h"
#include <cstdio>

static hipError_t fail_with = hipSuccess, last = hipSuccess;
extern "C" {
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipExtLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t, hipEvent_t, hipEvent_t, int)
{
    if (fail_with != hipSuccess) last = fail_with;   // an error stays until it is asked for
    return fail_with;
}
hipError_t hipGetLastError(void)
{
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t) { return "made to fail"; }
}

static void kern(int) {}

static int launch(kg_ctx* c, unsigned blocks = 1)
{
    if (int rc = kg_launch_begin(c, "kern")) return rc;
    kg_launch(c, kern, dim3(blocks), dim3(256), 0, 1);
    return kg_launch_end(c);
}

int main()
{
    kg_ctx c{};
%(body)s
}
'''


def run(tmp_path, body):
    csrc = ROOT / "kernelgen-perf-tests_amd" / "csrc"
    src = tmp_path / "t.hip"
    src.write_text(HIP % {"csrc": csrc, "body": body})
    flags = ["--offload-host-only", "-std=c++17", "-O1", "-w"]
    preload = tmp_path / "p.hip"
    names = "stencil3d tricubic stencil2d matmul util life typed batch poisson vecmath".split()
    preload.write_text(f'#include "{csrc}/kg_internal.h"\n'
                       + "".join(f"int kg_preload_{n}() {{ return 0; }}\n" for n in names)
                       + "size_t kg_stats_scratch_bytes() { return 8; }\nint kg_poisson_static_setup(int) { return 0; }\n")
    exe = tmp_path / "t"
    objs = []
    for s in (src, preload, csrc / "kg_runtime.hip"):
        o = tmp_path / (s.stem + ".o")
        subprocess.run(["/opt/rocm/bin/hipcc", *flags, "-c", str(s), "-o", str(o)], check=True, timeout=120)
        objs.append(str(o))
    subprocess.run(["/opt/rocm/bin/hipcc", *objs, "-o", str(exe)], check=True, timeout=120)
    return subprocess.run([str(exe)], capture_output=True, text=True, timeout=60).stdout.split()


def test_a_failed_launch_is_not_the_next_ones_error(tmp_path):
    got = run(tmp_path, r'''
    const int a = launch(&c);
    fail_with = hipErrorInvalidConfiguration;
    const int b = launch(&c);
    fail_with = hipSuccess;
    const int d = launch(&c);
    printf("%d %d %d\n", a == KG_OK, b == KG_ERR_HIP, d == KG_OK);
''')
    assert got == ["1", "1", "1"]
