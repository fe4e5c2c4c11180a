"""The build's check that the kernels which must not spill registers do not
(csrc/spills.awk), on the compiler's own reports: of a kernel that spills, of one
that does not, and of a source without either."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "tealeaf_ref_amd", "csrc")
HIPCC = "/opt/rocm/bin/hipcc"

# N doubles live over a barrier that they cannot be formed after
SOURCE = """
#include <hip/hip_runtime.h>
__global__ __launch_bounds__(1024) void k_%s(double *a) {
  double v[%d];
  for (int i = 0; i < %d; ++i) v[i] = a[i * 1024 + threadIdx.x];
  __syncthreads();
  for (int i = 0; i < %d; ++i) a[((i * 7) %% %d) * 1024 + threadIdx.x] = v[i] * v[(i + 5) %% %d];
}
"""


def _check(report, *options):
    return subprocess.run(["awk", *[x for o in options for x in ("-v", o)], "-f",
                           os.path.join(CSRC, "spills.awk"), str(report)],
                          capture_output=True, text=True)


@pytest.mark.skipif(not shutil.which(HIPCC), reason="needs hipcc")
@pytest.mark.parametrize("n,spills", [(8, False), (120, True)])
def test_compiler_reports(tmp_path, n, spills):
    src = tmp_path / "k.hip"
    src.write_text(SOURCE % ("res_c", n, n, n, n, n))
    r = subprocess.run([HIPCC, "-O3", "--offload-arch=gfx950", "-Rpass-analysis=kernel-resource-usage",
                        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                        "-c", str(src), "-o", str(tmp_path / "k.o")], capture_output=True, text=True,
                       check=True)
    report = tmp_path / "k.res"
    report.write_text(r.stderr)
    got = _check(report, "KERNELS=k_res_[cjp]", "VECTORS=1")
    assert (got.returncode != 0) == spills, got.stdout
    assert ("k_res_c" in got.stdout and "Spill" in got.stdout) == spills
    # a kernel that is not watched may; and none watched is a fault of the check
    assert _check(report, "KERNELS=k_deep_", "SCALARS=1").returncode != 0
    assert "no kernel" in _check(report, "KERNELS=k_deep_").stdout


def test_each_rule(tmp_path):
    """Vector moves, scalar moves and scratch, each alone."""
    for line, options, fails in (
            ("VGPRs Spill: 4", ("VECTORS=1",), True), ("VGPRs Spill: 4", ("SCALARS=1",), False),
            ("SGPRs Spill: 9", ("VECTORS=1",), False), ("SGPRs Spill: 9", ("SCALARS=1",), True),
            ("ScratchSize [bytes/lane]: 16", (), True), ("VGPRs: 256", ("VECTORS=1",), False)):
        report = tmp_path / "r"
        report.write_text("a.hpp:1:1: remark: Function Name: _Z6k_deep_x [-Rpass]\n"
                          f"a.hpp:1:1: remark:     {line} [-Rpass]\n")
        assert (_check(report, "KERNELS=k_deep_", *options).returncode != 0) == fails, line


def test_the_build_uses_it():
    """The rules of the sources that hold such kernels; their reports, where they
    have been built, pass."""
    make = open(os.path.join(CSRC, "Makefile")).read()
    for name, options in (("tl_resident", ("KERNELS=k_res_[cjp]", "VECTORS=1")),
                          ("tl_loops", ("KERNELS=k_deep_", "SCALARS=1")),
                          ("tl_mixed", ("KERNELS=k_deep_", "SCALARS=1"))):
        rule = next(l for l in make.splitlines() if f"{name}.o" in l and "WATCH" in l)
        assert all(f"-v {o}" in rule for o in options)
        report = os.path.join(CSRC, "_build", name + ".res")
        if os.path.exists(report):
            got = _check(report, *options)
            assert got.returncode == 0, got.stdout
