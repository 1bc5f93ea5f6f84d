"""The workgroup factorization of a diagonal block (potrf_block) with its waves
in either order between barriers.

The device code is compiled for the CPU (tests/emul): every lane a fiber, a
wave's lanes in lockstep at its cross-lane operations, and the four waves one
after the other from barrier to barrier, first 0, 1, 2, 3, then 3, 2, 1, 0.  Any
two waves that touch one LDS entry without a barrier between meet in both
orders, so the factor and the inverse are right, and the same bit for bit, only
if every such access is ordered.  Widths: one panel, part of one, all four.
"""
import pathlib
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parent.parent
CLANG = pathlib.Path("/opt/rocm/llvm/bin/clang++")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not CLANG.exists():
        pytest.skip(f"{CLANG} not installed")
    out = tmp_path_factory.mktemp("emul") / "diag_block"
    subprocess.run([CLANG, "-x", "c++", "-std=c++17", "-O2", "-w", f"-I{ROOT / 'tests' / 'emul'}",
                    f"-I{ROOT / 'suitesparse_amd' / 'csrc'}", ROOT / "tests" / "emul" / "diag_block.cpp",
                    "-o", out], check=True)
    return out


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nb", [9, 16, 17, 37, 48, 64])
def test_factor_and_inverse_do_not_depend_on_wave_order(program, precision, nb):
    out = subprocess.run([program, precision, str(nb)], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout + out.stderr


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nb,bad", [(9, 0), (16, 15), (37, 20), (64, 5), (64, 63)])
def test_non_positive_pivot_is_replaced_by_one(program, precision, nb, bad):
    """The factor and the inverse of a block with a negative diagonal entry stay
    finite: the pivot is reported and 1 takes its place."""
    out = subprocess.run([program, precision, str(nb), str(bad)], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout + out.stderr


def test_published_block_is_released_by_every_wave(program):
    """The flag of a folding tail says that the block's L and inverse are in memory
    for workgroups on other CUs: every wave has released its own stores before it."""
    out = subprocess.run([program, "publish"], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout + out.stderr
