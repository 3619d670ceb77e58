"""Every address that the direct-load GEMM tiles ask for, walked on the host by the functions the device code calls: nothing
outside the operands' allocations is read, and every element that counts comes from where it lies.  No GPU."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    compiler = shutil.which("g++")
    assert compiler, "needs a host C++ compiler"
    exe = str(tmp_path_factory.mktemp("gemm") / "check")
    subprocess.run([compiler, "-O2", "-std=c++17", "-Wall", "-Werror", os.path.join(HERE, "gemm_addresses_check.cpp"), "-o", exe], check=True)
    return lambda *args: subprocess.run([exe, *map(str, args)], stdout=subprocess.PIPE, text=True)


# M, N, K, layout (0 = B (K,N), 1 = B (N,K), 2 = A (K,M)), gap behind the rows of A and of B, rows of B missing, split of K
CASES = [
    (1000, 200, 4104, 0, 0, 0, 0, 8), (1000, 200, 4104, 1, 0, 0, 0, 8), (1000, 200, 4101, 2, 0, 0, 0, 8),   # K in parts, the last with a tail
    (129, 264, 2056, 0, 0, 0, 5, 3), (64, 128, 1160, 1, 0, 0, 0, 2), (65, 131, 1160, 1, 24, 8, 0, 2), (8, 8, 129, 2, 0, 0, 0, 2),
    (300, 264, 72, 0, 0, 0, 0, -2), (257, 258, 104, 1, 0, 0, 0, -2), (300, 264, 72, 0, 8, 16, 0, -2),                # K in halves
    (1, 8, 8, 0, 0, 0, 0, 0), (1, 1, 8, 1, 0, 0, 0, 0), (8, 8, 1, 2, 0, 0, 0, 0), (131, 264, 72, 0, 0, 0, 7, 0),      # one workgroup per tile
    (131, 259, 200, 1, 0, 0, 0, 0), (131, 259, 200, 1, 8, 40, 0, 0), (131, 264, 200, 0, 8, 40, 0, 0), (136, 264, 33, 2, 0, 0, 0, 0),
    (1, 8, 32, 0, 0, 0, 0, -3), (129, 136, 96, 0, 0, 0, 0, -3), (300, 264, 64, 0, 0, 0, 0, -3), (129, 131, 96, 1, 0, 0, 0, -3), (257, 1, 32, 1, 0, 0, 0, -3),   # three planes
    (45, 33, 70, 2, 3, 7, 0, 0),                                                                                     # ragged, rows padded to chunks
]


@pytest.mark.parametrize("M,N,K,layout,gap_a,gap_b,missing,split", CASES)
def test_no_read_outside_the_operands(check, M, N, K, layout, gap_a, gap_b, missing, split):
    lda, ldb = (M if layout == 2 else K) + gap_a, (K if layout == 1 else N) + gap_b
    assert lda % 8 == 0 and ldb % 8 == 0
    got = check(M, N, K, lda, ldb, layout, K - missing, split)
    assert got.returncode == 0, got.stdout


@pytest.mark.parametrize("M,N,K,layout,gap_a,gap_b,split", [(1000, 200, 4104, 0, 0, 0, 8), (64, 128, 1160, 1, 0, 0, 2), (300, 264, 72, 0, 0, 0, -2),
                                                           (131, 259, 200, 1, 8, 40, 0)])
def test_buffers_sized_by_their_strides_would_be_too_long(check, M, N, K, layout, gap_a, gap_b, split):
    """rows * stride as the buffer's size: a part's end lies k0 elements past the operand's, the gap behind the last row inside it."""
    got = check(M, N, K, K + gap_a, (K if layout == 1 else N) + gap_b, layout, K, split, 1)
    assert got.returncode == 1 and "reads up to element" in got.stdout
