"""The rule that sends an fp32 product to the split-operand GEMM (csrc/gemm_split_rule.h), on the CPU:
what the kernel can't address goes to the vendor library, and what it takes is cut into K ranges
that cover K without an empty one and whose partial products fit the workspace."""
import ctypes
import random
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "inferno_amd" / "csrc"
WS = 32 << 20


@pytest.fixture(scope="module")
def ranges(tmp_path_factory):
    d = tmp_path_factory.mktemp("rule")
    (d / "rule.cpp").write_text(
        '#include "gemm_split_rule.h"\n'
        'extern "C" int ranges(int ta, int tb, int64_t M, int64_t N, int64_t K, int64_t batch, int64_t lda, int64_t ldb,'
        ' size_t ws) { return inf::gemm_split_ranges(ta, tb, M, N, K, batch, lda, ldb, ws); }\n')
    subprocess.run(["g++", "-std=c++17", "-O1", "-fsanitize=undefined", "-fno-sanitize-recover", "-shared", "-fPIC",
                    f"-I{CSRC}", str(d / "rule.cpp"), "-o", str(d / "rule.so")], check=True)
    f = ctypes.CDLL(str(d / "rule.so")).ranges
    f.argtypes = [ctypes.c_int] * 2 + [ctypes.c_int64] * 6 + [ctypes.c_size_t]
    return lambda ta, tb, M, N, K, batch=1, lda=None, ldb=None, ws=WS: f(
        ta, tb, M, N, K, batch, lda or (M if ta else K), ldb or (K if tb else N), ws)


@pytest.mark.parametrize("K", [2**30 + 1, 2**31 - 64, 2**31 - 32, 2**31 - 31, 2**31 - 16, 2**31 - 1, 2**31, 2**33])
@pytest.mark.parametrize("M,N", [(1, 1), (256, 128), (4096, 4096)])
def test_a_k_past_32_bit_steps_goes_to_the_library(ranges, K, M, N):
    assert ranges(1, 0, M, N, K) == 0


@pytest.mark.parametrize("M,N", [(2**30 + 1, 128), (128, 2**30 + 1), (2**31, 2**20), (2**40, 1)])
def test_rows_and_columns_past_32_bits_go_to_the_library(ranges, M, N):
    assert ranges(1, 0, M, N, 64, lda=1 << 20, ldb=1 << 20) == 0


def test_what_the_kernel_cannot_read_goes_to_the_library(ranges):
    assert ranges(0, 0, 4096, 4096, 4096) and ranges(1, 0, 4096, 4096, 4095)
    for ta, tb in ((0, 0), (0, 1), (1, 1)):
        assert ranges(ta, tb, 4096, 4096, 4095) == 0  # a K-contiguous operand, 4 elements at a time
    assert ranges(1, 0, 4096, 4096, 4096, lda=(1 << 20) + 4) == 0 and ranges(1, 0, 4096, 4096, 4096, ldb=(1 << 20) + 4) == 0


def test_ranges_cover_k_and_fit_the_workspace(ranges):
    rng = random.Random(5)
    taken = 0
    for _ in range(4000):
        M, N, K = (int(2 ** rng.uniform(0, e)) for e in (15, 15, 17))
        batch, ws = rng.choice([1, 1, 1, 3, 40]), rng.choice([0, 1 << 20, WS])
        ks = ranges(1, 0, M, N, K, batch=batch, lda=max(M, 1), ldb=max(N, 1), ws=ws)
        assert 0 <= ks <= 8
        if ks:
            taken += 1
            nk = -(-K // 32)
            chunk = -(-nk // ks) * 32
            n = -(-K // chunk)
            assert 1 <= n <= ks and (n - 1) * chunk < K <= n * chunk
            assert ks == 1 or (batch == 1 and ks * M * N * 4 <= ws)
    assert taken > 200
