"""The fp32 GEMM on three bf16 parts per operand (gemm_split.hip), at the sizes where a tile, a K step,
a K range or the route to the vendor library ends, and at magnitudes far apart, against 64-bit torch.

Bar: operands are held exactly, a product of them is within 2^-25 and an MFMA rounds 16 of them at
once, so a result lies within a few 1e-7 of the norm of its terms; with terms of either sign
that norm is the result's own on average: 2e-6 (measured 1e-7 to 7e-7, what fp32 sums give too)."""
import math

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

BAR = 2e-6


@pytest.fixture(scope="module")
def ia():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import inferno_amd

    inferno_amd.lib()
    return inferno_amd


def make(M, N, K, ta, tb, seed=0, pad=0):
    g = torch.Generator().manual_seed(seed)
    def mat(r, c):
        return torch.randn((r, c + pad), generator=g).cuda()[:, :c]
    return mat(*((K, M) if ta else (M, K))), mat(*((N, K) if tb else (K, N)))


def ref(a, b, ta, tb):
    return (a.double().t() if ta else a.double()).contiguous() @ (b.double().t() if tb else b.double()).contiguous()


def rel(x, r):
    return ((x.double() - r).norm() / r.norm()).item()


# whole and ragged 256 x 128 tiles; K steps whole and ragged (K % 4 != 0 goes to
# the library unless both operands are K-strided); one
# range of K and several; operands wider than their rows
@pytest.mark.parametrize("M,N,K", [(2048, 1536, 768), (2049, 1537, 776), (2303, 1023, 1000), (1793, 1665, 2056),
                                   (300, 2900, 4108), (770, 3070, 8192), (1999, 2001, 1001), (257, 129, 20000)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("pad", [0, 12])
def test_sizes(ia, M, N, K, ta, tb, pad):
    print(f"[case] gemm split M{M} N{N} K{K} ta{ta} tb{tb} pad{pad}", flush=True)
    a, b = make(M, N, K, ta, tb, pad=pad)
    bias = torch.randn(N, device="cuda")
    out = torch.full((M, N), math.nan, device="cuda")
    got = ia.gemm(a, b, trans_a=bool(ta), trans_b=bool(tb), bias=bias, out=out)
    r = ref(a, b, ta, tb)
    assert rel(got, r + bias.double()) <= BAR
    again = ia.gemm(a, b, trans_a=bool(ta), trans_b=bool(tb), bias=bias)
    assert torch.equal(got, again)  # sums in one order
    c = torch.randn(M, N, device="cuda")
    want = 0.5 * c.double() - 2.0 * r
    assert rel(ia.gemm(a, b, trans_a=bool(ta), trans_b=bool(tb), alpha=-2.0, beta=0.5, out=c), want) <= BAR


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_rows_of_any_magnitude(ia, ta, tb):
    """Rows of A and columns of B scaled over 2^60, and K growing by 2^40 along the sum: every row
    and column keeps its own precision, and the accumulators follow the growing scale."""
    M, N, K = 2048, 1600, 1024
    a, b = make(M, N, K, ta, tb, seed=1)
    rs = torch.exp2(torch.linspace(-30, 30, M, device="cuda"))
    cs = torch.exp2(torch.linspace(30, -30, N, device="cuda"))
    a = a * (rs if ta else rs[:, None])
    b = b * (cs[:, None] if tb else cs)
    r = ref(a, b, ta, tb)
    got = ia.gemm(a, b, trans_a=bool(ta), trans_b=bool(tb))
    scaled = (got.double() - r) / rs.double()[:, None] / cs.double()
    base = r / rs.double()[:, None] / cs.double()
    assert (scaled.norm(dim=1) / base.norm(dim=1)).max() <= BAR and (scaled.norm(dim=0) / base.norm(dim=0)).max() <= BAR
    grow = torch.exp2(torch.linspace(-20, 20, K, device="cuda"))
    a2 = a * (grow[:, None] if ta else grow)
    r2 = ref(a2, b, ta, tb)
    got2 = ia.gemm(a2, b, trans_a=bool(ta), trans_b=bool(tb))
    e = (got2.double() - r2) / rs.double()[:, None] / cs.double()
    assert (e.norm(dim=1) / (r2 / rs.double()[:, None] / cs.double()).norm(dim=1)).max() <= BAR


@pytest.mark.parametrize("ea,eb", [(118, -118), (-118, 118), (118, -20), (-100, 20)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 1)])
def test_operands_at_the_ends_of_the_range(ia, ta, tb, ea, eb):
    """One operand near the largest floats, the other near the smallest: their products are ordinary
    numbers, and nothing on the way to them overflows or underflows."""
    a, b = make(2048, 1600, 1024, ta, tb, seed=4)
    a, b = a * 2.0**ea, b * 2.0**eb
    got = ia.gemm(a, b, trans_a=bool(ta), trans_b=bool(tb))
    assert got.isfinite().all() and rel(got, ref(a, b, ta, tb)) <= BAR


def test_nonfinite(ia):
    """Infinities and NaN reach the results that they reach in fp32, as what they are there."""
    M, N, K = 2048, 1600, 1024
    a, b = make(M, N, K, 0, 0, seed=2)
    clean = ia.gemm(a, b)
    a[100, 7] = math.inf
    b[9, 200] = math.nan
    a[:, 11] = a[:, 11].abs() + 0.1
    base = ia.gemm(a, b)
    b[11, 300] = -math.inf
    got = ia.gemm(a, b)
    keep_m = [i for i in range(M) if i != 100]
    keep_n = [i for i in range(N) if i not in (200, 300)]
    want = ref(a, b, 0, 0)
    assert rel(got[keep_m][:, keep_n], want[keep_m][:, keep_n]) <= BAR
    assert torch.isnan(got[:, 200]).all() and torch.isneginf(got[keep_m][:, 300]).all()
    sign = torch.sign(b[7]).double()
    fin = torch.tensor(keep_n, device="cuda")
    assert torch.equal(got[100][fin].double(), (sign * math.inf)[fin])
    assert clean.isfinite().all() and base.shape == got.shape


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_sums_of_results(ia, ta, tb):
    """Sums over thousands of results (a bias gradient): rounding that favours one direction would add
    up there, independent rounding stays at the error of one result."""
    a, b = make(8192, 2048, 768, ta, tb, seed=3)
    r, got = ref(a, b, ta, tb), ia.gemm(a, b, trans_a=bool(ta), trans_b=bool(tb)).double()
    for d in (0, 1):
        assert ((got.sum(d) - r.sum(d)).norm() / r.sum(d).norm()).item() <= 8e-7  # twice the measured 2e-7 to 4e-7


def test_batched(ia):
    B, M, N, K = 8, 512, 768, 512
    a = torch.randn(B, M, K, device="cuda")
    b = torch.randn(B, K, N, device="cuda")
    c = torch.empty(B, M, N, device="cuda")
    ws = torch.empty(ia.nn_workspace_bytes(ia.OP_GEMM), dtype=torch.uint8, device="cuda")
    st = ia.lib().inf_gemm(0, 0, M, N, K, 1.0, a.data_ptr(), K, M * K, b.data_ptr(), N, K * N, 0.0, c.data_ptr(), N,
                           M * N, B, None, ia.INF_F32, ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream)
    assert st == 0
    for i in range(B):
        assert rel(c[i], ref(a[i], b[i], 0, 0)) <= BAR


@pytest.mark.parametrize("e", [10, 13, 15, 30])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_columns_of_a_against_rows_of_b(ia, ta, tb, e):
    """Columns of A and rows of B scaled against each other by up to 2^e either way, in any order
    (features in unlike units with weights learnt for them): the terms are of one size again, so
    every row and column of C is as exact as without the scales."""
    M, N, K = 2048, 1600, 1024
    a, b = make(M, N, K, ta, tb, seed=6)
    s = torch.exp2(torch.linspace(-e, e, K).round()[torch.randperm(K, generator=torch.Generator().manual_seed(e))]).cuda()
    a = a * (s[:, None] if ta else s)
    b = b / (s if tb else s[:, None])
    got, r = ia.gemm(a, b, trans_a=bool(ta), trans_b=bool(tb)), ref(a, b, ta, tb)
    d = got.double() - r
    assert (d.norm(dim=1) / r.norm(dim=1)).max() <= BAR and (d.norm(dim=0) / r.norm(dim=0)).max() <= BAR


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_products_with_a_permutation_are_exact(ia, ta, tb):
    """A times a permutation matrix is A's columns in that order, bit for bit, whatever stands beside an
    element in its row: an outlier of 2^40, zeros, subnormal numbers; and a permutation times B."""
    M, N, K = 2048, 1536, 1536
    a, b = make(M, N, K, ta, tb, seed=7)
    a = a.contiguous()
    rows = a if not ta else a.t()
    rows[:, 0] = 2.0**40
    rows[5] *= 1e-38
    rows[7] = torch.tensor([2.0**-149, -3 * 2.0**-140, 0.0, 1.0]).cuda().repeat(K // 4)
    rows[9] *= 1e25
    perm = torch.randperm(K, generator=torch.Generator().manual_seed(8)).cuda()
    eye = torch.zeros(K, K, device="cuda")
    eye[perm, torch.arange(K, device="cuda")] = 1.0  # column j picks element perm[j]
    got = ia.gemm(a, eye.t().contiguous() if tb else eye, trans_a=bool(ta), trans_b=bool(tb))
    assert torch.equal(got, rows[:, perm])
    pick = torch.zeros(M, K, device="cuda")
    src = torch.randint(0, K, (M,), generator=torch.Generator().manual_seed(9)).cuda()
    pick[torch.arange(M, device="cuda"), src] = 1.0
    b = b.contiguous()
    cols = b if not tb else b.t()
    cols[0] = -(2.0**40)
    got = ia.gemm(pick.t().contiguous() if ta else pick, b, trans_a=bool(ta), trans_b=bool(tb))
    assert torch.equal(got, cols[src])


def test_results_past_the_operands_factors(ia):
    """Results and operands whose size times the kernel's factors is past the largest float."""
    M, N, K = 2048, 1600, 1024
    for ea, eb in ((110, 10), (60, 40), (10, 110), (126, -126)):
        a, b = make(M, N, K, 0, 0, seed=10)
        a, b = a.clamp(-1.9, 1.9) * 2.0**ea, b.clamp(-1.9, 1.9) * 2.0**eb
        got = ia.gemm(a, b)
        assert got.isfinite().all() and rel(got, ref(a, b, 0, 0)) <= BAR, (ea, eb)


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(2048, 1600, 1024), (2049, 1537, 776), (770, 3070, 8192)])
def test_results_beside_nonfinite_ones(ia, ta, tb, M, N, K):
    """Infinities of one sign in a row and NaN in a column, in the middle and at the ragged ends (the last
    row, column and k): what they don't reach, in the same tile and K range, is an ordinary result."""
    a, b = make(M, N, K, ta, tb, seed=11)
    rows, cols = (a.t() if ta else a), (b.t() if tb else b)
    rows[100, K - 1] = math.inf
    rows[M - 1, 3] = -math.inf
    cols[K - 1, N - 1] = math.nan
    got = ia.gemm(a, b, trans_a=bool(ta), trans_b=bool(tb))
    km = [i for i in range(M) if i not in (100, M - 1)]
    want = ref(a, b, ta, tb)
    assert rel(got[km, :N - 1], want[km, :N - 1]) <= BAR
    assert torch.isnan(got[:, N - 1]).all()
    assert torch.equal(got[100, :N - 1], torch.sign(cols[K - 1, :N - 1]) * math.inf)
    assert torch.equal(got[M - 1, :N - 1], torch.sign(cols[3, :N - 1]) * -math.inf)
