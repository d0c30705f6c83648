"""The fp32 attention kernels' products on three bf16 parts per operand: magnitudes far from 1 and
far apart, within a tile, a row or a column, blocks of zeros, non-finite inputs, and the sizes where
a tile, a key block or the choice between the wide and the narrow backward ends, against 64-bit torch.

Bar: operands are held exactly and a product of them is within 2^-25, so a score carries the fp32
rounding of its sum, below 2^-22 of the largest score's terms (at most ~8 here, so a probability is
within ~2e-6 absolutely); sums over keys and queries add rounding of either sign.  1e-5 of a tensor's
norm is several times what such errors add up to (measured: 2e-7 to 7e-7), and a part dropped shows
at 1e-4 or more.
"""
import math

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

BAR = 1e-5


@pytest.fixture(scope="module")
def ia():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import inferno_amd

    inferno_amd.lib()
    return inferno_amd


def make(B, H, Tq, Tk, D, seed=0, qs=1.0, ks=1.0, vs=1.0, gs=1.0):
    g = torch.Generator().manual_seed(seed)
    rn = lambda t, s: (torch.randn((B, H, t, D), generator=g) * s).cuda()
    return rn(Tq, qs), rn(Tk, ks), rn(Tk, vs), rn(Tq, gs)


def exact(q, k, v, do, scale, causal=True):
    q, k, v, do = (x.double().requires_grad_(n < 3) for n, x in enumerate((q, k, v, do)))
    Tq, Tk = q.shape[2], k.shape[2]
    s = (q.unsqueeze(3) * k.unsqueeze(2)).sum(-1) * scale if Tq * Tk < 20000 else torch.matmul(
        q, k.transpose(2, 3).contiguous()) * scale
    if causal:
        s = s.masked_fill(torch.ones(Tq, Tk, dtype=torch.bool, device="cuda").triu(1 + Tk - Tq), -math.inf)
    o = torch.matmul(torch.softmax(s, -1), v)
    o.backward(do)
    return o.detach(), torch.logsumexp(s, -1).detach(), q.grad, k.grad, v.grad


def rel(x, r):
    return ((x.double() - r).norm() / r.norm()).item()


def run(ia, q, k, v, do, scale, causal=True):
    o, lse = ia.attn_fwd(q, k, v, causal=causal, scale=scale)
    return (o, lse, *ia.attn_bwd(q, k, v, o, do, lse, causal=causal, scale=scale))


# edges of the 32 / 64 / 128 / 256-row and -key tiles, one and several key blocks, small grids
# (128 keys per backward workgroup) and a larger one (256), causal and not, Tq < Tk
@pytest.mark.parametrize("B,H,Tq,Tk,D,causal", [
    (1, 1, 1, 1, 32, False), (1, 2, 31, 33, 64, True), (2, 1, 65, 127, 32, True), (1, 2, 129, 129, 128, True),
    (1, 3, 255, 257, 64, True), (2, 2, 257, 257, 32, True), (1, 1, 300, 513, 64, True), (1, 2, 40, 300, 64, False),
    (2, 8, 1030, 1030, 64, True), (3, 16, 520, 520, 32, True), (1, 2, 513, 515, 128, True), (8, 16, 300, 300, 64, False),
])
@pytest.mark.parametrize("det", [False, True])
def test_sizes(ia, B, H, Tq, Tk, D, causal, det):
    print(f"[case] split sizes B{B} H{H} Tq{Tq} Tk{Tk} D{D} causal={causal} det={det}", flush=True)
    q, k, v, do = make(B, H, Tq, Tk, D)
    c = 1 / math.sqrt(D)
    ia.set_deterministic(det)
    try:
        got = run(ia, q, k, v, do, c, causal)
    finally:
        ia.set_deterministic(False)
    for n, x, r in zip(("o", "lse", "dq", "dk", "dv"), got, exact(q, k, v, do, c, causal)):
        if r.norm() > 1e-12:  # one key: dq and dk are 0
            assert rel(x, r) <= BAR, n


# q and k scaled against each other (the scores stay), values and gradients of any magnitude
@pytest.mark.parametrize("qs,ks,vs,gs", [(1e-6, 1e6, 1.0, 1e-8), (3e4, 3e-5, 1e-12, 1.0), (1e-15, 1e15, 1e10, 1e-15),
                                         (7.9, 0.13, 31.9, 32.1)])
@pytest.mark.parametrize("D", [32, 64, 128])
def test_magnitudes(ia, qs, ks, vs, gs, D):
    q, k, v, do = make(1, 3, 300, 300, D, seed=1, qs=qs, ks=ks, vs=vs, gs=gs)
    c = 1 / math.sqrt(D)
    for det in (False, True):
        ia.set_deterministic(det)
        try:
            got = run(ia, q, k, v, do, c)
        finally:
            ia.set_deterministic(False)
        for n, x, r in zip(("o", "lse", "dq", "dk", "dv"), got, exact(q, k, v, do, c)):
            assert rel(x, r) <= BAR, (n, det)


def test_classes_grow(ia):
    """Magnitudes that grow along the sequence by 2^40: the running scales of K, V, dS and the
    accumulators kept in their units move several times, and every row's O keeps its precision."""
    q, k, v, do = make(1, 2, 700, 700, 64, seed=2)
    grow = torch.exp2(torch.linspace(-20, 20, 700, device="cuda")).view(1, 1, -1, 1)
    v, do = v * grow, do / grow
    c = 0.125
    got, ref = run(ia, q, k, v, do, c), exact(q, k, v, do, c)
    row = ((got[0].double() - ref[0]).norm(dim=-1) / ref[0].norm(dim=-1)).max().item()
    assert row <= BAR
    for n, x, r in zip(("lse", "dq", "dk", "dv"), got[1:], ref[1:]):
        assert rel(x, r) <= BAR, n


@pytest.mark.parametrize("D", [32, 64, 128])
def test_nonfinite_forward(ia, D):
    """A key that scores -inf has probability 0; +inf or NaN spoils the rows that see it and no
    other; an infinite value reaches the rows that see it as an infinity."""
    q, k, v, _ = make(1, 2, 400, 400, D, seed=3)
    c = 1 / math.sqrt(D)
    q[..., 0] = q[..., 0].abs() + 0.1
    clean, clean_lse = ia.attn_fwd(q, k, v, scale=c)
    k2 = k.clone()
    k2[:, :, 250, 0] = -math.inf
    o, lse = ia.attn_fwd(q, k2, v, scale=c)
    hidden = k.clone()
    hidden[:, :, 250] = 0
    s = torch.matmul(q.double(), hidden.double().transpose(2, 3).contiguous()) * c
    s[..., 250] = -math.inf
    s = s.masked_fill(torch.ones(400, 400, dtype=torch.bool, device="cuda").triu(1), -math.inf)
    assert rel(o, torch.matmul(torch.softmax(s, -1), v.double())) <= BAR
    assert rel(lse, torch.logsumexp(s, -1)) <= BAR
    for bad in (math.inf, math.nan):
        k3 = k.clone()
        k3[:, :, 250, 0] = bad
        o, lse = ia.attn_fwd(q, k3, v, scale=c)
        assert torch.isnan(o[:, :, 250:]).all() and torch.isnan(lse[:, :, 250:]).all()
        assert rel(o[:, :, :250], clean[:, :, :250].double()) <= BAR
        assert rel(lse[:, :, :250], clean_lse[:, :, :250].double()) <= BAR
    v2 = v.clone()
    v2[:, :, 250, 3] = math.inf
    o, _ = ia.attn_fwd(q, k, v2, scale=c)
    assert torch.isposinf(o[:, :, 250:, 3]).all()
    rest = [i for i in range(D) if i != 3]
    assert rel(o[..., rest], clean[..., rest].double()) <= BAR and rel(o[:, :, :250], clean[:, :, :250].double()) <= BAR


def test_nonfinite_gradient_stays_local(ia):
    """An infinity in one dO row makes that row's dQ and the sums over queries non-finite; the other
    rows' dQ keep their precision (the infinity does not set the head's scale)."""
    q, k, v, do = make(1, 2, 300, 300, 64, seed=4)
    o, lse = ia.attn_fwd(q, k, v)
    ref = ia.attn_bwd(q, k, v, o, do, lse)
    do[:, :, 100, 5] = math.inf
    dq, dk, dv = ia.attn_bwd(q, k, v, o, do, lse)
    keep = [i for i in range(300) if i != 100]
    assert rel(dq[:, :, keep], ref[0][:, :, keep].double()) <= BAR
    assert not torch.isfinite(dq[:, :, 100]).all() and not torch.isfinite(dv[:, :, :101, 5]).any()


def row_err(x, r, skip=None):
    """The largest relative error of a row (2-norms over the last dim; rows of zeros must be zeros)."""
    d, n = (x.double() - r).norm(dim=-1), r.norm(dim=-1)
    e = torch.where(n > 0, d / n.clamp(min=1e-300), d)
    if skip is not None:
        e = e[..., skip:]
    return e.max().item() if e.isfinite().all() else math.inf


def both_modes(ia, q, k, v, do, scale, causal=True):
    for det in (False, True):
        ia.set_deterministic(det)
        try:
            yield det, run(ia, q, k, v, do, scale, causal)
        finally:
            ia.set_deterministic(False)


# Blocks of zero keys (padding) where a wave's, a pair's or a tile's keys are: an all-zero operand beside
# ordinary ones.  Wide key blocks (64 keys to a pair of waves, else 32): D = 32 with (8, 16), D = 64 with
# (24, 12), both without a mask with (8, 16).
@pytest.mark.parametrize("B,H", [(1, 3), (8, 16), (24, 12)])
@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("what", ["k", "v", "kv"])
def test_zero_key_blocks(ia, B, H, D, causal, what):
    c = 1 / math.sqrt(D)
    for a, n in ((0, 64), (64, 64), (32, 32), (96, 32), (128, 128), (192, 108)):
        print(f"[case] zero {what} keys {a}..{a + n - 1} B{B} H{H} D{D} causal={causal}", flush=True)
        q, k, v, do = make(B, H, 300, 300, D, seed=5)
        for t, name in ((k, "k"), (v, "v")):
            if name in what:
                t[:, :, a:a + n] = 0
        want = exact(q, k, v, do, c, causal)
        for det, got in both_modes(ia, q, k, v, do, c, causal):
            for n_, x, r in zip(("o", "lse", "dq", "dk", "dv"), got, want):
                assert torch.isfinite(x).all() and rel(x, r) <= BAR, (n_, det)


@pytest.mark.parametrize("D", [32, 64, 128])
def test_probabilities_that_underflow(ia, D):
    """Scores hundreds apart: whole blocks of keys have probabilities of 0 or next to it for every query.
    A score of 300 is rounded by up to 2^-16, which moves its probability by as much: 1e-4."""
    q, k, v, do = make(1, 3, 300, 300, D, seed=6, qs=8.0, ks=8.0)
    c = 1 / math.sqrt(D)
    q[..., 0] = q[..., 0].abs() + 8
    k[:, :, 64:128, 0] -= 300 * math.sqrt(D) / 8
    want = exact(q, k, v, do, c)
    for det, got in both_modes(ia, q, k, v, do, c):
        for n_, x, r in zip(("o", "lse", "dq", "dk", "dv"), got, want):
            assert torch.isfinite(x).all() and rel(x, r) <= 1e-4, (n_, det)


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("factor", [2.0**20, 1e30])
def test_a_key_that_is_hidden(ia, D, factor):
    """A key 2^20 or 1e30 times as large as the others, in k, in v and in both, changes nothing for the
    rows that the mask keeps from it: every row by itself, forward and backward."""
    T, j = 500, 300
    c = 1 / math.sqrt(D)
    q, k, v, do = make(1, 2, T, T, D, seed=7)
    do[:, :, j:] = 0  # the rows that see the key send no gradient back
    want = exact(q, k, v, do, c)
    for kf, vf in ((factor, 1.0), (1.0, factor), (factor, factor)):
        k2, v2 = k.clone(), v.clone()
        k2[:, :, j] *= kf
        v2[:, :, j] *= vf
        o, lse = ia.attn_fwd(q, k2, v2, scale=c)
        assert row_err(o[:, :, :j], want[0][:, :, :j]) <= BAR, (kf, vf)
        assert rel(lse[:, :, :j], want[1][:, :, :j]) <= BAR
        if factor > 1e9:
            continue  # past the largest float in the rows that see the key
        for det, got in both_modes(ia, q, k2, v2, do, c):
            assert row_err(got[2][:, :, 1:j], want[2][:, :, 1:j]) <= 3 * BAR, (kf, vf, det)
            for x, r in zip(got[3:], want[3:]):
                assert row_err(x[:, :, :j], r[:, :, :j]) <= 3 * BAR, (kf, vf, det)


@pytest.mark.parametrize("D", [32, 64, 128])
def test_rows_and_columns_of_unlike_size(ia, D):
    """Rows and columns far below the largest of their tensor keep their own precision: the first value
    rows, single columns of v and dO, single rows of q, dO rows that alone see the last keys, q and k
    scaled against each other by column.  Bar: fp32 rounding of scores of about 10 to 30 and of the
    differences that make up a row of dS: 3e-5 of a row."""
    T, c, bar = 400, 1 / math.sqrt(D), 3e-5
    print(f"[case] unlike rows and columns D{D}", flush=True)
    q, k, v, do = make(1, 2, T, T, D, seed=8)
    small = v.clone()
    small[:, :, :3] *= 1e-9
    o, _ = ia.attn_fwd(q, k, small, scale=c)
    assert row_err(o[:, :, :3], exact(q, k, small, do, c)[0][:, :, :3]) <= 2e-6
    # a large column of v: the others, each by itself
    wide = v.clone()
    wide[..., 5] *= 2.0**24
    o, _ = ia.attn_fwd(q, k, wide, scale=c)
    e = exact(q, k, wide, do, c)[0]
    assert row_err(o.transpose(2, 3), e.transpose(2, 3)) <= 2e-6
    # columns of q against those of k (the scores stay)
    s = torch.exp2(torch.linspace(-15, 15, D, device="cuda"))[torch.randperm(D, generator=torch.Generator().manual_seed(9)).cuda()]
    cases = {"columns": (q * s, k / s, v, do)}
    # one row of q 1e6 times the others, where it sees its own key only at the end of a long row
    ql = q.clone()
    ql[:, :, 37] *= 1e6
    cases["q row"] = (ql, k, v, do)
    # the last rows' gradients 1e9 times smaller: the last keys are seen by them alone
    dl = do.clone()
    dl[:, :, 200:] *= 1e-9
    cases["dO rows"] = (q, k, v, dl)
    for name, args in cases.items():
        want = exact(*args, c)
        for det, got in both_modes(ia, *args, c):
            keep = [i for i in range(1, T) if not (name == "q row" and i == 37)]
            assert row_err(got[2][:, :, keep], want[2][:, :, keep]) <= bar, (name, det)
            lo = 38 if name == "q row" else 0
            # (the last key is seen by the last row alone: its dK row is one cancelling difference)
            assert row_err(got[3][:, :, lo:T - 8], want[3][:, :, lo:T - 8]) <= bar, (name, det)
            assert row_err(got[4][:, :, lo:], want[4][:, :, lo:]) <= bar, (name, det)


@pytest.mark.parametrize("B,H", [(1, 3), (8, 16)])
@pytest.mark.parametrize("D", [32, 64, 128])
def test_a_key_that_scores_minus_infinity_backward(ia, B, H, D):
    """Its probability is 0, so its dK and dV are 0 and nothing else changes: only the column of dQ
    that multiplies the infinity is 0 * inf.  Among the first keys (whose rows have their own row
    dots) and far from them; every query sees it or not."""
    c = 1 / math.sqrt(D)
    for causal in (True, False):
        for j in (5, 40, 250):
            print(f"[case] -inf key {j} B{B} H{H} D{D} causal={causal}", flush=True)
            q, k, v, do = make(B, H, 300, 300, D, seed=10)
            q[..., 0] = q[..., 0].abs() + 0.1
            k2 = k.clone()
            k2[:, :, j, 0] = -math.inf
            keep = [i for i in range(300) if i != j]
            # without the key: causal rows before it see the same keys, rows behind it one less
            mask = torch.ones(300, 300, dtype=torch.bool, device="cuda").triu(1) if causal else torch.zeros(
                300, 300, dtype=torch.bool, device="cuda")
            mask[:, j] = True
            qd, kd, vd = (x.double().requires_grad_() for x in (q, k, v))
            s = torch.matmul(qd, kd.transpose(2, 3).contiguous()) * c
            s = s.masked_fill(mask, -math.inf)
            o = torch.matmul(torch.softmax(s, -1), vd)
            o.backward(do.double())
            for det, got in both_modes(ia, q, k2, v, do, c, causal):
                assert rel(got[0], o.detach()) <= BAR, det
                assert (got[3][:, :, j] == 0).all() and (got[4][:, :, j] == 0).all(), det
                assert rel(got[3][:, :, keep], kd.grad[:, :, keep]) <= BAR, det
                assert rel(got[4][:, :, keep], vd.grad[:, :, keep]) <= BAR, det
                assert rel(got[2][..., 1:], qd.grad[..., 1:]) <= BAR, det


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("B,H,Tq,Tk,causal", [(1, 2, 1100, 1100, True), (2, 3, 130, 700, False), (1, 2, 100, 1030, True)])
def test_rows_beside_nonfinite_keys(ia, B, H, Tq, Tk, causal, D):
    """Rows that are formed again in plain fp32 (a key at -inf that all of them see, before many others):
    whole blocks of visible keys, the diagonal's, the ragged end, chunks of a split key range."""
    c = 1 / math.sqrt(D)
    q, k, v, _ = make(B, H, Tq, Tk, D, seed=11)
    q[..., 0] = q[..., 0].abs() + 0.1
    k2 = k.clone()
    k2[:, :, 17, 0] = -math.inf
    mask = torch.ones(Tq, Tk, dtype=torch.bool, device="cuda").triu(1 + Tk - Tq) if causal else torch.zeros(
        Tq, Tk, dtype=torch.bool, device="cuda")
    mask[:, 17] = True
    s = torch.matmul(q.double(), k.double().transpose(2, 3).contiguous()) * c
    s = s.masked_fill(mask, -math.inf)
    o, lse = ia.attn_fwd(q, k2, v, causal=causal, scale=c)
    assert row_err(o, torch.matmul(torch.softmax(s, -1), v.double())) <= BAR
    assert rel(lse, torch.logsumexp(s, -1)) <= BAR


@pytest.mark.parametrize("B,H", [(1, 3), (1, 288)])
@pytest.mark.parametrize("which", ["q", "k", "v", "do"])
def test_largest_row_stride(ia, B, H, which):
    """Rows 2^22 elements apart, the largest stride that is taken: a tile of rows spans just less than 2^31
    bytes (narrow key blocks, and wide ones with 288 heads).  The same results as from dense rows: the
    same bits, but for the order in which dQ's atomics arrive."""
    D, T, c = 64, 300, 0.125
    print(f"[case] row stride 2^22 of {which} H{H}", flush=True)
    q, k, v, do = make(B, H, T, T, D, seed=12)
    want = run(ia, q, k, v, do, c)
    buf = torch.empty(((T - 1) << 22) + H * D, device="cuda")
    t = {"q": q, "k": k, "v": v, "do": do}
    far = buf.as_strided((B, H, T, D), (0, D, 1 << 22, 1))
    far.copy_(t[which])
    t[which] = far
    got = run(ia, t["q"], t["k"], t["v"], t["do"], c)
    for n, x, r in zip(("o", "lse", "dq", "dk", "dv"), got, want):
        assert (rel(x, r.double()) <= 1e-6) if n == "dq" else torch.equal(x, r), n
