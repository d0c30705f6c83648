"""The fp32 attention kernels' products on two fp16 parts per operand: magnitudes far from 1 and
far apart, non-finite inputs, and the sizes where a tile, a key block or the choice between the
wide and the narrow backward ends, against 64-bit torch.

Bar: a split operand is within 2^-22.7 of its value, so a score is within about D 2^-21.7 max|q k|
in the worst case and sqrt(D) times that for terms of either sign, below 3e-6 of the largest score
(at most ~8 here, so a probability is within ~3e-6 absolutely); sums over keys and queries add
rounding of either sign.  1e-5 of a tensor's norm is several times what such errors add up to
(measured: 2e-7 to 7e-7), and a part dropped or a scale missed shows at 1e-4 or more."""
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
