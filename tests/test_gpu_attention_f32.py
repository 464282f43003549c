"""fp32 attention on the matrix cores (each factor in three bf16 parts, fp32
products where those do not reach) at head dims 64 and 128: causal or not, grouped heads,
lengths that are not multiples of the 64-position tiles, more or fewer keys
than queries.  Forward (o, lse) and backward (dq, dk, dv) against the float64
oracle on the same inputs, to the fp32 tolerance; and the kernels that ran
are the matrix-core ones."""
import pytest
import torch

from conftest import announce
from oracle import interpret
from oracle.data import relative
from test_gpu_attention_general import TOL_F32, _check, _np, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,H,KV,S,Sk,B,causal", [
    (64, 4, 2, 300, 300, 2, True), (64, 2, 2, 96, 250, 2, False), (64, 2, 2, 100, 180, 1, True),
    (128, 2, 1, 129, 129, 2, True), (128, 3, 3, 200, 77, 1, False), (64, 8, 8, 1024, 1024, 1, True),
    (128, 2, 2, 256, 256, 2, True)])
def test_fp32_attention_on_matrix_cores(target, D, H, KV, S, Sk, B, causal):
    announce("attn fp32 mfma", D, H, KV, S, Sk, B, causal)
    gen = torch.Generator(device="cuda").manual_seed(D * 7 + S + Sk + H)
    q = torch.randn(B, S, H, D, device="cuda", generator=gen) * 0.5
    k = torch.randn(B, Sk, KV, D, device="cuda", generator=gen) * 0.5
    v = torch.randn(B, Sk, KV, D, device="cuda", generator=gen)
    g = torch.randn(B, S, H, D, device="cuda", generator=gen)
    outs, (fwd, bwd) = _run(q, k, v, g, causal, True)
    assert f"f32_attn_fwd_d{D}" in fwd.describe(), fwd.describe()
    assert f"f32_attn_dkdv_d{D}" in bwd.describe() and f"f32_attn_dq_d{D}" in bwd.describe(), bwd.describe()
    _check(outs, q, k, v, g, causal, TOL_F32)


def test_fp32_attention_replays_bitwise(target):
    """No atomics: the same inputs give the same bits on every run."""
    announce("attn fp32 mfma repeat")
    gen = torch.Generator(device="cuda").manual_seed(5)
    q, k, v, g = (torch.randn(2, 384, 4, 64, device="cuda", generator=gen) for _ in range(4))
    (o, lse, dq, dk, dv), (fwd, bwd) = _run(q, k, v, g, True, True)
    first = [t.clone() for t in (o, lse, dq, dk, dv)]
    for _ in range(3):
        fwd()
        bwd()
    torch.cuda.synchronize()
    for a, b in zip(first, (o, lse, dq, dk, dv)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("D,B,H,KV,S,causal,split", [
    (64, 1, 2, 2, 700, True, True), (128, 1, 2, 1, 300, False, True), (64, 4, 16, 16, 512, True, False)])
def test_fp32_split_and_whole_sweeps(target, D, B, H, KV, S, causal, split):
    """A grid under one workgroup a CU splits each sweep into parts (partial
    results combined or summed in part order); a grid that fills the device
    sweeps whole.  Both against the float64 oracle."""
    announce("attn fp32 mfma split", D, B, H, KV, S, causal, split)
    gen = torch.Generator(device="cuda").manual_seed(17 * D + S + H)
    q = torch.randn(B, S, H, D, device="cuda", generator=gen) * 0.5
    k = torch.randn(B, S, KV, D, device="cuda", generator=gen) * 0.5
    v = torch.randn(B, S, KV, D, device="cuda", generator=gen)
    g = torch.randn(B, S, H, D, device="cuda", generator=gen)
    outs, (fwd, bwd) = _run(q, k, v, g, causal, True)
    assert ("f32_attn_combine" in fwd.describe()) == split, fwd.describe()
    assert ("f32_attn_sum_dk" in bwd.describe() and "f32_attn_sum_dq" in bwd.describe()) == split, bwd.describe()
    _check(outs, q, k, v, g, causal, TOL_F32)


@pytest.mark.parametrize("D,S,causal", [(64, 65, True), (64, 128, False), (64, 63, True), (128, 129, True),
                                        (128, 64, False), (64, 1, True)])
def test_fp32_values_out_of_the_parts_reach(target, D, S, causal):
    """Tiles computed again with fp32 products: an infinity in V gives infinity
    where it is seen and leaves the other features alone; and gradients scaled far
    down keep their relative accuracy, at the edges of tiles."""
    announce("attn fp32 parts", D, S, causal)
    gen = torch.Generator(device="cuda").manual_seed(D + S)
    r = lambda: torch.randn(2, S, 2, D, device="cuda", generator=gen) * 0.5  # noqa: E731
    q, k, v, g = r(), r(), r(), r()
    outs, _ = _run(q, k, v, g, causal, True)
    _check(outs, q, k, v, g, causal, TOL_F32)
    small = g * 1e-30
    outs, _ = _run(q, k, v, small, causal, True)
    want = interpret.attention_bwd(*(_np(t) for t in (q, k, v, g)), causal)
    for got, ref in zip(outs[2:], want):
        assert relative(_np(got) * 1e30, ref) < TOL_F32, relative(_np(got) * 1e30, ref)
    v[0, 0, 1, 3] = float("inf")
    v[1, 0, 0, 5] = float("-inf")
    outs, _ = _run(q, k, v, g, False, True)
    o = outs[0]
    assert torch.isposinf(o[0, :, 1, 3]).all() and torch.isneginf(o[1, :, 0, 5]).all()
    rest = torch.ones_like(o, dtype=torch.bool)
    rest[0, :, 1, 3] = rest[1, :, 0, 5] = False
    clean = torch.where(torch.isfinite(v), v, torch.zeros_like(v))
    ro, _ = interpret.attention_fwd(_np(q), _np(k), _np(clean), False)
    keep = rest.cpu().numpy()
    assert relative(_np(o)[keep], ro[keep]) < TOL_F32


@pytest.mark.parametrize("D,S", [(64, 1024), (128, 300)])
@pytest.mark.parametrize("what,e", [("dout", -110), ("dout", -119), ("v", -119), ("features", 122)])
def test_fp32_attention_over_fp32s_range(target, D, S, what, e):
    """dO, or V, of about 2^e; and a quarter of the features 2^e in Q, 2^-e in K:
    the same results as at ordinary sizes, scaled (a power of two, so exactly what
    fp32 products of the scaled factors give), where the lower parts of a factor
    lie under bf16's least subnormal."""
    announce("attn fp32 range", D, S, what, e)
    gen = torch.Generator(device="cuda").manual_seed(D + S + e)
    q, k, v, g = (torch.randn(1, S, 2, D, device="cuda", generator=gen) * 0.5 for _ in range(4))
    t = 2.0 ** e
    up = torch.ones(D, device="cuda")
    if what == "features":
        up[::4] = t
    scaled = [q * up, k / up, v * t if what == "v" else v, g * t if what == "dout" else g]
    (o, _, dq, dk, dv), _ = _run(*scaled, True, True)
    ro, _ = interpret.attention_fwd(_np(q), _np(k), _np(v), True)
    want = interpret.attention_bwd(_np(q), _np(k), _np(v), _np(g), True)
    u = _np(up).astype("f8")
    so, sg, sv = t if what == "v" else 1.0, t if what in ("v", "dout") else 1.0, t if what == "dout" else 1.0
    for name, got, ref in (("o", _np(o).astype("f8") / so, ro), ("dq", _np(dq).astype("f8") / sg * u, want[0]),
                           ("dk", _np(dk).astype("f8") / sg / u, want[1]), ("dv", _np(dv).astype("f8") / sv, want[2])):
        print("   ", name, relative(got, ref), flush=True)
        assert relative(got, ref) < 4e-6, (name, relative(got, ref))


@pytest.mark.parametrize("e", [20, 30])
def test_fp32_attention_at_small_scales(target, e):
    """Q and K of 2^e under a scale of 2^-2e / 8: in three parts down to a scale
    of 2^-50, in fp32 products under it, the same results as at e = 0 either way."""
    import tempest_hip.launch as L
    announce("attn fp32 scale", e)
    gen = torch.Generator(device="cuda").manual_seed(e)
    q, k, v, g = (torch.randn(1, 200, 2, 64, device="cuda", generator=gen) for _ in range(4))
    t = 2.0 ** e
    o, dq, dk, dv = (torch.empty_like(q) for _ in range(4))
    lse = torch.empty(1, 200, 2, device="cuda")
    qt, kt = q * t, k * t
    p = [x.data_ptr() for x in (qt, kt, v, o, lse)]
    extra = {"causal": True, "head_dim": 64, "f32": True, "scale": t ** -2 / 8}
    L.attention_fwd(1, 2, 2, 200, *p, **extra)()
    L.attention_bwd(1, 2, 200, *p, g.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), kv_heads=2, **extra)()
    torch.cuda.synchronize()
    ro, _ = interpret.attention_fwd(_np(q), _np(k), _np(v), True)
    want = interpret.attention_bwd(_np(q), _np(k), _np(v), _np(g), True)
    for name, got, ref in (("o", _np(o), ro), ("dq", _np(dq) * t, want[0]), ("dk", _np(dk) * t, want[1]),
                           ("dv", _np(dv), want[2])):
        assert relative(got, ref) < 4e-6, (name, relative(got, ref))
