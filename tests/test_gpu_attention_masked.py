"""bf16 attention at head dims 64 and 128 under device-held masks on the matrix
cores (mfma_attn_*_masked): packed documents whose cuts fall on and off the
kernels' blocks of 64 and 128, first keys in no order, key counts, keys more
or fewer than queries, grouped heads, rows at odd addresses.  Forward and
backward against the float64 oracle.  P and dS are fp32's (three bf16 parts
each), so the forward's error is its result's rounding (2^-9 of each element) and
a gradient's that and o's, which enters through delta."""
import numpy as np
import pytest
import torch

from conftest import announce
from oracle import interpret
from oracle.data import relative

pytestmark = pytest.mark.gpu

TOL_O = 2.0 ** -9 + 2.0 ** -14
TOL_GRAD = 2.0 ** -8


def _np(t):
    return t.float().cpu().numpy().astype(np.float64)


def _documents(S, cuts):
    cuts = [0] + [c for c in cuts if 0 < c < S] + [S]
    return [lo + 1 for lo, hi in zip(cuts, cuts[1:]) for _ in range(lo, hi)]


def _run(q, k, v, g, causal, lengths=None):
    """o, lse, dq, dk and dv."""
    import tempest_hip.launch as L
    (B, S, H, D), (_, Sk, KV, _) = q.shape, k.shape
    o, dq, dk, dv, lse = *map(torch.empty_like, (q, q, k, v)), torch.empty(B, S, H, device="cuda")
    extra = {"causal": causal, "head_dim": D, "kv_seq": Sk, "lengths": lengths.data_ptr()}
    p = [t.data_ptr() for t in (q, k, v, o, lse)]
    fwd = L.attention_fwd(B, H, KV, S, *p, **extra)
    bwd = L.attention_bwd(B, H, S, *p, g.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), kv_heads=KV, **extra)
    assert "mfma_attn_fwd_masked" in fwd.describe() and "mfma_attn_dkdv_masked" in bwd.describe()
    fwd()
    bwd()
    torch.cuda.synchronize()
    return o, lse, dq, dk, dv


def _check(D, B, H, KV, S, Sk, causal, starts=None, lengths=None, offset=0, seed=0):
    import tempest_hip.launch as L
    gen = torch.Generator(device="cuda").manual_seed(D + S + Sk + H + seed)

    def array(*shape):
        n = int(np.prod(shape))
        t = torch.empty(n + offset, device="cuda", dtype=torch.bfloat16)[offset:].view(*shape)
        return t.copy_(torch.randn(*shape, device="cuda", generator=gen))
    q, g, o, dq = (array(B, S, H, D) for _ in range(4))
    k, v, dk, dv = (array(B, Sk, KV, D) for _ in range(4))
    lse = torch.empty(B, S, H, device="cuda")
    st = None if starts is None else torch.tensor(np.asarray(starts), dtype=torch.int32, device="cuda")
    ln = None if lengths is None else torch.tensor(lengths, dtype=torch.int32, device="cuda")
    extra = {n: t.data_ptr() for n, t in (("starts", st), ("lengths", ln)) if t is not None}
    p = [t.data_ptr() for t in (q, k, v, o)]
    fwd = L.attention_fwd(B, H, KV, S, *p, lse.data_ptr(), causal=causal, head_dim=D, kv_seq=Sk, **extra)
    bwd = L.attention_bwd(B, H, S, *p, lse.data_ptr(), g.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(),
                          causal=causal, kv_heads=KV, head_dim=D, kv_seq=Sk, **extra)
    assert "mfma_attn_fwd" in fwd.describe() and "mfma_attn_dkdv_masked" in bwd.describe()
    fwd()
    bwd()
    torch.cuda.synchronize()
    ro, rl = interpret.attention_fwd(_np(q), _np(k), _np(v), causal, None, starts, lengths)
    want = interpret.attention_bwd(_np(q), _np(k), _np(v), _np(g), causal, None, starts, lengths)
    assert relative(_np(o), ro) < TOL_O, relative(_np(o), ro)
    assert np.max(np.abs(_np(lse) - rl)) < 1e-5 * max(1.0, np.abs(rl).max())
    for name, got, ref in zip(("dq", "dk", "dv"), (dq, dk, dv), want):
        assert relative(_np(got), ref) < TOL_GRAD, (name, relative(_np(got), ref))
    return q, k, v, g, (o, lse, dq, dk, dv), (fwd, bwd), st


@pytest.mark.parametrize("D,B,H,KV,S,cuts", [
    (64, 2, 4, 2, 300, ([64, 128, 129], [7, 200])), (64, 1, 2, 2, 1000, ([63, 64, 65, 511, 512, 900],)),
    (128, 2, 2, 1, 257, ([128, 256], [1, 2, 3, 255])), (128, 1, 3, 3, 515, ([500],)), (64, 1, 1, 1, 17, ([16],)),
    (64, 1, 2, 1, 2048, (list(range(100, 2048, 100)),))])
def test_packed_documents(target, D, B, H, KV, S, cuts):
    announce("attn masked documents", D, B, H, KV, S)
    starts = np.stack([_documents(S, c) for c in cuts])
    q, k, v, g, outs, (fwd, bwd), st = _check(D, B, H, KV, S, S, True, starts)
    first = [t.clone() for t in outs]
    fwd()  # and again, bit for bit
    bwd()
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(first, outs))


@pytest.mark.parametrize("D,S,Sk,causal,lengths", [
    (64, 200, 200, False, [200, 1]), (64, 130, 333, False, [70, 333]), (128, 333, 130, True, [129, 64]),
    (128, 100, 1000, False, [999, 128]), (64, 64, 64, True, [63, 64])])
def test_key_counts(target, D, S, Sk, causal, lengths):
    announce("attn masked lengths", D, S, Sk, causal, lengths)
    _check(D, 2, 4, 2, S, Sk, causal, lengths=np.array(lengths))
    # and first keys in no order, none past the last key its query sees
    rng = np.random.default_rng(S)
    top = np.minimum(np.arange(S)[None, :] + 1 if causal else Sk, np.array(lengths)[:, None])
    starts = np.floor(rng.random((2, S)) * top).astype(np.int64) + 1
    _check(D, 2, 4, 2, S, Sk, causal, starts, np.array(lengths), seed=1)


def test_odd_addresses_and_sequences_without_keys(target):
    """Arrays that start at odd elements; and a sequence that holds no key,
    whose keys take no gradient."""
    announce("attn masked odd")
    _check(64, 1, 2, 2, 150, 150, True, np.array([_documents(150, [70])]), offset=1)
    import tempest_hip.launch as L
    q, k, v, g = (torch.randn(2, 100, 2, 128, device="cuda").to(torch.bfloat16) for _ in range(4))
    o, dq, dk, dv = (torch.full_like(q, 7.0) for _ in range(4))
    lse = torch.empty(2, 100, 2, device="cuda")
    ln = torch.tensor([0, 100], dtype=torch.int32, device="cuda")
    p = [t.data_ptr() for t in (q, k, v, o, lse)]
    fwd = L.attention_fwd(2, 2, 2, 100, *p, causal=True, lengths=ln.data_ptr())
    bwd = L.attention_bwd(2, 2, 100, *p, g.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), causal=True,
                          lengths=ln.data_ptr())
    fwd()
    bwd()
    torch.cuda.synchronize()
    assert torch.isnan(o[0]).all() and torch.isneginf(lse[0]).all()
    assert not dk[0].any() and not dv[0].any() and not dq[0].any()
    want = interpret.attention_bwd(_np(q[1:]), _np(k[1:]), _np(v[1:]), _np(g[1:]), True)
    for got, ref in zip((dq, dk, dv), want):
        assert relative(_np(got[1:]), ref) < TOL_GRAD


@pytest.mark.parametrize("D,H,KV,S,Sk", [(64, 2, 2, 64, 64), (64, 4, 1, 130, 200), (128, 2, 1, 200, 330)])
def test_weights_and_their_gradients_hold_fp32s_bits(target, D, H, KV, S, Sk):
    """Keys in pairs, and queries, the second one bf16 step from the first in
    one feature, its value (its gradient) the negative: every result is a sum of
    differences of weights, or of dS, 2^-13 apart.  fp32's scores, exponentials
    and sums leave each within about 2^-22, so 2^-9 of that difference, o's
    rounding in delta as much, and the result's rounding 2^-9; weights of
    16 bits would leave 2^-5.  (The stepped feature itself has a larger term.)"""
    announce("attn masked weights", D, H, KV, S, Sk)
    gen = torch.Generator(device="cuda").manual_seed(D + S)
    r = lambda *n: torch.randn(*n, device="cuda", generator=gen).to(torch.bfloat16)  # noqa: E731
    q, k, v, g = r(2, S, H, D) * 0.25, r(2, Sk, KV, D), r(2, Sk, KV, D), r(2, S, H, D)
    for x, y in ((k, v), (q, g)):
        x[:, 1::2], y[:, 1::2] = x[:, ::2], -y[:, ::2]
        x[:, 1::2, :, 0] = x[:, ::2, :, 0] * (1 + 2.0 ** -7)
    lengths = torch.tensor([Sk, Sk // 4 * 2], dtype=torch.int32, device="cuda")
    o, _, dq, dk, dv = _run(q, k, v, g, False, lengths)
    ln = lengths.cpu().numpy()
    want, _ = interpret.attention_fwd(_np(q), _np(k), _np(v), False, None, None, ln)
    wants = (want, *interpret.attention_bwd(_np(q), _np(k), _np(v), _np(g), False, None, None, ln))
    for name, got, ref, lo in zip(("o", "dq", "dk", "dv"), (o, dq, dk, dv), wants, (0, 1, 1, 0)):
        err = relative(_np(got)[..., lo:], ref[..., lo:])
        print("   ", name, err, flush=True)
        assert err < 2.0 ** -7, (name, err)


def test_infinite_values_stay_infinite(target):
    """A value of +-inf that a query sees makes its feature of the output that
    infinity, and a gradient of +-inf its feature of dV, as a sum weighted in
    fp32 does; the other features are as without it."""
    announce("attn masked infinite")
    gen = torch.Generator(device="cuda").manual_seed(3)
    q, k, v, g = (torch.randn(1, 100, 2, 64, device="cuda", generator=gen).to(torch.bfloat16) for _ in range(4))
    q[0, ::2] = 0.0  # rows whose weights are alike
    lengths = torch.tensor([90], dtype=torch.int32, device="cuda")
    inf = float("inf")
    plain = _run(q, k, v, g, False, lengths)
    w = v.clone()
    w[0, 7, 0, 5], w[0, 89, 1, 63] = inf, -inf
    o = _run(q, k, w, g, False, lengths)[0]
    assert torch.isposinf(o[0, :, 0, 5]).all() and torch.isneginf(o[0, :, 1, 63]).all()
    o[0, :, 0, 5], o[0, :, 1, 63] = plain[0][0, :, 0, 5], plain[0][0, :, 1, 63]
    assert torch.equal(o, plain[0])
    h = g.clone()
    h[0, 8, 0, 5], h[0, 99, 1, 63] = inf, -inf
    dv = _run(q, k, v, h, False, lengths)[4]
    assert torch.isposinf(dv[0, :90, 0, 5]).all() and torch.isneginf(dv[0, :90, 1, 63]).all()
    dv[0, :90, 0, 5], dv[0, :90, 1, 63] = plain[4][0, :90, 0, 5], plain[4][0, :90, 1, 63]
    assert torch.equal(dv, plain[4])  # (zeros past the length)


@pytest.mark.parametrize("D,S,lo,hi", [(64, 300, 32, 192), (64, 300, 96, 64), (128, 257, 160, 256), (64, 1000, 512, 576)])
def test_what_no_query_sees_may_be_anything(target, D, S, lo, hi):
    """Causal, NaN in every array from position `hi` on leaves the outputs before
    it as they are (hi a multiple of 64), and NaN before `lo`, in a document of its own,
    the document that starts there (lo a multiple of 32; from the next multiple of 64
    on): the general kernels sweep no further than that."""
    import tempest_hip.launch as L
    announce("attn masked garbage", D, S, lo, hi)
    gen = torch.Generator(device="cuda").manual_seed(S + lo)
    r = lambda: torch.randn(1, S, 2, D, device="cuda", generator=gen).to(torch.bfloat16)  # noqa: E731
    arrays = [r() for _ in range(4)]

    def run(arrays, starts):
        q, k, v, g = arrays
        o, dq, dk, dv = (torch.empty_like(q) for _ in range(4))
        lse = torch.empty(1, S, 2, device="cuda")
        st = torch.tensor(starts, dtype=torch.int32, device="cuda")
        p = [t.data_ptr() for t in (q, k, v, o, lse)]
        extra = {"causal": True, "head_dim": D, "starts": st.data_ptr()}
        fwd = L.attention_fwd(1, 2, 2, S, *p, **extra)
        bwd = L.attention_bwd(1, 2, S, *p, g.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), **extra)
        assert "masked" in fwd.describe() and "masked" in bwd.describe()
        fwd()
        bwd()
        torch.cuda.synchronize()
        return o, lse, dq, dk, dv

    def broken(at):
        out = [t.clone() for t in arrays]
        for t in out:
            t[:, at] = float("nan")
        return out

    one = [[1] * S]
    for got, want in list(zip(run(broken(slice(hi, S)), one), run(arrays, one)))[:3]:  # o, lse, dq
        assert torch.equal(got[:, :hi], want[:, :hi])
    two = [_documents(S, [lo])]
    at = (lo + 63) // 64 * 64
    for got, want in zip(run(broken(slice(0, lo)), two), run(arrays, two)):
        assert torch.equal(got[:, at:], want[:, at:])
