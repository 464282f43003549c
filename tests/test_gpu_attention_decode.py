"""Decode: a few bf16 queries over a long cache (mfma_attn_fwd_decode), with
and without the device-held masks, at the edges of its blocks of 32 keys,
steps of 128 and parts, against the float64 oracle.  The weights are fp32's
(three bf16 parts each), so what is left is the result's one rounding to bf16:
at most 2^-9 of each element."""
import numpy as np
import pytest
import torch

from conftest import announce
from oracle import interpret
from oracle.data import relative

pytestmark = pytest.mark.gpu

TOL = 2.0 ** -9 + 2.0 ** -14  # the rounding, and fp32 sums over the keys


def _np(t):
    return t.float().cpu().numpy().astype(np.float64)


def _case(D, B, H, KV, S, Sk, offset=0, seed=0):
    gen = torch.Generator(device="cuda").manual_seed(D + H + S + Sk + seed)

    def array(*shape):  # starting `offset` elements into its allocation
        n = int(np.prod(shape))
        t = torch.empty(n + offset, device="cuda", dtype=torch.bfloat16)[offset:].view(*shape)
        return t.copy_(torch.randn(*shape, device="cuda", generator=gen))
    return array(B, S, H, D), array(B, Sk, KV, D), array(B, Sk, KV, D), array(B, S, H, D)


def _launch(q, k, v, o, lse, causal=False, starts=None, lengths=None):
    import tempest_hip.launch as L
    extra = {n: t.data_ptr() for n, t in (("starts", starts), ("lengths", lengths)) if t is not None}
    f = L.attention_fwd(q.shape[0], q.shape[2], k.shape[2], q.shape[1], q.data_ptr(), k.data_ptr(), v.data_ptr(),
                        o.data_ptr(), lse.data_ptr(), causal=causal, head_dim=q.shape[3], kv_seq=k.shape[1], **extra)
    assert "mfma_attn_fwd_decode" in f.describe(), f.describe()
    return f


def _check(q, k, v, o, lse, causal=False, starts=None, lengths=None):
    st = None if starts is None else starts.cpu().numpy()
    ln = None if lengths is None else lengths.cpu().numpy()
    ro, rl = interpret.attention_fwd(_np(q), _np(k), _np(v), causal, None, st, ln)
    assert relative(_np(o), ro) < TOL, relative(_np(o), ro)
    assert np.max(np.abs(_np(lse) - rl)) < 1e-5 * max(1.0, np.abs(rl).max())


@pytest.mark.parametrize("D,B,H,KV,S,Sk", [
    (64, 2, 2, 2, 1, 1), (64, 3, 8, 2, 1, 31), (128, 2, 4, 4, 1, 32), (64, 2, 16, 1, 1, 33), (128, 1, 8, 1, 2, 127),
    (128, 2, 8, 2, 4, 128), (64, 2, 4, 1, 3, 129), (128, 3, 3, 1, 5, 1000), (64, 1, 1, 1, 16, 4099),
    (128, 40, 32, 8, 1, 3000)])
def test_decode_at_the_edges(target, D, B, H, KV, S, Sk):
    announce("attn decode", D, B, H, KV, S, Sk)
    q, k, v, o = _case(D, B, H, KV, S, Sk)
    lse = torch.empty(B, S, H, device="cuda")
    _launch(q, k, v, o, lse)()
    torch.cuda.synchronize()
    _check(q, k, v, o, lse)
    lengths = torch.randint(1, Sk + 1, (B,), dtype=torch.int32, device="cuda", generator=None)
    lengths[0] = Sk
    starts = torch.randint(1, Sk // 2 + 2, (B, S), dtype=torch.int32, device="cuda").clamp(max=lengths[:, None])
    for b in range(B):  # what a cache holds past its length is anything
        k[b, int(lengths[b]):] = float("nan")
        v[b, int(lengths[b]):] = float("inf")
    f = _launch(q, k, v, o, lse, lengths=lengths)
    f()
    f2 = _launch(q, k, v, o2 := torch.empty_like(o), lse2 := torch.empty_like(lse), starts=starts, lengths=lengths)
    f2()
    torch.cuda.synchronize()
    keep = [torch.nan_to_num(x, nan=0.0, posinf=0.0) for x in (k, v)]
    _check(q, *keep, o, lse, lengths=lengths)
    _check(q, *keep, o2, lse2, starts=starts, lengths=lengths)


def test_decode_causal_unaligned_and_empty(target):
    """Causal (query j sees keys 0..j), arrays that start at odd elements, a
    sequence that holds no key (its row is 0/0 and its lse -inf, as the
    general kernels leave it), and lengths beyond the cache."""
    announce("attn decode unaligned")
    q, k, v, o = _case(64, 3, 4, 2, 6, 40, offset=1)
    lse = torch.empty(3, 6, 4, device="cuda")
    lengths = torch.tensor([40, 1000, 3], dtype=torch.int32, device="cuda")
    _launch(q, k, v, o, lse, causal=True, lengths=lengths)()
    torch.cuda.synchronize()
    _check(q, k, v, o, lse, causal=True, lengths=lengths.clamp(max=40))
    q, k, v, o = _case(128, 2, 4, 2, 1, 700, offset=3)
    lse = torch.empty(2, 1, 4, device="cuda")
    lengths = torch.tensor([0, 700], dtype=torch.int32, device="cuda")
    _launch(q, k, v, o, lse, lengths=lengths)()
    torch.cuda.synchronize()
    assert torch.isnan(o[0]).all() and torch.isneginf(lse[0]).all()
    _check(q[1:], k[1:], v[1:], o[1:], lse[1:])


def test_decode_recorded_before_its_first_run(target):
    """A caller's own graph records the launch before it has a workspace, and
    every replay reads the lengths the device then holds."""
    import ctypes
    from tempest_hip._lib import call
    announce("attn decode recorded")
    q, k, v, o = _case(64, 4, 8, 2, 1, 2000)
    lse = torch.empty(4, 1, 8, device="cuda")
    lengths = torch.tensor([5, 2000, 129, 640], dtype=torch.int32, device="cuda")
    f = _launch(q, k, v, o, lse, lengths=lengths)
    was = ctypes.c_void_p()
    call("th_get_stream", ctypes.byref(was))
    graph = torch.cuda.CUDAGraph()
    try:
        with torch.cuda.graph(graph):
            call("th_set_stream", ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
            f()
    finally:
        call("th_set_stream", was)
    for n in ([5, 2000, 129, 640], [2000, 1, 64, 999], [31, 32, 33, 128]):
        lengths.copy_(torch.tensor(n, dtype=torch.int32))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        _check(q, k, v, o, lse, lengths=lengths)
        got = o.clone()
        f()
        torch.cuda.synchronize()
        assert torch.equal(got, o)


@pytest.mark.parametrize("D,H,KV,S,Sk", [(64, 2, 2, 1, 64), (128, 8, 2, 2, 1000)])
def test_decode_weights_hold_fp32s_bits(target, D, H, KV, S, Sk):
    """Keys in pairs, the second one bf16 step from the first in one feature,
    its value the negative: the output is the difference of weights 2^-13
    apart.  fp32's score, exponential and sums leave each weight within about
    2^-22, so 2^-9 of that difference, and the result's rounding another 2^-9;
    weights of 16 bits would leave 2^-5."""
    announce("attn decode weights", D, H, KV, S, Sk)
    q, k, v, o = _case(D, 2, H, KV, S, Sk)
    q *= 0.25
    k[:, 1::2], v[:, 1::2] = k[:, ::2], -v[:, ::2]
    k[:, 1::2, :, 0] = torch.where(k[:, ::2, :, 0] == 0, 0.0, k[:, ::2, :, 0] * (1 + 2.0 ** -7))
    lse = torch.empty(2, S, H, device="cuda")
    lengths = torch.tensor([Sk, Sk // 4 * 2], dtype=torch.int32, device="cuda")
    _launch(q, k, v, o, lse, lengths=lengths)()
    torch.cuda.synchronize()
    ro, _ = interpret.attention_fwd(_np(q), _np(k), _np(v), False, None, None, lengths.cpu().numpy())
    assert np.linalg.norm(ro) < 2.0 ** -8 * np.linalg.norm(_np(v)) / Sk ** 0.5
    assert relative(_np(o), ro) < 2.0 ** -7, relative(_np(o), ro)


def test_decode_an_infinite_value_stays_one(target):
    """A value of +-inf that a query sees makes its feature of the output that
    infinity, as a weighted sum in fp32 does, and leaves the others as they are."""
    announce("attn decode infinite")
    q, k, v, o = _case(64, 1, 4, 2, 2, 500)
    lse = torch.empty(1, 2, 4, device="cuda")
    v[0, 3, 0, 5], v[0, 499, 1, 63] = float("inf"), -float("inf")
    k[0, 3] = 0.0  # (a weight whose nearest bf16 it may well be)
    q[0, 1] = 0.0  # every weight 1
    _launch(q, k, v, o, lse)()
    torch.cuda.synchronize()
    assert torch.isposinf(o[0, :, :2, 5]).all() and torch.isneginf(o[0, :, 2:, 63]).all()
    finite = v.nan_to_num(posinf=0.0, neginf=0.0)
    _launch(q, k, finite, o2 := torch.empty_like(o), lse)()
    torch.cuda.synchronize()
    o[0, :, :2, 5], o[0, :, 2:, 63] = o2[0, :, :2, 5], o2[0, :, 2:, 63]
    assert torch.equal(o, o2)


@pytest.mark.parametrize("lo", [32, 96, 128, 160, 544])
def test_decode_reads_nothing_into_what_lies_before_the_first_key(target, lo):
    """A cache padded on the left: what lies before the first key (a multiple
    of 32, as far as the general kernels skip) may be anything."""
    announce("attn decode left padding", lo)
    q, k, v, o = _case(64, 1, 4, 2, 1, 700)
    lse = torch.empty(1, 1, 4, device="cuda")
    starts = torch.tensor([[lo + 1]], dtype=torch.int32, device="cuda")
    _launch(q, k, v, o, lse, starts=starts)()
    torch.cuda.synchronize()
    _check(q, k, v, o, lse, starts=starts)
    want = o.clone()
    k[:, :lo], v[:, :lo] = float("nan"), float("nan")
    _launch(q, k, v, o, lse, starts=starts)()
    torch.cuda.synchronize()
    assert torch.equal(o, want)
