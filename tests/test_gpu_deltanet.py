"""Config 5 on the GPU: chunked gated DeltaNet forward and gradient against
the oracle (float64, on the same bf16/fp32 inputs)."""
import numpy as np
import pytest
import torch

from conftest import announce
from oracle import interpret
from oracle.data import relative

pytestmark = pytest.mark.gpu

TOL = 2e-2


def _inputs(B, T, H, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda *s: torch.randn(*s, device="cuda", generator=gen)  # noqa: E731
    unit = lambda x: x / x.norm(dim=-1, keepdim=True)  # noqa: E731
    q = unit(r(B, T, H, 128)).to(torch.bfloat16)
    k = unit(r(B, T, H, 128)).to(torch.bfloat16)
    v = r(B, T, H, 128).to(torch.bfloat16)
    a = -torch.nn.functional.softplus(r(B, T, H))
    beta = torch.sigmoid(r(B, T, H))
    do = r(B, T, H, 128).to(torch.bfloat16)
    return q, k, v, a.contiguous(), beta.contiguous(), do


def _np(t):
    return t.float().cpu().numpy()


# (1, 8192, 2): config 5's sequence length, 128 chunks of state hand-off
# through the split-bf16 products.
@pytest.mark.parametrize("B,T,H", [(1, 64, 1), (1, 256, 2), (2, 192, 3), (1, 8192, 2)])
def test_forward_and_gradient_match_oracle(target, B, T, H):
    import tempest_hip as th
    announce("deltanet", B, T, H)
    q, k, v, a, beta, do = _inputs(B, T, H, T + H)
    comp = th.compile(th.programs.deltanet(B, H, T), target, q, k, v, a, beta, do)
    o, dq, dk, dv, da, dbeta = comp(q, k, v, a, beta, do)
    args = [_np(x) for x in (q, k, v, a, beta)]
    ro = interpret.deltanet_chunked(*args)
    assert relative(_np(o).reshape(B, T, H, 128), ro) < TOL
    grads = interpret.deltanet_grad(*args, _np(do))
    got = [_np(x) for x in (dq, dk, dv)] + [_np(da), _np(dbeta)]
    shapes = [(B, T, H, 128)] * 3 + [(B, T, H)] * 2
    for name, g, s, r in zip(("dq", "dk", "dv", "da", "dbeta"), got, shapes, grads):
        assert relative(g.reshape(s), r) < TOL, name


def test_forward_alone_matches_the_token_rule(target):
    import tempest_hip.launch as L
    announce("deltanet fwd")
    B, T, H = 1, 128, 2
    q, k, v, a, beta, _ = _inputs(B, T, H, 5)
    o = torch.empty_like(q)
    l = L.deltanet(B, H, T, q.data_ptr(), k.data_ptr(), v.data_ptr(), a.data_ptr(), beta.data_ptr(), o.data_ptr())
    l()
    torch.cuda.synchronize()
    ref = interpret.deltanet_sequential(*(_np(x) for x in (q, k, v, a, beta)))
    assert relative(_np(o).reshape(B, T, H, 128), ref) < TOL


def test_config5_full_size_sampled_sequences(target):
    """B4 H16 T8192: every output computed on the GPU; two (batch, head)
    sequences checked against the float64 oracle."""
    import tempest_hip as th
    announce("deltanet config5 full")
    B, T, H = 4, 8192, 16
    q, k, v, a, beta, do = _inputs(B, T, H, 55)
    comp = th.compile(th.programs.deltanet(B, H, T), target, q, k, v, a, beta, do)
    o, dq, dk, dv, da, dbeta = comp(q, k, v, a, beta, do)
    for b, h in ((0, 0), (3, 9)):
        pick = lambda t: _np(t.view(B, T, H, -1)[b:b + 1, :, h:h + 1])  # noqa: E731
        pickg = lambda t: _np(t.view(B, T, H)[b:b + 1, :, h:h + 1])  # noqa: E731
        args = [pick(q), pick(k), pick(v), pickg(a), pickg(beta)]
        assert relative(pick(o), interpret.deltanet_chunked(*args)) < TOL
        grads = interpret.deltanet_grad(*args, pick(do))
        for name, g, r in zip(("dq", "dk", "dv", "da", "dbeta"),
                              (pick(dq), pick(dk), pick(dv), pickg(da), pickg(dbeta)), grads):
            assert relative(g, r) < TOL, (b, h, name)


@pytest.mark.parametrize("B,T,H,decay", [(1, 64, 1, 1.0), (1, 192, 2, 0.0), (2, 128, 3, 0.3), (1, 320, 1, 1.0)])
def test_gate_gradients_to_the_products_precision(target, B, T, H, decay):
    """da and dbeta are fp32 and depend on every product of a chunk's gradient,
    each exact to about 2^-16: through the at most six products in a row of
    the longest path, 6 x 2^-16 < 1e-4 of the float64 oracle, norm-wise; from
    no decay at all to about e^-51 over a chunk."""
    import tempest_hip as th
    announce("deltanet gates", B, T, H, decay)
    q, k, v, a, beta, do = _inputs(B, T, H, 3 * T + H)
    a = (a * decay).contiguous()
    comp = th.compile(th.programs.deltanet(B, H, T), target, q, k, v, a, beta, do)
    out = comp(q, k, v, a, beta, do)
    grads = interpret.deltanet_grad(*[_np(x).astype(np.float64) for x in (q, k, v, a, beta, do)])
    for name, got, ref in (("da", out[4], grads[3]), ("dbeta", out[5], grads[4])):
        err = relative(_np(got).reshape(B, T, H), ref)
        assert err < 1e-4, (name, err)


@pytest.mark.parametrize("B,T,H,decay", [(1, 128, 2, 3.0), (1, 192, 1, 10.0)])
def test_gates_that_decay_past_fp32_within_a_chunk(target, B, T, H, decay):
    """A chunk's decay of e^-150 and e^-500, whose inverse fp32 does not
    hold: every gradient finite and, where the last state is gone, the
    oracle's."""
    import tempest_hip as th
    announce("deltanet strong gates", B, T, H, decay)
    q, k, v, a, beta, do = _inputs(B, T, H, 7 * T + H)
    a = (a * decay).contiguous()
    comp = th.compile(th.programs.deltanet(B, H, T), target, q, k, v, a, beta, do)
    out = [_np(x) for x in comp(q, k, v, a, beta, do)]
    args = [_np(x).astype(np.float64) for x in (q, k, v, a, beta)]
    assert np.abs(args[3].reshape(B, T // 64, 64, H).sum(axis=2)).max() > 88 * decay / 3
    refs = [interpret.deltanet_chunked(*args), *interpret.deltanet_grad(*args, _np(do).astype(np.float64))]
    for name, got, ref in zip(("o", "dq", "dk", "dv", "da", "dbeta"), out, refs):
        assert np.isfinite(got).all() and np.isfinite(ref).all(), name
        # bf16 results: TOL; the fp32 ones as in the test above.
        err = relative(got.reshape(ref.shape), ref)
        assert err < (1e-4 if name in ("da", "dbeta") else TOL), (name, err)
