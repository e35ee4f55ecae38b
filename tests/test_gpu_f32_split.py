"""The float32 kernels' split products (three bf16 pieces per operand) at the edges of their tiles, with
one and two groups of waves per work item, and on inputs that take the float32 matrix instructions
instead (Q and K from 2^43, sums that are not finite)."""
import numpy as np
import pytest

from _cases import FP32_TOL, assert_close, inputs, oracle_fwd_bwd, to_np, to_torch

pytestmark = pytest.mark.gpu


def _run(pf, q, k, v, do, mask, tiles=None):
    import torch
    q, k, v, do = (to_torch(x, "fp32") for x in (q, k, v, do))
    for t in (q, k, v):
        t.requires_grad_(True)
    bm = None if mask is None else pf.create_block_mask(mask, q.shape[0], q.shape[1], q.shape[2], k.shape[2], 128)
    opts = None if tiles is None else {"BLOCK_M": tiles}
    o = pf.flex_attention(q, k, v, block_mask=bm, enable_gqa=q.shape[1] != k.shape[1], kernel_options=opts)
    return [to_np(x) for x in (o.detach(),) + torch.autograd.grad(o, (q, k, v), do)]


# one and two groups: at most 512 work items share theirs between two (256 CUs), B 9 H 64 has 576 and more
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,D,causal,tiles", [
    (1, 2, 2, 1, 1, 64, False, None), (1, 2, 1, 33, 31, 32, False, None), (1, 2, 2, 127, 127, 64, True, None),
    (1, 2, 2, 129, 129, 128, True, None), (2, 2, 1, 257, 257, 64, True, None), (1, 2, 2, 95, 289, 64, False, None),
    (1, 2, 2, 200, 200, 128, True, 64), (1, 2, 2, 160, 160, 32, True, 64), (9, 64, 64, 40, 40, 32, True, None),
    (9, 64, 32, 33, 65, 64, False, None)])
def test_tile_edges(B, Hq, Hkv, Sq, Skv, D, causal, tiles):
    import pallas_flexattn as pf
    q, k, v, do = inputs(31 + Sq, B, Hq, Hkv, Sq, Skv, D, "fp32")
    got = _run(pf, q, k, v, do, pf.causal_mask if causal else None, tiles)
    dense = np.broadcast_to(np.tril(np.ones((Sq, Skv), bool)) if causal else np.ones((Sq, Skv), bool),
                            (B, Hq, Sq, Skv))
    o, _, grads = oracle_fwd_bwd(q, k, v, do, dense)
    for name, a, b in zip("o dq dk dv".split(), got, (o,) + tuple(grads)):
        assert_close(name, a, b, FP32_TOL)


@pytest.mark.parametrize("S,D", [(70, 64), (300, 64), (130, 128)])
def test_large_and_infinite_inputs_take_the_float32_instructions(S, D):
    import pallas_flexattn as pf
    rng = np.random.default_rng(5)
    q, k, v, do = (rng.standard_normal((1, 2, S, D)).astype(np.float32) for _ in range(4))
    v[0, 0, 3, 7] = np.inf   # every row sees key 3: column 7 of head 0 is inf, the rest as without it
    v[0, 1, 5, 2] = 3.0e38   # no bf16 piece holds it
    k[0, 1, 9] = 0.0
    q[0, 1, 4] *= 2.0 ** 31  # a one-hot row in the limit; its scores are far apart
    o = _run_fwd(pf, q, k, v)
    s = q.astype(np.float64) @ k.astype(np.float64).transpose(0, 1, 3, 2) / np.sqrt(D)
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    vf = np.where(np.isinf(v), 0.0, v).astype(np.float64)
    want = p @ vf
    assert np.all(np.isposinf(o[0, 0, :, 7]))
    got = o.astype(np.float64)
    got[0, 0, :, 7] = want[0, 0, :, 7]
    # per element, relative to the magnitudes summed (3e38 in one column)
    scale = p @ np.abs(vf)
    assert np.max(np.abs(got - want) / scale) < 1e-5


def _run_fwd(pf, q, k, v):
    return to_np(pf.flex_attention(*(to_torch(x, "fp32") for x in (q, k, v))))


def _exact(q, k, v, do, scale, causal):
    """float64 O, dQ, dK, dV and the magnitudes their sums are made of."""
    q, k, v, do = (x.astype(np.float64) for x in (q, k, v, do))
    t = lambda x: x.swapaxes(-1, -2)  # noqa: E731
    s = q @ t(k) * scale
    if causal:
        s = np.where(np.tril(np.ones(s.shape[-2:], bool)), s, -np.inf)
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    o = p @ v
    ds = p * (do @ t(v) - (o * do).sum(-1, keepdims=True))
    mds = p * (np.abs(do) @ t(np.abs(v)) + ((p @ np.abs(v)) * np.abs(do)).sum(-1, keepdims=True))
    return ((o, ds @ k * scale, t(ds) @ q * scale, t(p) @ do),
            (p @ np.abs(v), mds @ np.abs(k) * scale, t(mds) @ np.abs(q) * scale, t(p) @ np.abs(do)))


# D 32: two groups in all three kernels, 64: in forward and dQ, 128: none
@pytest.mark.parametrize("S,D,e", [(130, 32, 44), (300, 64, 44), (200, 128, 44), (300, 64, 33), (200, 128, 33),
                                   (130, 32, 42)])
def test_backward_of_large_inputs(S, D, e):
    """Finite values from 2^e in V, dO and K, each in a head of its own next to a head without.  From 2^43 on the
    work items that meet the K run on the float32 instructions, the others on the split, in one launch; below, and
    with V and dO, all on the split (the sums stay finite)."""
    import pallas_flexattn as pf
    rng = np.random.default_rng(S)
    q, k, v, do = (rng.standard_normal((1, 4, S, D)).astype(np.float32) for _ in range(4))
    v[0, 0, S // 3] *= np.float32(2.0 ** e)
    do[0, 1, S - 5, 3] = np.float32(2.0 ** e)
    q[0, 2, :, 0] = 0.0                            # (scores as without)
    k[0, 2, S // 2, 0] = np.float32(2.0 ** e)
    got = _run(pf, q, k, v, do, pf.causal_mask)
    want, mag = _exact(q, k, v, do, D ** -0.5, True)
    for name, a, b, m in zip("o dq dk dv".split(), got, want, mag):
        err = np.abs(a.astype(np.float64) - b)
        assert np.all(np.isfinite(a)) and np.max(err / np.maximum(m, 1e-30)) < 1e-5, name


@pytest.mark.parametrize("S,D", [(130, 32), (300, 64), (200, 128)])
def test_backward_whose_scaled_sums_overflow(S, D):
    """Inputs of some 2^42 (below the line) in K, V and dO of one key and one query: dQ and dK pass 2^95, where sums of
    2^32 times their value are infinite and the work items run again."""
    import pallas_flexattn as pf
    rng = np.random.default_rng(S)
    q, k, v, do = (rng.standard_normal((1, 2, S, D)).astype(np.float32) for _ in range(4))
    big = np.float32(2.0 ** 42)
    v[0, 0, 5] *= big
    do[0, 0, S - 3] *= big
    q[0, 0, :, 0] = 0.0
    k[0, 0, S // 2, 0] = big
    got = _run(pf, q, k, v, do, None)
    want, mag = _exact(q, k, v, do, D ** -0.5, False)
    assert np.max(np.abs(want[1])) > 2.0 ** 95
    for name, a, b, m in zip("o dq dk dv".split(), got, want, mag):
        err = np.abs(a.astype(np.float64) - b)
        assert np.all(np.isfinite(a)) and np.max(err / np.maximum(m, 1e-30)) < 1e-5, name


@pytest.mark.parametrize("what", ["v", "do", "v-and-do", "columns", "probabilities"])
@pytest.mark.parametrize("S,D", [(96, 32), (300, 64), (200, 128)])
def test_small_inputs_keep_their_bits(S, D, what):
    """Values close to the smallest normal number: no piece of an operand, of P or of dS is cut.  Every column of O
    and the gradients within 4e-6 (2-norm) of float64, eight times what the kernels show at ordinary magnitudes (a
    piece cut at 2^-133 is 2^-13 of 2^-120); probabilities of 2^-124 (where a cut costs 2^-7) within 2^-10: the
    sums of their scores round up to 96 times by 2^-24 of 124."""
    import pallas_flexattn as pf
    rng = np.random.default_rng(D + S)
    q, k, v, do = (rng.standard_normal((1, 3, S, D)).astype(np.float32) for _ in range(4))
    tol = 4e-6
    if what == "v":
        v *= np.float32(2.0 ** -120)
    elif what == "do":
        do *= np.float32(2.0 ** -120)
    elif what == "v-and-do":  # dS far below its factors
        v *= np.float32(2.0 ** -60)
        do *= np.float32(2.0 ** -60)
    elif what == "columns":
        for x in (q, k, v, do):
            x[..., 1::2] *= np.float32(2.0 ** -118)
    else:  # the last 32 keys get 2^-124 of every row but have V to themselves in column 0
        q *= np.float32(0.05)
        q[..., 0], k[..., 0] = np.float32(D ** 0.5), 0.0
        k[:, :, -32:, 0] = np.log(S - 32) - 86.0
        v[:, :, :-32, 0] = 0.0
        tol = 2.0 ** -10
    got = _run(pf, q, k, v, do, None if what == "probabilities" else pf.causal_mask)
    want, _ = _exact(q, k, v, do, D ** -0.5, what != "probabilities")
    for name, a, b in zip("o dq dk dv".split(), got, want):
        if what == "probabilities" and name in ("dk", "dv"):  # (these keys' rows alone)
            a, b = a[:, :, -32:], b[:, :, -32:]
        if what == "probabilities" and name == "o":
            a, b = a[..., :1], b[..., :1]
        err = np.linalg.norm(a.astype(np.float64) - b, axis=2) / np.linalg.norm(b, axis=2)
        assert np.max(err) < tol, (name, np.max(err))
