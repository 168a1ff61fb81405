"""Branches of the head-space MABA-SA prefill that only some selections or shapes take, against
the float64 oracle (rtol = atol = 2e-3, as test_gpu_prefill_attention.py): distinct blocks read
from bits, a union too long for them, references that move far, rows whose offsets need 64 bits."""
import numpy as np
import pytest
import torch

from _helpers import assert_close, to_np
from oracle import sparse_attn as osa
from test_gpu_prefill_attention import _case, _hip

pytestmark = pytest.mark.gpu


def _distinct(B, Lq, nb, K, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.rand(B, Lq, nb, generator=g).argsort(dim=-1)[..., :K]


def _check(dev, case, scale, what, **kw):
    q, k, v, kh, vh, early, idx, gate = case
    d = lambda t: None if t is None else t.to(dev)  # noqa: E731
    out = _hip().hip_maba_sa_prefill(*(d(t) for t in case), scale=scale, out_dtype=torch.float32, **kw)
    exp = osa.maba_sa_prefill_heads(*(to_np(t) if t is not None else None for t in (q, k, v, kh, vh, early)), idx.numpy(),
                                    to_np(gate), window=kw.get("window", 128), n_sink=kw.get("n_sink", 4), scale=scale)
    assert_close(out, exp, 2e-3, 2e-3, what)


@pytest.mark.parametrize("dh", [32, 64, 128])
@pytest.mark.parametrize("Lq,Lkv,K", [(100, 100, 1), (100, 2500, 7), (65, 4160, 64)])
def test_distinct_blocks(dev, dh, Lq, Lkv, K):
    case = list(_case(1, 2, Lq, Lkv, dh, K, dh + Lkv))
    case[6] = _distinct(1, Lq, (Lkv + 63) // 64, K, 1)
    _check(dev, case, dh ** -0.5, f"distinct {dh} {Lkv}")


def test_union_beyond_the_bits(dev):
    """64 queries of 64 distinct blocks each among 700: more than 512 in the union."""
    Lq, Lkv = 64, 64 * 700
    case = list(_case(1, 1, Lq, Lkv, 64, 64, 3))
    case[6] = _distinct(1, Lq, 700, 64, 2)
    assert case[6].unique().numel() > 512
    _check(dev, case, 0.125, "long union")


@pytest.mark.parametrize("scale", [4.0, 0.0, -1.0])
@pytest.mark.parametrize("dup", [False, True])
def test_references_that_move(dev, scale, dup):
    """Scores of hundreds of log2 units, so the running reference moves at most tiles; scores all
    equal; a negative scale (masked keys stay masked)."""
    case = list(_case(1, 2, 150, 1000, 64, 8, 7, dup=dup))
    if not dup:
        case[6] = _distinct(1, 150, 16, 8, 4)
    _check(dev, case, scale, f"scale {scale}")


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("channels", [1, 64])
@pytest.mark.parametrize("scale", [0.125, -0.125])
@pytest.mark.parametrize("dup", [False, True])
def test_non_finite_key_stays_with_its_block(dev, bad, channels, scale, dup):
    """A key whose scores are infinite (either sign) or NaN changes nothing for the queries that do
    not list its block."""
    case = list(_case(1, 2, 150, 1000, 64, 4, 8, dup=dup))
    if not dup:
        case[6] = _distinct(1, 150, 16, 4, 5)
    q, k, v, kh, vh, early, idx, gate = case
    others = (idx[0] != 5).all(dim=-1).nonzero()[:, 0]   # block 5 is outside every query's window too
    assert 50 < others.numel() < 150
    exp = osa.maba_sa_prefill_heads(*(to_np(t) if t is not None else None for t in (q, k, v, kh, vh, early)), idx.numpy(),
                                    to_np(gate), window=128, n_sink=4, scale=scale)
    case[1] = k.clone()
    case[1][:, :, 5 * 64 + 7, :channels] = bad
    d = lambda t: None if t is None else t.to(dev)  # noqa: E731
    out = _hip().hip_maba_sa_prefill(*(d(t) for t in case), scale=scale, out_dtype=torch.float32)
    assert_close(out[:, :, others.to(dev)], exp[:, :, others.numpy()], 2e-3, 2e-3, f"{bad} {channels}")


def test_far_rows(dev):
    """Key rows 2^23 elements apart."""
    q, k, v, kh, vh, early, idx, gate = _case(1, 1, 70, 70, 64, 2, 9)
    buf = torch.empty(70, 1 << 23, dtype=torch.bfloat16, device=dev)
    far = buf[:, :64].view(1, 1, 70, 64)
    far.copy_(k)
    d = lambda t: None if t is None else t.to(dev)  # noqa: E731
    args = [d(t) for t in (q, k, v, kh, vh, early, idx, gate)]
    want = _hip().hip_maba_sa_prefill(*args, scale=0.125)
    args[1] = far
    assert torch.equal(_hip().hip_maba_sa_prefill(*args, scale=0.125), want)


@pytest.mark.parametrize("B,Lq,K,nb", [(1, 16, 1, 1), (1, 31, 32, 40), (2, 200, 64, 16384), (3, 77, 5, 33), (1, 70000, 7, 900)])
def test_prefill_union_counts(dev, B, Lq, K, nb):
    """Distinct blocks per 16 queries, dense and permuted index strides, more groups than one
    round of workgroups, and values that are no block (counted as one)."""
    from maba_sparse.kernels import hip_backend as hb
    g = torch.Generator().manual_seed(B + Lq)
    idx = torch.randint(0, nb, (B, Lq, K), generator=g)
    idx[:, 3::16, 0] = nb - 1
    if Lq == 77:
        idx[:, ::5, 1] = -1
    want = sum(len(set(r)) for r in idx[:, : Lq // 16 * 16].reshape(-1, 16 * K).tolist())
    d = idx.to(dev)
    assert sum(hb.hip_prefill_union(d).tolist()) == want
    assert sum(hb.hip_prefill_union(d.permute(2, 0, 1).contiguous().permute(1, 2, 0)).tolist()) == want


@pytest.mark.parametrize("form", ["heads", "latent"])
@pytest.mark.parametrize("T", [40, 777])
def test_layer_output_in_64_bits(dev, form, T):
    """The bf16 layer's output through either kernel, from its input to after ``o_proj``, against the
    whole in 64 bits (given the selections, which depend on rounding).  The 2-norm of the difference:
    seven bf16 roundings in a row (q; the latent rows; keys or absorbed queries; values; means; the
    heads' output; the layer's) of 2^-9 / sqrt(3) each and their effect on the scores; 4e-3 expected,
    1.5e-2 allowed."""
    from maba_sparse.layers import MabaSparseAttention
    torch.manual_seed(3)
    H, dh, D = 5, 64, 320
    layer = MabaSparseAttention(dim=D, n_heads=H, d_head=dh, d_c=128, d_idx=32, top_k=6).to(dev, torch.bfloat16).eval()
    layer.prefill_form = form
    seen = {}
    fused = layer._fused_prefill
    layer._fused_prefill = lambda x, q, c, idx: (seen.update(idx=idx), fused(x, q, c, idx))[1]
    x = torch.randn(2, T, D, device=dev).bfloat16()
    with torch.no_grad():
        y, _ = layer(x)
    lin = lambda t, m: t @ to_np(m.weight).T + (0 if m.bias is None else to_np(m.bias))  # noqa: E731
    heads = lambda t: t.reshape(2, -1, H, dh).transpose(0, 2, 1, 3)  # noqa: E731
    xd = to_np(x)
    c = lin(xd, layer.kv_down_proj)
    nc = T // 64
    means = c[:, : nc * 64].reshape(2, nc, 64, 128).mean(axis=2)
    n_early = min(T, 63)
    early = c[:, :n_early].cumsum(axis=1) / np.arange(1, n_early + 1)[:, None]
    kh, vh = (heads(lin(means, m)) if nc else None for m in (layer.k_up_proj, layer.v_up_proj))
    o = osa.maba_sa_prefill_heads(heads(lin(xd, layer.q_proj)), heads(lin(c, layer.k_up_proj)), heads(lin(c, layer.v_up_proj)),
                                  kh, vh, heads(lin(early, layer.v_up_proj)), seen["idx"].cpu().numpy(),
                                  lin(xd, layer.stream_gate), scale=dh ** -0.5)
    want = lin(o.transpose(0, 2, 1, 3).reshape(2, T, H * dh), layer.o_proj)
    err = np.linalg.norm(to_np(y) - want) / np.linalg.norm(want)
    assert err < 1.5e-2, err
    print(f"{form} {T}: {err:.2e}")


@pytest.mark.parametrize("dh,scale,bound", [(64, 0.25, 9.7e-7), (32, 0.5, 8.3e-7), (128, 0.25, 8.6e-7)])
def test_fp32_output_error(dev, dh, scale, bound):
    """Relative 2-norm of the error before the output's rounding.  A query's heaviest key is exact in
    the probabilities' bf16 hi + lo parts while the running reference is its score; a reference that
    lags far behind leaves it a rounding of 2^-17 as well.  Bounds: 6 % above the errors with the
    reference always at the largest score (9.14e-7, 7.63e-7, 7.94e-7); with one lagging by up to 2^8
    1.03e-6, 8.9e-7, 9.2e-7."""
    case = list(_case(1, 4, 1000, 1000, dh, 8, 21))
    case[6] = _distinct(1, 1000, 16, 8, 6)
    q, k, v, kh, vh, early, idx, gate = case
    d = lambda t: None if t is None else t.to(dev)  # noqa: E731
    out = to_np(_hip().hip_maba_sa_prefill(*(d(t) for t in case), scale=scale, out_dtype=torch.float32))
    exp = osa.maba_sa_prefill_heads(*(to_np(t) if t is not None else None for t in (q, k, v, kh, vh, early)), idx.numpy(),
                                    to_np(gate), window=128, n_sink=4, scale=scale)
    err = np.linalg.norm((out - exp)[:, :, 64:]) / np.linalg.norm(exp[:, :, 64:])
    assert err < bound, err
