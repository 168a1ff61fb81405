"""How the sub-chunk DGDA prefill cuts a sequence: segments as the workspace allows, in-place
buffers across the launches, and sub-chunks on both sides of the decay range its matrix products
take.  Tolerances as in test_gpu_dgda_prefill.py: rtol = atol = 2e-3 against the float64
recurrence; where only the cut differs, the last bits of fp32 sums of products split to 16
mantissa bits (observed 1e-5)."""
import numpy as np
import pytest
import torch

from _helpers import assert_close, dgda_inputs, oracle_dgda_args, to_np
from oracle import dgda as odgda

pytestmark = pytest.mark.gpu


def _call(inp, nbytes, s0=None, sf=None):
    """maba_hip_dgda_prefill with a workspace of ``nbytes``."""
    from maba_sparse import _native as N
    lib = N.load()
    q, v = inp["q"], inp["v"]
    B, H, L, dk = q.shape
    dv = v.shape[3]
    out = torch.empty(B, H, L, dv, device=q.device)
    sf = torch.empty(B, H, dk, dv, device=q.device) if sf is None else sf
    ws = torch.full((max(int(nbytes), 16),), 0xff, dtype=torch.uint8, device=q.device)   # NaN patterns
    rc = lib.maba_hip_dgda_prefill(N.desc(q), N.desc(inp["k"]), N.desc(v), None, N.desc(inp["log_alpha"]),
                                   N.desc(inp["b"]), N.desc(inp["w"]), N.desc(s0), N.desc(out), N.desc(sf), 16,
                                   ws.data_ptr(), int(nbytes), N.stream_ptr(q.device))
    N.check(rc, "dgda_prefill")
    return out, sf


def _sizes(inp):
    from maba_sparse import _native as N
    lib = N.load()
    d = [N.desc(inp[n]) for n in ("q", "v", "log_alpha", "b")]
    return lib.maba_hip_dgda_prefill_workspace_size(*d), lib.maba_hip_dgda_prefill_workspace_preferred(*d)


@pytest.mark.parametrize("dk,dv", [(64, 64), (32, 32), (128, 128)])
@pytest.mark.parametrize("decay", ["baseline", "slow"])
def test_segments_follow_the_workspace(dev, dk, dv, decay):
    """The least workspace, the preferred one and two between give the recurrence's result."""
    inp = dgda_inputs(1, 2, 1300, dk=dk, dv=dv, seed=3, decay=decay, gates="channel", device=dev, with_state=True)
    eo, eS = odgda.dgda_prefill_seq(**oracle_dgda_args(inp))
    least, best = _sizes(inp)
    assert 16 < least < best
    for nbytes in (least, (least + best) // 2, best - 1, best):
        o, S = _call(inp, nbytes, s0=inp["initial_state"])
        assert_close(o, eo, 2e-3, 2e-3, f"out {nbytes}")
        assert_close(S, eS, 2e-3, 2e-3, f"state {nbytes}")


@pytest.mark.parametrize("B,H,L", [(1, 1, 14 * 64), (1, 2, 14 * 64 + 1), (2, 3, 16 * 64), (3, 1, 16 * 64 + 1), (1, 3, 2100),
                                   (65, 1, 1000), (1, 1, 300 * 64), (1, 10, 7000)])
@pytest.mark.parametrize("decay", ["baseline", "slow"])
def test_chunk_segments_follow_the_workspace(dev, B, H, L, decay):
    """Per-token gates: slots of four chunks with the preferred workspace, of sixteen with any
    smaller one, at the lengths where the cut begins and changes."""
    inp = dgda_inputs(B, H, L, seed=7, decay=decay, gates="scalar", device=dev, with_state=True)
    assert inp["log_alpha"].stride(3) == 0 and inp["q"].dtype == torch.bfloat16
    least, best = _sizes(inp)
    assert (best > least) == (14 * 64 < L and B * H < 65)
    eo, eS = odgda.dgda_prefill_seq(**oracle_dgda_args(inp))
    for nbytes in sorted({least, best - 1, best} - {least - 1}):
        o, S = _call(inp, nbytes, s0=inp["initial_state"])
        assert_close(o, eo, 2e-3, 2e-3, f"out {nbytes}")
        assert_close(S, eS, 2e-3, 2e-3, f"state {nbytes}")


@pytest.mark.parametrize("decay", ["baseline", "slow"])
def test_state_in_place_across_segments(dev, decay):
    inp = dgda_inputs(2, 3, 900, seed=5, decay=decay, gates="channel", device=dev, with_state=True)
    _, best = _sizes(inp)
    o, S = _call(inp, best, s0=inp["initial_state"])
    buf = inp["initial_state"].clone()
    o2, S2 = _call(inp, best, s0=buf, sf=buf)
    assert torch.equal(o, o2) and torch.equal(S, S2)


@pytest.mark.parametrize("L", [1, 2, 3, 17, 700])
def test_layer_history_in_place(dev, L):
    """The new conv history over the old one's buffers, one segment and several."""
    from maba_sparse.kernels import hip_backend as hb
    g = torch.Generator().manual_seed(L)
    rn = lambda *s: torch.randn(*s, generator=g).bfloat16().to(dev)  # noqa: E731
    projs, convs = rn(2, L, 6 * 128).split(128, dim=-1), [rn(128, 1, 4) for _ in range(3)]
    hist = [rn(2, 128, 3) for _ in range(3)]
    o, S, new = hb.hip_dgda_layer_prefill(projs, convs, hist)
    for s in range(3):
        want = torch.cat([hist[s].transpose(1, 2), projs[s]], dim=1)[:, -3:].transpose(1, 2)
        assert torch.equal(new[s], want)
    buf = [h.clone() for h in hist]
    o2, S2, new2 = hb.hip_dgda_layer_prefill(projs, convs, buf, out_history=buf)
    assert torch.equal(o, o2) and torch.equal(S, S2) and all(torch.equal(a, b) for a, b in zip(new, new2))


@pytest.mark.parametrize("per_token", [-3.999, -4.001, -8.0, -30.0, -200.0, 3.999, 4.001])
@pytest.mark.parametrize("dk", [32, 64, 128])
def test_decay_range_of_the_products(dev, per_token, dk):
    """One channel in four decays by ``per_token`` at every token, so a sub-chunk's range is sixteen
    times that: 64 is where the products end and the pairwise sums begin.  Growth is kept to one
    sub-chunk with a written state of order one."""
    L = 16 if per_token > 0 else 70
    inp = dgda_inputs(1, 2, L, dk=dk, dv=64, seed=9, decay="slow", gates="channel", qkv_dtype=torch.float32, device=dev)
    la = inp["log_alpha"].clone()
    la[..., ::4] = per_token
    inp["log_alpha"] = la
    eo, eS = odgda.dgda_prefill_seq(**oracle_dgda_args(inp))
    o, S = _call(inp, _sizes(inp)[1])
    for a, e in ((o, eo), (S, eS)):   # relative to the largest value: growth reaches e^64
        scale = max(1.0, float(np.abs(e).max()))
        assert_close(a / scale, e / scale, 2e-3, 2e-3, f"{per_token}")


def test_layer_strong_decay_gates(dev):
    """Decay projections far up: every sub-chunk of the fused layer leaves the products' range, its
    decays at the e^-14 floor."""
    from maba_sparse.kernels import hip_backend as hb
    g = torch.Generator().manual_seed(2)
    rn = lambda *s: torch.randn(*s, generator=g).bfloat16()  # noqa: E731
    x = list(rn(1, 300, 6 * 64).split(64, dim=-1))
    x[3] = (x[3].float() * 40).bfloat16()
    convs = [rn(64, 1, 4) for _ in range(3)]
    o, S, _ = hb.hip_dgda_layer_prefill([t.to(dev).contiguous() for t in x], [w.to(dev) for w in convs],
                                        state_dtype=torch.float32)
    f = lambda t: t.double().numpy()  # noqa: E731
    q, k, v, la, _, b, w, _ = odgda.layer_prologue(*[f(t) for t in x], *[f(c[:, 0]) for c in convs], n_heads=1)
    eo, eS = odgda.dgda_prefill_seq(*(t[:, None] for t in (q, k, v)), alpha=np.exp(la)[:, None], b=b[:, None], w=w[:, None])
    assert_close(o.float().view(1, 300, 1, 64).transpose(1, 2), eo, 1e-2, 1e-2, "out")   # bf16 output
    assert_close(S, eS, 2e-3, 2e-3, "state")


@pytest.mark.parametrize("fast", [0, 64])
@pytest.mark.parametrize("per_token", [-3.0, -200.0])
def test_transition_that_vanishes_by_half(dev, fast, per_token):
    """d_k = 128: the transition's columns of one half of the channels vanish, the other half's do
    not.  Two waves form a map, and the one whose columns vanish stores nothing."""
    inp = dgda_inputs(1, 2, 1300, dk=128, dv=64, seed=11, decay="slow", gates="channel", device=dev, with_state=True)
    inp["log_alpha"][..., fast: fast + 64] = per_token
    eo, eS = odgda.dgda_prefill_seq(**oracle_dgda_args(inp))
    for nbytes in _sizes(inp):
        o, S = _call(inp, nbytes, s0=inp["initial_state"])
        assert_close(o, eo, 2e-3, 2e-3, f"out {nbytes}")
        assert_close(S, eS, 2e-3, 2e-3, f"state {nbytes}")


def test_rows_beyond_32_bits(dev):
    """600 tokens 4 MiB apart: the sequence's bytes leave 32 bits, a sub-chunk's do not."""
    inp = dgda_inputs(1, 2, 600, seed=4, decay="slow", gates="channel", qkv_dtype=torch.float32, device=dev)
    buf = torch.empty(600, 1 << 20, device=dev)
    far = {}
    for i, n in enumerate(("q", "k", "v", "log_alpha", "b", "w")):
        far[n] = buf[:, 128 * i: 128 * (i + 1)].view(1, 600, 2, 64).transpose(1, 2)
        far[n].copy_(inp[n])
    best = _sizes(inp)[1]
    assert _sizes(far)[1] == best > 16   # the same kernel and cut
    o, S = _call(inp, best)
    o2, S2 = _call(far, best)
    assert torch.equal(o, o2) and torch.equal(S, S2)


def test_layer_rows_beyond_32_bits(dev):
    """600 tokens of projections 4 MiB apart: their bytes leave 31 bits, their elements do not."""
    from maba_sparse.kernels import hip_backend as hb
    g = torch.Generator().manual_seed(6)
    x = torch.randn(1, 600, 6 * 64, generator=g).bfloat16().to(dev)
    convs = [torch.randn(64, 1, 4, generator=g).bfloat16().to(dev) for _ in range(3)]
    far = torch.empty(600, 1 << 21, dtype=torch.bfloat16, device=dev)[None, :, : 6 * 64]
    far.copy_(x)
    want = hb.hip_dgda_layer_prefill(x.split(64, dim=-1), convs)
    got = hb.hip_dgda_layer_prefill(far.split(64, dim=-1), convs)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    assert all(torch.equal(a, b) for a, b in zip(got[2], want[2]))


@pytest.mark.parametrize("L", [1, 15, 100, 300])
def test_layer_columns_per_wave(dev, L):
    """Few heads take 32 value columns per wave, many 64: the same heads give the same bits."""
    from maba_sparse.kernels import hip_backend as hb
    g = torch.Generator().manual_seed(L)
    rn = lambda *s: torch.randn(*s, generator=g).bfloat16().to(dev)  # noqa: E731
    x, convs, hist = rn(1, L, 6 * 128), [rn(128, 1, 4) for _ in range(3)], [rn(1, 128, 3) for _ in range(3)]
    many = 600   # 1,200 heads: more waves than SIMDs, one segment
    args = lambda n: (x.expand(n, -1, -1).contiguous().split(128, dim=-1), convs, [h.expand(n, -1, -1).contiguous() for h in hist])  # noqa: E731
    one, all_ = hb.hip_dgda_layer_prefill(*args(1)), hb.hip_dgda_layer_prefill(*args(many))
    for a, b in zip((one[0], one[1], *one[2]), (all_[0], all_[1], *all_[2])):
        if L <= 100:   # one segment either way
            assert torch.equal(b, a.expand_as(b))
        else:
            assert_close(b[0], to_np(a[0]), 1e-2, 1e-2, "cut differs")
            assert torch.equal(b, b[:1].expand_as(b))
