"""How finely the DGDA prefill cuts a sequence with the preferred workspace, read from its size (no
GPU: 256 CUs are assumed).  Where a state remembers, every segment's start costs a step that waits
for the one before, so the number of segments is bounded."""
import os

import pytest

from maba_sparse import _native as N
from test_capi_boundary import _t

pytestmark = pytest.mark.skipif(not os.path.exists(N.LIB_PATH), reason="libmaba_hip.so not built")
CUS = 256


def _nbytes(B, H, T, d, gates, which, dv=None):
    q, v = _t([B, H, T, d]), _t([B, H, T, dv or d])
    token = [H * T, T, 1, 0]
    gate = lambda: _t([B, H, T, d], N.MABA_F32, token if gates == "token" else None)  # noqa: E731
    return getattr(N.load(), f"maba_hip_dgda_prefill_workspace_{which}")(q, v, gate(), gate())


def _chunk_segments(BH, T, which="preferred"):
    return _nbytes(1, BH, T, 64, "token", which) / (BH * (64 * 128 + 1) * 4)


@pytest.mark.parametrize("BH", [1, 2, 3, 4, 6, 8, 10, 16, 20, 40, 80])
def test_chunk_cut_is_bounded(BH):
    for nch in [*range(15, 70), 128, 157, 256, 300, 512, 600, 1024, 2048, 4096, 16384]:
        least, n = _chunk_segments(BH, nch * 64, "size"), _chunk_segments(BH, nch * 64)
        assert n == int(n) or n < 1            # whole segments, or 16 bytes for one
        if nch > 16:
            assert n >= least
        # ends inside slots add one
        assert n <= max(29, least), f"{nch} chunks"
        if n > 14 and BH * nch <= 16 * CUS:    # a long walk: one workgroup per CU
            assert BH * nch / (n - 1) >= min(16, BH * nch / CUS) - 1, f"{nch} chunks"


def test_chunk_cut_where_walks_are_short():
    """Two heads' short prompts are still cut into slots of four chunks."""
    assert _chunk_segments(20, 2048) == 9 and _chunk_segments(40, 1500) == 7


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("BH", [1, 2, 4, 10, 40, 160])
def test_sub_chunk_cut_is_bounded(BH, d):
    for T in (100, 1000, 4096, 10007, 32768, 65536):   # longer, the least size is the larger one
        n = _nbytes(1, BH, T, d, "channel", "preferred") / (BH * (d * 2 * d * 4 + 8))
        assert n <= {32: 256, 64: 192, 128: 96}[d], f"{T} tokens"


@pytest.mark.parametrize("dk,dv,BH,T,segments", [
    (64, 64, 160, 200, 1), (64, 64, 160, 240, 1), (64, 64, 320, 200, 1), (64, 64, 320, 500, 1), (64, 64, 320, 1000, 1),
    (64, 64, 160, 320, 4), (64, 64, 10, 200, 3), (64, 64, 40, 320, 4), (64, 64, 320, 1100, 3), (64, 64, 160, 1000, 6),
    (128, 64, 160, 170, 1), (128, 64, 160, 250, 1), (128, 64, 10, 170, 3), (128, 64, 160, 1000, 6), (128, 128, 160, 170, 3),
    (32, 32, 10, 170, 1), (32, 32, 160, 200, 1), (32, 32, 10, 250, 4), (32, 32, 640, 320, 1), (32, 32, 160, 320, 4)])
def test_sub_chunk_short_sequences(dk, dv, BH, T, segments):
    """Many heads' short sequences stay whole, few heads' and long ones are cut."""
    n = _nbytes(1, BH, T, dk, "channel", "preferred", dv) / (BH * (dk * (dv + dk) * 4 + 8))
    assert max(1, n) == segments
