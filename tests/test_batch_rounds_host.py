"""The batch's brick layout where an item has more segments than one round stages,
checked on the host: the only brick of 4 x 4 x 8 is crossed by every ray and rows
are cut into at most 64 slices, so 150,000 rays leave more than two cuts of 1024
segments in every item."""
import numpy as np

CUT = 1024  # segments between the recorded positions a round may start from
MAX_SLICES = 64


def test_layout_of_items_with_several_rounds(P, monkeypatch):
    """The self-check walks the items round by round through their cuts and
    compares with the CSC before any device call; without a GPU creation then
    stops at the device (code 4)."""
    monkeypatch.setenv("PLSQR_TILE_CHECK", "1")
    rays = 150000
    s = P.generate(4, 4, 8, rays, P.GEOM_OPPOSITE_FACES, 3, 0.02, 0.1)
    assert np.unique(s.k_row_idx).size == rays and rays / MAX_SLICES > 2 * CUT
    for n_rhs in (1, 4):
        try:
            P.Batch([s], n_rhs, flags=P.BATCH_NO_TUNE).close()
        except P.PlsqrError as e:
            assert e.code == 4 and "self-check" not in str(e), str(e)
