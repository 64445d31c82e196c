"""Default chunks of harmonics of the eccentric realizations (CPU).  Every chunk draws under a seed of its
own, so the chunks of given sizes are part of what a seed means and stay what they are."""
import pytest


@pytest.mark.parametrize("B,F,H,R,chunk", [
    (1, 1, 1, 1, 1), (52111, 20, 30, 100, 30), (189771, 40, 100, 100, 12), (744471, 40, 100, 500, 3),
    (744471, 1, 100, 2000, 100), (127551, 10, 90, 1500, 69), (79296, 16, 93, 467, 72), (124215, 18, 93, 75, 41),
    (118275, 6, 159, 53, 129), (174824, 22, 173, 857, 23), (71712, 39, 193, 47, 33), (202500, 7, 174, 26, 65),
    (273240, 22, 93, 775, 15), (75768, 22, 164, 195, 55), (58344, 25, 182, 196, 63), (37044, 22, 195, 286, 111),
])
def test_default_chunks_stay(B, F, H, R, chunk):
    from holodeck_amd import engine
    assert engine.eccen_harm_chunk(B, F, H, R) == chunk
