"""Film read-back: the channels the device makes from the accumulators, at
pixel counts around the block size and past one launch's pixels."""
import numpy as np
import pytest

import rrhip
import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height", [(1, 1), (63, 1), (257, 1), (513, 512)])
def test_film_channels_follow_the_accumulator(width, height):
    s = scenes.box_room(width, height)
    p = rrhip.RenderParams.make(max_depth=3)
    with rrhip.Context(0) as ctx:
        ps = rrhip.PtScene(ctx, s.desc())
        se = ps.session(p)
        se.set_film(True)
        assert not se.film().any()  # no samples: every channel zero
        for start in (0, 1):  # a second read after more samples
            se.render(start, 1)
            f, a = se.film(), se.accum()
            assert f.shape == (width * height, rrhip.FILM_CHANNELS)
            # the same two float64 operations per channel, so bit for bit
            assert np.array_equal(f[:, 0:3], a[:, 0:3] / a[:, 6:7])
            assert np.array_equal(f[:, 6:9], np.maximum(f[:, 0:3] - f[:, 3:6], 0.0))
            # counts over samples: 0, 1/2 or 1
            assert np.isin(f[:, 17], [0.0, 0.5, 1.0]).all()
            assert (f[:, 15] > 0).any()
        se.close()
        ps.close()
