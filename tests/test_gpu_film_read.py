"""Film read-back: the channels the device makes from the accumulators, at
pixel counts around the block size and past one launch's pixels."""
import numpy as np
import pytest
import torch

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


def test_reading_the_film_takes_no_device_memory():
    """Film mode's buffers are there when it is switched on: a read after a
    long render must not fail for want of memory (38 MB at this size)."""
    s = scenes.box_room(513, 512)
    p = rrhip.RenderParams.make(max_depth=1, samples_per_pass=1)
    with rrhip.Context(0) as ctx:
        ps = rrhip.PtScene(ctx, s.desc())
        for first in (True, False):  # the first session's read loads the kernel's code
            se = ps.session(p)
            se.set_film(True)
            se.render(0, 1)
            free = torch.cuda.mem_get_info(0)[0]
            se.film()
            if not first:
                assert torch.cuda.mem_get_info(0)[0] == free
            se.close()
        ps.close()
