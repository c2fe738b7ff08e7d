"""What the workspace of a convolution's weight gradient holds: 256 floats per tile of sums, for 64 sets of tiles for the reduction
and for as many more as shares of 32 steps of a row give up to 32768 of them (layers of up to 16 (channel, kernel row) pairs) or
some 8192 (wider ones).  The kernel cuts the line it walks to the room there is (test_gpu_synapse_walk.py)."""
import pytest

# (N, Ci, Co, H, W, T), kernel, padding -> shares of the time axis, tiles of a wave
CASES = [((64, 1, 16, 32, 32, 300), 3, 1, 10, 3),                # 2048 rows x 10 visits
         ((32, 4, 16, 32, 32, 302), 3, 1, 10, 3),
         ((8, 4, 64, 64, 64, 300), 3, 1, 10, 3),                 # four blocks of channels
         ((32, 2, 16, 64, 64, 900), 5, 2, 15, 5),                # 2048 rows: two visits of 29 a share
         ((2, 1, 16, 4, 4, 31), 3, 1, 1, 3),
         ((32, 8, 16, 32, 32, 300), 3, 1, 5, 6)]                 # 24 pairs


@pytest.mark.parametrize('size,kernel,pad,shares,tiles', CASES)
def test_shares_of_the_time_axis(size, kernel, pad, shares, tiles):
    from lava_dl_amd.slayer import _native
    n, ci, co, h, w, t = size
    waves = n * h * shares
    floats = _native.lib().slayer_conv_synapse_wgrad_workspace(n, ci, co, h, w, t, kernel, kernel, 1, pad, 1)
    assert floats == (waves + 64) * ((co + 15) // 16) * tiles * 256
