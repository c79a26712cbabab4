"""The kernels that run fp32 contractions on the f16 matrix cores by splitting
each operand into two f16 parts under a power-of-two row scale (s2s_split.hip),
against the oracle's fp32: at the sizes where their tiling changes, and over
input magnitudes far outside f16's range."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def run_stage(pkg, orc, c, heads, ratio, depth, hp, wp, scale=1.0, seed=5):
    """max |device - oracle| of one stage, over max |oracle|."""
    M = pkg.model
    arch = M.Arch(upsampler="pixelshuffle", scale=2, embed=c, heads=heads, mlp_ratio=ratio,
                  depths=[depth])
    wts = M.make_weights(arch, seed=seed, perturb=True)
    x = np.random.default_rng(seed).standard_normal((hp * wp, c), dtype=np.float32)
    x = (x * np.float32(scale)).astype(np.float32)
    nchw = np.ascontiguousarray(x.reshape(hp, wp, c).transpose(2, 0, 1))
    want = orc.rstb(arch, wts, orc.plan_explicit(hp, wp, 8, c), 0, nchw)
    be = pkg.HipBackend(arch, wts)
    try:
        got = be.test_rstb(0, hp, wp, x)
    finally:
        be.close()
    got = got.reshape(hp, wp, c).transpose(2, 0, 1)
    assert np.isfinite(got).all()
    return np.abs(got - want).max() / np.abs(want).max()


# (C, heads, mlp ratio, plane): one to four row blocks of 16 tokens per task,
# with row counts that leave a partial last task, a plane of one window, widths
# that end in a partial k step (180 = 5 x 32 + 20) and inside a 16-column tile
# (60, 36), the largest width (192) and other hidden widths. 1e-4 of the largest
# value is the bar of the other stage tests.
@pytest.mark.parametrize("c,heads,ratio,hp,wp", [
    (180, 6, 2, 8, 8), (180, 6, 2, 8, 40), (180, 6, 2, 96, 96), (180, 6, 2, 128, 136),
    (60, 6, 2, 8, 8), (60, 6, 2, 144, 152), (60, 6, 2, 224, 232),
    (120, 6, 2, 16, 24), (192, 6, 1, 16, 24), (36, 3, 3, 16, 24), (24, 2, 4, 8, 16),
])
def test_token_half_sizes(pkg, orc, c, heads, ratio, hp, wp):
    assert run_stage(pkg, orc, c, heads, ratio, 1, hp, wp) < 1e-4


# magnitudes that f16 cannot hold unscaled (largest 65,504, smallest 6e-8)
@pytest.mark.parametrize("c", [180, 60])
@pytest.mark.parametrize("scale", [0.0, 1e-20, 1e-6, 1e6, 1e15])
def test_token_half_magnitudes(pkg, orc, c, scale):
    assert run_stage(pkg, orc, c, 6, 2, 2, 16, 24, scale) < 1e-4
