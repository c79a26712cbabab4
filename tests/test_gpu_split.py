"""The kernels that run fp32 contractions on the f16 matrix cores by splitting
each operand into two f16 parts under a power-of-two row scale (s2s_split.hip),
against the oracle's fp32: at the sizes where their tiling changes, and over
input magnitudes far outside f16's range."""
import numpy as np
import pytest

import refimpl as R

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


# (C, heads, mlp ratio, plane): a plane of one window up to more tasks than run at
# once, row counts that leave a partial last task, widths
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


# Each build of the token half: every count of row blocks per task (`rb`) at every
# width class, with a partial last task and with more tasks than run at once.
@pytest.mark.parametrize("c,heads,hp,wp,rb", [
    (60, 6, 40, 72, 1), (60, 6, 144, 152, 2), (60, 6, 200, 200, 3), (36, 3, 264, 264, 3),
    (120, 6, 40, 72, 1), (128, 4, 96, 96, 2), (120, 6, 128, 136, 3), (192, 6, 40, 72, 1), (180, 6, 96, 96, 2),
    (192, 6, 136, 128, 3),
])
def test_token_half_row_blocks(pkg, orc, c, heads, hp, wp, rb):
    assert pkg.abi.split_tiles(hp, wp, c, c)[0] == rb
    assert run_stage(pkg, orc, c, heads, 2, 1, hp, wp) < 1e-4


# magnitudes that f16 cannot hold unscaled (largest 65,504, smallest 6e-8)
@pytest.mark.parametrize("c", [180, 60])
@pytest.mark.parametrize("scale", [0.0, 1e-20, 1e-6, 1e6, 1e15])
def test_token_half_magnitudes(pkg, orc, c, scale):
    assert run_stage(pkg, orc, c, 6, 2, 2, 16, 24, scale) < 1e-4


# A bias far above the rows' deviation in front of each LayerNorm, and weights with a
# large common part besides: the norm takes the row's mean off, and what it leaves is
# at the bar of the other stage tests (an fp32 sum would carry the mean's rounding,
# 2^-24 of it over the deviation: 2e-3 at 3e4).
@pytest.mark.parametrize("c", [180, 60, 24])
@pytest.mark.parametrize("where", ["attn.proj", "mlp.fc2"])
@pytest.mark.parametrize("offset", [3e2, -3e3, 3e4, 1e8])
def test_token_half_row_offset(pkg, c, where, offset):
    M = pkg.model
    hp, wp, heads = 8, 16, 2 if c == 24 else 6
    arch = M.Arch(upsampler="pixelshuffle", scale=2, embed=c, heads=heads, mlp_ratio=2, depths=[1])
    wts = M.make_weights(arch, seed=5, perturb=True)
    p = "layers.0.residual_group.blocks.0." + where
    wts[p + ".bias"] = (wts[p + ".bias"] + np.float32(offset)).astype(np.float32)
    if offset < 0:
        wts[p + ".weight"] = (wts[p + ".weight"] + np.float32(8)).astype(np.float32)
    x = np.random.default_rng(c).standard_normal((c, hp, wp)).astype(np.float32)
    want = R.rstb(x.astype(np.float64), wts, 0, 1, 8, heads)
    be = pkg.HipBackend(arch, wts)
    try:
        got = be.test_rstb(0, hp, wp, np.ascontiguousarray(x.transpose(1, 2, 0).reshape(hp * wp, c)))
    finally:
        be.close()
    err = np.abs(got.reshape(hp, wp, c).transpose(2, 0, 1) - want).max() / np.abs(want).max()
    assert err < 1e-4, err


# One unit of the hidden layer with an fc1 row 2^12 times the others', or shut by a
# bias far below 0, and no part in fc2: with the scale that the units share, the rest
# is no further from 64 bits than the fp32 GEMMs were (6.9e-7 and 3.1e-7; the seed
# and the sums' order move it by a tenth).
@pytest.mark.parametrize("c", [180, 60])
@pytest.mark.parametrize("row,bias", [(1.0, 0.0), (2.0 ** 12, 0.0), (1.0, -2.0 ** 20)])
def test_token_half_hidden_outlier(pkg, c, row, bias):
    M = pkg.model
    hp, wp, p = 16, 24, "layers.0.residual_group.blocks.0.mlp."
    arch = M.Arch(upsampler="pixelshuffle", scale=2, embed=c, heads=6, mlp_ratio=2, depths=[1])
    wts = M.make_weights(arch, seed=5, perturb=True)
    for k in ("fc1.weight", "fc1.bias", "fc2.weight"):
        wts[p + k] = wts[p + k].copy()
    wts[p + "fc1.weight"][7] *= np.float32(row)
    wts[p + "fc1.bias"][7] += np.float32(bias)
    wts[p + "fc2.weight"][:, 7] = 0
    x = np.random.default_rng(c).standard_normal((c, hp, wp)).astype(np.float32)
    want = R.rstb(x.astype(np.float64), wts, 0, 1, 8, 6)
    be = pkg.HipBackend(arch, wts)
    try:
        got = be.test_rstb(0, hp, wp, np.ascontiguousarray(x.transpose(1, 2, 0).reshape(hp * wp, c)))
    finally:
        be.close()
    d = got.reshape(hp, wp, c).transpose(2, 0, 1) - want
    rel = np.linalg.norm(d) / np.linalg.norm(want)
    assert rel < (6.9e-7 if c == 180 else 3.1e-7), rel


def attention_f64(x, w, b, ls, cpb, hp, wp, heads, hd, shift, norms=False):
    """qkv projection and window attention in 64 bits, on [hp*wp][c] rows; with
    norms, of the norms of each head's v in the place of its values."""
    c = heads * hd
    X = x.astype(np.float64).reshape(hp, wp, c)
    X = np.roll(X, (-shift, -shift), (0, 1))
    win = lambda t: t.reshape(hp // 8, 8, wp // 8, 8, -1).transpose(0, 2, 1, 3, 4).reshape(-1, 64, t.shape[-1])
    qkv = win(X) @ w.astype(np.float64).T + b
    q, k, v = (t.reshape(-1, 64, heads, hd).transpose(0, 2, 1, 3) for t in np.split(qkv, 3, -1))
    q, k = (t / np.maximum(np.linalg.norm(t, axis=-1, keepdims=True), 1e-12) for t in (q, k))
    if norms:
        v = np.repeat(np.linalg.norm(v, axis=-1, keepdims=True), hd, -1)
    s = q @ k.transpose(0, 1, 3, 2)
    s = s * np.exp(np.minimum(ls.astype(np.float64), np.log(100.0)))[None, :, None, None]
    s += cpb.astype(np.float64).reshape(64, 64, heads).transpose(2, 0, 1)
    if shift:
        band = lambda n: (np.arange(n) >= n - 8).astype(int) + (np.arange(n) >= n - shift)
        reg = win((band(hp)[:, None] * 3 + band(wp)[None, :])[..., None])[..., 0]
        s -= 100.0 * (reg[:, :, None] != reg[:, None, :])[:, None]
    p = np.exp(s - s.max(-1, keepdims=True))
    o = (p / p.sum(-1, keepdims=True)) @ v
    o = o.transpose(0, 2, 1, 3).reshape(hp // 8, wp // 8, 8, 8, c).transpose(0, 2, 1, 3, 4)
    return np.roll(o.reshape(hp, wp, c), (shift, shift), (0, 1)).reshape(hp * wp, c)


# planes of one window, of fewer windows than XCDs, of one window column, and of
# more items than workgroups at once (256 CUs x 2, a third of it windows). The
# bar is per window: x of each window scaled by its own power of ten. A logit of
# 100 x 1.44 in fp32 carries 100 x 1.44 x 6e-8 = 9e-6 into each probability, and
# a cosine of 30 terms a few roundings more: 5e-5 of the window's largest value.
@pytest.mark.parametrize("hd", [30, 10])
@pytest.mark.parametrize("hp,wp", [(8, 8), (8, 40), (72, 8), (120, 136)])
@pytest.mark.parametrize("shift", [0, 4])
@pytest.mark.parametrize("spread", [0, 12])
def test_window_attention(pkg, hd, hp, wp, shift, spread):
    heads, c = 6, 6 * hd
    rng = np.random.default_rng(hp * 1000 + wp + hd + shift + spread)
    x = rng.standard_normal((hp, wp, c))
    mag = 10.0 ** rng.uniform(-spread, spread, size=(hp // 8, wp // 8))
    x = np.roll(x, (-shift, -shift), (0, 1)) * np.kron(mag, np.ones((8, 8)))[..., None]
    x = np.roll(x, (shift, shift), (0, 1)).reshape(hp * wp, c).astype(np.float32)
    w = (rng.standard_normal((3 * c, c)) * 0.05).astype(np.float32)
    b = np.zeros(3 * c, np.float32)
    if not spread:
        b = rng.uniform(-0.1, 0.1, 3 * c).astype(np.float32)
        b[c:2 * c] = 0
    ls = np.linspace(0.0, 5.5, heads).astype(np.float32)
    cpb = (16 / (1 + np.exp(-rng.standard_normal((4096, heads))))).astype(np.float32)
    got = pkg.abi.test_block_attention(hp, wp, heads, hd, shift, x, w, b, ls, cpb)
    want = attention_f64(x, w, b, ls, cpb, hp, wp, heads, hd, shift)
    win = lambda t: np.roll(t.reshape(hp, wp, c), (-shift, -shift), (0, 1)).reshape(
        hp // 8, 8, wp // 8, 8, c).transpose(0, 2, 1, 3, 4).reshape(-1, 64 * c)
    err = np.abs(win(got - want)).max(1) / np.abs(win(want)).max(1)
    assert err.max() < 5e-5, err.max()


# Tokens of a window apart by up to 2^50: a row of the plane that the shift mask
# parts from the rest of its windows, single tokens, and every token. An output's
# error is held against the sum of its probabilities times the norms of v, to which
# fp32's is in proportion, so a large token that a query hardly sees costs it
# nothing. 5e-5 as above.
@pytest.mark.parametrize("hd", [30, 10])
@pytest.mark.parametrize("shift", [0, 4])
@pytest.mark.parametrize("span", [4, 7, 20, 50])
@pytest.mark.parametrize("where", ["rows", "token", "all"])
def test_window_attention_tokens_apart(pkg, hd, shift, span, where):
    heads, c, hp, wp = 6, 6 * hd, 24, 40
    rng = np.random.default_rng(hd + shift + span)
    x = rng.standard_normal((hp, wp, c))
    if where == "rows":
        x[20:] *= 2.0 ** span
    elif where == "token":
        x[3::8, 5::8] *= 2.0 ** span
    else:
        x *= 2.0 ** rng.integers(-span, 1, (hp, wp, 1))
    x = x.reshape(hp * wp, c).astype(np.float32)
    w = (rng.standard_normal((3 * c, c)) * 0.05).astype(np.float32)
    b = np.zeros(3 * c, np.float32)
    ls = np.linspace(0.0, 5.5, heads).astype(np.float32)
    cpb = (16 / (1 + np.exp(-rng.standard_normal((4096, heads))))).astype(np.float32)
    got = pkg.abi.test_block_attention(hp, wp, heads, hd, shift, x, w, b, ls, cpb)
    want = attention_f64(x, w, b, ls, cpb, hp, wp, heads, hd, shift)
    size = attention_f64(x, w, b, ls, cpb, hp, wp, heads, hd, shift, norms=True)
    err = (np.abs(got - want) / size).max()
    assert err < 5e-5, err


# the tile is 8 pixels by 2 to 16 rows: planes smaller than one, of one column of
# tiles, ragged in both directions, and of more tiles than workgroups (2 x 256);
# widths that end inside a k step and inside a column tile. Sums of 9 cin products
# in fp32 on unit-normal data: sqrt(1620) roundings of 6e-8 of at most 5 would be
# 1.2e-5.
@pytest.mark.parametrize("cin,cout,h,w", [
    (180, 180, 1, 1), (180, 180, 7, 9), (180, 180, 96, 100), (180, 180, 130, 124),
    (120, 120, 40, 72), (60, 60, 3, 50), (60, 60, 150, 133), (180, 64, 50, 37),
    (120, 32, 64, 65), (60, 4, 17, 70),
])
@pytest.mark.parametrize("epilogue", [0, 2, 5])
def test_split_conv(pkg, cin, cout, h, w, epilogue):
    import torch
    rng = np.random.default_rng(cin + cout + h + w)
    x = rng.standard_normal((h * w, cin), dtype=np.float32)
    wt = (rng.uniform(-1, 1, (cout, cin, 3, 3)) * (1 / (3 * cin)) ** 0.5).astype(np.float32)
    b = rng.standard_normal(cout, dtype=np.float32)
    res = rng.standard_normal((h * w, cout), dtype=np.float32)
    got = pkg.abi.test_conv3x3_winograd(x, h, w, wt, b, epilogue, res if epilogue == 2 else None, 0.2)
    t = torch.from_numpy
    want = torch.nn.functional.conv2d(t(x.astype(np.float64).reshape(h, w, cin)).permute(2, 0, 1)[None],
                                      t(wt.astype(np.float64)), t(b.astype(np.float64)), padding=1)
    want = want[0].permute(1, 2, 0).reshape(h * w, cout).numpy()
    if epilogue == 2:
        want = want + res
    if epilogue == 5:
        want = np.where(want < 0, 0.2 * want, want)
    assert np.abs(got - want).max() < 2e-5


# Each build of the conv: every count of row blocks per wave (`rb`) of every shape,
# and the tiles shared by all of a wave's column tiles (`share`).
@pytest.mark.parametrize("cin,cout,h,w,rb,share", [
    (60, 60, 37, 70, 1, 2), (60, 60, 67, 129, 1, 1), (60, 60, 161, 163, 2, 1), (60, 60, 199, 211, 3, 1),
    (60, 60, 251, 259, 3, 1), (60, 60, 230, 250, 4, 1), (120, 32, 37, 70, 1, 2), (120, 32, 99, 131, 1, 1),
    (120, 32, 150, 133, 2, 1), (120, 32, 170, 190, 3, 1), (180, 64, 37, 70, 1, 2), (180, 64, 170, 190, 1, 1),
    (180, 64, 161, 163, 2, 1), (120, 120, 3, 50, 1, 2), (120, 120, 37, 70, 1, 1), (120, 120, 67, 129, 2, 1),
    (120, 120, 130, 124, 3, 1), (120, 120, 161, 163, 4, 1), (180, 180, 3, 50, 1, 3), (180, 180, 37, 70, 1, 1),
    (180, 180, 67, 129, 2, 1), (180, 180, 130, 124, 3, 1),
])
def test_split_conv_row_blocks(pkg, cin, cout, h, w, rb, share):
    assert pkg.abi.split_tiles(h, w, cin, cout)[1:] == (rb, share)
    rng = np.random.default_rng(cin + cout + h + w)
    x = rng.standard_normal((h * w, cin), dtype=np.float32)
    wt = (rng.uniform(-1, 1, (cout, cin, 3, 3)) * (1 / (3 * cin)) ** 0.5).astype(np.float32)
    b = rng.standard_normal(cout, dtype=np.float32)
    res = rng.standard_normal((h * w, cout), dtype=np.float32)
    got = pkg.abi.test_conv3x3_winograd(x, h, w, wt, b, 2, res, 0.0).reshape(h, w, cout)
    assert np.abs(got - conv_f64(x, wt, b, h, w) - res.reshape(h, w, cout)).max() < 2e-5


# A non-finite value reaches the outputs whose footprint holds it and no other.
@pytest.mark.parametrize("cin,cout", [(180, 180), (60, 60)])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_split_conv_nonfinite(pkg, cin, cout, bad):
    h, w = 40, 33
    rng = np.random.default_rng(7)
    x = rng.standard_normal((h * w, cin), dtype=np.float32)
    wt = (rng.uniform(-1, 1, (cout, cin, 3, 3)) * (1 / (3 * cin)) ** 0.5).astype(np.float32)
    b = rng.standard_normal(cout, dtype=np.float32)
    clean = pkg.abi.test_conv3x3_winograd(x, h, w, wt, b, 0).reshape(h, w, cout)
    x[17 * w + 12, 5] = bad
    got = pkg.abi.test_conv3x3_winograd(x, h, w, wt, b, 0).reshape(h, w, cout)
    near = np.zeros((h, w), bool)
    near[16:19, 11:14] = True
    assert not np.isfinite(got[near]).any()
    # (the scale may differ by the clean value's part in the maximum)
    assert np.abs(got[~near] - clean[~near]).max() < 2e-5


def conv_f64(x, wt, b, h, w):
    import torch
    t = torch.from_numpy
    y = torch.nn.functional.conv2d(t(x.astype(np.float64).reshape(h, w, -1)).permute(2, 0, 1)[None],
                                   t(wt.astype(np.float64)), t(b.astype(np.float64)), padding=1)
    return y[0].permute(1, 2, 0).numpy()


# Pixels of one tile apart by up to 2^60, one of them alone among small ones: an
# output owes nothing to pixels outside its footprint, as in fp32, so each output's
# error is held against its own footprint's largest pixel. 2e-5 as above.
@pytest.mark.parametrize("cin,cout,h,w", [(180, 180, 13, 11), (180, 180, 96, 100), (120, 120, 9, 20),
                                          (60, 60, 40, 33), (180, 64, 50, 37), (120, 32, 17, 9)])
@pytest.mark.parametrize("spread", [20, 60])
def test_split_conv_pixels_apart(pkg, cin, cout, h, w, spread):
    rng = np.random.default_rng(cin + cout + h + spread)
    mag = 2.0 ** -rng.integers(0, spread, (h, w))
    mag[h // 2 - 3:h // 2 + 4, w // 2 - 3:w // 2 + 4] = 2.0 ** -spread
    mag[h // 2, w // 2] = 1.0
    x = (rng.standard_normal((h, w, cin)) * mag[..., None]).astype(np.float32).reshape(h * w, cin)
    wt = (rng.uniform(-1, 1, (cout, cin, 3, 3)) * (1 / (3 * cin)) ** 0.5).astype(np.float32)
    got = pkg.abi.test_conv3x3_winograd(x, h, w, wt, np.zeros(cout, np.float32), 0).reshape(h, w, cout)
    want = conv_f64(x, wt, np.zeros(cout), h, w)
    pad = np.pad(mag, 1)
    near = np.max([pad[i:i + h, j:j + w] for i in range(3) for j in range(3)], 0)
    err = (np.abs(got - want) / near[..., None]).max()
    assert err < 2e-5, err


# An infinity is that infinity times the weight's sign in every output whose
# footprint holds it, a NaN or two opposite infinities in one tap sum a NaN.
@pytest.mark.parametrize("cin,cout", [(180, 180), (60, 60), (180, 64)])
@pytest.mark.parametrize("epilogue", [0, 5])
def test_split_conv_infinities(pkg, cin, cout, epilogue):
    h, w = 40, 33
    rng = np.random.default_rng(9)
    x = rng.standard_normal((h * w, cin), dtype=np.float32)
    wt = (rng.uniform(-1, 1, (cout, cin, 3, 3)) * (1 / (3 * cin)) ** 0.5).astype(np.float32)
    b = rng.standard_normal(cout, dtype=np.float32)
    x[3 * w + 5, 7], x[17 * w + 12, 5], x[30 * w + 32, cin - 1], x[22 * w, 3] = np.inf, -np.inf, np.inf, np.nan
    x[30 * w + 32, 1] = 3e38
    got = pkg.abi.test_conv3x3_winograd(x, h, w, wt, b, epilogue, None, 0.2).reshape(h, w, cout)
    with np.errstate(invalid="ignore"):
        want = conv_f64(x, wt, b, h, w)
    if epilogue == 5:
        want = np.where(want < 0, 0.2 * want, want)
    bad = ~np.isfinite(want)
    assert np.array_equal(got[bad], want[bad].astype(np.float32), equal_nan=True)
    assert np.abs(got[~bad] - want[~bad]).max() < 2e-5


# Output channels apart by up to 2^40: each one's error against its own weights.
@pytest.mark.parametrize("cin,cout", [(180, 180), (120, 120), (60, 60), (180, 64), (60, 4)])
def test_split_conv_channels_apart(pkg, cin, cout):
    h, w = 20, 33
    rng = np.random.default_rng(cin + cout)
    x = rng.standard_normal((h * w, cin), dtype=np.float32)
    mag = 2.0 ** -rng.permutation(np.linspace(0, 40, cout).astype(int))
    wt = rng.uniform(-1, 1, (cout, cin, 3, 3)) * (1 / (3 * cin)) ** 0.5
    wt = (wt * mag[:, None, None, None]).astype(np.float32)
    got = pkg.abi.test_conv3x3_winograd(x, h, w, wt, np.zeros(cout, np.float32), 0).reshape(h, w, cout)
    err = (np.abs(got - conv_f64(x, wt, np.zeros(cout), h, w)) / mag).max()
    assert err < 2e-5, err


# A non-finite token costs its window (every query of it sees the token's key) and
# nothing outside: the rest is bit for bit what it is without.
@pytest.mark.parametrize("hd", [30, 10])
@pytest.mark.parametrize("shift", [0, 4])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_window_attention_nonfinite(pkg, hd, shift, bad):
    heads, c, hp, wp = 6, 6 * hd, 24, 40
    rng = np.random.default_rng(hd)
    x = rng.standard_normal((hp, wp, c)).astype(np.float32)
    w = (rng.standard_normal((3 * c, c)) * 0.05).astype(np.float32)
    b = np.zeros(3 * c, np.float32)
    ls = np.linspace(0.0, 5.5, heads).astype(np.float32)
    cpb = rng.uniform(0, 16, (4096, heads)).astype(np.float32)
    run = lambda: pkg.abi.test_block_attention(hp, wp, heads, hd, shift, x.reshape(-1, c), w, b, ls,
                                               cpb).reshape(hp, wp, c)
    clean = run()
    x[shift + 9, shift + 18, 7] = bad
    got = run()
    hit = np.zeros((hp, wp), bool)
    hit[shift + 8:shift + 16, shift + 16:shift + 24] = True
    assert not np.isfinite(got[hit]).any()
    assert np.array_equal(got[~hit], clean[~hit])


# ... and through the token half (row by row) and the stage's closing conv (one
# pixel further).
@pytest.mark.parametrize("c", [180, 60])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_stage_nonfinite(pkg, c, bad):
    M = pkg.model
    hp, wp = 40, 48
    arch = M.Arch(upsampler="pixelshuffle", scale=2, embed=c, heads=6, mlp_ratio=2, depths=[1])
    x = np.random.default_rng(c).standard_normal((hp, wp, c)).astype(np.float32)
    be = pkg.HipBackend(arch, M.make_weights(arch, seed=5, perturb=True))
    try:
        clean = be.test_rstb(0, hp, wp, x.reshape(-1, c)).reshape(hp, wp, c)
        x[9, 18, 7] = bad
        got = be.test_rstb(0, hp, wp, x.reshape(-1, c)).reshape(hp, wp, c)
    finally:
        be.close()
    hit = np.zeros((hp, wp), bool)
    hit[7:17, 15:25] = True
    assert not np.isfinite(got[hit]).any()
    assert np.array_equal(got[~hit], clean[~hit])
