"""The decode on the FP32 matrix cores (k_decode_mfma) against the VALU decode: the same values bit for bit, as floats, as
bytes and as squared 8-bit differences, over image sizes around its 16-pixel tiles and 64- and 256-pixel rounds, extents,
numbers of outputs and layers, leaks and models with NaN and infinite weights."""
import numpy as np
import pytest

from gpu_common import LAYOUTS, data, say, trainer
from neural_block_textures_amd.trainer import Layout

pytestmark = pytest.mark.gpu


def both(lay, z, p, tgt):
    """(float image, bytes, error of the whole image, error of a smaller extent) on the matrix cores, then on the VALU"""
    got = []
    for on in (True, False):
        tr = trainer(lay, z, p, tgt, max_pairs=1, max_batch=16)
        tr.set_matrix_cores(on)
        out = [tr.decode_full(), tr.decode_full(z[::-1].copy()), tr.decode_rgb8()]
        if lay.nout % 3 == 0:
            for ew, eh in ((0, 0), (max(1, lay.W - 3), max(1, lay.H - 1))):
                a, b = tr.decode_error(ew, eh), tr.decode_error_noalloc(ew, eh)
                assert a[1] == b[1] or (np.isnan(a[1]) and np.isnan(b[1]))
                out += [np.asarray(a[0]), np.asarray([a[1]])]
        tr.close()
        got.append(out)
    return got


def same(lay, z, p, tgt):
    a, b = both(lay, z, p, tgt)
    for x, y in zip(a, b):
        assert x.dtype == y.dtype and x.tobytes() == y.tobytes()


@pytest.mark.parametrize("name", sorted(n for n in LAYOUTS if not n.endswith("_valu")))
def test_decode_same_bits(name):
    lay = LAYOUTS[name]
    z, p, tgt = data(lay, 31)
    say("decode", name)
    same(lay, z, p, tgt)


@pytest.mark.parametrize("W,H", [(1, 1), (15, 1), (16, 1), (17, 1), (63, 1), (64, 1), (65, 1), (255, 1), (257, 3), (640, 480)])
@pytest.mark.parametrize("levels,hidden,T,leak", [([(4, 8, False)], [16, 16], 1, 0.0), ([(1, 2, True), (4, 4, False)], [32, 32], 4, 0.01),
                                                  ([(2, 4, False), (8, 8, False)], [64, 64], 4, 0.0)])
def test_decode_sizes(W, H, levels, hidden, T, leak):
    lay = Layout(W, H, [(-(-W // d), -(-H // d), c, near) for d, c, near in levels], hidden, T=T, leak=leak)
    z, p, tgt = data(lay, 32)
    say("decode", W, H, hidden)
    same(lay, z, p, tgt)


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf, 3e38])
def test_decode_values(value):
    """a weight of the second hidden layer and, in another model, a latent that is not finite or overflows"""
    lay = LAYOUTS["material"]
    z, p, tgt = data(lay, 33)
    q = p.copy()
    q[lay.nin * lay.hidden[0] + lay.hidden[0] + 3] = value
    say("decode value", value)
    # the sign of a NaN is the operation's own affair: values, and NaN in the same places
    for zz, pp in ((z, q), (np.where(np.arange(z.size) == 5, np.float32(value), z).astype(np.float32), p)):
        a, b = both(lay, zz, pp, tgt)
        for x, y in zip(a, b):
            assert np.array_equal(x, y, equal_nan=x.dtype.kind == "f")


@pytest.mark.parametrize("leak,clamp", [(1.5, False), (-0.25, True)])
def test_decode_leak(leak, clamp):
    lay = Layout(70, 9, [(18, 3, 4, False)], [24, 24], T=2, leak=leak, clamp_out=clamp)
    z, p, tgt = data(lay, 34)
    same(lay, z, p, tgt)


@pytest.mark.parametrize("hidden,T", [([32], 1), ([64], 4), ([24] * 3, 1), ([32] * 4, 4), ([64] * 3, 1), ([64] * 4, 4)])
def test_decode_layers(hidden, T):
    """one, three and four hidden layers: kernels of fewer waves, and (the last two) models whose layers do not fit the registers,
    which the VALU decode takes"""
    lay = Layout(131, 37, [(33, 10, 4, False), (9, 3, 4, False)], hidden, T=T, leak=0.01)
    z, p, tgt = data(lay, 35)
    say("decode layers", hidden, T)
    same(lay, z, p, tgt)


@pytest.mark.parametrize("W,H", [(512, 511), (512, 513), (1030, 520)])
def test_decode_floats_on_a_full_chip(W, H):
    """at most 4 outputs as floats: images below a full chip, on one and on two (the matrix cores on the first and last)"""
    lay = Layout(W, H, [(-(-W // 4), -(-H // 4), 8, False), (-(-W // 16), -(-H // 16), 4, False)], [32, 32], leak=0.0)
    z, p, tgt = data(lay, 36)
    say("decode floats", W, H)
    same(lay, z, p, tgt)
