"""INT4_RESIDUAL pages of the quantiser (csrc/quantize.hip): the packed arithmetic of
finite pages against the oracle bit for bit, over scales from the smallest float16
subnormal to the largest finite value and values at the codes' ties, and the plain form
of the pages it leaves over (infinities, NaN, a scale that underflows to zero)."""
import numpy as np
import pytest

from oracle import quant as Q

pytestmark = pytest.mark.gpu


def _quantize(x):
    import torch
    from intent_attention import quantize_pages
    codes, scales = quantize_pages(torch.from_numpy(x).cuda(), "INT4_RESIDUAL")
    return codes.cpu().numpy(), scales.cpu().numpy()


def _check(x, codes, scales):
    for p in range(x.shape[0]):
        (q1, q2), (s1, s2) = Q.quantize_page(x[p], "INT4_RESIDUAL")
        assert np.array_equal(codes[p], Q.pack_int4_residual(q1, q2)), p
        assert scales[p, 0] == np.float32(s1[0]) and scales[p, 1] == s2[0], p


@pytest.mark.parametrize("D", [64, 128])
def test_scales_and_ties(D):
    rng = np.random.default_rng(D)
    mags = np.concatenate([2.0 ** np.arange(-24, 16), [65504.0, 127.0, 63.5, 6e-6, 7.6e-6]])
    x = (rng.uniform(-1, 1, (2 * len(mags) + 1, 16, D)) * np.tile(mags, 3)[:2 * len(mags) + 1, None, None]).astype(np.float16)
    x[::3, 0, 0] = np.repeat(mags, 3)[:len(x[::3])].astype(np.float16)
    # scale 1 (absmax 127): every base tie k + 1/2, and their float16 neighbours
    t = np.resize(np.concatenate([np.arange(-8, 8) + 0.5, np.arange(-8, 9)]), 16 * D).astype(np.float16)
    near = np.nextafter(t, np.float16(200) * np.resize([1, -1], t.size).astype(np.float16))
    ties = np.stack([t, near]).reshape(2, 16, D)
    ties[:, 15, D - 1] = 127
    x = np.concatenate([x, ties])
    _check(x, *_quantize(x))


@pytest.mark.parametrize("D", [64, 128])
def test_pages_left_to_the_plain_form(D):
    rng = np.random.default_rng(D + 1)
    x = rng.standard_normal((7, 16, D)).astype(np.float16)
    x[1, 3, 5] = x[1, 15, D - 1] = np.nan          # drops out of the maxima, code 0
    x[2, 0, 0] = np.inf                            # scale inf: every code 0
    x[3, 15, D - 1] = -np.inf
    x[4] = 0
    x[5] = (rng.integers(-40, 41, (16, D)) * 2.0 ** -24).astype(np.float16)   # scale underflows to zero
    codes, scales = _quantize(x)
    zeroed = np.where(np.isnan(x), np.float16(0), x)
    keep = [0, 1, 4, 5, 6]
    _check(zeroed[keep], codes[keep], scales[keep])
    for p in (2, 3):
        assert (codes[p] == 0x88).all() and np.isinf(scales[p, 0]) and scales[p, 1] == np.float32(1e-8)
