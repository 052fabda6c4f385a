"""Fused chirp-z row and column passes at the edges of their convolution
lengths (n = 2^k + 1, where M doubles, and n = 2^k - 1), with one axis a power
of two, rows and tiles that don't fill a block, and batches whose blocks run
several rows and tiles, against the oracle in 64 bits.  The bound is the one the
other sizes have (1e-5: each line transform is two float32 FFTs, about 3e-7, and
there are up to twelve per image here)."""
import numpy as np
import pytest
import torch

import emsim_amd
from emsim_amd.backend.slice_builder_hip import MultiSlicesBuilder
from oracle import emsim_oracle as orc

pytestmark = pytest.mark.gpu
TOL = 1e-5
LAM, GAMMA = orc.wavelength_and_gamma(200.0)


def _inputs(shape, seed):
    rng = np.random.default_rng(seed)
    w = (1.0 + 0.3 * rng.standard_normal(shape) + 0.3j * rng.standard_normal(shape))
    return w.astype(np.complex64), rng


@pytest.mark.parametrize("n1,n2,batch", [(9, 9, 1), (15, 17, 3), (33, 65, 2), (129, 8, 1),
                                         (64, 127, 5), (257, 100, 2), (511, 512, 1),
                                         (1025, 16, 1), (9, 1023, 2), (2047, 24, 1)])
def test_multislice_and_lens(hip, n1, n2, batch):
    prop = emsim_amd.wave.get_raw_wave_propagator((n1, n2), 1.0, 200)
    w, rng = _inputs((batch, n1, n2), n1 + n2)
    shared = rng.uniform(0, 20, (2, n1, n2)).astype(np.float32)
    own = rng.uniform(0, 20, (batch, 2, n1, n2)).astype(np.float32)
    for v, per_image in ((shared, False), (own, True)):
        got = prop.multislice_propagate(w, v, 2.0)
        img = prop.lens_intensity(got, 1.3, 700.0, 10e-3).cpu().numpy()
        got = got.cpu().numpy()
        for b in range(batch):
            vb = v[b] if per_image else v
            ref = orc.multislice_f64(w[b].astype(np.complex128), vb.astype(np.float64), 2.0, LAM,
                                     GAMMA, 1.0, 1.0)
            ref_i = np.abs(orc.lens_propagate_f64(ref, LAM, 1.3, 700.0, 10e-3, 1.0, 1.0)) ** 2
            e, ei = orc.rel_l2(got[b], ref), orc.rel_l2(img[b], ref_i)
            assert e < TOL and ei < TOL, (b, e, ei)


@pytest.mark.parametrize("n,batch", [(33, 300), (75, 200), (150, 40)])
def test_batch_equals_single(hip, n, batch):
    """Blocks that run several rows and column tiles, and narrow against wide
    tiles (one image takes the narrow ones): the same bits."""
    prop = emsim_amd.wave.get_raw_wave_propagator((n, n), 1.0, 200)
    w, rng = _inputs((3, n, n), n)
    v = rng.uniform(0, 20, (2, n, n)).astype(np.float32)
    many = prop.multislice_propagate(np.tile(w, (batch // 3 + 1, 1, 1))[:batch], v, 2.0)
    for b in (0, 1, 2, batch - 1):
        one = prop.multislice_propagate(w[b % 3], v, 2.0)
        assert torch.equal(one, many[b])


@pytest.mark.parametrize("n,slices,elems", [(9, 1, [6]), (33, 3, [1, 8]), (75, 40, [1, 6, 7, 8]),
                                            (100, 2, [1, 6, 7, 8, 16, 79])])
def test_slices(hip, n, slices, elems):
    builder = MultiSlicesBuilder(elems, slices, n, n, 2.0, 1.0, 1.0)
    rng = np.random.default_rng(n)
    hist = rng.poisson(0.05, (len(elems), slices, n, n)).astype(np.float32)
    sf = orc.scattering_factors_half(elems, n, n, 1.0, 1.0)
    for limit in (True, False):
        got = builder.make_multi_slices(hist, limit).cpu().numpy()
        ref = orc.make_multi_slices_f64(hist, sf, limit)
        assert orc.rel_l2(got, ref) < TOL


@pytest.mark.parametrize("n1,n2,slices", [(75, 75, 6), (33, 64, 5), (9, 100, 7)])
def test_slices_do_not_mix(hip, n1, n2, slices):
    """Each slice of a grid of odd n1 comes from its own counts alone: the same
    bits with one slice or several to a launch, and with infinite counts in the
    slice before it."""
    elems = [1, 6]
    rng = np.random.default_rng(n1)
    hist = rng.poisson(0.2, (len(elems), slices, n1, n2)).astype(np.float32)
    limit = n1 == n2
    builder = MultiSlicesBuilder(elems, slices, n1, n2, 2.0, 1.0, 1.0)
    one = MultiSlicesBuilder(elems, 1, n1, n2, 2.0, 1.0, 1.0)
    got = builder.make_multi_slices(hist, limit)
    for s in range(slices):
        alone = one.make_multi_slices(np.ascontiguousarray(hist[:, s:s + 1]), limit)
        assert torch.equal(alone[0], got[s]), s
    hist[1, 2, n1 // 2, 3] = np.inf
    again = builder.make_multi_slices(hist, limit)
    for s in range(slices):
        assert s == 2 or torch.equal(again[s], got[s]), s
