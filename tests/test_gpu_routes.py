"""The batched path picks its kernels by the batch's size: slices per launch of
the spectrum pass (up to a bound of plane memory) and pass A in one kernel or
two (up to a bound of pixels).  Every choice runs the same operations on the
same values, so a molecule's result is the same bits in any batch."""
from ctypes import POINTER, c_int64, c_uint64

import numpy as np
import pytest
import torch

import emsim_amd
from emsim_amd import synth
from emsim_amd.backend import hip_ext
from emsim_amd.backend._device import ptr, stream_handle
from emsim_amd.backend.slice_builder_hip import MultiSlicesBuilder
from emsim_amd.backend.wave_propagator_hip import WavePropagator
from emsim_amd.batch import BatchPipe
from oracle import emsim_oracle as orc
from tests._chain import pipe_oracle

pytestmark = pytest.mark.gpu
ELEMS = [1, 6, 7, 8, 16]
SPLIT_PIXELS = 2 * 512 * 512   # the library's bound for pass A in two kernels


def _tem():
    return emsim_amd.tem.TEM(electron_dose=20, beam_energy_kev=200, cs_mm=1.3, defocus=700,
                             aperture=10e-3)


# (n, molecules beyond the bound, slices): one slice, fewer and more slices than
# a launch takes (8 for the largest batch here, 19 at 128^2, all 40 alone)
@pytest.mark.parametrize("n,over,slices", [(128, 1, 1), (128, 1, 40), (256, 1, 9),
                                           (512, 1, 21), (64, 1, 3), (8, 1, 2)])
def test_image_does_not_depend_on_the_batch(hip, n, over, slices):
    batch = SPLIT_PIXELS // (n * n) + over
    base = [synth.protein_cloud(400 + 150 * k, 40 + k) for k in range(4)]
    pipe = BatchPipe(_tem(), 1.0, 2.0, n, slices, ELEMS)
    prepared = [pipe.prepare(m) for m in base]
    together = pipe.upload([prepared[k % 4] for k in range(batch)])
    images = pipe.run(together)
    waves, v = pipe.exit_waves_and_slices(together)
    for k in range(4 if batch >= 4 else batch):
        alone = pipe.upload([prepared[k]])
        assert torch.equal(pipe.run(alone)[0], images[k])
        w1, v1 = pipe.exit_waves_and_slices(alone)
        assert torch.equal(w1[0], waves[k]) and torch.equal(v1[0], v[k])
    assert torch.equal(images[batch - 1], images[(batch - 1) % 4])


def test_rectangular_grid_does_not_depend_on_the_batch(hip):
    """n1 != n2 (no band-limit disk), through the C ABI: rows and columns of
    different length on both routes."""
    n1, n2, slices = 128, 256, 5
    builder = MultiSlicesBuilder(ELEMS, slices, n1, n2, 2.0, 1.0, 1.0).backend
    prop = WavePropagator(n1, n2, 1.0, 1.0, 200.0).backend
    square = BatchPipe(_tem(), 1.0, 2.0, 128, slices, ELEMS)
    prepared = [square.prepare(synth.protein_cloud(500 + 100 * k, 60 + k)) for k in range(3)]

    def run(batch):
        out = torch.empty((len(batch), n1, n2), device="cuda")
        n_atoms = batch.coords.shape[0]
        need = hip_ext.raw("emsim_hip_simulate_workspace_size")(builder.h, len(batch), n_atoms, 0)
        ws = torch.empty(need, dtype=torch.uint8, device="cuda")
        args = (builder.h, prop.h, ptr(batch.coords), n_atoms,
                batch.mol_off.ctypes.data_as(POINTER(c_int64)),
                batch.counts.ctypes.data_as(POINTER(c_int64)), len(batch), 4.5, 1.3, 700.0, 10e-3,
                0, ptr(out), None, 0, ptr(ws))
        # one byte less than the size function asks for is refused
        rc = hip_ext.raw("emsim_hip_simulate")(*args, need - 1, stream_handle())
        assert rc == hip_ext.EWORKSPACE
        hip_ext.call("emsim_hip_simulate", *args, need, stream_handle())
        return out

    count = SPLIT_PIXELS // (n1 * n2) + 1
    many = run(square.upload([prepared[k % 3] for k in range(count)]))
    for k in range(3):
        assert torch.equal(run(square.upload([prepared[k]]))[0], many[k])
    assert np.isfinite(many.cpu().numpy()).all()


# (n1, n2, waves): the column pass takes quarter, half or full tiles by the
# number of full tiles (bounds 48 and 128; 512 rows: half up to 48).  n2 = 8 is
# narrower than a tile; the waves put the batch on one side of a bound and the
# waves alone on the other.
@pytest.mark.parametrize("n1,n2,waves", [(128, 8, 49), (128, 8, 129), (128, 512, 9),
                                         (256, 256, 3), (256, 256, 8), (256, 16, 49),
                                         (256, 256, 9), (512, 512, 2), (512, 8, 49),
                                         (512, 64, 7)])
def test_wave_does_not_depend_on_the_batch(hip, n1, n2, waves):
    prop = WavePropagator(n1, n2, 1.0, 1.0, 200.0)
    gen = torch.Generator(device="cuda").manual_seed(n1 + n2 + waves)
    v = 40 * torch.rand((waves, 3, n1, n2), generator=gen, device="cuda")
    psi0 = prop.init_wave(20.0, batch=waves)
    psi = prop.multislice_propagate(psi0, v, 2.0)
    image = prop.lens_intensity(psi, 1.3, 700.0, 10e-3)
    for k in {0, waves // 2, waves - 1}:
        alone = prop.multislice_propagate(psi0[k], v[k], 2.0)
        assert torch.equal(alone, psi[k])
        assert torch.equal(prop.lens_intensity(alone, 1.3, 700.0, 10e-3), image[k])


# Columns that the propagator zeroes whole are left out between the slices: none
# at n2 = 8 within a tile, part of a tile, many tiles; a potential of NaN in one
# wave must not reach another, and a given output holds nothing of before.
@pytest.mark.parametrize("n1,n2,d2", [(64, 8, 1.0), (128, 64, 1.0), (64, 128, 2.0),
                                      (256, 512, 0.5), (8, 1024, 1.0)])
def test_multislice_equals_slice_by_slice(hip, n1, n2, d2):
    prop = WavePropagator(n1, n2, 1.0, d2, 200.0)
    gen = torch.Generator(device="cuda").manual_seed(n1 + n2)
    v = 40 * torch.rand((2, 4, n1, n2), generator=gen, device="cuda")
    psi = prop.init_wave(20.0, batch=2)
    many = prop.multislice_propagate(psi, v, 2.0)
    one = psi
    for s in range(4):
        one = prop.space_propagate(prop.slice_transmit(one, v[:, s].contiguous()), 2.0)
    # float32 transforms: one rounding per pass and slice, log2(n1 n2) passes
    tol = 4 * np.log2(n1 * n2) * 2.0 ** -24 * 4
    assert float((many - one).norm() / one.norm()) < tol
    v[1, 1, 3, 3] = float("nan")
    again = prop.multislice_propagate(psi, v, 2.0)
    assert torch.equal(again[0], many[0]) and not torch.isfinite(again[1]).any()


# The spectrum pass leaves out the eighths of the rows beyond the middle quarter
# or half if an element has no atoms there: atoms up to just inside and just
# beyond those borders, all columns and both transform kinds (leading radix 8 at
# 64 and 512 rows, 4 at 256, 2 at 128).  The bound is the other sizes' (1e-5).
@pytest.mark.parametrize("n", [64, 128, 256, 512])
@pytest.mark.parametrize("eighths,out", [(1, -0.6), (1, 0.6), (2, -0.6), (2, 0.6), (4, -1.6)])
def test_rows_in_the_middle_of_the_box(hip, n, eighths, out):
    half = n * eighths / 8 + out
    rng = np.random.default_rng(n + eighths)
    count = 60
    xyz = np.stack([rng.uniform(-3.5, 3.5, count), rng.uniform(-half, half, count),
                    rng.uniform(-n / 2 + 2, n / 2 - 2, count)], 1).astype(np.float32)
    xyz[0, 1], xyz[1, 1] = -half, half          # one element spans the range,
    xyz[2::3, 1] *= 0.1                         # another stays in the middle
    zs = np.where(np.arange(count) % 3 == 2, 8, 6)
    mol = emsim_amd.atoms.AtomList(zs, xyz)
    pipe = BatchPipe(_tem(), 1.0, 2.0, n, 4, [6, 8])
    image = pipe.run(pipe.upload([pipe.prepare(mol)]))[0].cpu().numpy()
    _, exact, _, _ = pipe_oracle(mol, _tem(), 2.0, 2.0, (n, n))
    assert orc.rel_l2(image, exact) < 1e-5


# The water path: hydrogen and oxygen rows from one transform, the others from
# their buckets.  Rows shorter than a wave and longer than one, more elements than
# threads per row, both routes of pass A, several launches of the spectrum pass, the
# packed column of 2048 rows, rectangles.  Potentials against the dense ones of
# the same counts (the bound is the other sizes', 1e-5).
@pytest.mark.parametrize("n1,n2,slices,elems,count", [
    (8, 8, 3, [1, 6, 8], 2), (16, 64, 2, [1, 8], 3), (64, 16, 9, [1, 6, 7, 8, 16], 2),
    (128, 128, 5, [1, 6, 7, 8, 16], 40), (256, 256, 21, [1, 6, 7, 8, 16], 9),
    (1024, 32, 2, [1, 6, 8], 1), (512, 1024, 1, [1, 8], 1), (2048, 64, 2, [1, 6, 8], 2)])
def test_water_potentials_equal_dense_ones(hip, n1, n2, slices, elems, count):
    dz, d1, d2 = 2.0, 1.0, 1.0
    builder = MultiSlicesBuilder(elems, slices, n1, n2, dz, d1, d2)
    prop = WavePropagator(n1, n2, d1, d2, 200.0).backend
    rng = np.random.default_rng(n1 + n2)
    counts = rng.integers(0, 60, (count, len(elems))).astype(np.int64)
    off = np.concatenate([[0], np.cumsum(counts.sum(axis=1))]).astype(np.int64)
    n_atoms = int(off[-1])
    half = np.array([slices * dz, n1 * d1, n2 * d2]) / 2
    coords = torch.from_numpy(rng.uniform(-half, half, (n_atoms, 3)).astype(np.float32)).cuda()
    seeds = rng.integers(0, 2 ** 62, count).astype(np.uint64)
    band = 1 if n1 == n2 else 0
    image = torch.empty((count, n1, n2), device="cuda")
    v = torch.full((count, slices, n1, n2), -1.0, device="cuda")
    need = hip_ext.raw("emsim_hip_simulate_water_workspace_size")(builder.backend.h, count,
                                                                   n_atoms, 0)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    args = (builder.backend.h, prop.h, ptr(coords), n_atoms, off.ctypes.data_as(POINTER(c_int64)),
            np.ascontiguousarray(counts).ctypes.data_as(POINTER(c_int64)), count, 4.5, 1.3, 700.0,
            10e-3, band, elems.index(1), elems.index(8),
            emsim_amd.physics.water_num_dens * d1 * d2 * dz,
            seeds.ctypes.data_as(POINTER(c_uint64)), ptr(image), ptr(v), 0, ptr(ws))
    rc = hip_ext.raw("emsim_hip_simulate_water")(*args, need - 1, stream_handle())
    assert rc == hip_ext.EWORKSPACE
    hip_ext.call("emsim_hip_simulate_water", *args, need, stream_handle())
    for b in range(count):
        hist = builder.backend.bin_atoms(coords[off[b]:off[b + 1]], counts[b])
        hist = builder.add_water(hist, seed=int(seeds[b]))
        ref = builder.backend.make_slices(hist, bool(band))
        assert float((v[b] - ref).norm() / ref.norm()) < 1e-5, b
    assert torch.isfinite(image).all()


# Row sums run over the atoms in a fixed order: the bits don't depend on the
# order the atoms come in.  Rows sorted by a thread and by a wave (on both sides
# of sqrt(8 n) atoms), ranges up to the sorting kernel's LDS (16384 atoms) and
# beyond; boxes of 8 to 2048 bins.
@pytest.mark.parametrize("n,per_row", [(64, [3] * 40), (64, [22, 23, 700] * 9), (8, [8, 9, 90, 2]),
                                       (64, [9000, 1, 0, 7000, 380, 2, 1]), (64, [17000, 3, 1, 30]),
                                       (512, [64, 24, 65, 0, 63] * 9), (2048, [300, 129, 26])])
def test_image_does_not_depend_on_the_atoms_order(hip, n, per_row):
    rng = np.random.default_rng(sum(per_row))
    x = np.concatenate([np.full(c, k - len(per_row) // 2 + 0.5) for k, c in enumerate(per_row)])
    xyz = np.stack([np.zeros_like(x), x, rng.uniform(-0.47 * n, 0.47 * n, len(x))],
                   1).astype(np.float32)
    zs = np.full(len(x), 6)
    pipe = BatchPipe(_tem(), 1.0, 2.0, n, 2, [6, 8])
    images = []
    for order in (np.arange(len(x)), rng.permutation(len(x))):
        mol = emsim_amd.atoms.AtomList(zs[order], xyz[order])
        images.append(pipe.run(pipe.upload([pipe.prepare(mol)]))[0])
    assert torch.isfinite(images[0]).all() and torch.equal(images[0], images[1])


# Rows of 1024 points and more are transformed by several waves, and a block runs
# several rows: a row's last LDS reads come before the next row's writes.  The
# same inputs give the same bits, and the image is the squared wave.
@pytest.mark.parametrize("n1,n2,batch", [(512, 1024, 8), (2048, 2048, 1), (4096, 4096, 1),
                                         (64, 4096, 40)])
def test_long_rows_are_reproducible(hip, n1, n2, batch):
    prop = WavePropagator(n1, n2, 1.0, 1.0, 200.0)
    gen = torch.Generator(device="cuda").manual_seed(n1 + n2)
    psi = torch.view_as_complex(torch.randn((batch, n1, n2, 2), generator=gen, device="cuda"))
    wave = prop.lens_propagate(psi, 1.3, 700.0, 10e-3)
    image = prop.lens_intensity(psi, 1.3, 700.0, 10e-3)
    for _ in range(4):
        assert torch.equal(prop.lens_propagate(psi, 1.3, 700.0, 10e-3), wave)
        assert torch.equal(prop.lens_intensity(psi, 1.3, 700.0, 10e-3), image)
    # float32 against float32 of the same wave: a few roundings of the square
    square = wave.abs().double() ** 2
    assert float((image.double() - square).norm() / square.norm()) < 1e-6


def _workspace_bytes(n, slices, batch, water):
    builder = MultiSlicesBuilder(ELEMS, slices, n, n, 2.0, 1.0, 1.0).backend
    name = f"emsim_hip_simulate{'_water' if water else ''}_workspace_size"
    return hip_ext.raw(name)(builder.h, batch, 1000, 0)


# Planes of several slices are workspace that a batch of one slice at a time does
# not need: 2 GiB of them at most, and none beyond the first slice where that one
# is larger.  (The atoms' row table: 2 x 4 bytes a row, 4 per molecule, and a sum of 4
# bytes per tile of its scan, 2048 rows.)
@pytest.mark.parametrize("n,batch", [(256, 64), (512, 64), (2048, 16), (2048, 64), (4096, 1),
                                     (4096, 100)])
@pytest.mark.parametrize("water", [False, True])
def test_workspace_of_several_slices_is_bounded(hip, n, batch, water):
    slices = 16
    rows = (slices - 1) * batch * len(ELEMS) * n
    tables = 8 * rows + 4 * (rows // 2048) + 4 * (slices - 1) * batch + 4096
    one = _workspace_bytes(n, 1, batch, water)
    more = _workspace_bytes(n, slices, batch, water) - one - tables
    plane = batch * n * (n // 2 + 1) * 8 * (3 if water else 1)
    assert more <= (2 << 30) - plane or (plane > 1 << 30 and more <= 0)


def test_image_does_not_depend_on_the_bounded_planes(hip):
    """16 images of 2048^2: seven slices to a launch by that bound, eleven alone."""
    pipe = BatchPipe(_tem(), 1.0, 2.0, 2048, 9, ELEMS)
    prepared = [pipe.prepare(synth.protein_cloud(2000 + 300 * k, 70 + k)) for k in range(2)]
    images = pipe.run(pipe.upload([prepared[k % 2] for k in range(16)]))
    for k in range(2):
        assert torch.equal(pipe.run(pipe.upload([prepared[k]]))[0], images[k])


# 512 to 2048 rows: where two slices' planes fit the cache behind the L2s (192 MiB
# of them), a launch takes no more than fit it.
@pytest.mark.parametrize("n,batch", [(512, 16), (512, 64), (1024, 16), (2048, 2), (2048, 4)])
def test_planes_that_fit_the_cache_stay_in_it(hip, n, batch):
    slices = 16
    rows = (slices - 1) * batch * len(ELEMS) * n
    tables = 8 * rows + 4 * (rows // 2048) + 4 * (slices - 1) * batch + 4096
    more = _workspace_bytes(n, slices, batch, False) - _workspace_bytes(n, 1, batch, False)
    assert more - tables <= (192 << 20) - batch * n * (n // 2 + 1) * 8
