"""The work that programs using this package have it do, as timed cases.

Each case is one call, or one short sequence of calls, through the public entry
points, at the sizes of this repository's own configurations, tests and
benchmark: single images from host molecules (``Pipe``), batches of prepared
molecules (``BatchPipe``), molecules of mixed wave sizes (``MixedBatch``),
propagation through given potentials (the wave propagator), the learned
coarse-slice pipeline (``LearnedPipe``) and the gradients of a training step
(``FNO``).  ``exact`` computes the same results in 64 bits from the inputs
alone, with plain torch and numpy.
"""
import math
from pathlib import Path

import numpy as np
import torch

from emsim_amd import atoms, tem, wave
from emsim_amd.backend import hip_ext
from emsim_amd.backend._device import ptr, stream_handle
from emsim_amd.batch import BatchPipe, MixedBatch
from emsim_amd.learned import FNO, CoarseFinePairs, LearnedPipe
from emsim_amd.pipe import Pipe

DATA = Path(__file__).resolve().parent.parent / "emsim_amd" / "data"
NETWORK = DATA / "fno_512.npz"

# the protein mix of the synthetic specimens: H, C, N, O, S
ELEMENTS = (1, 6, 7, 8, 16)
FRACTIONS = (0.49, 0.32, 0.09, 0.095, 0.005)
# the microscope of the benchmark, the tests and the training
DOSE, ENERGY, CS_MM, DEFOCUS, APERTURE = 20.0, 200.0, 1.3, 700.0, 10e-3
# the network's coarse slices (fno_512.npz: 4 x 25 A for a 100 A box)
COARSE_DZ, COARSE_SLICES = 25.0, 4


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the first thing anyone runs: five atoms in a row, weak-phase-object
        # image of 512^2 pixels; all launch latency
        {"name": "five_atoms_wpo", "kind": "wpo", "n": 512, "atoms": 5, "pixel": 1.0},
        # a small molecule from host atoms to an image, one at a time
        {"name": "pipe_128", "kind": "pipe", "n": 128, "atoms": 5000, "pixel": 1.0, "dz": 2.0},
        # the same at a lateral size that is not a power of two
        {"name": "pipe_150", "kind": "pipe", "n": 150, "atoms": 10000, "pixel": 1.0, "dz": 2.0},
        # one image of a 50k-atom cloud, 45 slices: latency of the batched path
        {"name": "single_256", "kind": "batch", "n": 256, "atoms": 50000, "batch": 1,
         "slices": 45, "dz": 2.0, "pixel": 1.0},
        # the same cloud size, 64 molecules at once
        {"name": "batch_256", "kind": "batch", "n": 256, "atoms": 50000, "batch": 64,
         "slices": 45, "dz": 2.0, "pixel": 1.0},
        # the benchmark: 64 molecules of uneven size, 512^2, 100 slices of 1 A
        {"name": "batch_512", "kind": "batch", "n": 512, "atoms": 40000, "batch": 64,
         "slices": 100, "dz": 1.0, "pixel": 1.0},
        # a 20 A cut of the large water slab: 2048^2 pixels of 0.5 A, dense slices
        {"name": "slab_2048", "kind": "slab", "n": 2048, "slices": 20, "dz": 1.0, "pixel": 0.5},
        # the reference's default image: every empty voxel filled with water
        {"name": "water_256", "kind": "water", "n": 256, "atoms": 30000, "batch": 16,
         "slices": 40, "dz": 2.0, "pixel": 1.0},
        # molecules of mixed size as they come from the host, three wave sizes
        {"name": "mixed_24", "kind": "mixed", "atoms": 30000, "batch": 24, "dz": 2.0,
         "pixel": 1.0},
        # propagation and lens through potentials the program already has
        {"name": "propagate_512", "kind": "propagate", "n1": 512, "n2": 512, "batch": 16,
         "slices": 50, "dz": 1.0, "pixel": 1.0},
        # the learned pipeline: 4 coarse slices, the network, its checks
        {"name": "learned_512", "kind": "learned", "atoms": 40000, "batch": 64},
        # forward, loss and backward of one training step of that network
        {"name": "train_512", "kind": "train", "n": 512, "atoms": 30000, "batch": 8},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["wpo", "pipe", "pipe", "batch", "batch", "batch", "slab", "water",
                       "mixed", "propagate", "propagate", "learned", "train"])
    if kind == "wpo":
        return {"kind": kind, "n": rng.choice([128, 256, 512, 300, 511]),
                "atoms": _log_int(rng, 5, 20000), "pixel": rng.choice([0.5, 1.0])}
    if kind == "pipe":
        n = rng.choice([64, 128, 256, 512, rng.randint(75, 511), rng.randint(75, 300)])
        return {"kind": kind, "n": n, "atoms": _log_int(rng, 500, 50000),
                "pixel": rng.choice([0.5, 1.0]), "dz": rng.choice([1.0, 2.0, 4.0])}
    if kind == "batch":
        n = rng.choice([128, 256, 512])
        return {"kind": kind, "n": n, "atoms": _log_int(rng, 5000, 60000),
                "batch": _log_int(rng, 1, 64), "slices": rng.randint(10, 90),
                "dz": rng.choice([1.0, 2.0]), "pixel": 1.0}
    if kind == "slab":
        return {"kind": kind, "n": rng.choice([1024, 2048]), "slices": rng.randint(3, 20),
                "dz": rng.choice([1.0, 2.0]), "pixel": 0.5}
    if kind == "water":
        n = rng.choice([128, 256, 512])
        return {"kind": kind, "n": n, "atoms": _log_int(rng, 3000, 60000),
                "batch": _log_int(rng, 1, 16 if n < 512 else 8), "slices": rng.randint(10, 45),
                "dz": 2.0, "pixel": 1.0}
    if kind == "mixed":
        return {"kind": kind, "atoms": _log_int(rng, 8000, 40000), "batch": rng.randint(3, 40),
                "dz": rng.choice([2.0, 4.0]), "pixel": 1.0}
    if kind == "propagate":
        sides = rng.choice([(128, 128), (256, 256), (512, 512), (1024, 1024), (256, 512),
                            (300, 256), (96, 200), (rng.randint(75, 511),) * 2])
        cap = 16 * 512 * 512 // (sides[0] * sides[1])
        return {"kind": kind, "n1": sides[0], "n2": sides[1],
                "batch": _log_int(rng, 1, max(1, min(32, cap))), "slices": rng.randint(4, 50),
                "dz": rng.choice([1.0, 2.0, 4.0]), "pixel": rng.choice([0.5, 1.0])}
    if kind == "learned":
        return {"kind": kind, "atoms": _log_int(rng, 10000, 60000),
                "batch": _log_int(rng, 2, 64)}
    return {"kind": kind, "n": rng.choice([256, 512]), "atoms": _log_int(rng, 8000, 40000),
            "batch": rng.randint(1, 8)}


# ---------------------------------------------------------------------------
# specimens
# ---------------------------------------------------------------------------
def _cloud(rng, count):
    """A protein-like cloud: a sphere of the specimens' density (90 A across at
    50k atoms) of atoms at least 1 A apart (a jittered lattice), turned at
    random, elements in the protein mix and in random order."""
    step = (math.pi / 6 * 90.0 ** 3 / 50000.0) ** (1.0 / 3.0)
    radius = 45.0 * (count / 50000.0) ** (1.0 / 3.0)
    half = int(math.ceil(radius / step)) + 2
    axis = np.arange(-half, half + 1, dtype=np.float64)
    pts = np.stack(np.meshgrid(axis, axis, axis, indexing="ij"), -1).reshape(-1, 3)
    pts = (pts + rng.uniform(-0.5, 0.5, 3)) * step
    near = np.argpartition(np.einsum("ij,ij->i", pts, pts), count)[:count]
    pts = pts[near] + rng.uniform(-0.48, 0.48, (count, 3))
    turn, _ = np.linalg.qr(rng.standard_normal((3, 3)))
    zs = np.repeat(np.asarray(ELEMENTS), rng.multinomial(count, FRACTIONS))
    return atoms.AtomList(rng.permutation(zs), (pts @ turn).astype(np.float32))


def _five_atoms(rng):
    """C, Si, Cu, Au, U in a row, 10 A apart, a little off the grid."""
    xyz = np.array([[0, 0, 5], [0, 0, 15], [0, 0, 25], [0, 0, 35], [0, 0, 45]], np.float32)
    return atoms.AtomList(np.array([6, 14, 29, 79, 92]),
                          xyz + rng.uniform(-2, 2, (5, 3)).astype(np.float32))


def _water_slab(rng, thickness, side):
    """Amorphous water filling a box, with a cut through one protein cloud."""
    count = int(round(0.0334 * thickness * side * side))
    box = np.array([thickness, side, side])
    oxygen = rng.uniform(-box / 2, box / 2, (count, 3))
    u = rng.standard_normal((count, 3))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    v = np.cross(u, rng.standard_normal((count, 3)))
    v /= np.linalg.norm(v, axis=1, keepdims=True)
    a, b = 0.96 * math.cos(math.radians(52.25)), 0.96 * math.sin(math.radians(52.25))
    xyz = np.concatenate([oxygen, oxygen + a * u + b * v, oxygen + a * u - b * v])
    zs = np.repeat([8, 1, 1], count)
    cloud = _cloud(rng, 50000)
    cut = np.abs(cloud.coordinates[:, 0]) < thickness / 2 - 0.1
    xyz = np.concatenate([xyz.astype(np.float32), cloud.coordinates[cut]])
    order = rng.permutation(len(xyz))
    return atoms.AtomList(np.concatenate([zs, cloud.elements[cut]])[order], xyz[order])


def _sizes(case, rng):
    """Uneven atom counts, log-uniform over a factor of six about case['atoms']."""
    spread = np.exp(rng.uniform(-0.9, 0.9, case["batch"])) if case["batch"] > 1 else np.ones(1)
    return np.maximum(8, (case["atoms"] * spread).astype(int))


def _molecules(case, seed):
    rng = np.random.default_rng(seed)
    if case["kind"] in ("wpo", "pipe"):
        return [_five_atoms(rng) if case["atoms"] <= 5 else _cloud(rng, case["atoms"])]
    if case["kind"] == "slab":
        return [_water_slab(rng, case["slices"] * case["dz"], case["n"] * case["pixel"])]
    return [_cloud(rng, int(k)) for k in _sizes(case, rng)]


def _wave_sizes(case):
    """Every molecule's wave size: the three sizes in turn."""
    return [(256, 512, 128)[i % 3] for i in range(case["batch"])]


def _given_potentials(case, seed):
    """(batch, slices, n1, n2) float32 potentials: Gaussian blobs of about an
    atom's width on random positions, as strong as protein slices are."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    shape = (case["n1"], case["n2"])
    f1 = torch.fft.fftfreq(shape[0], case["pixel"], device="cuda", dtype=torch.float64)
    f2 = torch.fft.rfftfreq(shape[1], case["pixel"], device="cuda", dtype=torch.float64)
    blob = torch.exp(-6.0 * (f1[:, None] ** 2 + f2[None, :] ** 2)) * 60.0
    out = torch.empty((case["batch"], case["slices"]) + shape, device="cuda")
    for b in range(case["batch"]):
        for s in range(0, case["slices"], 8):
            k = min(8, case["slices"] - s)
            hit = torch.rand((k,) + shape, generator=gen, device="cuda") < 0.02
            v = torch.fft.irfft2(torch.fft.rfft2(hit.double()) * blob, s=shape)
            out[b, s:s + k] = v.clamp_(min=0).float()
    return out


def _network_inputs(case, seed):
    """Coarse exit waves, their potentials and the fine exit waves (1 A
    slices) of the case's molecules, computed here in 64 bits."""
    shifted = [_centred(m) for m in _molecules(case, seed)]
    n, grid = case["n"], (case["n"], case["n"], 1.0)
    coarse, v = _exit_waves(shifted, ELEMENTS, grid, COARSE_DZ, COARSE_SLICES, keep=True)
    fine = _exit_waves(shifted, ELEMENTS, grid, 1.0, 100)
    assert coarse.shape[1:] == (n, n)
    return coarse.to(torch.complex64), v.float(), fine.to(torch.complex64)


def _start_weights(case, seed):
    """Weights a training run starts from: uniform +-1/sqrt(fan in), spectral
    weights U(0, 1) / C^2, a small projection."""
    rng = np.random.default_rng(seed + 77)
    c, m, cin = 32, 16, 2 + COARSE_SLICES

    def uni(shape, fan):
        return rng.uniform(-1, 1, shape) / math.sqrt(fan)

    lift = np.zeros((16, c))
    lift[:cin] = uni((cin, c), cin)
    p = {"lift_w": lift, "lift_b": uni((c,), cin), "w": [], "b": [], "r": [],
         "proj_w": 0.1 * uni((c, 2), c), "proj_b": np.zeros(2)}
    for _ in range(4):
        p["w"].append(uni((c, c), c))
        p["b"].append(uni((c,), c))
        r = rng.uniform(0, 1, (2, 2 * m, m, c, c)) / c ** 2
        p["r"].append(r[0] + 1j * r[1])
    return p


# ---------------------------------------------------------------------------
# what a program has in hand, and one pass
# ---------------------------------------------------------------------------
def _tem():
    return tem.TEM(DOSE, ENERGY, CS_MM, DEFOCUS, APERTURE)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("wpo", "pipe"):
        pipe = Pipe(_tem(), 2.0 * case["pixel"], case.get("dz", 1.0), roi=case["n"],
                    add_water=False)
        return {"kind": kind, "pipe": pipe, "mol": _molecules(case, seed)[0]}
    if kind in ("batch", "slab", "water"):
        pipe = BatchPipe(_tem(), case["pixel"], case["dz"], case["n"], case["slices"], ELEMENTS,
                         add_water=kind == "water")
        batch = pipe.upload(pipe.prepare_many(_molecules(case, seed)))
        return {"kind": kind, "pipe": pipe, "batch": batch, "seeds": _seeds(case, seed)}
    if kind == "mixed":
        mixed = MixedBatch(_tem(), case["pixel"], case["dz"], ELEMENTS)
        sizes = _wave_sizes(case)
        return {"kind": kind, "mixed": mixed,
                "items": [(m, int(n)) for m, n in zip(_molecules(case, seed), sizes)]}
    if kind == "propagate":
        prop = wave.get_raw_wave_propagator((case["n1"], case["n2"]), case["pixel"], ENERGY)
        return {"kind": kind, "prop": prop, "slices": _given_potentials(case, seed),
                "dz": case["dz"], "batch": case["batch"]}
    if kind == "learned":
        pairs = CoarseFinePairs(_tem(), coarse_dz=COARSE_DZ, coarse_slices=COARSE_SLICES)
        pipe = LearnedPipe(FNO.load(str(NETWORK)), pairs)
        batch = pairs.fine.upload(pairs.fine.prepare_many(_molecules(case, seed)))
        return {"kind": kind, "pipe": pipe, "batch": batch}
    fno = FNO(case["n"], 2 + COARSE_SLICES)
    fno.set_params(_start_weights(case, seed))
    coarse, v, fine = _network_inputs(case, seed)
    lam, gamma = _beam()
    return {"kind": kind, "fno": fno, "coarse": coarse, "v": v, "fine": fine,
            "psi0": float(np.float32(math.sqrt(DOSE))),
            "sigma": float(np.float32(lam) * np.float32(gamma)),
            "grads": torch.empty(fno.n_params, device="cuda")}


def _seeds(case, seed):
    return [int(s) for s in np.random.default_rng(seed + 5).integers(0, 2 ** 62,
                                                                      case.get("batch", 1))]


def run(state):
    kind = state["kind"]
    if kind == "pipe":
        return state["pipe"].run(state["mol"])
    if kind == "wpo":
        return state["pipe"].run_wpo(state["mol"])
    if kind in ("batch", "slab"):
        return state["pipe"].run(state["batch"])
    if kind == "water":
        return state["pipe"].run(state["batch"], seeds=state["seeds"])
    if kind == "mixed":
        return state["mixed"].run(state["items"])
    if kind == "propagate":
        prop = state["prop"]
        psi = prop.init_wave(DOSE, batch=state["batch"])
        psi = prop.multislice_propagate(psi, state["slices"], state["dz"])
        return prop.lens_intensity(psi, CS_MM, DEFOCUS, APERTURE, overwrite_wave=True)
    if kind == "learned":
        return state["pipe"].run(state["batch"])[0]
    # a training step up to its gradients (the optimiser's update is one
    # elementwise kernel; leaving it out keeps every pass on the same weights)
    fno, psi0 = state["fno"], state["psi0"]
    x = fno.pack(state["coarse"], state["v"], psi0, state["sigma"])
    out = fno.forward(x, training=True)
    psi = fno.apply(state["coarse"], out, psi0)
    loss, dout = fno.loss(psi, state["fine"], psi0, grad=True)
    fno.backward(x, dout)
    hip_ext.call("emsim_hip_fno_get_grads", fno.h, ptr(state["grads"]), stream_handle())
    return {"loss": loss, "wave": psi, "grads": state["grads"]}


def _thickness(case, seed):
    """(slices of each wave size) of a mixed batch: the thickest molecule's."""
    sizes, ns = _wave_sizes(case), {}
    for m, n in zip(_molecules(case, seed), sizes):
        z = _centred(m)[0][:, 0]
        k = int(math.ceil(float(z.max() - z.min()) / case["dz"]))
        ns[int(n)] = max(ns.get(int(n), 1), k)
    return ns


def work(case):
    """Bytes: atoms, given potentials and weights read once, images and
    gradients written once.  Flops: the FFTs of the algorithm -- per slice and
    image one real 2-D transform per element and one back, and two complex
    ones -- or the network's multiply-adds."""
    kind = case["kind"]

    def images(count, n1, n2, slices, built=True):
        pix = n1 * n2
        real = 2.5 * (len(ELEMENTS) + 1) if built else 0.0
        return count * pix * math.log2(pix) * (slices * (real + 10.0) + 10.0)

    def network(count, n):
        pix, c, m = n * n, 32, 16
        layer = pix * (2 * c * c + 8 * m * c) + 16 * m * m * n * c + 16 * m * m * c * c
        return count * (4 * layer + pix * 2 * c * (2 + COARSE_SLICES + 2))

    if kind in ("wpo", "pipe"):
        n, count = case["n"], case["atoms"]
        across = 90.0 * (count / 50000.0) ** (1.0 / 3.0)
        ns = 1 if kind == "wpo" else max(1, math.ceil(across / case["dz"]))
        return {"bytes": 20.0 * count + 4.0 * n * n, "flops": images(1, n, n, ns)}
    if kind in ("batch", "water"):
        n, b = case["n"], case["batch"]
        return {"bytes": b * (12.0 * case["atoms"] + 4.0 * n * n),
                "flops": images(b, n, n, case["slices"])}
    if kind == "slab":
        n = case["n"]
        count = 0.1 * case["slices"] * case["dz"] * (n * case["pixel"]) ** 2
        return {"bytes": 12.0 * count + 4.0 * n * n, "flops": images(1, n, n, case["slices"])}
    if kind == "mixed":
        across = 90.0 * (case["atoms"] / 50000.0) ** (1.0 / 3.0)
        ns = math.ceil(1.3 * across / case["dz"])
        per = case["batch"] / 3.0
        return {"bytes": case["batch"] * (13.0 * case["atoms"] + 4.0 * 114688),
                "flops": sum(images(per, n, n, ns) for n in (128, 256, 512))}
    if kind == "propagate":
        pix = case["batch"] * case["n1"] * case["n2"]
        return {"bytes": pix * 4.0 * (case["slices"] + 1),
                "flops": images(case["batch"], case["n1"], case["n2"], case["slices"], False)}
    if kind == "learned":
        b, n = case["batch"], 512
        return {"bytes": b * (12.0 * case["atoms"] + 4.0 * n * n),
                "flops": images(b, n, n, COARSE_SLICES) + images(1, n, n, 100) + network(b, n)}
    n, b = case["n"], case["batch"]
    weights = 8.0 * 4 * 2 * 16 * 16 * 32 * 32
    return {"bytes": b * n * n * (8.0 + 4.0 * COARSE_SLICES + 8.0 + 8.0) + weights,
            "flops": 3.0 * network(b, n)}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _beam():
    """Wavelength (A) and relativistic gamma of the beam, CGS constants."""
    c, e = 29979245800.0, 1.602176634e-19
    rest = 9.1093835611e-28 * c ** 2 * 1e-7 / e / 1000.0
    return (6.62607015e-27 * c * 0.01 / e / math.sqrt(ENERGY ** 2 + 2 * rest * ENERGY),
            1 + ENERGY / rest)


def _centred(mol):
    """Coordinates with the box centre moved to the origin (in float32, which
    decides the bins) and the atomic numbers."""
    xyz = mol.coordinates
    lo, hi = xyz.min(axis=0), xyz.max(axis=0)
    return xyz + (-lo - (hi - lo) / np.float32(2.0)), np.asarray(mol.elements)


def _bins(x, n, d):
    """numpy.histogram's bin of float32 x on n bins of width d about 0, or -1."""
    start = -d * (n // 2)
    edges = np.arange(start, start + n * d + d, d)
    b = np.searchsorted(edges, x.astype(np.float64), side="right") - 1
    b[x == edges[-1]] = n - 1
    b[(b >= n) | ~(x == x)] = -1
    return b


def _form_factors(elements, n1, n2, d):
    table = np.loadtxt(DATA / "kirkland_params.txt", comments="#")
    q2 = np.fft.fftfreq(n1, d)[:, None] ** 2 + np.fft.rfftfreq(n2, d)[None, :] ** 2
    out = []
    for z in elements:
        p = table[int(z) - 1, 2:].astype(np.float32).astype(np.float64)
        a, b, c, g = p[0:3], p[3:6], p[6:9], p[9:12]
        f = sum(a[i] / (q2 + b[i]) + c[i] * np.exp(-g[i] * q2) for i in range(3))
        out.append(np.where(q2 < 16, f, 0.0))
    return torch.from_numpy(np.stack(out)).cuda()


def _freq(n):
    return np.where(np.arange(n) < (n + 1) // 2, np.arange(n), np.arange(n) - n)


def _masks_and_f2(n1, n2, d):
    """(2/3 band mask, aperture mask, f^2): the masks as float32 arithmetic
    decides them, f^2 in 64 bits."""
    lam = np.float32(_beam()[0])
    d32 = np.float32(d)
    one = np.float32(1.0)
    fx = _freq(n1).astype(np.float32) * (one / d32 / np.float32(n1))
    fy = _freq(n2).astype(np.float32) * (one / d32 / np.float32(n2))
    f32 = (fx * fx)[:, None] + (fy * fy)[None, :]
    band = np.float32(0.6667) * (np.float32(0.5) / d32)
    aper = np.float32(APERTURE) / lam
    f2 = (_freq(n1) / (n1 * d))[:, None] ** 2 + (_freq(n2) / (n2 * d))[None, :] ** 2
    return (torch.from_numpy(f32 <= band * band).cuda(),
            torch.from_numpy(f32 <= aper * aper).cuda(), torch.from_numpy(f2).cuda())


def _splitmix(x):
    """SplitMix64 of int64 tensors holding unsigned 64-bit values."""
    def shr(v, k):
        return (v >> k) & ((1 << (64 - k)) - 1)

    x = x + (0x9E3779B97F4A7C15 - (1 << 64))
    x = (x ^ shr(x, 30)) * (0xBF58476D1CE4E5B9 - (1 << 64))
    x = (x ^ shr(x, 27)) * (0x94D049BB133111EB - (1 << 64))
    return x ^ shr(x, 31)


def _poisson(bits, mean):
    u = ((bits >> 40) & 0xFFFFFF).float() / 16777216.0
    lam, p = np.float32(mean), np.float32(math.exp(-mean))
    cdf, k = p, torch.zeros_like(u, dtype=torch.float64)
    for i in range(1, 65):   # the sampler's inversion stops at 64
        more = u >= float(cdf)
        if not bool(more.any()):
            break
        k += more
        q = np.float32(lam / np.float32(i))
        p = np.float32(p * q)
        cdf = np.float32(cdf + p)
    return k


def _add_water(hist, seeds, s, elements, cell):
    """Poisson water in the voxels empty of every element (slice s), drawn from
    SplitMix64 of each molecule's seed and the voxel's number."""
    b, _, n1, n2 = hist.shape
    vox = torch.arange(n1 * n2, device="cuda", dtype=torch.int64) + s * n1 * n2
    key = _splitmix(torch.tensor(seeds, device="cuda")[:, None] ^ _splitmix(vox)[None, :])
    empty = (hist.sum(dim=1) == 0).reshape(b, -1)
    for z, mean, turn in ((8, 0.031 * cell, 1), (1, 2 * 0.031 * cell, 2)):
        drawn = _poisson(_splitmix(key + turn), mean) * empty
        hist[:, list(elements).index(z)] += drawn.reshape(b, n1, n2)


def _exit_waves(mols, elements, grid, dz, slices, seeds=None, one_slice=False, keep=False):
    """Exit waves (complex128) of centred molecules in boxes of the same slice
    count, a few molecules at a time; with keep also the potentials."""
    n1, n2, d = grid
    step = max(1, min(16, 16 * 512 * 512 // (n1 * n2)))
    if len(mols) > step:
        parts = [_exit_waves(mols[i:i + step], elements, grid, dz, slices,
                             seeds[i:i + step] if seeds else None, one_slice, keep)
                 for i in range(0, len(mols), step)]
        if keep:
            return torch.cat([p[0] for p in parts]), torch.cat([p[1] for p in parts])
        return torch.cat(parts)
    lam, gamma = _beam()
    ff = _form_factors(elements, n1, n2, d)
    index = {int(z): i for i, z in enumerate(elements)}
    at, layer = [], []
    for b, (xyz, zs) in enumerate(mols):
        s = np.zeros(len(xyz), int) if one_slice else _bins(xyz[:, 0], slices, dz)
        x, y = _bins(xyz[:, 1], n1, d), _bins(xyz[:, 2], n2, d)
        e = np.array([index[int(z)] for z in range(1, 104) if z in index])
        lut = np.zeros(104, int)
        lut[[z for z in sorted(index)]] = e
        ok = (s >= 0) & (x >= 0) & (y >= 0)
        at.append((((b * len(elements) + lut[zs]) * n1 + x) * n2 + y)[ok])
        layer.append(s[ok])
    at, layer = np.concatenate(at), np.concatenate(layer)
    order = np.argsort(layer, kind="stable")
    ends = np.searchsorted(layer[order], np.arange(slices + 1))
    at = torch.from_numpy(at[order]).cuda()
    band, _, f2 = _masks_and_f2(n1, n2, d)
    prop = torch.polar(band.double(), -math.pi * lam * (0.0 if one_slice else dz) * f2)
    i1, i2 = (torch.from_numpy((np.arange(n) + n // 2) % n - (n + 1) // 2).cuda()
              for n in (n1, n2))
    half = n2 // 2 + 1
    disk = (i1[:, None] ** 2 + i2[None, :half] ** 2 <= (min(n1, n2) // 2) ** 2).double()
    if n1 != n2:
        disk = torch.ones_like(disk)
    psi = torch.full((len(mols), n1, n2), math.sqrt(DOSE * d * d), dtype=torch.complex128,
                     device="cuda")
    kept = []
    for s in range(slices):
        hist = torch.zeros(len(mols) * len(elements) * n1 * n2, dtype=torch.float64,
                           device="cuda")
        mine = at[int(ends[s]):int(ends[s + 1])]
        hist.scatter_add_(0, mine, torch.ones_like(mine, dtype=torch.float64))
        hist = hist.reshape(len(mols), len(elements), n1, n2)
        if seeds:
            _add_water(hist, seeds, s, elements, d * d * dz)
        spec = (torch.fft.rfft2(hist) * ff).sum(dim=1) * disk
        rows = torch.fft.ifft(spec, dim=-2)
        rows[..., 0].imag.zero_()
        if n2 % 2 == 0:
            rows[..., -1].imag.zero_()
        v = torch.fft.irfft(rows, n=n2, dim=-1).clamp_(min=1e-13)
        if keep:
            kept.append(v)
        psi = _through(psi, v, lam * gamma, prop)
    return (psi, torch.stack(kept, dim=1)) if keep else psi


def _through(psi, v, factor, prop):
    return torch.fft.ifft2(torch.fft.fft2(psi * torch.polar(torch.ones_like(v), factor * v)) * prop)


def _images(psi, d):
    """|psi|^2 after the lens, float64."""
    n1, n2 = psi.shape[-2:]
    lam, _ = _beam()
    _, aper, f2 = _masks_and_f2(n1, n2, d)
    chi = 0.5 * math.pi * CS_MM * 1e7 * lam ** 3 * f2 ** 2 - math.pi * DEFOCUS * lam * f2
    lens = torch.polar(aper.double(), -chi)
    return torch.cat([torch.fft.ifft2(torch.fft.fft2(p[None]) * lens).abs() ** 2 for p in psi])


def _blocks(c, m, layers, cin_pad):
    """(name, shape) of the parameter blocks, each starting on a multiple of 64."""
    out = [("lift_w", (cin_pad, c)), ("lift_b", (c,))]
    for l in range(layers):
        out += [(("w", l), (c, c)), (("b", l), (c,)), (("r", l), (2 * m, m, c, c, 2))]
    return out + [("proj_w", (c, 2)), ("proj_b", (2,))]


def _network(x, p, layers, m):
    """The network in 64 bits: x (B, n, n, channels) -> (B, n, n, 2)."""
    n = x.shape[1]
    k1 = list(range(m)) + list(range(n - m, n))
    v = x @ p["lift_w"] + p["lift_b"]
    for l in range(layers):
        spec = torch.fft.rfft2(v, dim=(1, 2))[:, k1, :m]
        r = torch.view_as_complex(p["r", l])
        mixed = torch.einsum("bxkc,xkcd->bxkd", spec, r)
        full = torch.zeros((x.shape[0], n, n // 2 + 1, v.shape[-1]), dtype=mixed.dtype,
                           device=x.device)
        full = full.index_put((torch.arange(x.shape[0], device=x.device)[:, None, None],
                               torch.tensor(k1, device=x.device)[None, :, None],
                               torch.arange(m, device=x.device)[None, None, :]), mixed)
        back = torch.fft.ifft(full, dim=1)
        first = torch.zeros(n // 2 + 1, dtype=torch.float64, device=x.device)
        first[0] = 1.0
        back = torch.complex(back.real, back.imag * (1.0 - first)[None, None, :, None])
        u = torch.fft.irfft(back, n=n, dim=2)
        v = v @ p["w", l] + p["b", l] + u
        if l + 1 < layers:
            v = torch.nn.functional.gelu(v)
    return v @ p["proj_w"] + p["proj_b"]


def _inputs(psi, v, psi0, sigma):
    x = torch.zeros(psi.shape + (16,), dtype=torch.float64, device="cuda")
    x[..., 0], x[..., 1] = psi.real / psi0, psi.imag / psi0
    x[..., 2:2 + v.shape[1]] = sigma * v.permute(0, 2, 3, 1)
    return x


def _exact_learned(case, seed):
    with np.load(NETWORK, allow_pickle=False) as z:
        flat = torch.from_numpy(z["params"].astype(np.float64)).cuda()
        n, _, c, m, layers, _ = (int(k) for k in z["config"])
    p, off = {}, 0
    for name, shape in _blocks(c, m, layers, 16):
        size = int(np.prod(shape))
        p[name] = flat[off:off + size].reshape(shape)
        off += (size + 63) // 64 * 64
    lam, gamma = _beam()
    psi0 = math.sqrt(DOSE)
    mols = [_centred(m_) for m_ in _molecules(case, seed)]
    out = []
    for i in range(0, len(mols), 4):
        psi, v = _exit_waves(mols[i:i + 4], ELEMENTS, (n, n, 1.0), COARSE_DZ, COARSE_SLICES,
                             keep=True)
        fix = _network(_inputs(psi, v, psi0, lam * gamma), p, layers, m)
        out.append(_images(psi + psi0 * torch.complex(fix[..., 0], fix[..., 1]), 1.0))
    return torch.cat(out)


def _exact_train(case, seed):
    coarse, v, fine = _network_inputs(case, seed)
    weights, layers, m = _start_weights(case, seed), 4, 16
    p = {}
    for name, shape in _blocks(32, m, layers, 16):
        a = weights[name[0]][name[1]] if isinstance(name, tuple) else weights[name]
        a = np.stack([a.real, a.imag], -1) if np.iscomplexobj(a) else a
        p[name] = torch.from_numpy(a).float().double().cuda().requires_grad_()
    lam, gamma = _beam()
    psi0, batch = math.sqrt(DOSE), case["batch"]
    losses, waves = [], []
    for b in range(batch):
        a, t = coarse[b:b + 1].to(torch.complex128), fine[b:b + 1].to(torch.complex128)
        out = _network(_inputs(a, v[b:b + 1].double(), psi0, lam * gamma), p, layers, m)
        psi = a + psi0 * torch.complex(out[..., 0], out[..., 1])
        norm = t.abs().square().sum()
        rel = (psi - t).abs().square().sum() / norm
        (rel / batch).backward()
        losses.append([float(rel), float(norm), float(psi.detach().abs().square().sum())])
        waves.append(psi.detach())
    flat = []
    for name, shape in _blocks(32, m, layers, 16):
        g = p[name].grad.reshape(-1)
        flat += [g, g.new_zeros(-g.numel() % 64)]
    return {"loss": torch.tensor(losses, dtype=torch.float64), "wave": torch.cat(waves),
            "grads": torch.cat(flat)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "learned":
        return _exact_learned(case, seed)
    if kind == "train":
        return _exact_train(case, seed)
    d = case["pixel"]
    if kind == "propagate":
        lam, gamma = _beam()
        n1, n2 = case["n1"], case["n2"]
        band, _, f2 = _masks_and_f2(n1, n2, d)
        prop = torch.polar(band.double(), -math.pi * lam * case["dz"] * f2)
        slices, out = _given_potentials(case, seed), []
        for b in range(case["batch"]):
            psi = torch.full((n1, n2), math.sqrt(DOSE * d * d), dtype=torch.complex128,
                             device="cuda")
            for s in range(case["slices"]):
                psi = _through(psi, slices[b, s].double(), lam * gamma, prop)
            out.append(psi)
        return _images(torch.stack(out), d)
    mols = [_centred(m) for m in _molecules(case, seed)]
    if kind == "mixed":
        sizes, ns = _wave_sizes(case), _thickness(case, seed)
        out = [None] * len(mols)
        for n in ns:
            mine = [i for i in range(len(mols)) if int(sizes[i]) == n]
            psi = _exit_waves([mols[i] for i in mine], ELEMENTS, (n, n, d), case["dz"], ns[n])
            for i, image in zip(mine, _images(psi, d)):
                out[i] = image
        return out
    n = case["n"]
    if kind in ("wpo", "pipe"):
        zs = sorted(int(z) for z in np.unique(mols[0][1]))
        z = mols[0][0][:, 0]
        ns = 1 if kind == "wpo" else max(1, int(math.ceil(float(z.max() - z.min()) / case["dz"])))
        psi = _exit_waves(mols, zs, (n, n, d), case.get("dz", 1.0), ns, one_slice=kind == "wpo")
        return _images(psi, d)[0]
    psi = _exit_waves(mols, ELEMENTS, (n, n, d), case["dz"], case["slices"],
                      _seeds(case, seed) if kind == "water" else None)
    return _images(psi, d)
