"""An exchange's LDS reads come before the barrier behind them, also where a
transform of few threads is spread over several waves (columns side by side) and
its results are used under a block-uniform condition only: read off the
assembly of a kernel of that form, compiled here, and by repeating passes whose
blocks run many column tiles."""
import re
import shutil
import subprocess

import pytest
import torch

from emsim_amd.backend.wave_propagator_hip import WavePropagator
from emsim_amd.csrc import build

KERNEL = r"""
#include <hip/hip_runtime.h>
#include "fft_lds.hpp"
using namespace emsim;
template <int N, int C>
__global__ __launch_bounds__(N / 8 * C) void k_columns(const float2* in, float2* out, int ld,
                                                       int n_tiles, int run, const float2* tw) {
    constexpr int EPT = 8, T = N / EPT, W = LdsLayout<N>::kStride;
    __shared__ float re[C * W], im[C * W];
    const int c = threadIdx.x % C, t = threadIdx.x / C;
    TwCache<N, EPT> twc;
    twc.load(tw, t);
    for (int r = 0; r < run; ++r) {
        const int tile = blockIdx.x * run + r;
        const bool ok = tile < n_tiles;
        const int j = (ok ? tile : 0) * C + c;
        float2 v[EPT];
        for (int m = 0; m < EPT; ++m) v[m] = in[(int64_t)(t + m * T) * ld + j];
        fft_n<N, EPT, false>(v, re + c * W, im + c * W, t, twc);
        if (ok)
            for (int m = 0; m < EPT; ++m) out[(int64_t)(t + m * T) * ld + j] = v[m];
    }
}
template __global__ void k_columns<N_, C_>(const float2*, float2*, int, int, int, const float2*);
"""


@pytest.mark.skipif(not shutil.which(build.hipcc()), reason="no hipcc")
@pytest.mark.parametrize("n,columns", [(64, 16), (128, 16), (256, 8), (512, 8), (1024, 4)])
def test_reads_stay_ahead_of_their_barrier(tmp_path, n, columns):
    src, asm = tmp_path / "k.hip", tmp_path / "k.s"
    src.write_text(KERNEL.replace("N_", str(n)).replace("C_", str(columns)))
    subprocess.run([build.hipcc(), *build.FLAGS, f"-I{build.HERE}", "--cuda-device-only", "-S",
                    str(src), "-o", str(asm)], check=True, capture_output=True, timeout=100)
    ops = re.findall(r"^\s*(ds_read|ds_write|s_barrier)", asm.read_text(), re.M)
    events = "".join({"ds_read": "r", "ds_write": "w", "s_barrier": "b"}[op] for op in ops)
    # every exchange: writes, barrier, reads, barrier; nothing behind the last
    assert re.fullmatch(r"(w+br+b)+", events), events


@pytest.mark.gpu
@pytest.mark.parametrize("n1,n2,batch", [(75, 75, 400), (150, 150, 100), (250, 250, 40),
                                         (64, 512, 300)])
def test_column_tiles_are_reproducible(hip, n1, n2, batch):
    prop = WavePropagator(n1, n2, 1.0, 1.0, 200.0)
    gen = torch.Generator(device="cuda").manual_seed(n1 + n2)
    psi = torch.view_as_complex(torch.randn((batch, n1, n2, 2), generator=gen, device="cuda"))
    v = 40 * torch.rand((2, n1, n2), generator=gen, device="cuda")
    wave = prop.multislice_propagate(psi, v, 2.0)
    image = prop.lens_intensity(psi, 1.3, 700.0, 10e-3)
    for _ in range(3):
        assert torch.equal(prop.multislice_propagate(psi, v, 2.0), wave)
        assert torch.equal(prop.lens_intensity(psi, 1.3, 700.0, 10e-3), image)
