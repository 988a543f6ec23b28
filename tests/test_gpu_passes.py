"""Mixed-radix kernels whose first pass reads and last pass writes HBM directly, at the sizes where a
schedule can go wrong (gpu): every butterfly radix, one-pass and many-pass lengths, workgroups with idle
lanes, batch tails, the longest one-workgroup lengths, and the four-step over mixed factors."""
from __future__ import annotations

import numpy as np
import pytest

import kfr_amd
import oracle
from tests.common import bound_fp64

pytestmark = pytest.mark.gpu

# one pass (9, 15); pairs of composite radices (14*12, 15*12, 15*16, 10*9); odd powers; lengths whose
# thread count is no multiple of a wave; the longest of one workgroup (f32 7680, f64 2560); four-step
LENGTHS = [9, 15, 45, 90, 168, 180, 225, 240, 686, 729, 945, 960, 1080, 1372, 2187, 2401, 2560, 3125, 6300, 7680,
           10080, 30240, 44100]


@pytest.mark.parametrize("n", LENGTHS)
@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
def test_mixed_passes(n, dtype):
    torch = pytest.importorskip("torch")
    batch = 7 if n < 5000 else 3  # tails: no multiple of the transforms per workgroup
    x = oracle.complex_uniform(600 + n, (batch, n), dtype)
    p = kfr_amd.dft_plan(n, dtype)
    rdt = np.float32 if dtype == np.complex64 else np.float64
    xd = torch.from_numpy(x.view(rdt).copy()).cuda()
    for inverse in (False, True):
        ref = np.fft.ifft(x.astype(np.complex128)) * n if inverse else np.fft.fft(x.astype(np.complex128))
        yd = torch.full_like(xd, float("nan"))
        p.execute_batch(yd, xd, batch, inverse=inverse)
        zd = xd.clone()
        p.execute_batch(zd, zd, batch, inverse=inverse)  # in place
        y = yd.cpu().numpy().view(dtype).reshape(batch, n)
        err = max(oracle.rel_rms(y[b], ref[b]) for b in range(batch))
        print(f"n={n} {np.dtype(dtype).name} inv={inverse} rel_rms_fp64={err:.3e}", flush=True)
        assert err <= bound_fp64(n, dtype)
        assert torch.equal(yd, zd)


@pytest.mark.parametrize("n", [30, 180, 1920, 2160, 12600])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_mixed_real(n, dt):
    torch = pytest.importorskip("torch")
    batch = 5
    x = oracle.gaussian(700 + n, batch * n, dt).reshape(batch, n)
    cdt = np.complex64 if dt == np.float32 else np.complex128
    p = kfr_amd.dft_plan_real(n, kfr_amd.CCs, dt)
    xd = torch.from_numpy(x.copy()).cuda()
    yd = torch.full((batch, 2 * (n // 2 + 1)), float("nan"), dtype=xd.dtype, device="cuda")
    zd = torch.full_like(xd, float("nan"))
    p.execute_batch(yd, xd, batch)
    p.execute_batch(zd, yd, batch, inverse=True)
    y = yd.cpu().numpy().view(cdt)
    ref = np.fft.rfft(x.astype(np.float64))
    bound = bound_fp64(n, dt)
    assert max(oracle.rel_rms(y[b], ref[b]) for b in range(batch)) <= bound
    assert oracle.rel_rms(zd.cpu().numpy() / n, x) <= 2 * bound


# axes transformed along their stride: mixed and power-of-two lengths before odd and narrow dimensions,
# more and fewer columns than a workgroup takes, batches of arrays, one-pass axes; (97, 33) and (6, 5, 100)
# run a direct prime pass and a one-pass axis, (30, 12, 4) has an axis below the 64-byte run
MD_SHAPES = [(1080, 241), (45, 128), (64, 45, 33), (9, 8), (97, 33), (6, 5, 100), (30, 12, 4), (512, 15, 9), (5, 1, 80)]


@pytest.mark.parametrize("shape", MD_SHAPES)
@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
def test_strided_axes(shape, dtype):
    torch = pytest.importorskip("torch")
    n = int(np.prod(shape))
    rng = np.random.default_rng(n)
    x = (rng.standard_normal((2,) + shape) + 1j * rng.standard_normal((2,) + shape)).astype(dtype)
    axes = tuple(range(1, len(shape) + 1))
    p = kfr_amd.dft_plan_md(shape, dtype)
    xd = torch.from_numpy(x).cuda()
    for inverse in (False, True):
        ref = np.fft.ifftn(x.astype(np.complex128), axes=axes) * n if inverse else np.fft.fftn(
            x.astype(np.complex128), axes=axes)
        yd = torch.full_like(xd, float("nan"))
        p.execute_batch(yd, xd, 2, inverse)
        zd = xd.clone()
        p.execute_batch(zd, zd, 2, inverse)
        assert oracle.rel_rms(yd.cpu().numpy(), ref) <= bound_fp64(n, dtype)
        assert torch.equal(yd, zd)


@pytest.mark.parametrize("shape", [(1080, 242), (45, 30, 16), (7, 64, 30), (1, 30)])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_strided_real_axes(shape, dt):
    torch = pytest.importorskip("torch")
    n = int(np.prod(shape))
    x = oracle.gaussian(800 + n, n, dt).reshape(shape)
    cdt = torch.complex64 if dt == np.float32 else torch.complex128
    p = kfr_amd.dft_plan_md_real(shape, False, dt)
    xd = torch.from_numpy(x.copy()).cuda()
    yd = torch.empty(p.complex_size(), dtype=cdt, device="cuda")
    keep = torch.full_like(xd, float("nan"))
    p.execute(yd, xd)
    spectrum = yd.clone()
    p.execute(keep, yd)
    assert torch.equal(yd, spectrum)  # the input spectrum is left as it was
    bound = bound_fp64(n, dt)
    assert oracle.rel_rms(yd.cpu().numpy(), np.fft.rfftn(x.astype(np.float64))) <= bound
    assert oracle.rel_rms(keep.cpu().numpy() / n, x) <= 4 * bound


# the longest one-workgroup powers of two run a few transforms as two kernels and many in one workgroup
# each (they change over at 80), and stay in one workgroup under capture
@pytest.mark.parametrize("n,dtype", [(1 << 14, np.complex64), (1 << 15, np.complex64), (1 << 14, np.complex128)])
@pytest.mark.parametrize("batch", [1, 79, 80, 95, 96])
def test_longest_one_workgroup_lengths(n, dtype, batch):
    torch = pytest.importorskip("torch")
    x = oracle.complex_uniform(620 + batch, (batch, n), dtype)
    p = kfr_amd.dft_plan(n, dtype)
    xd = torch.from_numpy(x).cuda()
    for inverse in (False, True):
        ref = np.fft.ifft(x.astype(np.complex128)) * n if inverse else np.fft.fft(x.astype(np.complex128))
        yd = torch.full_like(xd, float("nan"))
        p.execute_batch(yd, xd, batch, inverse)
        assert oracle.rel_rms(yd.cpu().numpy(), ref) <= bound_fp64(n, dtype)
    zd = torch.full_like(xd, float("nan"))
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        p.execute_batch(zd, xd, batch, inverse=True)
    for _ in range(3):
        zd.fill_(0)
        g.replay()
        torch.cuda.synchronize()
        assert oracle.rel_rms(zd.cpu().numpy(), ref) <= bound_fp64(n, dtype)
