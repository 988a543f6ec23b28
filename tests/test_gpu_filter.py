"""The streaming filter's time-domain kernel at the sizes where its tiles end (gpu): taps around a run of
eight, a lane's share and the lane counts, calls shorter and longer than a workgroup's outputs and than the
history, real and complex, against a direct convolution in FP64."""
from __future__ import annotations

import numpy as np
import pytest

import kfr_amd
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [np.float32, np.float64, np.complex64, np.complex128])
@pytest.mark.parametrize("nt", [1, 2, 8, 9, 64, 65, 129, 1000, 4096, 4097])
def test_filter_calls(nt, dt):
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(900 + nt)
    calls = [1, 7, 32, 33, 500, 2049, 3, 4500]
    total = sum(calls)

    def data(n):
        x = rng.standard_normal(n)
        return (x + 1j * rng.standard_normal(n) if np.dtype(dt).kind == "c" else x).astype(dt)

    h, x = data(nt), data(total)
    f = kfr_amd.convolve_filter(h, 1024)
    rdt = np.float32 if np.dtype(dt) in (np.dtype(np.float32), np.dtype(np.complex64)) else np.float64
    cx = 2 if np.dtype(dt).kind == "c" else 1
    ref = np.convolve(x.astype(np.complex128), h.astype(np.complex128))[:total]
    # rounding of sums of nt products in the data's precision, against the output's magnitude
    bound = 2e-6 if rdt == np.float32 else 2e-14
    out, pos = np.empty_like(x), 0
    for n in calls:
        if cx == 1:  # device buffers, real data
            xd = torch.from_numpy(x[pos:pos + n].copy()).cuda()
            yd = torch.full_like(xd, float("nan"))
            f.apply(yd, xd)
            out[pos:pos + n] = yd.cpu().numpy()
        else:
            y = np.empty(n, dtype=dt)
            f.apply(y, x[pos:pos + n].copy())
            out[pos:pos + n] = y
        pos += n
    err = oracle.rel_rms(out, ref if cx == 2 else ref.real)
    print(f"nt={nt} {np.dtype(dt).name} rel_rms_fp64={err:.3e}", flush=True)
    assert err <= bound
