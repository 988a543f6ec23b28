"""The engine's HIP kernels run on the CPU through an emulation of the HIP runtime (tests/cpu_emu):
every workgroup as host threads meeting at its barriers, its LDS as one heap block of exactly the
launch's size, device buffers as exact host allocations. Built with AddressSanitizer, any LDS or
global access outside its buffer aborts the run; the spectra are checked against numpy in FP64.

Cases: the generic four-step over factors 3, 5, 7 with workgroups that straddle batch items
(f32 at 16 points per thread), the power-of-two four-step, the mixed-radix menu lengths, Bluestein, a
real transform, a DCT, the one-kernel DCT-II/III and R2C/C2R, the R2C repack pass; half-precision storage; the
streaming filter, the convolution and its gradients, axes of multidimensional arrays; and the f64
generic kernels built at 16 points per thread (the geometry an earlier build ran on the GPU, where
lengths with radix-5 passes came out wrong) on those lengths.
Set KFR_AMD_EMU_TSAN=1 to also run a ThreadSanitizer build (a missing barrier shows as a race), and
KFR_AMD_EMU_FULL=1 for the 16-points-per-thread f64 build and the slowest f64 length."""
from __future__ import annotations

import os
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

HERE = Path(__file__).resolve().parent
sys.path.insert(0, str(HERE / "cpu_emu"))
import build as emu_build  # noqa: E402

import oracle  # noqa: E402
from tests.common import fp64_dct, fp64_rdft  # noqa: E402

pytestmark = pytest.mark.skipif(not Path(emu_build.CXX).exists(), reason="ROCm clang++ not found")


def _run(variant, tmp_path, args, x, out_dtype, env=None):
    exe = emu_build.build(variant)
    fin, fout = tmp_path / "in.bin", tmp_path / "out.bin"
    np.ascontiguousarray(x).tofile(fin)
    r = subprocess.run([str(exe)] + [str(a) for a in args] + [str(fin), str(fout)], capture_output=True, text=True,
                       timeout=900, env=None if env is None else dict(os.environ, **env))
    assert r.returncode == 0, r.stderr[-4000:]
    return np.fromfile(fout, dtype=out_dtype)


def _dft(variant, tmp_path, dtype, n, batch, inverse, seed):
    t = "f32" if dtype == np.complex64 else "f64"
    x = oracle.complex_uniform(seed, (batch, n), dtype)
    y = _run(variant, tmp_path, ["dft", t, n, batch, int(inverse)], x, dtype).reshape(batch, n)
    xx = x.astype(np.complex128)
    ref = np.fft.ifft(xx, axis=1) * n if inverse else np.fft.fft(xx, axis=1)
    return max(oracle.rel_rms(y[b], ref[b]) for b in range(batch))


# (n, batch): 59049 = 3^10 and 30240 = 2^5 3^3 5 7 run the generic four-step with odd column and row
# counts; 13440 = 2^7 3 5 7 and 62500 = 2^2 5^6 are the lengths that failed at 16 f64 points per
# thread; 65536 the power-of-two four-step; 3840 a menu length; 10007 chained Bluestein (M = 2^15); 97 a direct
# prime pass
F32_CASES = [(59049, 3), (30240, 3), (13440, 2), (1 << 16, 2), (3840, 3), (10007, 1), (97, 5)]
F64_CASES = [(13440, 3), (15360, 2), (30240, 3), (62500, 1)]
# the default run keeps the CPU suite to a few minutes: one sanitizer build, and f64 without its
# slowest length; KFR_AMD_EMU_FULL=1 adds 15360 and the 16-points-per-thread f64 build
FULL = os.environ.get("KFR_AMD_EMU_FULL") == "1"
F64_VARIANTS = ["asan", "asan_pm16"] if FULL else ["asan"]
if not FULL:
    F64_CASES = [c for c in F64_CASES if c[0] != 15360]


@pytest.mark.parametrize("n,batch", F32_CASES)
def test_emulated_f32_lengths(n, batch, tmp_path):
    for inverse in (False, True):
        e = _dft("asan", tmp_path, np.complex64, n, batch, inverse, 40 + n % 97)
        print(f"emulated f32 n={n} batch={batch} inv={inverse}: rel_rms_fp64={e:.3e}", flush=True)
        assert e <= 1e-6


@pytest.mark.parametrize("variant", F64_VARIANTS)
@pytest.mark.parametrize("n,batch", F64_CASES)
def test_emulated_f64_lengths(variant, n, batch, tmp_path):
    for inverse in (False, True):
        e = _dft(variant, tmp_path, np.complex128, n, batch, inverse, 50 + n % 89)
        print(f"emulated f64 ({variant}) n={n} batch={batch} inv={inverse}: rel_rms_fp64={e:.3e}", flush=True)
        assert e <= 1e-14


# the constants of the butterflies are the rounded values: within half a unit of the last place, and a sliver
# for the extended-precision reference's own rounding
@pytest.mark.parametrize("n", [3, 5, 7, 8, 9, 12, 14, 15, 16, 127])
def test_butterfly_constants(n, tmp_path):
    out = tmp_path / "c.bin"
    r = subprocess.run([str(emu_build.build("asan")), "constants", "f64", str(n), str(out)], timeout=900)
    assert r.returncode == 0
    got = np.fromfile(out, dtype=np.float64).reshape(n, 2)
    pi = np.longdouble(3.141592653589793116) + np.longdouble(1.2246467991473532e-16)
    # octants reduced in whole numbers, so that the extended sine and cosine see small angles
    k = np.arange(n)
    a = [(8 * v + n) // (2 * n) % 4 for v in k]                     # nearest quarter turn
    t = 2 * pi * np.array([4 * v - n * ((8 * v + n) // (2 * n)) for v in k], dtype=np.longdouble) / (4 * n)
    c, s = np.cos(t), np.sin(t)
    ref = np.array([[(c, -s, -c, s)[q][i], (s, c, -s, -c)[q][i]] for i, q in enumerate(a)])
    ulp = np.spacing(np.maximum(np.abs(ref.astype(np.float64)), 2.0 ** -60))
    assert np.all(np.abs(got - ref) <= 0.501 * ulp)


# the longest one-workgroup lengths: a few transforms as two kernels, with the plan's intermediate or a
# workspace and the same bits, and under capture in one workgroup, with its two-round LDS exchange
@pytest.mark.parametrize("dtype,n", [(np.complex64, 1 << 15), (np.complex64, 1 << 14), (np.complex128, 1 << 14)])
def test_emulated_longest_one_workgroup(dtype, n, tmp_path):
    t, batch = "f32" if dtype == np.complex64 else "f64", 2
    x = oracle.complex_uniform(64, (batch, n), dtype)
    for inverse in (False, True):
        xx = x.astype(np.complex128)
        ref = np.fft.ifft(xx) * n if inverse else np.fft.fft(xx)
        args = [t, n, batch, int(inverse)]
        two = _run("asan", tmp_path, ["dft"] + args, x, dtype)
        ws = _run("asan", tmp_path, ["ws"] + args + [4], x, dtype)
        one = _run("asan", tmp_path, ["dft"] + args, x, dtype, {"EMU_CAPTURING": "1"})
        assert np.array_equal(two, ws) and not np.array_equal(two, one)
        for y in (two, one):
            assert oracle.rel_rms(y.reshape(batch, n), ref) <= (1e-6 if t == "f32" else 1e-14)


# axes along their stride (mixed lengths, a power of two before an odd dimension, a short axis whose workgroups
# take a wave of columns, a batch of arrays) and the shapes that take transposes instead: runs under 32 bytes
# (2400 and 8192 points), the staged power-of-two kernel under 64 (256 x 40 f32), f64 powers of two from 4096
@pytest.mark.parametrize("t,shape,strided", [("f32", (1080, 40), True), ("f32", (3, 45, 9), True), ("f64", (9, 128, 33), True),
                                             ("f32", (128, 40), True), ("f32", (4, 300), True), ("f64", (256, 40), True),
                                             ("f32", (2400, 40), False), ("f32", (8192, 9), False),
                                             ("f32", (256, 40), False), ("f64", (2400, 9), False), ("f64", (4096, 9), False)])
def test_emulated_axes(t, shape, strided, tmp_path):
    dt = np.complex64 if t == "f32" else np.complex128
    rt = np.float32 if t == "f32" else np.float64
    bound = 1e-6 if t == "f32" else 1e-14
    rng = np.random.default_rng(91)
    fin, fout = tmp_path / "in.bin", tmp_path / "out.bin"

    def run(x, sh, real, inverse, out_dtype):
        x.tofile(fin)
        r = subprocess.run([str(emu_build.build("asan")), "md", t, ",".join(map(str, sh)), str(real), str(int(inverse)),
                            str(fin), str(fout)], capture_output=True, text=True, timeout=900)
        assert r.returncode == 0, r.stderr[-4000:]
        assert ("along its stride" in r.stdout) == strided, r.stdout
        return np.fromfile(fout, dtype=out_dtype)

    x = (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(dt)
    for inverse in (False, True):
        ref = np.fft.ifftn(x.astype(np.complex128)) * x.size if inverse else np.fft.fftn(x.astype(np.complex128))
        assert oracle.rel_rms(run(x, shape, 0, inverse, dt).reshape(shape), ref) <= bound
    if shape[-1] % 2 == 0 or not strided:  # a real last axis with as many spectrum values as columns above
        real = shape[:-1] + (2 * (shape[-1] - 1),)
        v = rng.standard_normal(real).astype(rt)
        ref = np.fft.rfftn(v.astype(np.float64))
        assert oracle.rel_rms(run(v, real, 1, False, dt).reshape(ref.shape), ref) <= bound
        assert oracle.rel_rms(run(ref.astype(dt), real, 1, True, rt).reshape(real) / v.size, v) <= 2 * bound


# lengths with direct passes, the only ones that the build with them runs: one or two primes after
# butterflies or alone, a schedule that takes more threads than the least (1032 = 24 * 43 in f64: 172)
@pytest.mark.parametrize("t,n", [("f32", 1032), ("f64", 1032), ("f32", 11), ("f64", 286), ("f32", 2431)])
def test_emulated_direct_passes(t, n, tmp_path):
    r = subprocess.run([str(emu_build.build("asan")), "schedule", t, str(n)], capture_output=True, text=True, timeout=900)
    if (t, n) == ("f64", 1032):
        assert "threads/transform=172" in r.stdout, r.stdout
    e = _dft("asan", tmp_path, np.complex64 if t == "f32" else np.complex128, n, 5, n % 2 == 0, 65)
    assert e <= (1e-6 if t == "f32" else 1e-14)


# the streaming filter's time-domain kernel: taps around a run of eight and a lane's share, calls shorter and
# longer than a workgroup's outputs and the history. One non-finite sample reaches the outputs of its own taps
# and no others, which keep every bit
@pytest.mark.parametrize("t", ["f32", "f64", "c32", "c64"])
@pytest.mark.parametrize("nt", [1, 9, 100, 130])
def test_emulated_filter(t, nt, tmp_path):
    rt = np.float32 if t in ("f32", "c32") else np.float64
    dt = np.result_type(rt, np.complex64) if t[0] == "c" else rt
    calls = [300, 7, 140, 1, 65]
    rng = np.random.default_rng(90 + nt)
    h, x = (rng.standard_normal(k) + (1j * rng.standard_normal(k) if t[0] == "c" else 0) for k in (nt, sum(calls)))
    h, x = h.astype(dt), x.astype(dt)
    h.tofile(tmp_path / "h.bin")

    def run(v):
        return _run("asan", tmp_path, ["filter", t, nt, ",".join(map(str, calls)), tmp_path / "h.bin"], v, dt)

    y = run(x)
    ref = np.convolve(x.astype(np.complex128), h.astype(np.complex128))[: len(x)]
    # sums of nt products in the data's precision
    assert oracle.rel_rms(y, ref if t[0] == "c" else ref.real) <= (2e-6 if rt == np.float32 else 2e-14)
    for at in (20, 290, 350):
        zero, bad = x.copy(), x.copy()
        zero[at], bad[at] = 0, np.nan if at != 290 else np.inf
        got, clean = run(bad), run(zero)
        hit = np.zeros(len(x), dtype=bool)
        hit[at:at + nt] = True
        assert not np.isfinite(got[hit]).any()
        assert np.array_equal(got[~hit].view(rt), clean[~hit].view(rt))


# calls on one plan run in order whatever streams they are on, with scratch or without: every launch waits
# for the one before, by its stream or by an event recorded after it. Streams 0 (the default one) and 5, 6; a
# caller's stream may be destroyed after its last call, so its work is recorded before the call returns; two
# calls in a row on the default stream without scratch record nothing
@pytest.mark.parametrize("calls", ["5-,6-", "0-,5-", "5-,0-", "0-,0-,5-,0-,6s,0-,0s,5-,5-,0-", "0s,5-,6-,0-,5s", "5s,6-,5-"])
def test_stream_order(calls, tmp_path):
    out = tmp_path / "log.txt"
    assert subprocess.run([str(emu_build.build("asan")), "order", calls, str(out)], timeout=900).returncode == 0
    log = [line.split() for line in out.read_text().split("\n") if line]
    seen, event, done = {}, set(), []      # launches each stream's next work runs after; those the event covers
    for k, (op, s) in enumerate(log):
        known = seen.setdefault(s, set())
        if op == "launch":
            assert set(done) <= known, (calls, log)
            done.append(k)
            known.add(k)
            if s != "0":
                assert log[k + 1] == ["record", s]
        elif op == "record":
            event = set(known)
        else:
            known |= event
    assert len(done) == len(calls.split(","))
    if calls.startswith("0-,0-"):
        assert [op for op, _ in log[:2]] == ["launch", "launch"]


def test_emulated_real_and_dct(tmp_path):
    n, batch = 1 << 14, 3
    x = oracle.gaussian(71, batch * n, np.float32).reshape(batch, n)
    for fmt in (0, 1):
        X = _run("asan", tmp_path, ["real", "f32", n, fmt, batch, 0], x, np.complex64).reshape(batch, -1)
        assert oracle.rel_rms(X, fp64_rdft(x.astype(np.float64), fmt)) <= 1e-6
        y = _run("asan", tmp_path, ["real", "f32", n, fmt, batch, 1], X, np.float32).reshape(batch, n)
        assert oracle.rel_rms(y / n, x) <= 1e-6
    m = 4096
    d = oracle.gaussian(72, 2 * m, np.float32).reshape(2, m)
    for inverse in (False, True):
        y = _run("asan", tmp_path, ["dct", "f32", m, 2, int(inverse)], d, np.float32).reshape(2, m)
        assert oracle.rel_rms(y, fp64_dct(d.astype(np.float64), inverse)) <= 2e-6


# R2C and C2R in one kernel for power-of-two halves that fit one workgroup (f32 2^8, 2^10, 2^13 and
# 2^15 halves, the last two with two-round LDS exchanges; f64 2^14), both pack formats
@pytest.mark.parametrize("t,n,batch", [("f32", 512, 5), ("f32", 2048, 3), ("f32", 1 << 14, 2), ("f32", 1 << 16, 2),
                                       ("f64", 1 << 15, 2)])
def test_emulated_real_one_kernel(t, n, batch, tmp_path):
    dt = np.float32 if t == "f32" else np.float64
    cdt = np.complex64 if t == "f32" else np.complex128
    bound = 1e-6 if t == "f32" else 1e-14
    for fmt in (0, 1):
        x = oracle.gaussian(75 + fmt, batch * n, dt).reshape(batch, n)
        X = _run("asan", tmp_path, ["real", t, n, fmt, batch, 0], x, cdt).reshape(batch, -1)
        ref = fp64_rdft(x.astype(np.float64), fmt)
        assert oracle.rel_rms(X, ref) <= bound
        y = _run("asan", tmp_path, ["real", t, n, fmt, batch, 1], ref.astype(cdt), dt).reshape(batch, n)
        assert oracle.rel_rms(y / n, x) <= bound


# C2R of lengths whose half does not fit one generic workgroup: the unpacking pass into plain
# half-length sequences, then the power-of-two kernels (2^16) or the generic four-step (30000)
@pytest.mark.parametrize("n,batch,fmt", [(1 << 16, 2, 1), (1 << 16, 3, 0), (30000, 2, 1)])
def test_emulated_c2r_unpack_pass(n, batch, fmt, tmp_path):
    x = oracle.gaussian(74 + fmt, batch * n, np.float32).reshape(batch, n)
    X = fp64_rdft(x.astype(np.float64), fmt).astype(np.complex64)
    y = _run("asan", tmp_path, ["real", "f32", n, fmt, batch, 1], X, np.float32).reshape(batch, n)
    assert oracle.rel_rms(y / n, x) <= 1e-6


# R2C whose half does not fit one workgroup: the complex 2^16-point half transform, then the repack
# pass over the half spectrum in global memory
@pytest.mark.parametrize("fmt", [0, 1])
def test_emulated_r2c_repack_pass(fmt, tmp_path):
    n, batch = 1 << 17, 1
    x = oracle.gaussian(76 + fmt, batch * n, np.float32).reshape(batch, n)
    X = _run("asan", tmp_path, ["real", "f32", n, fmt, batch, 0], x, np.complex64).reshape(batch, -1)
    assert oracle.rel_rms(X, fp64_rdft(x.astype(np.float64), fmt)) <= 1e-6


# DCT-II and DCT-III in one kernel: f32 at 2^8 points per half (16 threads per transform, the shortest
# fused length), 2^10 (mirrored first pass, LDS partner exchange) and 2^13, 2^15 (two-round LDS
# exchange, mirrored first and last passes), f64 at 2^13 and 2^14; 128 points f32 stays on the
# pack/FFT/post path
@pytest.mark.parametrize("t,m,batch", [("f32", 512, 5), ("f32", 256, 3), ("f32", 2048, 3), ("f32", 1 << 14, 2),
                                       ("f32", 1 << 16, 1), ("f64", 1 << 14, 2), ("f64", 1 << 15, 1)])
def test_emulated_fused_dct(t, m, batch, tmp_path):
    dt = np.float32 if t == "f32" else np.float64
    d = oracle.gaussian(73 + m % 7, batch * m, dt).reshape(batch, m)
    for inverse in (False, True):
        y = _run("asan", tmp_path, ["dct", t, m, batch, int(inverse)], d, dt).reshape(batch, m)
        e = oracle.rel_rms(y, fp64_dct(d.astype(np.float64), inverse))
        print(f"emulated dct {t} m={m} batch={batch} inverse={inverse}: rel_rms_fp64={e:.3e}", flush=True)
        assert e <= (1e-6 if t == "f32" else 1e-14)


def _to_half(x: np.ndarray, storage: str) -> np.ndarray:
    """complex values as interleaved 2-byte pairs: binary16, or bfloat16 rounded to nearest even"""
    f = np.stack([x.real, x.imag], -1).astype(np.float32)
    if storage == "f16":
        return f.astype(np.float16).view(np.uint16)
    u = f.view(np.uint32).astype(np.uint64)
    return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)


def _from_half(h: np.ndarray, storage: str) -> np.ndarray:
    if storage == "f16":
        f = h.view(np.float16).astype(np.float64)
    else:
        f = (h.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    return f[..., 0] + 1j * f[..., 1]


# half-precision storage: one workgroup (2^10), the two-kernel form of few transforms (2^15) and the multi-pass
# kernels with their f32 intermediates (2^15 and 2^16, selected through KFR_AMD_HALF_MULTIPASS_MIN_LOG)
@pytest.mark.parametrize("storage,n,batch,multi", [("bf16", 1 << 10, 3, False), ("bf16", 1 << 15, 2, False),
                                                   ("bf16", 1 << 15, 2, True), ("f16", 1 << 16, 1, True)])
def test_emulated_half_storage(storage, n, batch, multi, tmp_path):
    exe = emu_build.build("asan")
    rng = np.random.default_rng(n + batch)
    x = rng.standard_normal((batch, n)) + 1j * rng.standard_normal((batch, n))
    h = _to_half(x, storage)
    xq = _from_half(h, storage)
    fin, fout = tmp_path / "in.bin", tmp_path / "out.bin"
    h.tofile(fin)
    env = dict(os.environ, KFR_AMD_HALF_MULTIPASS_MIN_LOG="15" if multi else "99")
    for inverse in (False, True):
        r = subprocess.run([str(exe), "half", storage, str(n), str(batch), str(int(inverse)), str(fin), str(fout)],
                           capture_output=True, text=True, timeout=900, env=env)
        assert r.returncode == 0, r.stderr[-4000:]
        y = _from_half(np.fromfile(fout, dtype=np.uint16).reshape(batch, n, 2), storage)
        ref = np.fft.ifft(xq, axis=1) * n if inverse else np.fft.fft(xq, axis=1)
        e = np.linalg.norm(y - ref) / np.linalg.norm(ref)
        print(f"emulated {storage} n={n} multi={multi} inv={inverse}: rel_rms_fp64={e:.3e}", flush=True)
        assert e <= (2e-3 if storage == "bf16" else 5e-4)


def _conv(variant, tmp_path, t, nx, nh, batch, shared, seed, env=None):
    """relative errors of a convolution plan's output and its two gradients"""
    dt = np.float32 if t == "f32" else np.float64
    rng = np.random.default_rng(seed)
    ny = nx + nh - 1
    x, g = (rng.standard_normal((batch, n)).astype(dt) for n in (nx, ny))
    h = rng.standard_normal((1 if shared else batch, nh)).astype(dt)
    out = _run(variant, tmp_path, ["conv", t, nx, nh, batch, int(shared)], np.concatenate([x.ravel(), h.ravel(), g.ravel()]), dt, env)
    m = 1 << (ny + nh).bit_length()
    X, H, Gf = (np.fft.rfft(v.astype(np.float64), m) for v in (x, h, g))
    dh = np.fft.irfft(Gf * X.conj(), m)[:, :nh]
    ref = [np.fft.irfft(X * H, m)[:, :ny], np.fft.irfft(Gf * H.conj(), m)[:, :nx], dh.sum(0) if shared else dh]
    parts = np.split(out, [batch * ny, batch * (ny + nx)])
    return [oracle.rel_rms(a, r.ravel()) for a, r in zip(parts, ref)]


# the convolution and its gradients, overlap-save over blocks of 256 points: one segment and four, the last
# ragged, a shared filter; workgroups of the filter gradient with one, three and one, and all of the segments;
# a filter as long as the signal, through full-length transforms
@pytest.mark.parametrize("t,nx,nh,batch,shared,per", [("f32", 700, 30, 2, False, 0), ("f32", 700, 30, 3, False, 3),
                                                      ("f64", 700, 30, 2, True, 3), ("f64", 300, 80, 3, True, 9),
                                                      ("f32", 90, 40, 2, False, 0), ("f32", 200, 200, 2, True, 0)])
def test_emulated_convolution(t, nx, nh, batch, shared, per, tmp_path):
    env = {"KFR_AMD_CONV_SEGMENTS": str(per)} if per else None
    for e in _conv("asan", tmp_path, t, nx, nh, batch, shared, 92, env):
        assert e <= (1e-6 if t == "f32" else 1e-14)


@pytest.mark.skipif(os.environ.get("KFR_AMD_EMU_TSAN") != "1", reason="set KFR_AMD_EMU_TSAN=1")
@pytest.mark.parametrize("dtype,n,batch", [(np.complex64, 30240, 3), (np.complex64, 1 << 15, 1),
                                           (np.complex128, 13440, 2)])
def test_emulated_no_races(dtype, n, batch, tmp_path):
    e = _dft("tsan", tmp_path, dtype, n, batch, False, 60)
    assert e <= (1e-6 if dtype == np.complex64 else 1e-14)


# the one-workgroup kernel with its two-round exchange, the time-domain filter, the convolution kernels, a
# real transform unpacked in LDS and an axis along its stride
@pytest.mark.skipif(os.environ.get("KFR_AMD_EMU_TSAN") != "1", reason="set KFR_AMD_EMU_TSAN=1")
def test_emulated_no_races_in_shared_memory(tmp_path):
    x = oracle.complex_uniform(66, (1, 1 << 15), np.complex64)
    y = _run("tsan", tmp_path, ["dft", "f32", 1 << 15, 1, 0], x, np.complex64, {"EMU_CAPTURING": "1"})
    assert oracle.rel_rms(y, np.fft.fft(x.astype(np.complex128))[0]) <= 1e-6
    v = oracle.gaussian(67, 600, np.float32)
    h = oracle.gaussian(68, 130, np.float32)
    h.tofile(tmp_path / "h.bin")
    y = _run("tsan", tmp_path, ["filter", "f32", 130, "400,200", tmp_path / "h.bin"], v, np.float32)
    assert oracle.rel_rms(y, np.convolve(v.astype(np.float64), h.astype(np.float64))[:600]) <= 2e-6
    assert max(_conv("tsan", tmp_path, "f32", 700, 30, 2, False, 93, {"KFR_AMD_CONV_SEGMENTS": "3"})) <= 1e-6
    v = oracle.gaussian(69, 3 * 180, np.float32).reshape(3, 180)
    X = np.fft.rfft(v.astype(np.float64)).astype(np.complex64)
    assert oracle.rel_rms(_run("tsan", tmp_path, ["real", "f32", 180, 1, 3, 1], X, np.float32) / 180, v.ravel()) <= 1e-6
    x = oracle.complex_uniform(70, (45, 20), np.complex64)
    y = _run("tsan", tmp_path, ["md", "f32", "45,20", 0, 0], x, np.complex64)
    assert oracle.rel_rms(y, np.fft.fft2(x.astype(np.complex128)).ravel()) <= 1e-6
