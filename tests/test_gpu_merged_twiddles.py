"""Merged-twiddle butterflies: every radix, remainder radix and number of
passes that a transform is cut into, against 64-bit numpy.

The bound is on the rounding of the network itself.  A radix-2 level writes
each value after two roundings of at most half an ulp (three where the product
with the root is rounded first, two of them on the smaller product), whose
errors, u = 2^-24, have a variance of u^2/3 relative to the value; with the
rounding of the roots a level adds less than u^2, so log2 N levels stay below
u sqrt(log2 N) in the 2-norm.  A wrong or misplaced root gives an error of order
one.
"""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


def _run(pkg, gpu, n, batch, direction, executed, params, seed):
    import torch

    rng = np.random.default_rng(seed)
    x = (rng.standard_normal((batch, n)) + 1j * rng.standard_normal((batch, n))).astype(np.complex64)
    plan = pkg.ExecutionPlan(n=n, batch=batch, direction="dit", precision="fp32", selection_source="table",
                             reason="test", fallback=False, executed=executed, block=None, params=params,
                             transform_direction=direction, norm="ortho")
    y = pkg.execute_fft_plan(plan, torch.from_numpy(x).to(gpu)).cpu().numpy()
    e = (np.fft.fft if direction == "forward" else np.fft.ifft)(x.astype(np.complex128), norm="ortho")
    return float(np.linalg.norm(y - e) / np.linalg.norm(e))


@pytest.mark.parametrize("direction", ["forward", "inverse"])
@pytest.mark.parametrize("schedule", [0, 1, 3])
@pytest.mark.parametrize("l1,l2", [(4, 4), (5, 4), (4, 6), (6, 5), (7, 6), (8, 7), (7, 9), (9, 8), (10, 8), (10, 10)])
def test_four_step_split(pkg, gpu, l1, l2, schedule, direction):
    """Pass 2's roots carry W_N^(n2 k1): every pass length 16..1024 on either
    side, which takes first radices 4 to 32, middle radices 4 to 16 and last
    radices 2 to 32."""
    n = 1 << (l1 + l2)
    err = _run(pkg, gpu, n, 3, direction, "fft_four_step_batch", {"n1": 1 << l1, "schedule": schedule},
               1000 * l1 + l2)
    assert err <= U * math.sqrt(l1 + l2), err


@pytest.mark.parametrize("l1,l2", [(4, 4), (5, 6), (7, 5), (8, 9), (10, 9)])
def test_four_step_real(pkg, gpu, l1, l2):
    """The real epilogues' row passes take the same roots at permuted (R2C)
    and mirrored columns: forward and back returns the samples."""
    import torch

    n = 2 << (l1 + l2)
    x = np.random.default_rng(n).standard_normal((3, n)).astype(np.float32)
    common = dict(n=n, batch=3, direction="dit", precision="fp32", selection_source="table", reason="test",
                  fallback=False, executed="fft_four_step_batch", block=None, params={"n1": 1 << l1}, norm="ortho")
    spec = pkg.execute_fft_plan(pkg.ExecutionPlan(transform_type="r2c", **common), torch.from_numpy(x).to(gpu))
    e = np.fft.rfft(x.astype(np.float64), norm="ortho")
    levels = l1 + l2 + 2  # the core's, the stitch and the rounding of its roots
    assert np.linalg.norm(spec.cpu().numpy() - e) <= U * math.sqrt(levels) * np.linalg.norm(e)
    back = pkg.execute_fft_plan(pkg.ExecutionPlan(transform_type="c2r", transform_direction="inverse", **common), spec)
    assert np.linalg.norm(back.cpu().numpy() - x) <= U * math.sqrt(2 * levels) * np.linalg.norm(x)


@pytest.mark.parametrize("direction", ["forward", "inverse"])
@pytest.mark.parametrize("logn", [11, 12, 13, 14, 15])
def test_lds_32_elements(pkg, gpu, logn, direction):
    """Remainder radices 2, 4, 8, 16 and 32 after the radix-32 passes, and the
    last block's rows past a ragged batch."""
    err = _run(pkg, gpu, 1 << logn, 3, direction, "fft_lds_fused_batch", {"elems": 32}, logn)
    assert err <= U * math.sqrt(logn), err


@pytest.mark.parametrize("logn", [4, 5, 6, 7, 8, 9, 10, 11])
@pytest.mark.parametrize("batch", [1, 3, 257])
def test_lds_last_block_rows(gpu, logn, batch):
    """Several transforms a block: the threads of rows past the batch load its
    last row again, or nothing, and store nothing, in each mode with every
    element count it takes."""
    import torch

    from kunlunxin_fft_amd import native

    n, m = 1 << logn, (1 << (logn - 1)) + 1
    x = np.random.default_rng(n + batch).standard_normal((batch, n)).astype(np.float32)
    e = np.fft.fft(x.astype(np.float64), norm="ortho")
    tol = U * math.sqrt(2 * (logn + 2))
    xin = torch.from_numpy(x).to(gpu)
    stream = torch.cuda.current_stream().cuda_stream

    def run(kind, elems, src, out):
        plan = native.NativePlan(n, batch, kind, "inverse" if kind == "c2r" else "forward", norm="ortho",
                                 flow=native.FLOW_LDS_FUSED, params=[elems])
        assert plan.info.elems_per_thread == elems
        plan.execute(src.data_ptr(), out.data_ptr(), stream)
        torch.cuda.synchronize()
        return out.cpu().numpy()

    def close(y, ref):
        return np.linalg.norm(y - ref) <= tol * np.linalg.norm(ref)

    for elems in (4, 8, 16, 32):
        if elems < 32 or logn >= 10:
            cplx = xin.to(torch.complex64)
            assert close(run("c2c", elems, cplx, torch.empty_like(cplx)), e), elems
        if elems < 32 or logn >= 11:  # a real transform's core is n/2
            spec = torch.empty((batch, m), dtype=torch.complex64, device=gpu)
            assert close(run("r2c", elems, xin, spec), e[:, :m]), elems
            assert close(run("c2r", elems, spec, torch.empty_like(xin)), x), elems


MAX = float(np.finfo(np.float32).max)
RANGE_PLANS = [("fft_lds_fused_batch", 12, {"elems": 32}), ("fft_lds_fused_batch", 13, {"elems": 32}),
               ("fft_lds_fused_batch", 14, {"elems": 32}), ("fft_lds_fused_batch", 15, {"elems": 32}),
               ("fft_lds_fused_batch", 12, {"elems": 16}), ("fft_four_step_batch", 14, {"n1": 64}),
               ("fft_four_step_batch", 16, {"n1": 256}), ("fft_four_step_batch", 18, {"n1": 512}),
               ("fft_four_step_batch", 20, {"n1": 1024}), ("fft_four_step_batch", 20, {"n1": 1024, "schedule": 3})]


def _unscaled(pkg, gpu, executed, logn, params, x):
    import torch

    plan = pkg.ExecutionPlan(n=1 << logn, batch=len(x), direction="dit", precision="fp32", selection_source="table",
                             reason="test", fallback=False, executed=executed, block=None, params=params, norm="none")
    x = torch.from_numpy(x.astype(np.complex64)).to(gpu)
    return pkg.execute_fft_plan(plan, x[0] if len(x) == 1 else x).cpu().numpy().reshape(x.shape)


@pytest.mark.parametrize("executed,logn,params", RANGE_PLANS)
def test_overflow_stays_in_its_bins(pkg, gpu, executed, logn, params):
    """A tone whose own bin exceeds the float range 2^d to 2^(d+1) times: the
    first partial sums that overflow are those of n / 2^d samples, which only
    the 2^d bins k0 + i n / 2^d are computed from; the rest stays finite."""
    n, k0 = 1 << logn, 5
    for d in range(5):
        x = (1.5 * 2.0 ** d * MAX / n) * np.exp(2j * np.pi * k0 * np.arange(n) / n)
        y = _unscaled(pkg, gpu, executed, logn, params, x[None])[0]
        lost = np.flatnonzero(~(np.isfinite(y.real) & np.isfinite(y.imag)))
        assert set(lost) <= set((k0 + np.arange(1 << d) * (n >> d)) % n) and k0 in lost, (d, lost[:8])


@pytest.mark.parametrize("executed,logn,params", RANGE_PLANS)
def test_infinite_first_sample(pkg, gpu, executed, logn, params):
    """x[0] enters every bin with factor 1: an infinite real part makes every
    real part infinite and leaves the imaginary parts finite."""
    x = np.full((1, 1 << logn), 0.5 + 0j)
    x[0, 0] = np.inf
    y = _unscaled(pkg, gpu, executed, logn, params, x)
    assert np.all(np.isposinf(y.real)) and np.all(np.isfinite(y.imag))


@pytest.mark.parametrize("executed,logn,params", RANGE_PLANS)
def test_largest_values_in_range(pkg, gpu, executed, logn, params):
    """Bins up to 0.999 of the largest float come out, whatever the partial
    sums on the way to them."""
    n, batch = 1 << logn, max(1, (1 << 20) >> logn)
    rng = np.random.default_rng(logn)
    x = rng.standard_normal((batch, n)) + 1j * rng.standard_normal((batch, n))
    e = np.fft.fft(x)
    top = 0.999 * MAX / np.maximum(np.abs(e.real).max(-1), np.abs(e.imag).max(-1))[:, None]
    y = _unscaled(pkg, gpu, executed, logn, params, x * top)
    assert np.all(np.isfinite(y.real)) and np.all(np.isfinite(y.imag))
    e = e * top / MAX
    y = y.astype(np.complex128) / MAX
    # one rounding for the samples beside those of the network
    assert np.linalg.norm(y - e) <= U * math.sqrt(logn + 1) * np.linalg.norm(e)
