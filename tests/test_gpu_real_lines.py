"""Bin rows of n/2 + 1 values, which start anywhere in a 128-byte line, in the
real modes of the LDS kernel: several rows a block, a ragged last block, bins
stored straight or in whole lines, and nothing written outside the rows,
against 64-bit numpy.

The bound is that of the transform's own rounding: below u per radix-2 level
and for the stitch (u = 2^-24), so u sqrt(log2 n + 2) in the 2-norm; a bin in
a neighbour's place gives an error of order one.
"""
import math

import numpy as np
import pytest

from kunlunxin_fft_amd import native

pytestmark = pytest.mark.gpu

U = 2.0 ** -24
GUARD = 32  # bins or samples around the rows that must stay as they are

# (log2 n, elements per thread): 8 and 16 elements with one and with several
# transforms a block, float2 and split exchange, and 32 elements
CASES = [(10, 8), (11, 8), (12, 8), (11, 16), (12, 16), (13, 16), (14, 16), (15, 16),
         (12, 32), (13, 32), (14, 32), (15, 32), (16, 32)]


def _plan(n, batch, kind, elems):
    return native.NativePlan(n, batch, kind, "forward" if kind == "r2c" else "inverse", norm="ortho",
                             flow=native.FLOW_LDS_FUSED, params=[elems])


@pytest.mark.parametrize("batch,shift", [(1, 0), (3, 1), (5, 8), (2, 15)])
@pytest.mark.parametrize("logn,elems", CASES)
def test_bin_rows(gpu, logn, elems, batch, shift):
    import torch

    n, m = 1 << logn, (1 << (logn - 1)) + 1
    x = np.random.default_rng(100 * logn + elems + shift).standard_normal((batch, n)).astype(np.float32)
    e = np.fft.rfft(x.astype(np.float64), norm="ortho")
    tol = U * math.sqrt(logn + 2)
    stream = torch.cuda.current_stream().cuda_stream

    plan = _plan(n, batch, "r2c", elems)
    xin = torch.from_numpy(x).to(gpu)
    buf = torch.full((GUARD + shift + batch * m + GUARD,), 7.0 + 5.0j, dtype=torch.complex64, device=gpu)
    first = GUARD + shift
    plan.execute(xin.data_ptr(), buf[first:].data_ptr(), stream)
    torch.cuda.synchronize()
    got = buf.cpu().numpy()
    assert np.all(got[:first] == 7 + 5j) and np.all(got[first + batch * m:] == 7 + 5j)
    got = got[first:first + batch * m].reshape(batch, m)
    for r in range(batch):
        assert np.linalg.norm(got[r] - e[r]) <= tol * np.linalg.norm(e[r]), r

    plan = _plan(n, batch, "c2r", elems)
    spec = np.full((GUARD + shift + batch * m + GUARD,), np.nan + 1j * np.nan, dtype=np.complex64)
    bins = e.astype(np.complex64)
    bins[:, 0] += 3j  # the imaginary parts of bins 0 and n/2 are ignored
    bins[:, -1] -= 2j
    spec[first:first + batch * m] = bins.reshape(-1)
    sin = torch.from_numpy(spec).to(gpu)
    out = torch.full((batch * n + GUARD,), 7.0, dtype=torch.float32, device=gpu)
    plan.execute(sin[first:].data_ptr(), out.data_ptr(), stream)
    torch.cuda.synchronize()
    back = out.cpu().numpy()
    assert np.all(back[batch * n:] == 7.0)
    back = back[:batch * n].reshape(batch, n)
    for r in range(batch):
        assert np.linalg.norm(back[r] - x[r]) <= (tol + U) * np.linalg.norm(x[r]), r  # + the bins' own rounding


@pytest.mark.parametrize("kind", ["r2c", "c2r"])
@pytest.mark.parametrize("logn", [14, 15])
def test_default_kernel_is_the_same_at_every_batch(gpu, logn, kind):
    """Without an element count a row comes from the same kernel, so with the
    same bits, whatever the batch around it."""
    import torch

    n, batch = 1 << logn, 1 << (24 - logn)
    shape = (batch, n) if kind == "r2c" else (batch, n + 2)  # a row of samples, or of n/2 + 1 bins
    x = torch.from_numpy(np.random.default_rng(logn).standard_normal(shape).astype(np.float32)).to(gpu)
    stream = torch.cuda.current_stream().cuda_stream
    rows, elems = [], []
    for b in (1, batch):
        plan = native.NativePlan(n, b, kind, "forward" if kind == "r2c" else "inverse", norm="ortho",
                                 flow=native.FLOW_LDS_FUSED)
        out = torch.empty((b, n + 2 if kind == "r2c" else n), dtype=torch.float32, device=gpu)
        plan.execute(x.data_ptr(), out.data_ptr(), stream)
        torch.cuda.synchronize()
        rows.append(out[0].clone())
        elems.append(plan.info.elems_per_thread)
    assert elems[0] == elems[1], elems
    assert torch.equal(rows[0], rows[1])


# the lane-paired r2c kernels that store whole lines in large launches, and the
# first batch that does: 2^22 samples, past 2^25 at a core of 2^13
LINE_CASES = [(10, 8, 4096), (11, 16, 2048), (12, 16, 1024), (13, 8, 512), (13, 16, 512), (14, 16, 2049)]


@pytest.mark.parametrize("extra,shift", [(-1, 0), (0, 1), (3, 15)])
@pytest.mark.parametrize("logn,elems,first_batch", LINE_CASES)
def test_bin_rows_of_a_large_launch(gpu, logn, elems, first_batch, extra, shift):
    """One row below the launch size from which bins go out in whole lines, at
    it, and a ragged batch above it: every row has the bits that small launches
    give, and those of the edges and some between are right."""
    import torch

    n, m = 1 << logn, (1 << (logn - 1)) + 1
    batch = first_batch + extra
    stream = torch.cuda.current_stream().cuda_stream
    gen = torch.Generator(device=gpu)
    gen.manual_seed(100 * logn + elems)
    x = torch.randn((batch, n), device=gpu, generator=gen)
    first = GUARD + shift
    buf = torch.full((first + batch * m + GUARD,), 7.0 + 5.0j, dtype=torch.complex64, device=gpu)
    large = _plan(n, batch, "r2c", elems)
    large.execute(x.data_ptr(), buf[first:].data_ptr(), stream)
    small = torch.empty((batch, m), dtype=torch.complex64, device=gpu)
    plans = []
    for r in range(0, batch, 256):
        plans.append(_plan(n, min(256, batch - r), "r2c", elems))
        plans[-1].execute(x[r:].data_ptr(), small[r:].data_ptr(), stream)
    torch.cuda.synchronize()
    got = buf[first:first + batch * m].view(batch, m)
    assert torch.equal(torch.view_as_real(got), torch.view_as_real(small))
    assert torch.all(buf[:first] == 7 + 5j) and torch.all(buf[first + batch * m:] == 7 + 5j)
    rows = [0, 1, 2, 3, 4, batch // 3, batch // 2, batch - 5, batch - 4, batch - 3, batch - 2, batch - 1]
    e = np.fft.rfft(x[rows].cpu().numpy().astype(np.float64), norm="ortho")
    y = got[rows].cpu().numpy()
    assert np.all(np.linalg.norm(y - e, axis=1) <= U * math.sqrt(logn + 2) * np.linalg.norm(e, axis=1))
