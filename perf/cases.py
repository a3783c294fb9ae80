"""The transforms whose time is measured, as a user's program runs them.

A program plans once (``plan_fft`` with the device profile, so the measured
selector table chooses the kernels), keeps the plan, and calls
``execute_fft_plan`` on tensors that are already on the GPU.  ``run`` is one
such call (for ``real_round_trip`` the forward and the inverse call after each
other); planning and the inputs are ``prepare``.

Range: every transform the library runs, power-of-two N from 16 to 2^20, C2C
forward and inverse, R2C and C2R, the four norms, batches of any size from one
transform to 2^26 points per call.
"""
from __future__ import annotations

import math

import torch

import __graft_entry__

_PKG = __graft_entry__.load_package()

MIN_LOG_N, MAX_LOG_N = 4, 20
MAX_LOG_POINTS = 26  # 2^26 points: 512 MiB of complex64 in and out


def _case(kind: str, n: int, batch: int, norm: str = "backward", name: str | None = None) -> dict:
    c = {"kind": kind, "n": n, "batch": batch, "norm": norm}
    if name is not None:
        c["name"] = name
    return c


def listed() -> list:
    return [
        # one short transform at a time, waited for: interactive use, control
        # loops; the benchmark's latency row
        _case("c2c_forward", 2048, 1, name="c2c_n2048_b1"),
        # a small batch of short transforms (a block of audio or radar channels)
        _case("c2c_forward", 1024, 64, name="c2c_n1024_b64"),
        # spectral filtering of a few real signals: spectrum and back
        _case("real_round_trip", 4096, 64, name="real_round_trip_n4096_b64"),
        # one long transform (a whole capture)
        _case("c2c_forward", 1 << 20, 1, name="c2c_n2p20_b1"),
        # very many very short transforms, a ragged batch (per-pixel, per-window spectra)
        _case("c2c_forward", 64, 100003, name="c2c_n64_b100003"),
        # the throughput row: a batch past the caches, one pass over memory
        _case("c2c_forward", 4096, 8192, name="c2c_n4096_b8192"),
        # a medium batch of medium transforms: one workgroup per compute unit
        _case("c2c_inverse", 16384, 256, name="c2c_inverse_n16384_b256"),
        # the longest single-pass transform, a batch that is not a power of two
        _case("c2c_inverse", 32768, 1000, "ortho", name="c2c_inverse_ortho_n32768_b1000"),
        # a batch of long transforms, two passes over memory
        _case("c2c_forward", 65536, 256, name="c2c_n65536_b256"),
        # the longest transform, in batches: the largest call
        _case("c2c_forward", 1 << 20, 64, name="c2c_n2p20_b64"),
        # long real signals to half spectra, single pass
        _case("r2c", 16384, 4096, name="r2c_n16384_b4096"),
        # half spectra of very long signals back to samples, two passes
        _case("c2r", 1 << 18, 256, name="c2r_n2p18_b256"),
    ]


def draw(rng) -> dict:
    """One more case: N uniform over its powers of two, the batch spread over
    its logarithm up to 2^26 points, forward C2C as often as everything else."""
    kind = rng.choice(["c2c_forward", "c2c_forward", "c2c_forward", "c2c_inverse", "r2c", "c2r", "real_round_trip"])
    log_n = rng.randint(MIN_LOG_N, MAX_LOG_N)
    log_b = rng.uniform(0.0, MAX_LOG_POINTS - log_n)
    batch = max(1, int(2.0 ** log_b))
    norm = rng.choice(["backward", "backward", "ortho", "forward", "none"])
    if kind == "real_round_trip":
        batch = max(1, batch // 2)  # two transforms a pass
        norm = rng.choice(["backward", "ortho", "forward"])
    return _case(kind, 1 << log_n, batch, norm)


def _shape(batch: int, last: int) -> tuple:
    return (last,) if batch == 1 else (batch, last)


def _input(case: dict, seed: int) -> torch.Tensor:
    """iid N(0, 1) samples (real and imaginary parts); a C2R input is a half
    spectrum of such bins, its edge bins real as a real signal's are."""
    n, b, kind = case["n"], case["batch"], case["kind"]
    dev = torch.device("cuda", torch.cuda.current_device())
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    if kind in ("r2c", "real_round_trip"):
        return torch.randn(_shape(b, n), generator=g, device=dev, dtype=torch.float32)
    last = n // 2 + 1 if kind == "c2r" else n
    x = torch.view_as_complex(torch.randn(_shape(b, last) + (2,), generator=g, device=dev, dtype=torch.float32))
    if kind == "c2r":
        x.imag[..., 0] = 0.0
        x.imag[..., -1] = 0.0
    return x


def _plan(case: dict, kind: str):
    ttype, direction = {"c2c_forward": ("c2c", "forward"), "c2c_inverse": ("c2c", "inverse"),
                        "r2c": ("r2c", "forward"), "c2r": ("c2r", "inverse")}[kind]
    return _PKG.plan_fft("dit", case["n"], batch=case["batch"], profile_hash=_PKG.DeviceProfile.load().hash(),
                         transform_type=ttype, transform_direction=direction, norm=case["norm"])


def prepare(case: dict, seed: int) -> dict:
    kinds = ("r2c", "c2r") if case["kind"] == "real_round_trip" else (case["kind"],)
    return {"x": _input(case, seed), "plans": [_plan(case, k) for k in kinds]}


def run(state: dict):
    x = state["x"]
    outs = []
    for plan in state["plans"]:
        x = _PKG.execute_fft_plan(plan, x)
        outs.append(x)
    return outs


def work(case: dict) -> dict:
    """Input read once and output written once per transform; 5 N log2 N
    operations per complex transform and half of that per real one."""
    n, b, kind = case["n"], case["batch"], case["kind"]
    if kind in ("c2c_forward", "c2c_inverse"):
        return {"bytes": 16 * n * b, "flops": 5 * n * math.log2(n) * b}
    one = {"bytes": (4 * n + 8 * (n // 2 + 1)) * b, "flops": 2.5 * n * math.log2(n) * b}
    return one if kind != "real_round_trip" else {k: 2 * v for k, v in one.items()}


def tolerance(case: dict) -> dict:
    """About four times the error of the 32-bit transforms against 64 bits:
    measured 0.8e-7 to 2.2e-7 in the 2-norm; the largest single difference
    grows with the number of values and the transform length."""
    return {"rel": 8e-7, "max": 8e-6}


_EXACT = {
    "c2c_forward": lambda x, n, norm: torch.fft.fft(x, norm=norm),
    "c2c_inverse": lambda x, n, norm: torch.fft.ifft(x, norm=norm),
    "r2c": lambda x, n, norm: torch.fft.rfft(x, norm=norm),
    "c2r": lambda x, n, norm: torch.fft.irfft(x, n=n, norm=norm),
}


def exact(case: dict, seed: int):
    x = _input(case, seed).cpu()
    x = x.to(torch.complex128 if x.is_complex() else torch.float64)
    n, norm, kind = case["n"], case["norm"], case["kind"]
    kinds = ("r2c", "c2r") if kind == "real_round_trip" else (kind,)
    outs = []
    for k in kinds:
        # "none" scales neither direction
        named = norm if norm != "none" else ("forward" if k in ("c2c_inverse", "c2r") else "backward")
        x = _EXACT[k](x, n, named)
        outs.append(x)
    return outs
