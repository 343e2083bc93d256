"""GPU: clmi_field_stats_noalloc where its kernel cannot take two z-neighbours at a time: odd sides, whose pairs would
straddle rows, and arrays aligned to one double only.  The oracle is numpy in FP64.

Tolerance: every sum is of at most 65^3 terms, added in chains of a few sites per thread, then by lane, wave and row
(fewer than 200 dependent additions of values of one sign, 2^-53 each, and a few roundings per term): 1e-13 relative."""
import numpy as np
import pytest

from test_gpu_parity import say

pytestmark = pytest.mark.gpu


# the smallest sides, odd ones below and above one workgroup's sites, and even ones for the offset alone
@pytest.mark.parametrize("N,offset", [(2, 0), (3, 0), (5, 0), (7, 1), (33, 0), (33, 1), (65, 0), (2, 1), (32, 1), (64, 1)])
def test_field_stats_of_odd_sides_and_unaligned_arrays(gpu, N, offset):
    import torch

    say(f"case field stats forms N={N} offset={offset}")
    dx = 0.37
    f = 0.9 + 0.3 * np.random.default_rng(N).standard_normal((N, N, N))
    buf = torch.zeros(N ** 3 + offset, dtype=torch.float64, device="cuda")
    buf[offset:] = torch.from_numpy(f.ravel()).to("cuda")
    out = torch.full((3,), float("nan"), dtype=torch.float64, device="cuda")
    stream = torch.cuda.current_stream()
    gpu.field_stats_noalloc(buf.data_ptr() + 8 * offset, N, dx, out.data_ptr(), stream.cuda_stream)
    stream.synchronize()
    grad = sum(float(np.mean((np.roll(f, -1, ax) - f) ** 2)) for ax in range(3)) / dx ** 2
    for got, want in zip(out.cpu().numpy(), (float(np.mean(f)), float(np.mean(f * f)), grad)):
        assert float(got) == pytest.approx(want, rel=1e-13)
