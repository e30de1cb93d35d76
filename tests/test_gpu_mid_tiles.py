"""The staged 128 x 128 NF4 GEMMs (batches too small for the 256 x 256 ones) at the edges of their own tiles, against the
fp64 oracle. Each case first asserts that its workspace is the one these kernels ask for: the GEMM queries exceed the
plain ones exactly where they are taken and stage more than the other kernels would."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import nf4_oracle as O
from tests._util import assert_close_fro, bf16_values, np_f32, oracle_weight, seeded, uniform

import molt_amd
from molt_amd import _lib, ops

pytestmark = pytest.mark.gpu


def _weight(n, k, seed):
    packed, qs = molt_amd.quantize_4bit(seeded((n, k), seed, std=0.02, dtype=torch.float32))
    return packed.reshape(-1), molt_amd.resolved_nf4_scales(qs), qs, oracle_weight(packed, qs).dequant_bf16().astype(np.float64)


def _adapter(n, r, seed):
    """fp32 masters that bf16(2 B) rounds exactly as bf16(B) does."""
    return seeded((n, r), seed, std=0.01, dtype=torch.float32)


@pytest.mark.parametrize("r", [8, 24, 48])
def test_infinite_low_rank_value_stays_infinite(r):
    """An infinite T (U) entry makes its row of outputs infinite with the adapter's signs, not NaN: the ring's step of
    64 holds zero adapter rows past a shorter rank, which the row's own columns must not meet."""
    print(f"mid infinite T r={r}", flush=True)
    m, n, k = 130, 200, 3072
    packed, scales, qs, _ = _weight(n, k, 70)
    x, t, b = seeded((m, k), 71), seeded((m, r), 72), _adapter(n, r, 73)
    args = (packed, scales, qs.code, n, k, 1, 64)
    y = ops.nf4_lora_forward(x, *args, t, b, 2.0)
    t[3, r - 1] = float("inf")
    bad = ops.nf4_lora_forward(x, *args, t, b, 2.0)
    keep = [i for i in range(m) if i != 3]
    assert torch.equal(bad[keep], y[keep]) and torch.equal(bad[3].float(), b[:, r - 1].sign() * float("inf"))
    m, n, k = 70, 192, 320
    packed, scales, qs, _ = _weight(n, k, 74)
    dy, u, a = seeded((m, n), 75), seeded((m, r), 76), uniform((r, k), 77, 1.0 / np.sqrt(k))
    args = (packed, scales, qs.code, n, k, 1, 64)
    dx = ops.nf4_lora_backward_input(dy, *args, u, a, 1.0)
    u[3, 0] = float("-inf")
    bad = ops.nf4_lora_backward_input(dy, *args, u, a, 1.0)
    keep = [i for i in range(m) if i != 3]
    assert torch.equal(bad[keep], dx[keep]) and torch.equal(bad[3].float(), a[0].sign() * float("-inf"))


def test_low_rank_rows_far_apart():
    """U rows whose stride puts the last one past 4 GiB: past the reach of the DMA's 32-bit offsets, so the call takes
    the kernel that addresses them in 64 bits."""
    m, n, k, r, ld = 70, 192, 320, 16, 32 * 1024 * 1024 + 8
    (p0, s0, qs, w0), (p1, s1, _, w1) = _weight(n, k, 80), _weight(n, k, 81)
    u = torch.empty((m - 1) * ld + 2 * r, device="cuda", dtype=torch.bfloat16).as_strided((m, 2 * r), (ld, 1))
    u.copy_(seeded((m, 2 * r), 82))
    dy0, dy1 = seeded((m, n), 83), seeded((m, n), 84)
    a0, a1 = uniform((r, k), 85, 1.0 / np.sqrt(k)), uniform((r, k), 86, 1.0 / np.sqrt(k))
    dx = ops.nf4_lora_backward_input_pair(dy0, dy1, p0, s0, p1, s1, qs.code, n, k, 1, u[:, :r], u[:, r:], a0, a1)
    uu = bf16_values(u)
    ref = bf16_values(dy0) @ w0 + bf16_values(dy1) @ w1 + uu[:, :r] @ bf16_values(a0) + uu[:, r:] @ bf16_values(a1)
    assert_close_fro(np_f32(dx), ref, what="dX")
