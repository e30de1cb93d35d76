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
