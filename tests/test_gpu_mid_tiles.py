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


# row tails of 128, column tails of 64 and of N % 64 != 0, short, whole and no ranks, one range and several
@pytest.mark.parametrize("m,n,k,r", [(70, 72, 256, 16), (130, 200, 3072, 8), (400, 1544, 3072, 64), (300, 320, 4096, 48),
                                     (129, 264, 4096, 0), (70, 1000, 256, 128)])
def test_forward(m, n, k, r):
    print(f"mid forward m={m} n={n} k={k} r={r}", flush=True)
    lib = _lib.load()
    assert lib.molt_nf4_gemm_forward_workspace(m, n, k, r, 1) > lib.molt_nf4_lora_forward_workspace(m, n, k, r)
    packed, scales, qs, wo = _weight(n, k, 20)
    x, t, b = seeded((m, k), 21), seeded((m, r), 22) if r else None, _adapter(n, r, 23) if r else None
    args = (packed, scales, qs.code, n, k, 1, 64)
    y = ops.nf4_lora_forward(x, *args, t, b, 2.0)
    assert torch.equal(y, ops.nf4_lora_forward(x, *args, t, b, 2.0))
    ref = bf16_values(x) @ wo.T
    if r:
        ref = ref + 2.0 * (bf16_values(t) @ bf16_values(b).T)
    assert_close_fro(np_f32(y), ref, what="Y")


@pytest.mark.parametrize("m,n,k,r", [(70, 72, 512, 16), (130, 200, 1024, 8), (300, 1096, 512, 24), (200, 584, 1536, 64),
                                     (257, 64, 2048, 0)])
def test_gate_up_forward(m, n, k, r):
    print(f"mid gate/up m={m} n={n} k={k} r={r}", flush=True)
    lib = _lib.load()
    assert lib.molt_nf4_gemm_forward_workspace(m, n, k, r, 2) > lib.molt_nf4_gateup_forward_workspace(m, n, k, r)
    (pg, sg, qs, wg), (pu, su, _, wu) = _weight(n, k, 30), _weight(n, k, 31)
    x, t = seeded((m, k), 32), seeded((m, 2 * r), 33) if r else None
    bg, bu = (_adapter(n, r, 34), _adapter(n, r, 35)) if r else (None, None)
    gate, up, h = ops.nf4_gateup_forward(x, pg, sg, pu, su, qs.code, n, k, 1, t, bg, bu, 2.0, 0.5)
    rg, ru = bf16_values(x) @ wg.T, bf16_values(x) @ wu.T
    if r:
        tt = bf16_values(t)
        rg, ru = rg + 2.0 * (tt[:, :r] @ bf16_values(bg).T), ru + 0.5 * (tt[:, r:] @ bf16_values(bu).T)
    assert_close_fro(np_f32(gate), rg, what="gate")
    assert_close_fro(np_f32(up), ru, what="up")
    # h from the stored gate and up: its own rounding only
    assert_close_fro(np_f32(h), O.swiglu_forward(np_f32(gate).astype(np.float64), np_f32(up).astype(np.float64)), what="h")


# Kw % 256 != 0 and % 128 != 0 (a column tile of 64), one range and several; n % 64 != 0: the padded copies
@pytest.mark.parametrize("m,n,k,r", [(70, 192, 320, 16), (70, 192, 64, 8), (520, 192, 4096, 64), (700, 192, 576, 24),
                                     (300, 192, 1088, 0), (90, 136, 320, 16)])
def test_input_gradient(m, n, k, r):
    print(f"mid dX m={m} n={n} k={k} r={r}", flush=True)
    lib = _lib.load()
    assert lib.molt_nf4_gemm_backward_workspace(m, n, k, r, 1, 0) > lib.molt_nf4_lora_backward_workspace(m, n, k, 1)
    packed, scales, qs, wo = _weight(n, k, 40)
    dy, u = seeded((m, n), 41), seeded((m, r), 42) if r else None
    a = uniform((r, k), 43, 1.0 / np.sqrt(k)) if r else None
    dx = ops.nf4_lora_backward_input(dy, packed, scales, qs.code, n, k, 1, 64, u, a, 1.0)
    ref = bf16_values(dy) @ wo
    if r:
        ref = ref + bf16_values(u) @ bf16_values(a)
    assert_close_fro(np_f32(dx), ref, what="dX")


@pytest.mark.parametrize("m,n,k,r", [(70, 192, 320, 16), (130, 576, 576, 24), (520, 192, 4096, 8), (400, 576, 192, 64),
                                     (90, 200, 320, 8)])
def test_paired_input_gradient(m, n, k, r):
    """Both segments, whole and split between ranges that end inside one."""
    print(f"mid paired dX m={m} n={n} k={k} r={r}", flush=True)
    lib = _lib.load()
    assert lib.molt_nf4_gemm_backward_workspace(m, n, k, r, 2, 0) > lib.molt_nf4_lora_backward_workspace(m, n, k, 2)
    (p0, s0, qs, w0), (p1, s1, _, w1) = _weight(n, k, 50), _weight(n, k, 51)
    dy0, dy1, u = seeded((m, n), 52), seeded((m, n), 53), seeded((m, 2 * r), 54)
    a0, a1 = uniform((r, k), 55, 1.0 / np.sqrt(k)), uniform((r, k), 56, 1.0 / np.sqrt(k))
    dx = ops.nf4_lora_backward_input_pair(dy0, dy1, p0, s0, p1, s1, qs.code, n, k, 1, u[:, :r], u[:, r:], a0, a1)
    uu = bf16_values(u)
    ref = bf16_values(dy0) @ w0 + bf16_values(dy1) @ w1 + uu[:, :r] @ bf16_values(a0) + uu[:, r:] @ bf16_values(a1)
    assert_close_fro(np_f32(dx), ref, what="dX")


@pytest.mark.parametrize("m,n,k,r", [(70, 192, 320, 16), (300, 192, 1088, 8), (130, 192, 192, 64), (90, 72, 320, 16)])
def test_swiglu_backward(m, n, k, r):
    print(f"mid swiglu backward m={m} n={n} k={k} r={r}", flush=True)
    lib = _lib.load()
    assert lib.molt_nf4_gemm_backward_workspace(m, n, k, r, 1, 1) > lib.molt_nf4_lora_backward_workspace(m, n, k, 1)
    packed, scales, qs, wo = _weight(n, k, 60)
    dy, u, a = seeded((m, n), 61), seeded((m, r), 62), uniform((r, k), 63, 1.0 / np.sqrt(k))
    gate, up = seeded((m, k), 64), seeded((m, k), 65)
    dg, du = ops.nf4_swiglu_backward(dy, packed, scales, qs.code, n, k, 1, u, a, gate, up)
    dh = O.bf16_round(bf16_values(dy) @ wo + bf16_values(u) @ bf16_values(a)).astype(np.float64)
    rg, ru = O.swiglu_backward(bf16_values(gate), bf16_values(up), dh)
    # dh, its products and silu are each rounded to bf16 once more than the oracle's
    assert_close_fro(np_f32(dg), rg, tol=1e-2, what="dgate")
    assert_close_fro(np_f32(du), ru, tol=1e-2, what="dup")


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
