"""MXFP4 calls of a few tokens (T k <= 256 pairs of experts large enough, T k H I >= 1.2e8): grouped 4-row tiles whose activations enter as eight
E4M3 terms and whose rows stay fp32, against the oracle's fp32 experts and a float64 combine.

Bounds: y is rounded to bf16 once, at most 2^-9 of each value, so 2^-9 of the result's norm; the
fp32 sums and the terms (2^-32 of a block's maximum) get 2^-13 more. Rows or act kept in
16 bits would not pass: they add 2^-9 each.
"""
import ctypes

import numpy as np
import pytest
import torch

import whallm_amd as wa
from oracle import moe as M
from whallm_amd import _lib
from whallm_amd import synthetic as S
from whallm_amd.ops import _ptr, _stream

pytestmark = pytest.mark.gpu

BOUND = 2.0 ** -9 + 2.0 ** -13


def oracle_experts(a):
    return [M.MXFP4Expert(a["gate_up"][e], a["gate_up_scales"][e], a["down"][e], a["down_scales"][e])
            for e in range(len(a["gate_up"]))]


# one row an expert and none, 4, 5, 8 and 9 rows of one expert, up to 32 of each, as many pairs as the path
# takes; K of the fewest, odd and many steps, last column tiles of half width
@pytest.mark.parametrize("T,k,E,H,I", [(32, 8, 512, 1024, 512), (25, 10, 64, 1152, 640), (32, 8, 9, 384, 1280),
                                       (16, 16, 16, 1280, 384), (9, 2, 2, 4096, 2048), (8, 1, 1, 7168, 2432), (5, 4, 4, 4096, 2048),
                                       (3, 4, 4, 5120, 2304)])
def test_few_tokens_match_oracle(device, T, k, E, H, I):
    rng = np.random.default_rng(T + k + E + H + I)
    arrays, shared_arrays = S.mxfp4_experts_np(rng, E, H, I), S.mxfp4_experts_np(rng, 1, H, I)
    x_bits, g_bits = S.bf16_normal_np(rng, (T, H)), S.bf16_normal_np(rng, (H,), 0.02)
    x_bits[:, :32] = 0                       # a block of zeros
    x_bits[T - 1, 64:96] = (x_bits[T - 1, 64:96] & 0x807f) | np.uint16(2 << 7)  # tiny values
    ids = np.stack([rng.permutation(E)[:k] for _ in range(T)]).astype(np.int32)
    w = rng.random((T, k)).astype(np.float32) + 0.1
    routed, shared = S.experts_to_device(arrays, device), S.experts_to_device(shared_arrays, device)
    x, gate = S.bf16_bits_to_tensor(x_bits, device), S.bf16_bits_to_tensor(g_bits, device)
    i_d, w_d = torch.from_numpy(ids).to(device), torch.from_numpy(w).to(device)
    xf = S.bf16_bits_to_f32(x_bits)
    rows = M.routed_outputs(xf, ids, oracle_experts(arrays))
    want = M.combine(rows, w, M.expert_ffn(xf, oracle_experts(shared_arrays)[0]),
                     xf.astype(np.float64) @ S.bf16_bits_to_f32(g_bits).astype(np.float64))

    def close(got, ref):
        ref = np.asarray(ref, dtype=np.float64)
        assert np.linalg.norm(got.double().cpu().numpy() - ref) <= BOUND * np.linalg.norm(ref)

    close(wa.moe_mxfp4(x, i_d, w_d, routed, shared, gate), want)
    close(wa.experts_mxfp4(x, i_d, routed), rows)


def test_few_tokens_slots_masks_and_replays(device):
    """Non-resident and out-of-range experts add nothing (zero rows per pair), a masked pair adds nothing and leaves
    its row of `out` as it is, and a captured call gives the same bits on every replay."""
    rng = np.random.default_rng(7)
    T, k, E, H, I = 6, 4, 12, 2560, 2048
    slots = np.arange(E, dtype=np.int32)
    slots[2], slots[5] = 5, -1
    tab = S.experts_to_device(S.mxfp4_experts_np(rng, E, H, I), device, slots=torch.from_numpy(slots).to(device), experts=E)
    x = S.bf16_bits_to_tensor(S.bf16_normal_np(rng, (T, H)), device)
    ids = np.stack([rng.permutation(E)[:k] for _ in range(T)]).astype(np.int32)
    ids[0, 0], ids[1, 1], ids[2, 2] = 5, E, -1
    live = (ids != 5) & (ids != E) & (ids >= 0)
    i_d, w_d = torch.from_numpy(ids).to(device), torch.rand(T, k, device=device) + 0.1
    per_pair = wa.experts_mxfp4(x, i_d, tab, out=torch.full((T, k, H), 3.0, dtype=torch.bfloat16, device=device))
    assert bool((per_pair[2, 2] == 3).all())
    per_pair[2, 2] = 0
    per_pair = per_pair.double()
    assert bool((per_pair[torch.from_numpy(~live).to(device)] == 0).all())
    want = (per_pair * w_d.double()[..., None]).sum(1)
    got = wa.moe_mxfp4(x, i_d, w_d, tab)
    assert (got.double() - want).norm() <= 2 * BOUND * want.norm()  # the pairs' rows are rounded too
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        wa.moe_mxfp4(x, i_d, w_d, tab)
    torch.cuda.current_stream().wait_stream(side)
    with torch.cuda.graph(graph):
        captured = wa.moe_mxfp4(x, i_d, w_d, tab)
    for _ in range(3):
        captured.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured, got)
        assert torch.equal(wa.moe_mxfp4(x, i_d, w_d, tab), got)


def test_few_tokens_hold_act_in_32_bits(device):
    """Act enters the down product as fp32 holds it, also beside a value 2^16 times as large in its 32-value block:
    columns 32 n of gate_up carry 2^8 times the weights (gate and up) and none in down, so y is made
    of the others. The terms leave at most 2^-32 of the block's maximum, 2^-16 of those."""
    rng = np.random.default_rng(24)
    T, k, E, H, I = 6, 4, 8, 2560, 2048
    a = S.mxfp4_experts_np(rng, E, H, I)
    for base in (0, I):
        a["gate_up_scales"][:, base:base + I:32] += 8
    a["down"][..., ::4] &= ~a["down"].dtype.type(15)
    tab = S.experts_to_device(a, device)
    x_bits = S.bf16_normal_np(rng, (T, H))
    ids = np.stack([rng.permutation(E)[:k] for _ in range(T)]).astype(np.int32)
    got = wa.experts_mxfp4(S.bf16_bits_to_tensor(x_bits, device), torch.from_numpy(ids).to(device), tab)
    want = np.asarray(M.routed_outputs(S.bf16_bits_to_f32(x_bits), ids, oracle_experts(a)), dtype=np.float64)
    err = np.linalg.norm(got.double().cpu().numpy() - want, axis=-1) / np.linalg.norm(want, axis=-1)
    assert err.max() <= BOUND + 2.0 ** -16


@pytest.mark.parametrize("T,k,E,H,I", [(8, 10, 64, 2560, 640), (16, 8, 32, 4096, 2048)])
def test_few_tokens_sum_in_32_bits(device, T, k, E, H, I):
    """Rows are the 64-bit results' bf16 roundings but for about 1 in 2,000. A result off by r of its value before
    the rounding takes its neighbour with probability r 2^7 / ln 2 (bf16's steps are 2^-7 of the power of two below
    the value); fp32 sums and __expf leave r near 2^-19, 4e-4 of the values, and 2^-17.5 is the bound: 1e-3.
    Sums in 14 bits pass the norms above and fail here (1.4e-2). x spans 2^6 within its blocks."""
    rng = np.random.default_rng(H + I)
    a = S.mxfp4_experts_np(rng, E, H, I)
    x = (rng.standard_normal((T, H)) * 2.0 ** rng.integers(-6, 1, (T, H))).astype(np.float32)
    x = torch.from_numpy(x).to(torch.bfloat16)
    ids = np.stack([rng.permutation(E)[:k] for _ in range(T)]).astype(np.int32)
    got = wa.experts_mxfp4(x.to(device), torch.from_numpy(ids).to(device), S.experts_to_device(a, device))
    lut = np.array([0, .5, 1, 1.5, 2, 3, 4, 6, 0, -.5, -1, -1.5, -2, -3, -4, -6])

    def weights(words, scales):
        b = np.ascontiguousarray(words).view(np.uint8)
        v = np.stack([lut[b & 15], lut[b >> 4]], -1).reshape(words.shape[0], -1)
        return v * np.repeat(2.0 ** (scales.astype(np.float64) - 127), 32, axis=1)

    xd, off, n = x.double().numpy(), 0, 0
    for e in np.unique(ids):
        t, j = np.nonzero(ids == e)
        gu = xd[t] @ weights(a["gate_up"][e], a["gate_up_scales"][e]).T
        g, u = gu[:, :I], gu[:, I:]
        with np.errstate(over="ignore"):
            want = (g / (1 + np.exp(-g)) * u) @ weights(a["down"][e], a["down_scales"][e]).T
        rounded = torch.from_numpy(want).to(torch.float32).to(torch.bfloat16)
        off += int((got[t, j].cpu() != rounded).sum())
        n += rounded.numel()
    assert off <= 1e-3 * n, off / n


def test_few_tokens_read_nothing_for_what_is_not_resident(device):
    """With no expert resident, routed or shared, the call adds nothing and computes nothing: its act and output
    rows in the workspace stay untouched (every byte of the rows, 4 H T (k + 1), and more)."""
    rng = np.random.default_rng(3)
    T, k, E, H, I = 6, 4, 12, 2560, 2048
    gone = torch.full((E,), -1, dtype=torch.int32, device=device)
    tab = S.experts_to_device(S.mxfp4_experts_np(rng, E, H, I), device, slots=gone, experts=E)
    shared = S.experts_to_device(S.mxfp4_experts_np(rng, 1, H, I), device, slots=gone[:1], experts=1)
    x = S.bf16_bits_to_tensor(S.bf16_normal_np(rng, (T, H)), device)
    ids = torch.from_numpy(np.stack([rng.permutation(E)[:k] for _ in range(T)]).astype(np.int32)).to(device)
    w = torch.rand(T, k, device=device) + 0.1
    c, sc = tab.c_struct(), shared.c_struct()
    nbytes = _lib.load().wm_moe_mxfp4_workspace_size(T, k, ctypes.byref(c))
    ws = torch.full((nbytes,), 0x5a, dtype=torch.uint8, device=device)
    y = torch.full_like(x, 3.0)
    _lib.call("wm_moe_mxfp4", _ptr(x), T, _ptr(ids), _ptr(w), k, ctypes.byref(c), ctypes.byref(sc), None, _ptr(y),
              _ptr(ws), nbytes, _stream(device))
    torch.cuda.synchronize()
    assert bool((y == 0).all())
    assert int((ws == 0x5a).sum()) >= 4 * H * T * (k + 1) + 2 * I * T * (k + 1)


@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf")])
def test_few_tokens_keep_what_is_not_finite_to_its_token(device, value):
    """A NaN or an infinity in x makes its own token's results NaN, as in 64 bits (an infinity meets weights of
    both signs and zeros), and changes no bit of the others', in rows of the same tiles."""
    rng = np.random.default_rng(11)
    T, k, E, H, I = 8, 4, 6, 2560, 2048
    tab, shared = (S.experts_to_device(S.mxfp4_experts_np(rng, n, H, I), device) for n in (E, 1))
    x = S.bf16_bits_to_tensor(S.bf16_normal_np(rng, (T, H)), device)
    i = torch.from_numpy(np.stack([rng.permutation(E)[:k] for _ in range(T)]).astype(np.int32)).to(device)
    w = torch.rand(T, k, device=device) + 0.1
    bad = x.clone()
    bad[3, 100] = value
    rest = [t for t in range(T) if t != 3]
    for got, want in ((wa.moe_mxfp4(bad, i, w, tab, shared), wa.moe_mxfp4(x, i, w, tab, shared)),
                      (wa.experts_mxfp4(bad, i, tab), wa.experts_mxfp4(x, i, tab))):
        assert torch.equal(got[rest], want[rest])
        assert bool(got[3].isnan().all())
