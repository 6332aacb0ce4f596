"""The bf16 GEMM's kernels (small, split, 64 and 128 tiles), the streaming GEMVs beside them and
the two-launch norm-router at the sizes where they can go wrong: K of 32 and with half-filled
last steps, single and odd outputs, token counts at the edges of the tiles and of the dispatch.

References are float64 on the same bf16 operands. Bounds: an fp32 sum of K exact products in
any order is within K * 2^-24 * sum |x w| of it; rounding to bf16 (8 significant bits) moves a
value by at most 2^-8 of it, which the MLP does to act and to y (2^-12 more is allowed for the
fp32 sums, exp and reciprocal below them).
"""
import pytest
import torch

import whallm_amd as wa

pytestmark = pytest.mark.gpu


def bf16(g, *shape, std=1.0):
    return (torch.randn(*shape, device="cuda", generator=g) * std).to(torch.bfloat16)


def check_sums(got, x, w):
    x, w = x.double(), w.double()
    bound = (x.shape[1] + 8) * 2.0 ** -24 * (x.abs() @ w.abs().T)
    assert bool(((got.double() - x @ w.T).abs() <= bound).all())


# kernel for kernel: GEMV (<= 4 tokens), small, a wave per output and either side of its line, split, 64 x 64 tiles,
# 128 x 128 tiles
@pytest.mark.parametrize("T,K,N", [(1, 32, 1), (4, 2080, 33), (3, 1032, 4097), (2, 512, 65), (2, 520, 65),
                                   (5, 32, 1), (16, 96, 513), (17, 2592, 512), (64, 2048, 77),
                                   (17, 32, 1), (63, 1056, 65), (6000, 32, 4), (57, 8192, 32), (58, 8192, 32), (65536, 32, 1),
                                   (33, 32, 1000), (129, 160, 640), (300, 416, 520),
                                   (65, 96, 4100), (600, 2592, 517), (2049, 32, 130),
                                   (4097, 96, 1001), (8, 224, 33000)])
def test_linear_edges(T, K, N):
    g = torch.Generator(device="cuda")
    g.manual_seed(T * 7 + K + N)
    x, w = bf16(g, T, K), bf16(g, N, K)
    check_sums(wa.linear_bf16(x, w), x, w)


@pytest.mark.parametrize("T,H,I", [(1, 32, 32), (2, 2592, 96), (4, 2048, 2080), (5, 32, 32), (5, 1056, 544),
                                   (3, 544, 1056), (6, 544, 32), (33, 96, 160), (63, 2080, 640),
                                   (129, 288, 96), (700, 96, 544), (2049, 1056, 2080)])
@pytest.mark.parametrize("gated", [True, False])
def test_mlp_edges(T, H, I, gated):
    g = torch.Generator(device="cuda")
    g.manual_seed(T + H + I)
    x, add = bf16(g, T, H), bf16(g, T, H) if gated else None
    wg, wu, wd = bf16(g, I, H, std=H ** -0.5), bf16(g, I, H, std=H ** -0.5), bf16(g, H, I, std=I ** -0.5)
    gv = bf16(g, H, std=0.02) if gated else None
    got = wa.mlp_bf16(x, wg, wu, wd, gv, add).double()
    xd = x.double()
    act = torch.nn.functional.silu(xd @ wg.double().T) * (xd @ wu.double().T)
    gate = torch.sigmoid(xd @ gv.double())[:, None] if gated else 1.0
    want = gate * (act @ wd.double().T) + (add.double() if gated else 0.0)
    bound = (2.0 ** -8 + 2.0 ** -12) * (want.abs() + gate * (act.abs() @ wd.double().abs().T)) + 1e-6
    assert bool(((got - want).abs() <= bound).all())


@pytest.mark.parametrize("T,H,E,gated", [(7, 2048, 64, True), (8, 2048, 65, True), (15, 4128, 33, False), (16, 4128, 33, True),
                                         (40, 1024, 512, True), (301, 1056, 130, True), (9, 40, 16, True),
                                         (20, 10240, 32, True), (17, 10272, 16, True), (129, 9600, 64, True), (96, 9600, 64, True),
                                         (33, 9600, 256, False)])
def test_norm_router_edges(T, H, E, gated):
    g = torch.Generator(device="cuda")
    g.manual_seed(T + H + E)
    r, y = torch.randn(T, H, device="cuda", generator=g), bf16(g, T, H)
    w, gate, nw = bf16(g, E, H), bf16(g, H) if gated else None, bf16(g, H)
    v = torch.empty_like(r)
    x, logits, shared = wa.norm_router(r, y, w, gate, nw, 1e-6, v)
    want_v = r + y.float()
    assert torch.equal(v, want_v)
    vd = want_v.double()
    want_x = vd * torch.rsqrt(vd.square().mean(-1, keepdim=True) + 1e-6) * nw.double()
    # bf16 rounding (2^-8) and the fp32 sum of squares, root and products (H 2^-24 of the sum)
    assert bool(((x.double() - want_x).abs() <= (2.0 ** -8 + H * 2.0 ** -24) * 1.01 * want_x.abs()).all())
    check_sums(logits, x, w)  # from the x it returned
    if gated:
        check_sums(shared[:, None], x, gate[None])
