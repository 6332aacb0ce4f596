"""The grouped GEMM's row tiles of 128, 64 and 16 rows give the same rows: a call whose experts have
few rows against the same tokens in a longer call that gives every expert more than 64 rows (tiles
of 128 rows, which test_gpu_moe.py and test_gpu_fp8.py hold against the oracle).

Row counts at the edges of the tiles, K of an even and odd number of 128-wide steps, a last column tile
of half its width, both layouts, a slot map with an expert that is not resident, ids out of range.
All take the same products in the same order, so a row's bits do not depend on the tile that held it.
The second test has more 64-row tiles than an XCD's 32 workgroups, so that each goes from tile to tile, over an odd
number of K steps (its last weight unit is half of one), and with hot experts also through the tiles that
the workgroups without a 128-row tile take first and the rest after them.
"""
import numpy as np
import pytest
import torch

import whallm_amd as wa
from whallm_amd import synthetic as S

pytestmark = pytest.mark.gpu

EDGES = [1, 15, 16, 17, 63, 64, 65, 129]  # rows of the first experts, one choice a token
CALLS = {  # tokens, choices, experts
    "edges": (370, 1, 32),         # 64- and 128-row tiles
    "edges-sparse": (370, 1, 64),  # MXFP4: 16-row tiles (5.8 rows an expert)
    "even": (40, 8, 16),           # 20 rows an expert, the shared expert's 40 in one 64-row tile
    "even-sparse": (33, 8, 64),    # MXFP4: 4.1 rows an expert in 16-row tiles
}
FORMS = ["mxfp4", "fp8-128", "fp8-32"]


def tables(form, rng, device, n, hidden, inter, **kw):
    if form == "mxfp4":
        return S.experts_to_device(S.mxfp4_experts_np(rng, n, hidden, inter), device, **kw)
    return S.fp8_experts_to_device(S.fp8_experts_np(rng, n, hidden, inter, scale_format=int(form == "fp8-32")), device, **kw)


MANY = {  # tokens, choices, experts, Zipf exponent
    "even": (100, 8, 64, 0.0),       # 320 tiles of 64 rows in either GEMM (MXFP4: 12.5 rows an expert)
    "skewed": (600, 8, 256, 1.1),    # about 20 experts of more than 64 rows, 230 of fewer
}


@pytest.mark.parametrize("call", sorted(MANY))
@pytest.mark.parametrize("form", FORMS)
def test_row_tiles_agree_from_tile_to_tile(device, form, call):
    T, k, E, skew = MANY[call]
    hidden, inter = 1152, 640  # 9 and 5 K steps
    rng = np.random.default_rng(T + E)
    routed, shared = tables(form, rng, device, E, hidden, inter), tables(form, rng, device, 1, hidden, inter)
    lot = rng.gumbel(size=(T, E)) - skew * np.log(np.arange(1, E + 1))  # the k largest: a draw without replacement
    ids = np.argsort(-lot, axis=1)[:, :k]
    counts = np.bincount(ids.ravel(), minlength=E)
    assert (counts <= 64).sum() * 5 > 256 and (counts > 64).any() == (skew > 0)
    more = np.stack([(np.arange(9 * E) + j * 5) % E for j in range(k)], 1)  # 72 rows for every expert
    n = T + len(more)
    x = S.bf16_bits_to_tensor(S.bf16_normal_np(rng, (n, hidden)), device)
    i = torch.from_numpy(np.concatenate([ids, more]).astype(np.int32)).to(device)
    w = torch.rand(n, k, device=device) + 0.1
    moe = wa.moe_mxfp4 if form == "mxfp4" else wa.moe_fp8
    for a, b in ((routed, shared), (wa.prefill_layout(routed), wa.prefill_layout(shared))):
        assert torch.equal(moe(x[:T], i[:T], w[:T], a, b), moe(x, i, w, a, b)[:T])


@pytest.mark.parametrize("hidden,inter", [(384, 384), (640, 384), (384, 640), (256, 256), (512, 1152)])
@pytest.mark.parametrize("call", sorted(CALLS))
@pytest.mark.parametrize("form", FORMS)
def test_row_tiles_agree(device, form, call, hidden, inter):
    T, k, E = CALLS[call]
    rng = np.random.default_rng(T + E + hidden + inter)
    deepseek = inter == 640
    kw = dict(up_first=True, swiglu_limit=10.0) if deepseek else {}
    slots = np.arange(E, dtype=np.int32)
    slots[3], slots[4] = 4, -1  # expert 4 is not resident
    routed = tables(form, rng, device, E, hidden, inter, slots=torch.from_numpy(slots).to(device), experts=E, **kw)
    plain = tables(form, rng, device, E, hidden, inter, **kw)
    shared = tables(form, rng, device, 1, hidden, inter, **kw)
    if k == 1:
        ids = rng.permutation(np.repeat(np.arange(len(EDGES)), EDGES))[:, None]
    else:
        ids = np.stack([rng.permutation(E)[:k] for _ in range(T)])
    more = np.stack([(np.arange(66 * E) + j * 5) % E for j in range(k)], 1)  # 66 rows for every expert
    ids_long = np.concatenate([ids, more]).astype(np.int32)
    n = len(ids_long)
    x = S.bf16_bits_to_tensor(S.bf16_normal_np(rng, (n, hidden)), device)
    i, w = torch.from_numpy(ids_long).to(device), torch.rand(n, k, device=device) + 0.1
    i[2, 0] = E  # its pair is left out of every list
    gate = None if deepseek else S.bf16_bits_to_tensor(S.bf16_normal_np(rng, (hidden,), 0.05), device)
    moe, experts = (wa.moe_mxfp4, wa.experts_mxfp4) if form == "mxfp4" else (wa.moe_fp8, wa.experts_fp8)
    for tab, sh in ((routed, shared), (plain, shared), (wa.prefill_layout(plain), wa.prefill_layout(shared))):
        for got, want in ((moe(x[:T], i[:T], w[:T], tab, sh, gate), moe(x, i, w, tab, sh, gate)[:T]),
                          (experts(x[:T], i[:T], tab), experts(x, i, tab)[:T])):
            assert bool(torch.isfinite(got.float()).all())
            assert torch.equal(got, want)
