"""fp32 on the matrix cores (gemm_f32.hip, router_mfma_f32_kernel) against the
float64 oracle, at the edges of its tiles.

A dot product of K fp32 products, summed in any order, is off by at most
(K + 1) * 2^-24 * sum |w * x| (one rounding per product and per sum), so that
is the bound, element by element, with the rounding of the stored value."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import attention as oa
from oracle import moe as om

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


def _ids(rng, E, k, T, only=None):
    """Distinct experts per token; `only`: every token takes these."""
    if only is not None:
        return np.tile(np.asarray(only, np.int32)[:, None], (1, T))
    return np.stack([rng.permutation(E)[:k] for _ in range(T)], axis=1).astype(np.int32)


# (n_out, n_in, E, k, T, fixed experts): 1 to 4 groups of 16 rows and more
# than one 64-row tile; columns that fill no 16-, 32-, 64- or 128-column tile;
# one stage, an odd number of 32-input stages, and enough blocks for each tile
# width; experts without rows.
SHAPES = [
    (4, 32, 4, 1, 1, None), (36, 96, 4, 2, 3, None), (64, 64, 8, 2, 16, None), (132, 160, 3, 2, 17, None),
    (200, 64, 5, 1, 33, [2]), (64, 64, 3, 1, 90, [1]), (260, 128, 2, 1, 48, [1]), (96, 224, 4, 2, 65, [0, 3]), (1028, 96, 40, 4, 130, None),
    (2052, 64, 64, 6, 200, None), (520, 32, 16, 2, 1000, None),
]


@pytest.mark.parametrize("n_out,n_in,E,k,T,only", SHAPES)
def test_mul_mat_id_f32(fm, n_out, n_in, E, k, T, only):
    rng = np.random.default_rng(n_out * 7 + T)
    w = rng.standard_normal((n_out, n_in, E)).astype(np.float32)
    x = rng.standard_normal((n_in, k, T)).astype(np.float32)
    ids = _ids(rng, E, k, T, only)
    got = fm.mul_mat_id(torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda(), torch.from_numpy(ids).cuda())
    ref = om.mul_mat_id(w, x, ids)
    bound = (n_in + 1) * EPS * om.mul_mat_id(np.abs(w), np.abs(x), ids) + EPS * np.abs(ref)
    assert fm.lowlevel.lib().fmoe_last_gemm_path() == fm.lowlevel.PATH_TILED
    assert np.all(np.abs(got.cpu().numpy() - ref) <= bound)


# The block: SwiGLU epilogue, gathered token rows, weighted scatter; the same
# bound carried through the three products (|silu'| <= 1.1), doubled for the
# products of the two errors and the fp32 exp.
@pytest.mark.parametrize("T,H,F,E,k", [(1, 64, 36, 8, 2), (7, 96, 64, 4, 4), (70, 128, 160, 6, 3),
                                       (300, 64, 132, 40, 4), (129, 256, 1408, 64, 6)])
def test_block_f32(fm, wl, T, H, F, E, k):
    cfg = wl.Config("F32", H, F, E, k, (T,), "f32", "f32", True, 1e-6, seed=T)
    x, wr, _ = wl.router_inputs(cfg, T)
    rng = np.random.default_rng(T)
    up, gate, down = (rng.standard_normal(s).astype(np.float32) * 0.1 for s in ((F, H, E), (F, H, E), (H, F, E)))
    got = fm.moe_ffn_block(*(torch.from_numpy(a).cuda() for a in (x, wr, up, gate, down)), E, k, H, F, True)
    ref, ids, rw = om.moe_ffn_block(x, wr, up, gate, down, E, k, H, F, True, return_routing=True)
    gids, gw = fm.router(torch.from_numpy(x).cuda(), torch.from_numpy(wr).cuda(), k, True)
    np.testing.assert_array_equal(gids.cpu().numpy(), ids)
    np.testing.assert_allclose(gw.cpu().numpy(), rw, rtol=1e-5, atol=1e-7)
    bound = np.zeros_like(ref)
    ax = np.abs(x).astype(np.float64)
    for e in range(E):
        slot, tok = np.nonzero(ids == e)
        if tok.size == 0:
            continue
        u, g = x[tok] @ up[:, :, e].T.astype(np.float64), x[tok] @ gate[:, :, e].T.astype(np.float64)
        du, dg = ((H + 1) * EPS * (ax[tok] @ np.abs(m[:, :, e]).T) for m in (up, gate))
        s = u / (1 + np.exp(-u))
        dh = np.abs(s) * dg + 1.1 * np.abs(g) * du + 8 * EPS * np.abs(g * s)
        h = np.abs(g * s)
        per = dh @ np.abs(down[:, :, e]).T + (F + 4 + k) * EPS * (h @ np.abs(down[:, :, e]).T)
        np.add.at(bound, tok, per * (rw[slot, tok] * (1 + 1e-5))[:, None] + 1e-5 * rw[slot, tok][:, None] * (
            h @ np.abs(down[:, :, e]).T))
    assert np.all(np.abs(got.cpu().numpy() - ref) <= 2 * bound)


# Router: each expert-chunk count the kernel is built for and one past it,
# token counts around its 16-token blocks, odd numbers of 16-column trips.
@pytest.mark.parametrize("T,H,E,k", [(1, 16, 3, 1), (16, 48, 16, 4), (17, 400, 17, 2), (33, 2064, 33, 6),
                                     (100, 64, 64, 17), (250, 784, 65, 8), (31, 2048, 128, 8), (20, 96, 129, 4),
                                     (9, 40, 24, 2)])
def test_router_f32(fm, wl, T, H, E, k):
    cfg = wl.Config("RF", H, 64, E, k, (T,), "f32", "f32", True, 1e-6, seed=E)
    x, wr, _ = wl.router_inputs(cfg, T)
    ids, w = fm.router(torch.from_numpy(x).cuda(), torch.from_numpy(wr).cuda(), k, True)
    rids, rw = om.router(x, wr, k, True)
    np.testing.assert_array_equal(ids.cpu().numpy(), rids)
    np.testing.assert_allclose(w.cpu().numpy(), rw, rtol=1e-5, atol=1e-7)


# The block's router: partial logits of 512-column ranges of the hidden axis,
# kept in the block's y rows, then the top-k that sums them; on both sides of
# 64 tokens, with a last range of 16 and 32 columns, 5 ranges, each width of
# the top-k.  k = 1 with more ranges x experts than hidden columns: the
# partials do not fit, one kernel routes (up to 128 experts, and beyond).
@pytest.mark.parametrize("T,H,E,k", [(3, 2064, 64, 6), (64, 528, 65, 4), (65, 2064, 128, 8), (33, 544, 129, 6),
                                     (64, 2064, 16, 2), (100, 2064, 256, 8), (200, 64, 128, 1), (40, 64, 256, 1)])
def test_block_router_f32(fm, wl, T, H, E, k):
    cfg = wl.Config("RB", H, 32, E, k, (T,), "f32", "f32", True, 1e-6, seed=E)
    x, wr, _ = wl.router_inputs(cfg, T)
    dev = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    up, gate, down = (torch.zeros(s, device="cuda") for s in ((32, H, E), (32, H, E), (H, 32, E)))
    block = fm.MoEFFNBlock(dev(wr), up, gate, down, E, k, H, 32, True, act_dtype=torch.float32)
    block(dev(x))
    ids, w = block.routing()[:2]
    rids, rw = om.router(x, wr, k, True)
    np.testing.assert_array_equal(ids.cpu().numpy(), rids)
    np.testing.assert_allclose(w.cpu().numpy(), rw, rtol=1e-5, atol=1e-7)


# Attention projections: one expert's rows in order, K split into partials.
@pytest.mark.parametrize("B,n_embd,H,Hkv", [(1, 128, 2, 1), (16, 512, 4, 2), (65, 1024, 8, 8), (130, 256, 16, 2)])
def test_attention_projections_f32(fm, B, n_embd, H, Hkv):
    rng = np.random.default_rng(B)
    D = n_embd // H
    f = lambda *s: rng.standard_normal(s).astype(np.float32)  # noqa: E731
    w = [f(n_embd, n_embd), f(n_embd, Hkv * D), f(n_embd, Hkv * D), f(n_embd, n_embd)]
    w = [m * np.float32(n_embd ** -0.5) for m in w]
    x, kc, vc, pos = f(B, n_embd), f(B, 5, Hkv, D), f(B, 5, Hkv, D), np.arange(B, dtype=np.int64)
    got = fm.attention_block_decode(x, pos, kc, vc, *w, None, None, None, None, False, H, Hkv, n_embd)
    ref = oa.attention_block_decode(x, pos, kc, vc, *w, None, None, None, None, False, H, Hkv, n_embd)
    # v_new is a bare projection: the dot-product bound
    bound = (n_embd + 2) * EPS * (np.abs(x).astype(np.float64) @ np.abs(w[2])).reshape(B, Hkv, D)
    assert np.all(np.abs(got[2] - ref[2]) <= bound)
    for g, r in zip(got[:2], ref[:2]):
        np.testing.assert_allclose(g, r, rtol=1e-4, atol=1e-4 * np.sqrt(np.mean(r**2)))
