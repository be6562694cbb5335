"""Row tiles of at most 128 rows of the prefill GEMM (gemm_tiled256.hip:
narrow_k_loop; k_loop_f8's half stages and 2 x 4 waves) against the float64 oracle's
grouped products, every expert holding a chosen number of rows."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import moe as om
from oracle import numerics as nm
from helpers import assert_close_rms

pytestmark = pytest.mark.gpu

# Rows per expert: both sides of each 16-row group and of 64 and 128 rows, as
# an expert's only tile and as its last tile behind full ones; none.
COUNTS = [1, 15, 17, 33, 48, 63, 64, 65, 81, 112, 127, 128, 129, 0, 257, 320, 321, 384, 385]


# (H, F): fewer stages than the ring, an odd number of 64-input stages, partial
# column tiles; a K range longer than the rings, split in two for the down
# projection.  Tolerances: the repository's for each configuration (bf16 2e-2;
# two-term rows against the oracle on the same rows).
# (The two-term GEMMs take multiples of 128 inputs.)
@pytest.mark.parametrize("H,F,weights", [
    (H, F, w) for H, F in [(128, 128), (192, 320), (256, 384), (640, 2176)]
    for w in ("bf16", "fp8", "x2") if w != "x2" or (H, F) != (192, 320)])
def test_narrow_tiles(fm, gemm_path, H, F, weights):
    rng = np.random.default_rng(H + F)
    E, T = len(COUNTS), sum(COUNTS)
    experts = rng.permutation(np.repeat(np.arange(E), COUNTS))
    x = rng.standard_normal((T, H)).astype(np.float32)
    x[:, :E] = 0.0
    x[np.arange(T), experts] = 4.0  # logit 32 for the token's expert, 0 for the others
    x = nm.bf16_round(x)
    wr = np.zeros((E, H), np.float32)
    wr[np.arange(E), np.arange(E)] = 8.0
    dev = [torch.from_numpy((rng.standard_normal(s) * s[1] ** -0.5).astype(np.float32)).cuda().bfloat16()
           for s in ((F, H, E), (F, H, E), (H, F, E))]
    host = [w.float().cpu().numpy() for w in dev]
    if weights == "bf16":
        packed = [fm.pack_expert_weights(w) for w in dev]
    else:
        packed = [fm.quantize_expert_weights(w) for w in dev]
        host = [nm.dequantize_e4m3fn(*nm.quantize_per_channel_e4m3fn(w)) for w in host]
    ll = gemm_path
    ll.check(ll.lib().fmoe_set_gemm_path(ll.PATH_TILED_LARGE))
    dt = torch.bfloat16
    blk = fm.MoEFFNBlock(torch.from_numpy(wr).cuda().to(dt), *packed, E, 1, H, F, True, act_dtype=dt,
                         fp8_activations="x2" if weights == "x2" else False)
    out = blk(torch.from_numpy(x).cuda().to(dt)).float().cpu().numpy()
    ref, ids, _ = om.moe_ffn_block(x, wr, *host, E, 1, H, F, True, return_routing=True,
                                   **({"act_quant": "x2", "dtype": np.float32} if weights == "x2"
                                      else {"dtype": np.float64}))
    np.testing.assert_array_equal(np.bincount(ids.reshape(-1), minlength=E), COUNTS)
    for e in range(E):  # per expert: a fault in a small tile is not lost in the whole output's norm
        rows = experts == e
        if rows.any():
            assert_close_rms(out[rows], ref[rows], 2e-2, what=f"{COUNTS[e]} rows, H={H} F={F} {weights}")
