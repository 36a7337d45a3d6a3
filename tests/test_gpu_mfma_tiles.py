"""The tiled many-row GEMM (k_mfma_q8t, K a multiple of 128) at the edges of its
tiles: one row or column, rows and columns one short of and past a tile of each
shape (32 x 16, 32 x 32, 64 x 32: the widths and row counts that select them),
one to five stages of K (fewer than the loads run ahead, and a partial turn of
the four buffers), against the oracle's matmul, bit for bit."""
import numpy as np
import pytest

import oracle_lib as OL
from test_gpu_mfma import case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K,M", [(1, 128, 1), (33, 128, 16), (31, 256, 15), (95, 384, 17), (130, 640, 31),
                                   (32, 512, 32), (65, 1152, 33), (1000, 256, 63), (65600, 128, 33),
                                   (65537, 384, 64), (32800, 256, 100)])
def test_tile_edges_bit_exact(pkg, N, K, M):
    rng = np.random.default_rng(N + 3 * K + 5 * M)
    w, ws, x, xs = case(rng, N, K, M)
    w[-1, :] = -128                                          # the largest group sums: |acc| = 32 * 128 * 127
    out = np.zeros((M, N), np.float32)
    print(f"[case] tiled mfma N={N} K={K} M={M}", flush=True)
    assert pkg.hip_lib().l98_gemm_q8(w.ctypes.data, OL.fp(ws), N, K, x.ctypes.data, OL.fp(xs), M, OL.fp(out)) == 0
    want = np.zeros((M, N), np.float32)
    OL.lib().o_matmul_q8(OL.fp(want), x.ctypes.data, OL.fp(xs), w.ctypes.data, OL.fp(ws), K, N, M, None)
    bad = np.nonzero(out.view(np.uint32) != want.view(np.uint32))
    assert len(bad[0]) == 0, (bad[0][:5], bad[1][:5], out[bad][:5], want[bad][:5])
