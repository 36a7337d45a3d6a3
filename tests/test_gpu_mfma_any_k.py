"""The many-row GEMM for K not a multiple of 128 (k_mfma_q8, and k_mfma_q8n for
few columns over many weight rows) on both sides of the rule between them and at
the narrow tiles' edges, against the oracle's matmul; and experts of width 704
over a 352-wide latent (grouped launches, both banks in one) through a session
batch against single sessions.  Bit for bit."""
import ctypes as C
import os

import numpy as np
import pytest

import oracle_lib as OL
from test_gpu_mfma import case
from test_gpu_parity import same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K,M", [(16400, 32, 1), (16384, 96, 16), (16353, 96, 17), (16321, 32, 32), (8255, 352, 33),
                                   (5100, 1056, 15), (16385, 800, 128), (16400, 1056, 129), (2047, 704, 31)])
def test_any_k_bit_exact(pkg, N, K, M):
    rng = np.random.default_rng(N + 3 * K + 5 * M)
    w, ws, x, xs = case(rng, N, K, M)
    w[-1, :] = -128
    out = np.zeros((M, N), np.float32)
    print(f"[case] mfma any K N={N} K={K} M={M}", flush=True)
    assert pkg.hip_lib().l98_gemm_q8(w.ctypes.data, OL.fp(ws), N, K, x.ctypes.data, OL.fp(xs), M, OL.fp(out)) == 0
    want = np.zeros((M, N), np.float32)
    OL.lib().o_matmul_q8(OL.fp(want), x.ctypes.data, OL.fp(xs), w.ctypes.data, OL.fp(ws), K, N, M, None)
    bad = np.nonzero(out.view(np.uint32) != want.view(np.uint32))
    assert len(bad[0]) == 0, (bad[0][:5], bad[1][:5], out[bad][:5], want[bad][:5])


@pytest.mark.parametrize("sessions,rows", [(2, 1), (9, 4), (16, 7)])
def test_expert_width_704_batch_matches_single(pkg, model_root, sessions, rows):
    """64 experts, top-8: groups of 1 to about 14 columns."""
    path = os.path.join(model_root, "expert704")
    cfg = pkg.synth_config(0)
    cfg.n_experts, cfg.topk, cfg.latent, cfg.moe_inter, cfg.vocab, cfg.seq_len = 64, 8, 352, 704, 1024, 128
    if not os.path.exists(os.path.join(path, "model.bin")):
        pkg.write_model(path, 0, 77, cfg=cfg)
    print(f"[case] batch of {sessions} x {rows} rows, expert width 704", flush=True)
    eng = pkg.Engine(path, spec_k_max=7)
    rs = np.random.RandomState(sessions)
    states = [eng.add_session(seq_len=64, spec_k_max=7) for _ in range(sessions)]
    try:
        toks, pos = rs.randint(0, eng.V, (sessions, rows)).astype(np.int32), []
        for st in states:
            prompt = rs.randint(0, eng.V, rs.randint(5, 40))
            eng.session_start_on(st, prompt)
            pos.append(len(prompt))
        marks = [st.ssm_slot for st in states]
        got = eng.verify_batch(states, toks, pos)[1]
        for i, st in enumerate(states):
            st.ssm_slot = marks[i]
            one = np.ascontiguousarray(toks[i])
            assert eng.lib.lz_forward_verify(C.byref(eng.m), C.byref(st), one.ctypes.data_as(C.POINTER(C.c_int)), rows,
                                             pos[i]) == 0
            want = np.ctypeslib.as_array(st.mtp_logits, shape=(pkg.L98_SPEC_K_GPU + 1, eng.V))[:rows]
            assert same_bits(got[i][0], want), i
    finally:
        for st in states:
            eng.free_session(st)
        eng.close()
