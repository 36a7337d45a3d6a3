"""A run state's host mirrors (pinned, written by device copies): every call has
written what it returns through them by the time it returns; and their blocks
pass from freed sessions to new ones cleared, across threads, and outlive the
model."""
import ctypes as C
import threading

import numpy as np
import pytest

from test_gpu_parity import same_bits

pytestmark = pytest.mark.gpu


def mirror(st, field, *shape):
    return np.ctypeslib.as_array(getattr(st, field), shape=shape)


def mirrors(pkg, eng, st, chain=False):
    """The mirrors by name (the chain, which most calls read, only on demand)."""
    out = {"logits": mirror(st, "logits", eng.V), "rows": mirror(st, "mtp_logits", pkg.L98_SPEC_K_GPU + 1, eng.V),
           "hidden": mirror(st, "mtp_verify_hidden", pkg.L98_SPEC_K_GPU + 1, eng.d),
           "draft": mirror(st, "mtp_draft_logits", eng.V)}
    if eng.dspark:
        out["kdraft"] = mirror(st, "mtp_kdraft_logits", pkg.LZ_SPEC_K_MAX, eng.V)
    if chain:
        out["chain"] = mirror(st, "mtp_chain", eng.d)
    return out


@pytest.mark.parametrize("which", ["tiny", "subln", "ds_tiny"])
def test_calls_write_their_mirrors_before_they_return(pkg, request, which):
    """Each call twice after the same prompt, the mirrors full of NaN before it:
    what the first wrote, the second writes again, whole."""
    eng = pkg.Engine(request.getfixturevalue(which), spec_k_max=6)
    st, lib, n, k = eng.s, eng.lib, 300, 2
    prompt = pkg.prompt_tokens(4, n, eng.V)
    toks, pos, ms = np.array([3, 77, 1000, 5], np.int32), np.array([n], np.int32), C.c_float()
    ip, m, s, ptrs = C.POINTER(C.c_int), C.byref(eng.m), C.byref(st), eng._state_ptrs([st])
    tp, pp = toks.ctypes.data_as(ip), pos.ctypes.data_as(ip)
    # the call, whether it succeeded, the mirrors that it writes and how much of them
    calls = [("start", lambda: eng.session_start(prompt) >= 0, {"logits": eng.V, "chain": eng.d}),
             ("forward", lambda: lib.lz_forward(m, s, 3, n), {"logits": eng.V}),
             ("capture", lambda: lib.lz_forward_capture(m, s, 3, n), {"logits": eng.V, "chain": eng.d}),
             ("verify", lambda: lib.lz_forward_verify(m, s, tp, 4, n) == 0, {"rows": 4, "hidden": 4}),
             ("batch", lambda: lib.l98_verify_batch(m, ptrs, 1, tp, 4, pp, 1, C.byref(ms)) == 0, {"rows": 4, "hidden": 4}),
             ("round", lambda: eng.spec_round(3, n - 1, k)[0] >= 1,
              {"rows": k + 1, "hidden": k + 1, **({"kdraft": k} if eng.dspark else {"draft": eng.V})})]
    if eng.dspark:
        calls.append(("draft batch", lambda: lib.lz_mtp_draft_batch(m, s, 3, k), {"kdraft": k}))
    else:
        calls.append(("draft step", lambda: lib.lz_mtp_draft_step(m, s, 3, n), {"draft": eng.V}))
    try:
        for name, call, fields in calls:
            print(f"[case] mirrors after {name}, {which}", flush=True)
            got = []
            for _ in range(2):
                eng.session_start(prompt)
                for a in mirrors(pkg, eng, st, "chain" in fields).values():
                    a.fill(np.nan)
                assert call(), name
                now = mirrors(pkg, eng, st, True)
                got.append({f: now[f][:r].copy() for f, r in fields.items()})
            for f in fields:
                assert np.isfinite(got[0][f]).all() and same_bits(got[0][f], got[1][f]), (name, f)
    finally:
        eng.close()


def test_blocks_of_freed_sessions_come_back_cleared(pkg, micro):
    eng = pkg.Engine(micro)
    print("[case] mirrors of new sessions after freed ones", flush=True)

    def dirty_and_check():
        st = eng.add_session(seq_len=64)
        for a in mirrors(pkg, eng, st, True).values():
            assert not a.any()
            a.fill(7.0)
        return st
    try:
        for _ in range(3):
            held = [dirty_and_check() for _ in range(5)]
            for st in held:
                eng.free_session(st)
        bad = []

        def churn():
            try:
                for _ in range(8):
                    eng.free_session(dirty_and_check())
            except Exception as e:       # noqa: BLE001
                bad.append(e)
        threads = [threading.Thread(target=churn) for _ in range(4)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not bad, bad
    finally:
        eng.close()


def test_a_session_may_be_freed_after_its_model(pkg, micro):
    eng = pkg.Engine(micro)
    print("[case] sessions freed after the model", flush=True)
    held = [eng.add_session(seq_len=64) for _ in range(3)]
    eng.free_session(held.pop())
    eng.close()                          # the model goes
    for st in held:
        assert not mirror(st, "logits", 16).any()
        eng.free_session(st)
