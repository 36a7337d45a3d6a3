"""The work that a user of this library has it do, as timed cases.

Every case is a call of the C ABI of include/llama98_hip.h through the ctypes
bindings: a verify forward, a draft-verify-accept round, a prompt's prefill, a
whole generation, a batch of sessions.  The models are the synthetic ones of
csrc/synth.h, with the widths, vocabularies, head counts and expert counts
that bench.py and the tests run; `wide` and `dspark` keep eight layers of
theirs (two periods of three KDA layers and an attention layer), so that a
model is written and loaded in seconds.

The arithmetic is a contract: every result is bit-identical to the reference
engine's float-oracle mode, so every tolerance here is "exact".  Activations
are requantized to int8 several times per layer, and the quantization's
decisions belong to the fp32 rounding sequence: a 64-bit evaluation takes
other decisions, and its distance says nothing about either side.  exact()
therefore has no value for any output.

A pass can be repeated on its state: a verify or round writes ring slots after
the session's current one and K/V rows after its position, so setting the
state's slot and MTP position back (as a caller does that rejects a round)
gives the next pass the same inputs; sessions that run device-resident rounds
are started again from their prompts.
"""
import ctypes as C
import functools
import os
import tempfile

import numpy as np

from __graft_entry__ import load_package

pkg = load_package()

# model name: (id of csrc/synth.h, layers kept or 0, seq_len or 0)
MODELS = {
    "tiny": (0, 0, 0),          # d = 256, 4 layers, 16 experts top-2, V = 8192
    "subln": (5, 0, 0),         # the same shapes with SubLN norms and Hadamard blocks
    "base": (1, 0, 0),          # d = 1024, 24 layers, 64 experts top-6, V = 65536
    "dspark": (22, 8, 0),       # base's widths with a 6-slot DSpark head
    "wide": (23, 8, 5200),      # d = 2048, 128 experts top-8, V = 131072, skewed router
}
MODEL_SEED = 1234
DEPTH_K = 7                     # spec_k_max of every state: a ring of 8 slots


def _config(name):
    cid, layers, seq_len = MODELS[name]
    cfg = pkg.synth_config(cid)
    if layers:
        cfg.n_layers = layers
    if seq_len:
        cfg.seq_len = seq_len
    return cfg


def _model_dir(name):
    """The model's directory, written on first use (renamed into place whole)."""
    root = os.path.join(tempfile.gettempdir(), "l98_case_models_%d" % os.getuid())
    cid, layers, seq_len = MODELS[name]
    path = os.path.join(root, "%s_%d_%d_%d_%d" % (name, cid, layers, seq_len, MODEL_SEED))
    if not os.path.isdir(path):
        os.makedirs(root, exist_ok=True)
        tmp = tempfile.mkdtemp(dir=root)
        pkg.write_model(tmp, cid, MODEL_SEED, threads=8, cfg=_config(name))
        try:
            os.rename(tmp, path)
        except OSError:              # another process was faster
            if not os.path.isdir(path):
                raise
    return path


@functools.lru_cache(maxsize=None)
def _engine(name):
    """A program opens a model once and starts its sessions on it."""
    return pkg.Engine(_model_dir(name), spec_k_max=1, seq_len=64)


class _Session:
    """One run state of a model, freed with the object."""

    def __init__(self, eng, seq_len):
        self.eng = eng
        self.st = eng.add_session(seq_len=seq_len, spec_k_max=DEPTH_K)

    def __del__(self):
        try:
            self.eng.free_session(self.st)
        except Exception:
            pass


def _rows(s, field, *shape):
    """The state's buffer `field` as an array that keeps the session alive."""
    buf = (C.c_float * int(np.prod(shape))).from_address(C.addressof(getattr(s.st, field).contents))
    buf.session = s
    return np.frombuffer(buf, np.float32).reshape(shape)


# --------------------------------------------------------------- cases ---

def listed():
    return [
        # the smallest call: one token of a small model, a short chat just begun
        {"name": "step_tiny", "kind": "verify", "model": "tiny", "rows": 1, "ctx": 65},
        # plain decoding, one token at a time
        {"name": "step_base", "kind": "verify", "model": "base", "rows": 1, "ctx": 517},
        # the verify of a k = 3 draft after a 512-token prompt
        {"name": "verify_base_k3", "kind": "verify", "model": "base", "rows": 4, "ctx": 512},
        # one round at temperature 0.8, top-p 0.95, the widest draft, late in a session
        {"name": "round_temp_base_k6", "kind": "temp", "model": "base", "k": 6, "ctx": 1037},
        # a greedy reply to a short question: prefill, device-resident rounds, one host-driven round
        {"name": "generate_base", "kind": "generate", "model": "base", "k": 3, "prompt": 61, "rounds": 16},
        # reading a 512-token prompt: prefill, MTP prefill, first token
        {"name": "prefill_base_512", "kind": "prefill", "model": "base", "prompt": 512},
        # a round of the SubLN variant (Hadamard blocks, a norm per projection)
        {"name": "round_subln_k2", "kind": "round", "model": "subln", "k": 2, "ctx": 131},
        # a round with a DSpark head: one batch of draft slots
        {"name": "round_dspark_k5", "kind": "round", "model": "dspark", "k": 5, "ctx": 300},
        # the verify of a wide model deep in a long document
        {"name": "verify_wide_long", "kind": "verify", "model": "wide", "rows": 4, "ctx": 4099},
        # reading a long document into a wide model, an odd length
        {"name": "prefill_wide_long", "kind": "prefill", "model": "wide", "prompt": 4001},
        # a server's step: 32 sessions of mixed contexts verify together
        {"name": "server_verify_32", "kind": "batch", "model": "wide", "sessions": 32, "rows": 4, "lo": 256, "hi": 2048},
        # a burst of short requests: started one after another, then decoded together
        {"name": "server_burst_12", "kind": "burst", "model": "base", "sessions": 12, "k": 3, "lo": 17, "hi": 160,
         "rounds": 12},
    ]


def _log(rng, lo, hi):
    """A size in [lo, hi], uniform in its logarithm."""
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["verify", "verify", "verify_wide", "round", "temp", "generate", "prefill", "prefill_wide",
                       "batch", "burst"])
    if kind == "verify":
        model = rng.choice(["tiny", "subln", "base", "dspark"])
        return {"kind": "verify", "model": model, "rows": rng.randint(1, 7),
                "ctx": _log(rng, 17, 480 if model in ("tiny", "subln") else 1200)}
    if kind == "verify_wide":
        return {"kind": "verify", "model": "wide", "rows": rng.randint(1, 7), "ctx": _log(rng, 17, 4500)}
    if kind == "round":
        model = rng.choice(["tiny", "subln", "base", "dspark", "wide"])
        return {"kind": "round", "model": model, "k": rng.randint(1, 6),
                "ctx": _log(rng, 17, 480 if model in ("tiny", "subln") else 1200)}
    if kind == "temp":
        model = rng.choice(["tiny", "base", "dspark"])
        return {"kind": "temp", "model": model, "k": rng.randint(1, 6),
                "ctx": _log(rng, 17, 480 if model == "tiny" else 1200)}
    if kind == "generate":
        return {"kind": "generate", "model": rng.choice(["tiny", "subln", "base", "dspark"]), "k": rng.randint(1, 6),
                "prompt": _log(rng, 9, 240), "rounds": rng.randint(4, 24)}
    if kind == "prefill":
        model = rng.choice(["tiny", "subln", "base", "dspark"])
        return {"kind": "prefill", "model": model, "prompt": _log(rng, 9, 500 if model in ("tiny", "subln") else 1200)}
    if kind == "prefill_wide":
        return {"kind": "prefill", "model": "wide", "prompt": _log(rng, 9, 4001)}
    if kind == "batch":
        lo = _log(rng, 32, 400)
        return {"kind": "batch", "model": rng.choice(["tiny", "base", "wide"]), "sessions": _log(rng, 2, 32),
                "rows": rng.randint(1, 4), "lo": lo, "hi": rng.randint(lo, 480)}
    lo = _log(rng, 9, 100)
    return {"kind": "burst", "model": rng.choice(["tiny", "base"]), "sessions": _log(rng, 2, 12),
            "k": rng.randint(1, 4), "lo": lo, "hi": rng.randint(lo, 160), "rounds": rng.randint(4, 12)}


# ------------------------------------------------------------- prepare ---

def _tokens(rs, n, vocab):
    return np.ascontiguousarray(rs.randint(0, vocab, size=n), np.int32)


def _started(eng, prompt, seq_len):
    """A session that has read its prompt."""
    s = _Session(eng, seq_len)
    s.anchor = eng.session_start_on(s.st, prompt)
    s.pos = len(prompt) - 1
    s.mark = (s.st.ssm_slot, s.st.mtp_pos)
    s.chain = _rows(s, "mtp_chain", eng.d).copy()
    return s


def _back(eng, s):
    """The session as its prompt left it: the rounds since are rejected."""
    s.st.ssm_slot, s.st.mtp_pos = s.mark
    C.memmove(s.st.mtp_chain, s.chain.ctypes.data, 4 * eng.d)


def prepare(case, seed):
    rs = np.random.RandomState((int(seed) * 1000003 + 17) % (1 << 32))
    eng = _engine(case["model"])
    kind = case["kind"]
    state = {"case": case, "eng": eng}
    if kind in ("verify", "round", "temp"):
        room = case["ctx"] + 16
        state["s"] = _started(eng, _tokens(rs, case["ctx"], eng.V), room)
        if kind == "verify":
            state["tokens"] = _tokens(rs, case["rows"], eng.V)
        if kind == "temp":
            state["rng"] = int(rs.randint(1, 1 << 30))
    elif kind in ("prefill", "generate"):
        more = (case["rounds"] + 2) * (case["k"] + 1) + 16 if kind == "generate" else 16
        state["prompt"] = _tokens(rs, case["prompt"], eng.V)
        state["s"] = _Session(eng, case["prompt"] + more)
    else:
        n = case["sessions"]
        lens = rs.randint(case["lo"], case["hi"] + 1, size=n)
        prompts = [_tokens(rs, int(m), eng.V) for m in lens]
        if kind == "batch":
            ss = [_started(eng, p, len(p) + 16) for p in prompts]
            state["tokens"] = _tokens(rs, n * case["rows"], eng.V)
            state["pos"] = np.ascontiguousarray(lens, np.int32)
        else:
            more = (case["rounds"] + 2) * (case["k"] + 1) + 16
            ss = [_Session(eng, len(p) + more) for p in prompts]
            state["prompts"] = prompts
        state["ss"] = ss
        state["ptrs"] = eng._state_ptrs([s.st for s in ss])
    return state


# ----------------------------------------------------------------- run ---

def _verify(eng, s, tokens, pos):
    n = len(tokens)
    if eng.lib.lz_forward_verify(C.byref(eng.m), C.byref(s.st), pkg._ip(tokens), n, int(pos)) != 0:
        raise RuntimeError("lz_forward_verify failed")
    return {"logits": _rows(s, "mtp_logits", n, eng.V), "hidden": _rows(s, "mtp_verify_hidden", n, eng.d)}


def _round(eng, s, anchor, pos, k, samp=None):
    out = np.zeros(pkg.L98_SPEC_K_GPU + 1, np.int32)
    na, npos, ke = C.c_int(), C.c_int(), C.c_int()
    err = C.create_string_buffer(256)
    lib, m, st = eng.lib, C.byref(eng.m), C.byref(s.st)
    args = (m, st, int(anchor), int(pos), int(k), 0.0, 0, C.byref(samp) if samp is not None else None, 0)
    tail = (pkg._ip(out), C.byref(na), C.byref(npos), C.byref(ke), err, 256)
    if eng.dspark:
        f = lib.lz_spec_round_dspark if samp is None else lib.lz_spec_round_dspark_temp
        r = f(*args, *tail)
    else:
        f = lib.lz_spec_round if samp is None else lib.lz_spec_round_temp
        r = f(*args, 0, *tail)
    if r < 1:
        raise RuntimeError("the round failed: %d %s" % (r, err.value.decode()))
    out[na.value + 1:] = -1          # as many values whatever was accepted
    got = {"tokens": out, "accepted": na.value, "chain": _rows(s, "mtp_chain", eng.d)}
    if samp is None:
        got["logits"] = _rows(s, "mtp_logits", ke.value + 1, eng.V)
        got["hidden"] = _rows(s, "mtp_verify_hidden", ke.value + 1, eng.d)
        if not eng.dspark:
            got["draft"] = _rows(s, "mtp_draft_logits", eng.V)
    return got


def _temp_sampler(eng, rng):
    p = pkg.LZSampleParams()
    eng.lib.lz_sample_defaults(C.byref(p))
    p.temperature, p.topp, p.topk, p.minp = 0.8, 0.95, 0, 0.0
    p.presence_penalty, p.frequency_penalty, p.repetition_penalty, p.repeat_last_n = 0.0, 0.0, 1.0, 0
    samp = pkg.LZSampler()
    eng.lib.lz_sampler_init(C.byref(samp), eng.V, C.byref(p), rng)
    return samp


def _device_rounds(eng, s, k, n):
    cap = n * (k + 1)
    toks, acc, ms = np.zeros(cap, np.int32), np.zeros(n, np.int32), C.c_float()
    got = eng.lib.l98_greedy_rounds(C.byref(eng.m), C.byref(s.st), k, n, 1, pkg._ip(toks), cap, pkg._ip(acc),
                                    C.byref(ms))
    if got < 0:
        raise RuntimeError("l98_greedy_rounds failed: %d" % got)
    return toks, acc, got


def _verify_batch(eng, state, tokens, rows, pos):
    ms = C.c_float()
    n = len(state["ss"])
    if eng.lib.l98_verify_batch(C.byref(eng.m), state["ptrs"], n, pkg._ip(tokens), rows, pkg._ip(pos), 1,
                                C.byref(ms)) != 0:
        raise RuntimeError("l98_verify_batch failed")
    return n


def run(state):
    case, eng = state["case"], state["eng"]
    kind = case["kind"]
    if kind == "verify":
        s = state["s"]
        _back(eng, s)
        return _verify(eng, s, state["tokens"], s.pos + 1)
    if kind == "round":
        s = state["s"]
        _back(eng, s)
        return _round(eng, s, s.anchor, s.pos, case["k"])
    if kind == "temp":
        s = state["s"]
        _back(eng, s)
        samp = _temp_sampler(eng, state["rng"])
        got = _round(eng, s, s.anchor, s.pos, case["k"], samp)
        got["rng"] = np.array([samp.rng_state], np.uint64).view(np.int64)
        return got
    if kind == "prefill":
        s = state["s"]
        first = eng.session_start_on(s.st, state["prompt"])
        return {"token": first, "logits": _rows(s, "logits", eng.V), "chain": _rows(s, "mtp_chain", eng.d)}
    if kind == "generate":
        s = state["s"]
        first = eng.session_start_on(s.st, state["prompt"])
        toks, acc, n = _device_rounds(eng, s, case["k"], case["rounds"])
        got = _round(eng, s, toks[n - 1], len(state["prompt"]) - 1 + n, case["k"])
        got.update(first=first, rounds=toks, round_accepts=acc)
        return got
    n = len(state["ss"])
    if kind == "batch":
        for s in state["ss"]:
            _back(eng, s)
        _verify_batch(eng, state, state["tokens"], case["rows"], state["pos"])
        return {"logits": [_rows(s, "mtp_logits", case["rows"], eng.V) for s in state["ss"]],
                "hidden": [_rows(s, "mtp_verify_hidden", case["rows"], eng.d) for s in state["ss"]]}
    k, rounds = case["k"], case["rounds"]
    first = [eng.session_start_on(s.st, p) for s, p in zip(state["ss"], state["prompts"])]
    cap = rounds * (k + 1)
    toks, cnt, ms = np.zeros((n, cap), np.int32), np.zeros(n, np.int32), C.c_float()
    if eng.lib.l98_greedy_rounds_batch(C.byref(eng.m), state["ptrs"], n, k, rounds, pkg._ip(toks), cap, pkg._ip(cnt),
                                       C.byref(ms)) < 0:
        raise RuntimeError("l98_greedy_rounds_batch failed")
    pos = np.ascontiguousarray([len(p) - 1 + c for p, c in zip(state["prompts"], cnt)], np.int32)
    last = np.ascontiguousarray([toks[i, cnt[i] - 1] for i in range(n)], np.int32)
    _verify_batch(eng, state, last, 1, pos + 1)
    return {"first": np.array(first, np.int32), "tokens": toks, "counts": cnt,
            "logits": [_rows(s, "mtp_logits", 1, eng.V) for s in state["ss"]]}


# ---------------------------------------------------------------- work ---

def _weights(c):
    """Weight bytes of a layer's KDA, attention and expert-free MoE parts, of
    one expert, of the MTP block (with its head's fc) and of the lm_head."""
    d, kq = c.hidden, c.kda_heads * c.kd
    q, kv = c.n_heads * c.head_dim, c.n_kv_heads * c.head_dim
    attn = d * (2 * q + 2 * kv) + q * d
    kda = d * (2 * kq + 2 * kq + c.gate_rank + c.kda_heads) + kq * d + c.gate_rank * kq
    moe = d * (c.n_experts + 2 * c.latent) + 3 * d * c.shared_w
    expert = 3 * c.latent * c.moe_inter
    mtp = attn + 3 * d * c.mtp_inter + (3 if c.mtp_n_draft > 1 else 2) * d * d
    return attn, kda, moe, expert, mtp, c.vocab * d


def _trunk(c, rows, seqs, ctx):
    """Bytes and operations of one forward of `rows` rows in `seqs` sessions
    whose contexts sum to ctx: each weight read once (of the experts, the
    share that this many draws of top-k reach), the K/V rows and the KDA
    state read once, the new state written."""
    attn, kda, moe, expert, _, _ = _weights(c)
    na = c.n_layers // c.attn_period
    nk = c.n_layers - na
    hit = c.n_experts * (1.0 - (1.0 - c.topk / c.n_experts) ** rows)
    kv = 2 * c.n_kv_heads * c.head_dim * 1.125
    st = 4 * c.kda_heads * c.kd * c.vd
    by = na * attn + nk * kda + c.n_layers * (moe + hit * expert) + na * ctx * kv + nk * st * (seqs + seqs)
    macs = rows * (na * attn + nk * kda + c.n_layers * (moe + c.topk * expert))
    macs += na * (rows / seqs) * ctx * c.n_heads * c.head_dim * 2 + nk * rows * 3 * c.kda_heads * c.kd * c.vd
    return by, 2 * macs


def _one_round(c, k, seqs, ctx):
    """One greedy round: k draft steps of a row per session (a DSpark head:
    one batch of k), the verify of k + 1 rows, the lm_head each time."""
    mtp, head = _weights(c)[4:]
    steps = 1 if c.mtp_n_draft > 1 else k
    by, fl = _trunk(c, seqs * (k + 1), seqs, ctx)
    by += steps * (mtp + head) + head + 4 * seqs * c.vocab * (2 * k + 1)
    fl += 2 * seqs * (k * (mtp + head) + (k + 1) * head)
    return by, fl


def work(case):
    c = _config(case["model"])
    kind = case["kind"]
    mtp, head = _weights(c)[4:]

    def prefill(n):
        by, fl = _trunk(c, n, 1, n / 2)
        return by + head + mtp + 4 * n * c.hidden, fl + 2 * (head + n * (mtp - 3 * c.hidden * c.mtp_inter))

    if kind == "verify":
        by, fl = _trunk(c, case["rows"], 1, case["ctx"])
        by, fl = by + head + 4 * case["rows"] * c.vocab, fl + 2 * case["rows"] * head
    elif kind in ("round", "temp"):
        by, fl = _one_round(c, case["k"], 1, case["ctx"])
    elif kind == "prefill":
        by, fl = prefill(case["prompt"])
    elif kind == "generate":
        by, fl = prefill(case["prompt"])
        rb, rf = _one_round(c, case["k"], 1, case["prompt"])
        by, fl = by + (case["rounds"] + 1) * rb, fl + (case["rounds"] + 1) * rf
    else:
        n, mean = case["sessions"], (case["lo"] + case["hi"]) / 2
        if kind == "batch":
            by, fl = _trunk(c, n * case["rows"], n, n * mean)
            by, fl = by + head + 4 * n * case["rows"] * c.vocab, fl + 2 * n * case["rows"] * head
        else:
            by, fl = prefill(int(mean))
            rb, rf = _one_round(c, case["k"], n, n * mean)
            by, fl = n * by + case["rounds"] * rb, n * fl + case["rounds"] * rf
    return {"bytes": float(by), "flops": float(fl)}


# Bit-identical results are the library's contract, and its tests hold every
# path to it: no rounding differs, so nothing may differ here either.
def tolerance(case):
    return "exact"


# See the head of the file: no output has a 64-bit value to be compared with.
def exact(case, seed):
    return None
