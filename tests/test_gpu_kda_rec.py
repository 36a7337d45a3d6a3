"""The prefill's KDA recurrence (k_kda_rec): a head's state columns split over
lanes and blocks, tokens in stages of eight.  Small models of each key width
the kernel has an instance for, prompts around the stage size (one stage and a
remainder of 0, 1 and 7 tokens, several stages) and a second chunk that starts
from the first one's state, against the CPU restatement, bit for bit: hidden
rows, then the logits of a verify that reads the state the prefill left."""
import numpy as np
import pytest

from oracle_lib import Oracle
from test_gpu_parity import diff_report, same_bits
from test_gpu_shapes import SHAPES, shape_model

pytestmark = pytest.mark.gpu

for _kd in (32, 64, 128):
    SHAPES.setdefault(f"rec_kd{_kd}", dict(kda_heads=3, kd=_kd, vd=_kd, gate_rank=32))


@pytest.mark.parametrize("first,second", [(16, 0), (17, 0), (23, 0), (24, 41), (63, 18)])
@pytest.mark.parametrize("kd", [32, 64, 128])
def test_prefill_recurrence(pkg, model_root, kd, first, second):
    print(f"[case] kd {kd}, prefill of {first} then {second} tokens", flush=True)
    model = shape_model(pkg, model_root, f"rec_kd{kd}")
    n = first + second
    prompt = pkg.prompt_tokens(21, n, 512)
    eng, ora = pkg.Engine(model), Oracle(model)
    try:
        eng.reset()
        for lo, hi in ((0, first), (first, n)):
            if hi == lo:
                continue
            h, ho = eng.batch_capture(prompt[lo:hi], lo), ora.batch_capture(prompt[lo:hi], lo)
            assert h is not None and ho is not None
            assert same_bits(h, ho), "hidden rows: " + diff_report(h, ho)
        toks = np.array([5, 7, 300, 41], np.int32)
        v, vo = eng.verify(toks, n), ora.verify(toks, n)
        assert same_bits(v[0], vo[0]), "verify logits: " + diff_report(v[0], vo[0])
    finally:
        eng.close()
        ora.close()
