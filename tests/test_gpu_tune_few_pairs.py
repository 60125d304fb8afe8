"""The autotuner on few pairs: candidates are timed in the form a tuning
shapes, not in the one few pairs take whatever the tuning, where any of them
could win."""
import random

import pytest

import tweakseq_amd as ta
from test_gpu_parity import compare, mutate, oracle_results, rand_prot

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [ta.GLOBAL, ta.LOCAL])
def test_candidates_are_timed_in_their_own_form(mode, monkeypatch):
    # One pair: 0.3 ms in the few-pairs form, 2.5 ms in the other (TWEAKALIGN_COOP set asks for that).
    rng = random.Random(mode)
    a = rand_prot(rng, 1500)
    pairs = [(a, mutate(rng, a))]
    params = ta.engine.make_params(mode=mode, gap_open=-11, gap_extend=-1)
    eng = ta.Engine(0)
    try:
        monkeypatch.setenv("TWEAKALIGN_COOP", "1")
        _, want = eng.autotune(pairs, params, repeats=3)
        monkeypatch.delenv("TWEAKALIGN_COOP")
        _, got = eng.autotune(pairs, params, repeats=3)
        assert got > 0.5 * want, (got, want)
        compare(eng.align(pairs, params), oracle_results(params, pairs), params, pairs, "tuned")
    finally:
        eng.close()
