"""Batches planned by several host threads and written out by the GPU: every
result as the oracle has it, around the sizes where the shares begin."""
import random

import pytest

import tweakseq_amd as ta
from test_gpu_parity import compare, oracle_results, rand_prot

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = ta.Engine(0)
    yield e
    e.close()


@pytest.mark.parametrize("n", [4095, 4097, 8193])
@pytest.mark.parametrize("mode, traceback", [(ta.LOCAL, True), (ta.GLOBAL, True), (ta.GLOBAL, False)])
def test_shares(eng, n, mode, traceback):
    rng = random.Random(n + mode)
    seqs = [""] + [rand_prot(rng, rng.randint(1, 40)) for _ in range(200)]
    pairs = [(rng.choice(seqs), rng.choice(seqs)) for _ in range(n - 3)]
    pairs += [(rand_prot(rng, 70), rand_prot(rng, 75)), (rand_prot(rng, 129), seqs[5]), ("", "")]
    for lanes in (ta.engine.LANES_AUTO, ta.engine.LANES_I32):
        params = ta.engine.make_params(mode=mode, traceback=traceback, lanes=lanes)
        compare(eng.align(pairs, params), oracle_results(params, pairs), params, pairs, "plan %d" % lanes)


@pytest.mark.parametrize("alphabet", [ta.PROTEIN, ta.DNA])
@pytest.mark.parametrize("go, ge", [(-10, -1), (-5, -5), (-2, -1), (-7, -9), (0, 0), (-120, -100), (-130, -120)])
def test_score_only_couples(eng, alphabet, go, ge):
    """Scores of global couples around the edges of lanes, strips and blocks,
    unrelated and related, with gap costs on both sides of the packed forms' rule."""
    rng = random.Random(-go * 7 - ge + alphabet)
    letters = "ACGT" if alphabet == ta.DNA else "ARNDCQEGHILKMFPSTWYV"
    rand = lambda k: "".join(rng.choice(letters) for _ in range(k))
    pairs = []
    for lb in (1, 7, 8, 9, 16, 63, 64, 130):
        for la in (1, 8, 15, 16, 17, 63, 65, 127, 128, 129, 513):
            a = rand(la)
            pairs += [(a, (a + rand(lb))[:lb]), (a, rand(lb))]
    a = rand(1000)
    pairs += [(a, a), (a, rand(1000)), (a, a[:900])]
    params = ta.engine.make_params(mode=ta.GLOBAL, alphabet=alphabet, gap_open=go, gap_extend=ge, traceback=False)
    compare(eng.align(pairs, params), oracle_results(params, pairs), params, pairs, "couples %d %d" % (go, ge))
