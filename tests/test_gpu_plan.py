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
