"""Pairs whose int16 fill saturates, few among many: the int32 rerun replaces
the plane records of these pairs alone, run after run."""
import random

import pytest

import tweakseq_amd as ta
from test_gpu_parity import compare, mutate, oracle_results, rand_prot

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("at", [(0,), (8999,), (0, 1, 2, 4500, 8998, 8999), tuple(range(3000, 3400))])
def test_few_of_many_rerun(at):
    rng = random.Random(len(at) + at[0])
    pairs = []
    for _ in range(9000):  # too many strips for the few-pairs form, so the packed fill runs
        a = rand_prot(rng, rng.randint(1, 60))
        pairs.append((a, mutate(rng, a) or "A"))
    for q, k in enumerate(at):  # 11 a W: just below int16's limit of 32,745, past it twice, and unable to reach it
        w = "W" * (2976 + 5 * (q % 3))
        pairs[k] = (w, ("ACD" + w, w + "G", w[:1500] + "AC" + w[1500:])[q % 3]) if len(at) < 9 or q % 40 == 0 else \
            ("W" * 40, "W" * 44)
    params = ta.engine.make_params(mode=ta.LOCAL, gap_open=-11, gap_extend=-1)
    some = sorted(set(at[:6]) | set(at[::40]) | set(rng.sample(range(9000), 300)))
    want = oracle_results(params, [pairs[k] for k in some])
    eng = ta.Engine(0)
    try:
        b = eng.batch(pairs, params)
        first = None
        for _ in range(3):
            b.run()
            b.wait()
            got = b.results()
            compare([got[k] for k in some], want, params, [pairs[k] for k in some], "rerun")
            assert first is None or got == first
            first = got
        b.close()
        for k, (g, w) in zip(some, zip([first[k] for k in some], want)):
            assert bool(g.flags & ta.F_RERUN) == (w[0] > 32767 - 22), (k, w[0], g.flags)
    finally:
        eng.close()
