"""Phase times of long pairs that go in groups: the fill is the fill, the
traceback every group's."""
import random

import pytest

import tweakseq_amd as ta
from test_gpu_parity import mutate, rand_prot

pytestmark = pytest.mark.gpu


def phases(pairs, params, runs=5):
    eng = ta.Engine(0)
    try:
        b = eng.batch(pairs, params)
        out = []
        for _ in range(runs):
            b.run()
            b.wait()
            out.append(b.timings())
        b.graph(True)  # a captured run is timed as a whole
        b.run()
        b.wait()
        assert b.timings()[:3] == [-1.0] * 3 and b.timings()[3] > 0
        b.graph(False)
        b.run()
        b.run_plain()  # one phase, whose tracebacks are not told apart: none of the run before is
        b.wait()
        assert b.timings()[2] < 0.5 * min(t[2] for t in out)
        b.close()
    finally:
        eng.close()
    return [min(t[k] for t in out) for k in range(4)]


def test_tracebacks_of_all_groups(monkeypatch):
    # A traceback region is 120 us: the large pair has 24 of them (none ahead: no room), the small pair, whose
    # group is the last, one.  By the last group's alone the traceback would be a twentieth.
    rng = random.Random(4)
    params = ta.engine.make_params(mode=ta.GLOBAL, alphabet=ta.DNA, gap_open=-5, gap_extend=-2, match=2, mismatch=-3,
                                   lanes=ta.LANES_LONG)
    a, c = rand_prot(rng, 12000, "ACGT"), rand_prot(rng, 520, "ACGT")
    large, small = (a, mutate(rng, a, 0.1, 0.02, "ACGT")), (c, mutate(rng, c, 0.1, 0.02, "ACGT"))
    monkeypatch.setenv("TWEAKALIGN_LONG_BYTES", "0")
    alone, both = phases([large], params), phases([large, small], params)
    assert both[2] > 0.7 * alone[2], (alone, both)
    assert both[0] < alone[0] + 0.5 * alone[2], (alone, both)
    assert abs(sum(both[:3]) - both[3]) < 0.2 * both[3]
