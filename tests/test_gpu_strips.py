"""Batches of few pairs (a wave per strip, anywhere on the GPU): every result
and flag as the wave- and workgroup-per-task fill gives it
(TWEAKALIGN_COOP set keeps that form), and as the oracle has it."""
import random

import pytest

import tweakseq_amd as ta
from test_gpu_parity import compare, oracle_results, rand_prot, mutate

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = ta.Engine(0)
    yield e
    e.close()


def both(eng, pairs, params, monkeypatch, graph=False):
    monkeypatch.delenv("TWEAKALIGN_COOP", raising=False)
    monkeypatch.delenv("TWEAKALIGN_WALK_IN_FILL", raising=False)
    b = eng.batch(pairs, params)
    if graph:
        b.graph(True)
    got = []
    for _ in range(4 if graph else 2):
        b.run(); b.wait()
        got.append(b.results())
        if graph:
            eng.align([("ACDEF" * 30, "ACDF" * 40)] * 3, params)  # other work between the replays
    tasks = b.info()["tasks"]
    b.close()
    monkeypatch.setenv("TWEAKALIGN_COOP", "1")
    want = eng.align(pairs, params)
    for r in got:
        assert r == want
    return got[0], tasks


# Rows: strips of 128 (2 rows per lane); columns: blocks of 8, the 64-column window, the 128-column ring.
@pytest.mark.parametrize("mode", [ta.LOCAL, ta.GLOBAL])
@pytest.mark.parametrize("la", [1, 2, 63, 127, 128, 129, 256, 257, 640, 1025])
def test_strip_and_block_edges(eng, mode, la, monkeypatch):
    rng = random.Random(la + 7 * mode)
    a = rand_prot(rng, la)
    pairs = [(a, "")]
    for lb in (1, 7, 8, 9, 63, 64, 65, 127, 128, 129, 193, 1000):
        pairs.append((a, (mutate(rng, a) + rand_prot(rng, lb))[:lb]))
        pairs.append((a, rand_prot(rng, lb)))
    for go, ge in ((-11, -1), (-2, -7), (0, 0)):
        params = ta.engine.make_params(mode=mode, gap_open=go, gap_extend=ge)
        got, _ = both(eng, pairs, params, monkeypatch)
        compare(got, oracle_results(params, pairs), params, pairs, "strips %d %d" % (go, ge))


@pytest.mark.parametrize("mode", [ta.LOCAL, ta.GLOBAL])
@pytest.mark.parametrize("npairs, hi", [(1, 3000), (16, 5000), (300, 900), (3000, 100)])
def test_ragged_batches(eng, mode, npairs, hi, monkeypatch):
    rng = random.Random(npairs + hi + mode)
    pairs = []
    for k in range(npairs):
        a = rand_prot(rng, rng.randint(1, hi))
        pairs.append((a, mutate(rng, a) if k % 3 else rand_prot(rng, rng.randint(1, hi))))
    params = ta.engine.make_params(mode=mode, gap_open=-11)
    got, tasks = both(eng, pairs, params, monkeypatch, graph=npairs == 16)
    compare(got, oracle_results(params, pairs), params, pairs, "ragged")


def test_more_strips_than_waves_and_flags(eng, monkeypatch):
    # strips that wait for a wave; then int16 pairs and one past int16's range
    rng = random.Random(3)
    pairs = []
    for k in range(900):
        a = rand_prot(rng, rng.randint(600, 900))
        pairs.append((a, mutate(rng, a)))
    for mode in (ta.LOCAL, ta.GLOBAL):
        params = ta.engine.make_params(mode=mode)
        got, tasks = both(eng, pairs, params, monkeypatch)
        assert 5 * 900 <= tasks <= 8 * 900
        compare(got[:40], oracle_results(params, pairs[:40]), params, pairs[:40], "four rows")
    w = "W" * 3000  # 33,000 > 32,767: the packed lanes would saturate
    params = ta.engine.make_params(mode=ta.LOCAL)
    got, _ = both(eng, [(w, w), (w[:2000], w)], params, monkeypatch)
    assert got[0].flags == ta.F_I32 | ta.F_RERUN and got[1].flags == 0


@pytest.mark.parametrize("mode", [ta.LOCAL, ta.GLOBAL])
def test_dna_and_lanes(eng, mode, monkeypatch):
    rng = random.Random(11 + mode)
    pairs = []
    for _ in range(12):
        a = rand_prot(rng, rng.randint(1, 2500), "ACGT")
        pairs.append((a, mutate(rng, a, 0.1, 0.03, "ACGT")))
    for lanes in (ta.LANES_AUTO, ta.LANES_I16, ta.LANES_I32):
        params = ta.engine.make_params(mode=mode, alphabet=ta.DNA, gap_open=-5, gap_extend=-2, match=2, mismatch=-3,
                                       lanes=lanes)
        got, _ = both(eng, pairs, params, monkeypatch)
        compare(got, oracle_results(params, pairs), params, pairs, "dna")
    params = ta.engine.make_params(mode=mode, alphabet=ta.DNA, gap_open=-5, gap_extend=-2, match=2, mismatch=-3,
                                   traceback=0)
    both(eng, pairs, params, monkeypatch)
