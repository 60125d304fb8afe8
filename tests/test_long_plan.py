"""Memory of long pairs: plans stay within what a request is admitted for
(tests/native/long_plan_check.cpp, CPU), served long pairs keep to the budget,
and pairs that share memory in groups give the same results."""
import os
import random
import shutil
import subprocess
import time

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_plans_within_admission(tmp_path):
    exe = str(tmp_path / "long_plan_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-fsanitize=undefined", "-fno-sanitize-recover=all",
                    os.path.join(ROOT, "tests", "native", "long_plan_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "long plan ok" in r.stdout, r.stdout + r.stderr


def dna(rng, n):
    return "".join(rng.choice("ACGT") for _ in range(n))


def served(eng, pairs, params):
    t, n = eng.submit(pairs, params)
    t0 = time.time()
    while True:
        r = eng.poll(t, n, params.traceback)
        if r is not None:
            return r
        assert time.time() - t0 < 60, "request still pending"
        time.sleep(0.001)


@pytest.mark.gpu
def test_served_long_pairs_keep_to_the_budget():
    # 30,000 x 30,000: rows and columns 28.3 MB, a region's codes 0.3 MB, regions ahead 20 MB
    import tweakseq_amd as ta
    rng = random.Random(2)
    a = dna(rng, 30000)
    b = a[:9000] + dna(rng, 40) + a[9100:]
    b = (b + dna(rng, 200))[:30000]
    params = dict(mode=ta.GLOBAL, alphabet=ta.DNA, gap_open=-5, gap_extend=-2, match=2, mismatch=-3)
    eng = ta.Engine(0)
    try:
        p = ta.engine.make_params(**params)
        want = eng.align([(a, b)], p)
        assert want[0].flags & ta.F_LONG
        eng.serve_config(25 << 20, 2)
        with pytest.raises(RuntimeError, match="budget"):
            eng.submit([(a, b)], p)
        score = ta.engine.make_params(traceback=0, **params)  # no traceback memory: not refused
        assert served(eng, [(a, b)], score)[0].score == want[0].score
        eng.serve_config(30 << 20, 2)  # enough without regions ahead
        assert served(eng, [(a, b)], p) == want
        eng.serve_config(64 << 20, 2)
        assert served(eng, [(a, b), (b[:7000], a[:7000])], p) == want + eng.align([(b[:7000], a[:7000])], p)
    finally:
        eng.close()


@pytest.mark.gpu
@pytest.mark.parametrize("traceback", [0, 1])
@pytest.mark.parametrize("limit", [0, 700_000, 3_000_000, 40_000_000])
def test_groups_share_memory(limit, traceback, monkeypatch):
    # no room but for one pair at a time; for a few; for some regions ahead; for all
    import tweakseq_amd as ta
    from test_gpu_parity import compare, mutate, oracle_results, rand_prot

    rng = random.Random(limit % 1000 + 3)
    pairs = []
    for n in (3000, 60, 1024, 513, 2100, 512, 2999, 1, 1500):
        a = dna(rng, n)
        pairs.append((a, mutate(rng, a, 0.1, 0.02, "ACGT") or "A"))
        pairs.append((dna(rng, rng.randint(1, 2000)), a))
    params = ta.engine.make_params(mode=ta.GLOBAL, alphabet=ta.DNA, gap_open=-5, gap_extend=-2, match=2, mismatch=-3,
                                   lanes=ta.LANES_LONG, traceback=traceback)
    monkeypatch.setenv("TWEAKALIGN_LONG_BYTES", str(limit))
    eng = ta.Engine(0)
    try:
        b = eng.batch(pairs, params)
        want = oracle_results(params, pairs)
        for graph in (False, True):
            b.graph(graph)
            for _ in range(3):
                b.run()
                b.wait()
                compare(b.results(), want, params, pairs, "groups %d" % limit)
        b.run_plain(0, len(pairs))
        b.wait()
        compare(b.results(), want, params, pairs, "plain %d" % limit)
        b.close()
    finally:
        eng.close()
