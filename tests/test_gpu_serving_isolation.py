"""Serving: a request that cannot run fails alone, whatever shares its batch."""
import random
import time

import pytest

import tweakseq_amd as ta
from test_gpu_parity import compare, mutate, oracle_results, rand_prot

pytestmark = pytest.mark.gpu


@pytest.fixture(params=["device_queue", "batches"])
def path(request, monkeypatch):
    monkeypatch.setenv("TWEAKALIGN_DEVICE_QUEUE", "1" if request.param == "device_queue" else "0")
    return request.param


def outcome(eng, ticket, n):
    t0 = time.time()
    while True:
        try:
            r = eng.poll(ticket, n)
        except RuntimeError as e:
            return str(e)
        if r is not None:
            return r
        assert time.time() - t0 < 60, "request still pending"
        time.sleep(0.001)


@pytest.mark.parametrize("nreq, bad", [(2, {0: "letter"}), (9, {4: "letter"}), (16, {0: "letter", 7: "length", 15: "letter"}),
                                       (5, {k: "letter" for k in range(5)})])
def test_bad_requests_fail_alone(path, nreq, bad):
    rng = random.Random(nreq)
    params = ta.engine.make_params(mode=ta.LOCAL, gap_open=-11, gap_extend=-1)
    reqs = []
    for q in range(nreq):
        pairs = []
        for _ in range(rng.randint(1, 4)):
            a = rand_prot(rng, rng.randint(1, 200))
            pairs.append((a, mutate(rng, a) or "A"))
        if q in bad:
            pairs[rng.randrange(len(pairs))] = ("ACD#EF", "ACDEF") if bad[q] == "letter" else ("A" * 1000001, "ACD")
        reqs.append(pairs)
    eng = ta.Engine(0)
    try:
        # one slot, held by requests of other parameters while the burst arrives
        eng.serve_config(64 << 30, 1)
        other = ta.engine.make_params(mode=ta.GLOBAL, alphabet=ta.DNA, gap_open=-5, gap_extend=-2, match=2, mismatch=-3)
        hold = [eng.submit([(rand_prot(rng, 2000, "ACGT"), rand_prot(rng, 2000, "ACGT"))], other) for _ in range(2)]
        tickets = [eng.submit(pairs, params) for pairs in reqs]
        for q, (t, n) in enumerate(tickets):
            got = outcome(eng, t, n)
            if q in bad:
                why = "residue outside the alphabet" if bad[q] == "letter" else "invalid argument"
                assert isinstance(got, str) and why in got, "request %d: %r" % (q, got)
            else:
                assert not isinstance(got, str), "request %d: %s" % (q, got)
                compare(got, oracle_results(params, reqs[q]), params, reqs[q], "beside a bad request")
        for t, n in hold:
            assert not isinstance(outcome(eng, t, n), str)
    finally:
        eng.close()
