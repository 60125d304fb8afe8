"""Device-queue serving beside batches: requests that the queue takes go there
also while a batch gathers, and letter requests through the queue mix with
requests on resident sequences, which go to batches."""
import random
import time

import pytest

import tweakseq_amd as ta
import test_gpu_resident
from test_gpu_parity import compare, mutate, oracle_results, rand_prot

pytestmark = pytest.mark.gpu


def test_a_gathering_batch_leaves_queue_requests_alone(monkeypatch):
    # A request too long for the queue, then a stream of short ones with the same parameters.  In its batch they
    # would wait for it (its cells take 50 ms and more beside the queue's kernel); the queue takes 1 ms.
    monkeypatch.setenv("TWEAKALIGN_DEVICE_QUEUE", "1")
    rng = random.Random(3)
    params = ta.engine.make_params(mode=ta.LOCAL, gap_open=-11, gap_extend=-1)
    long_pairs = [(rand_prot(rng, 20000), rand_prot(rng, 12000)) for _ in range(4)]
    short = []
    for _ in range(100):
        a = rand_prot(rng, 40)
        short.append([(a, mutate(rng, a) or "A")])
    eng = ta.Engine(0)
    try:
        eng.serve_config(64 << 30, 4)
        for _ in range(2):  # the queue's kernel runs
            t, n = eng.submit(short[0], params)
            while eng.poll(t, n) is None:
                time.sleep(1e-4)
        first = eng.submit(long_pairs, params)
        tickets = [eng.submit(p, params) for p in short]
        got, t0 = [None] * len(short), time.time()
        long_res = None
        while any(g is None for g in got):
            assert long_res is None, "%d short requests waited for the long one" % sum(g is None for g in got)
            got = [eng.poll(t, n) if g is None else g for g, (t, n) in zip(got, tickets)]
            long_res = eng.poll(*first)
            assert time.time() - t0 < 60
        for p, g in zip(short, got):
            compare(g, oracle_results(params, p), params, p, "queue beside a batch")
        while long_res is None:
            long_res = eng.poll(*first)
            assert time.time() - t0 < 60
        assert long_res == eng.align(long_pairs, params)
    finally:
        eng.close()


@pytest.mark.parametrize("queue", ["0", "1"])
def test_resident_beside_letter_requests(queue, monkeypatch):
    monkeypatch.setenv("TWEAKALIGN_DEVICE_QUEUE", queue)
    eng = ta.Engine(0)
    try:
        test_gpu_resident.test_served_resident_requests_equal_oracle(eng)
    finally:
        eng.close()
