"""The traceback workgroup's cell (tweakseq_amd/csrc/long.h, long_tb_kernel):
why a barrier follows its reads.

Wave 0 walks a region and stores the cell the walk stopped at in two LDS
words; behind a barrier every wave reads them and decides from them whether
the next region is one computed ahead (no barriers) or is computed now (the
workgroup's barriers).  Between the reads and wave 0's next stores lies no
other barrier when the next region is one computed ahead: a wave that is late
then reads the next cell, or half of it, and the waves part.

On the CPU, a model of two waves is run in every order of their steps.  On the
GPU, walks that take one region ahead after the other are compared with the
oracle's."""
import random

import pytest

CELLS = [(9, 9), (7, 6), (4, 4), (0, 2)]  # where the walk of a region stops, region by region


def program(wave, ahead, barrier):
    """The steps of a wave: ("bar",) | ("put", word, value) | ("get", word).  It is sent what it reads."""
    seen, k = [], 0
    while True:
        if not ahead[k]:  # long_region
            yield ("bar",)
            yield ("bar",)
        if wave == 0:
            yield ("put", 0, CELLS[k][0])
            yield ("put", 1, CELLS[k][1])
        yield ("bar",)
        i = yield ("get", 0)
        j = yield ("get", 1)
        if barrier:
            yield ("bar",)
        seen.append((i, j))
        k += 1
        if i <= 0 or j <= 0:
            yield ("end", tuple(seen))
            return


def outcomes(ahead, barrier):
    """What both waves saw, over all orders of their steps (None: one waits at a barrier for good)."""
    def step(wave, sent):  # the wave's next step after the values it was sent
        g = program(wave, ahead, barrier)
        op = next(g)
        for v in sent:
            op = g.send(v)
        return op

    out, done = set(), set()
    todo = [((), (), (None, None))]
    while todo:
        state = todo.pop()
        if state in done:
            continue
        done.add(state)
        sent, words = list(state[:2]), state[2]
        ops = [step(w, sent[w]) for w in (0, 1)]
        if all(o[0] == "end" for o in ops):
            out.add((ops[0][1], ops[1][1]))
            continue
        if all(o[0] == "bar" for o in ops):
            todo.append((sent[0] + (None,), sent[1] + (None,), words))
            continue
        moved = False
        for w, o in enumerate(ops):
            if o[0] not in ("put", "get"):
                continue
            moved = True
            new, mem = [sent[0], sent[1]], list(words)
            if o[0] == "put":
                mem[o[1]] = o[2]
                new[w] += (None,)
            else:
                new[w] += (mem[o[1]],)
            todo.append((new[0], new[1], tuple(mem)))
        if not moved:
            out.add(None)
    return out


@pytest.mark.parametrize("ahead", [(True,) * 4, (False,) * 4, (False, True, True, False), (True, False, True, True)])
def test_every_wave_reads_the_same_cell(ahead):
    assert outcomes(ahead, True) == {(tuple(CELLS), tuple(CELLS))}


def test_without_the_barrier_the_waves_part():
    # two regions ahead in a row are enough; regions that are computed now bring barriers of their own
    assert len(outcomes((True,) * 4, False)) > 1
    assert outcomes((False,) * 4, False) == {(tuple(CELLS), tuple(CELLS))}


@pytest.mark.gpu
def test_walks_over_regions_ahead():
    import tweakseq_amd as ta
    from test_gpu_parity import compare, mutate, oracle_results, rand_prot

    rng = random.Random(17)
    pairs = []
    for n in (700, 2048, 4000, 6000, 6500, 7000):
        a = rand_prot(rng, n, "ACGT")
        pairs.append((a, mutate(rng, a, 0.1, 0.02, "ACGT")))
        pairs.append((a, rand_prot(rng, n, "ACGT")))
    params = ta.engine.make_params(mode=ta.GLOBAL, alphabet=ta.DNA, gap_open=-5, gap_extend=-2, match=2, mismatch=-3,
                                   lanes=ta.LANES_LONG)
    eng = ta.Engine(0)
    try:
        b = eng.batch(pairs, params)
        want = oracle_results(params, pairs)
        for _ in range(10):
            b.run()
            b.wait()
            compare(b.results(), want, params, pairs, "regions ahead")
        b.close()
    finally:
        eng.close()
