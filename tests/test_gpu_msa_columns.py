"""A join's second cluster has at most the columns whose bottom rows fit a
CU's LDS: the last that fits against the oracle, the next one refused before
any launch, and the context good afterwards."""
import random

import pytest

import tweakseq_amd as ta
from test_gpu_msa import oracle_rows

pytestmark = pytest.mark.gpu

MOST = 20017  # (163,840 - 2,560) bytes of 8 a column, 80 + 63 of skew, blocks of 8


@pytest.fixture(scope="module")
def eng():
    e = ta.Engine(0)
    yield e
    e.close()


@pytest.mark.parametrize("la", [3, 150])
@pytest.mark.parametrize("lb", [MOST - 1, MOST, MOST + 1, 2 * MOST])
def test_columns_of_a_join(eng, la, lb):
    rng = random.Random(la + lb)
    b = "".join(rng.choice("ACGT") for _ in range(lb))
    seqs = [b[lb // 2:lb // 2 + la], b]
    p = ta.engine.make_params(mode=ta.GLOBAL, alphabet=ta.DNA, gap_open=-5, gap_extend=-2)
    if lb > MOST:
        with pytest.raises(RuntimeError, match="invalid argument"):
            eng.msa(seqs, p)
        seqs[1] = b[:1000]
    rows, joins = eng.msa(seqs, p)
    want, wjoins = oracle_rows(seqs, alphabet=1, go=-5, ge=-2)
    assert joins == wjoins and rows == want
