"""The draw counter of a track is 32 bits and goes on at 0 after its last value:
draw d of a stream lies in random block d >> 1, also for the draws taken in
pairs, triples and runs across the end. Against the oracle, which draws one by
one; tolerances as in test_gpu_parity.
"""
import numpy as np
import pytest

from conftest import STEP_SEED
from test_gpu_parity import compare_step, ctx2, dev, gpu_step  # noqa: F401

pytestmark = pytest.mark.gpu


def _tracks(n, ptype):
    """All patterns of used-up interaction lengths, the counter 1 ... 64 draws
    before its end, energies over the whole range."""
    from g4hepem_amd.tracks import step_tracks
    t = step_tracks(n, 78, 4)
    i = np.arange(n)
    if ptype is not None:
        t["ptype"][:] = ptype
    rng = np.random.default_rng(6)
    nial = t["num_ia_left"].reshape(4, n)
    for k in range(4):
        nial[k] = np.where((i >> k) & 1, -1.0, rng.exponential(size=n) + 1e-3)
    t["rng_ctr"][:] = np.uint32(0xFFFFFFFF) - ((i >> 4) & 63).astype(np.uint32)
    return t


@pytest.mark.parametrize("ptype", [0, 1, 2, None], ids=["electrons", "positrons", "gammas", "mixed"])
@pytest.mark.parametrize("sort", [True, False], ids=["sorted", "fused"])
def test_draws_across_the_counters_end(tables2, ctx2, oracle, dev, ptype, sort):
    t = _tracks(8192, ptype)
    print(f"draw counter's end ptype={ptype} sort={sort}", flush=True)
    ctx2.set_process_sort(sort)
    try:
        tg, rg, rej = gpu_step(ctx2, STEP_SEED, t, dev)
    finally:
        ctx2.set_process_sort("auto")
    tr, rr = oracle.step(tables2, STEP_SEED, t, nthreads=4)
    assert rej == 0
    assert np.any(tr["rng_ctr"] < t["rng_ctr"])
    compare_step(t, tg, rg, tr, rr, label=f"ptype={ptype}")
