"""Draw order of the per-track streams: every pattern of used-up interaction
lengths from every position in a random block, against the oracle.

The kernels draw pairs and triples a random block at a time and hand the draws
of several interaction lengths out together; the draws a track takes, and the
count it stores, must be those of one-by-one drawing. Tolerances as in
test_gpu_parity (integers exact, floats within 1e-12 relative).
"""
import numpy as np
import pytest

from conftest import STEP_SEED
from test_gpu_parity import compare_step, ctx2, ctx2_32, dev, gpu_step  # noqa: F401

pytestmark = pytest.mark.gpu


def _tracks(n, ptype):
    """Tracks with all 16 patterns of used-up lengths x 8 draw counters, with
    and without a cached Gaussian, energies over the whole range."""
    from g4hepem_amd.tracks import step_tracks
    t = step_tracks(n, 77, 4, mix=(4, 1, 5))
    i = np.arange(n)
    if ptype is not None:
        t["ptype"][:] = ptype
    rng = np.random.default_rng(5)
    nial = t["num_ia_left"].reshape(4, n)
    for k in range(4):
        nial[k] = np.where((i >> k) & 1, -1.0, rng.exponential(size=n) + 1e-3)
    t["rng_ctr"][:] = (i >> 4) & 7
    t["rng_has_gauss"][:] = (i >> 7) & 1
    t["rng_gauss"][:] = np.where((i >> 7) & 1, rng.normal(size=n), 0.0)
    return t


@pytest.mark.parametrize("ptype", [0, 1, 2, None], ids=["electrons", "positrons", "gammas", "mixed"])
@pytest.mark.parametrize("sort", [True, False], ids=["sorted", "fused"])
def test_draw_order(tables2, ctx2, oracle, dev, ptype, sort):
    t = _tracks(2048, ptype)
    print(f"draw order ptype={ptype} sort={sort}", flush=True)
    ctx2.set_process_sort(sort)
    try:
        tg, rg, rej = gpu_step(ctx2, STEP_SEED, t, dev)
    finally:
        ctx2.set_process_sort("auto")
    tr, rr = oracle.step(tables2, STEP_SEED, t, nthreads=4)
    assert rej == 0
    compare_step(t, tg, rg, tr, rr, label=f"ptype={ptype}")


@pytest.mark.parametrize("n", [1, 3, 4, 5, 64, 255, 4093, 4095, 4096, 4097, 8191, 8195])
@pytest.mark.parametrize("ptype", [0, 2, None], ids=["electrons", "gammas", "mixed"])
def test_tile_layout_edges(tables2, ctx2, oracle, dev, n, ptype):
    """Ends of a thread's slots, of a wave's and of a tile's in the particle and
    process layouts: the sorted step against the oracle on every slot."""
    t = _tracks(n, ptype)
    print(f"tile layout n={n} ptype={ptype}", flush=True)
    tg, rg, rej = gpu_step(ctx2, STEP_SEED + 1, t, dev)
    tr, rr = oracle.step(tables2, STEP_SEED + 1, t, nthreads=4)
    assert rej == 0
    compare_step(t, tg, rg, tr, rr, label=f"n={n}")
