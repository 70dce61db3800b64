"""The process layout of a tile's pending interactions and its final states
(k_classify_tiles, k_interact_tiles) at the ends of a thread's slots, a wave's, a
tile's: batches of every size reach them through the split Perform with the
process sort, while hepem_step takes them for large batches only. Against the
split Perform without the sort bit for bit, in both forms, and in FP64 against
the oracle with the tolerances of test_gpu_parity.
"""
import numpy as np
import pytest

from conftest import STEP_SEED
from test_gpu_parity import compare_step

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", params=["fp64", "fp32"])
def ctx(request, tables2):
    from g4hepem_amd import HEPEM_FP32T, HEPEM_FP64, Context
    assert torch.cuda.is_available(), "GPU test run without a visible GPU"
    c = Context(tables2, HEPEM_FP64 if request.param == "fp64" else HEPEM_FP32T)
    c.form = request.param
    return c


def _tracks(n, kind):
    from g4hepem_amd.tracks import step_tracks
    t = step_tracks(n, 41, 4, lnemin=np.log(1e-2), lnemax=np.log(1e5))
    if kind == "electron":
        t["ptype"][:] = np.arange(n) % 5 == 4
    elif kind == "gamma":
        t["ptype"][:] = 2
    elif kind == "one process":  # 10 keV gammas in lead: nearly all take the photoelectric effect
        t["ptype"][:] = 2
        t["ekin"][:] = 1e-2
        t["imc"][:] = 1
    return t


def _split(ctx, t, sort, kind):
    from g4hepem_amd.tracks import HowFarSoA, StepOutSoA, TrackSoA
    n = len(t["ekin"])
    tr, hs, res = TrackSoA.from_numpy(t, "torch", "cuda"), HowFarSoA(n, "torch", "cuda"), StepOutSoA(n, "torch", "cuda")
    work = ctx.work_buffer(n, "cuda")
    kind = kind if kind in ("electron", "gamma") else "mixed"
    ctx.set_process_sort(sort)
    try:
        ctx.howfar(STEP_SEED, tr, hs, work, kind=kind)
        ctx.perform(STEP_SEED, tr, hs, res, work, kind=kind)
        rejected = ctx.rejected(work)
    finally:
        ctx.set_process_sort("auto")
    return tr, res, rejected


@pytest.mark.parametrize("kind", ["mixed", "electron", "gamma", "one process"])
@pytest.mark.parametrize("n", [1, 3, 4, 5, 63, 64, 65, 255, 257, 4093, 4095, 4096, 4097, 8191, 8195])
def test_process_layout_edges(ctx, tables2, oracle, n, kind):
    from g4hepem_amd.tracks import step_outputs_differ
    print(f"process layout {ctx.form} n={n} {kind}", flush=True)
    t = _tracks(n, kind)
    t_ref, r_ref, rej_ref = _split(ctx, t, False, kind)
    t_got, r_got, rej = _split(ctx, t, True, kind)
    assert rej == rej_ref == 0
    assert not step_outputs_differ(t_got["ptype"], t_got, r_got, t_ref, r_ref)
    if ctx.form == "fp64":
        to, ro = oracle.step(tables2, STEP_SEED, t, nthreads=4)
        compare_step(t, t_got.to_numpy(), r_got.to_numpy(), to, ro, label=f"n={n} {kind}")
