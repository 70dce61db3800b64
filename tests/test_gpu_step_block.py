"""The step in one launch (final states sorted by process within a block): at the
edges of its waves, blocks, tiles and, in FP64, of the sizes that take it, in
both forms, against the fused step without any sort, bit for bit, and in place.
"""
import numpy as np
import pytest

from conftest import STEP_SEED

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

ROUND = 256 * 3 * 256  # slots of one resident round: the largest FP64 batch stepped in one launch


@pytest.fixture(scope="module", params=["fp64", "fp32"])
def ctx(request, tables2):
    from g4hepem_amd import HEPEM_FP32T, HEPEM_FP64, Context
    assert torch.cuda.is_available(), "GPU test run without a visible GPU"
    return Context(tables2, HEPEM_FP64 if request.param == "fp64" else HEPEM_FP32T)


def _tracks(n, kind):
    from g4hepem_amd.tracks import step_tracks, type_ordered
    t = step_tracks(n, 31, 4, lnemin=np.log(1e-2), lnemax=np.log(1e5))
    if kind == "gammas":
        t["ptype"][:] = 2
    elif kind == "positrons":
        t["ptype"][:] = 1
    if n > 2:
        t["imc"][n // 2] = -1   # rejected
        t["on_boundary"][n - 1] = 1
    return type_ordered(t) if kind == "ordered" else t


def _step(ctx, t, sort, in_place=False):
    from g4hepem_amd.tracks import StepOutSoA, TrackSoA
    n = len(t["ekin"])
    tin = TrackSoA.from_numpy(t, "torch", "cuda")
    tout = tin if in_place else TrackSoA(n, "torch", "cuda")
    res = StepOutSoA(n, "torch", "cuda")
    work = ctx.work_buffer(n, "cuda")
    ctx.set_process_sort(sort)
    try:
        ctx.step(STEP_SEED, tin, tout, res, work)
        rejected = ctx.rejected(work)
    finally:
        ctx.set_process_sort("auto")
    return tin, tout, res, rejected


@pytest.mark.parametrize("kind", ["mixed", "ordered", "gammas", "positrons"])
@pytest.mark.parametrize("n", [1, 63, 255, 256, 257, 4095, 4097, ROUND, ROUND + 1])
def test_one_launch_step(ctx, n, kind):
    from g4hepem_amd.tracks import step_outputs_differ
    print(f"one-launch step n={n} {kind}", flush=True)
    t = _tracks(n, kind)
    tin, t_ref, r_ref, rej_ref = _step(ctx, t, False)
    _, t_got, r_got, rej = _step(ctx, t, True)
    assert rej == rej_ref == (1 if n > 2 else 0)
    assert not step_outputs_differ(tin["ptype"], t_got, r_got, t_ref, r_ref)
    _, t_got, r_got, _ = _step(ctx, t, True, in_place=True)
    assert not step_outputs_differ(tin["ptype"], t_got, r_got, t_ref, r_ref)
