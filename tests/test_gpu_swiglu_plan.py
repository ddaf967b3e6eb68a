"""GPU parity of SwiGLU plans whose members run as one grouped launch.

Members of one rate and codebook share a launch of two groups and one
activation launch over all rows; members that differ, and plans with diagnostic
buffers, launch one by one.  Every form gives the bits of the two strix_gemv
outputs through the activation's host restatement, for one row to eight, a
hidden view wider than its rows, widths that are no multiple of the activation
kernel's 256 columns, and a layer of a single input split.
"""
import numpy as np
import pytest

import synth
from oracle import moe

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from strix_trellis import runtime  # noqa: E402

DEV = "cuda:0"


@pytest.fixture(scope="module")
def ctx():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    c = runtime.Context(0)
    yield c
    torch.cuda.synchronize()


@pytest.mark.parametrize("I,H,bits,codebooks,rows", [
    (1024, 256, (4, 4), ("mul1", "mul1"), 1), (2048, 384, (5, 5), ("mcg", "mcg"), 8),
    (128, 128, (3, 3), ("mul1", "mul1"), 5), (1024, 384, (4, 5), ("mul1", "mul1"), 3),
    (1024, 256, (4, 4), ("mul1", "3inst"), 2)])
def test_swiglu_plan_forms(ctx, I, H, bits, codebooks, rows):
    print(f"swiglu plan {I}->{H} K={bits} {codebooks} R={rows}", flush=True)
    ws = [runtime.Weights(ctx, *synth.layer(I, H, k, 8200 + I + i, bias=i == 1), cb)
          for i, (k, cb) in enumerate(zip(bits, codebooks))]
    x = torch.from_numpy(synth.activations(rows, I, 8201)).to(DEV)
    parts = []
    for w in ws:
        y = torch.empty((rows, H), device=DEV)
        runtime.gemv(w, x, y)
        parts.append(y.cpu().numpy())
    want = moe.swiglu(*parts).view(np.uint32)
    wide = torch.full((rows, H + 96), 7.0, device=DEV)
    plan = runtime.TpSwigluPlan(*ws, x, wide[:, :H])
    for _ in range(3):
        wide[:, :H] = float("nan")
        plan.submit()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(wide[:, :H].cpu().numpy().view(np.uint32), want)
    assert bool((wide[:, H:] == 7.0).all())
    # replayed from a graph, inputs rewritten in between
    g = torch.cuda.CUDAGraph()
    s = torch.cuda.Stream()
    hidden = torch.empty((rows, H), device=DEV)
    cap = runtime.TpSwigluPlan(*ws, x, hidden, stream=s)
    with torch.cuda.graph(g, stream=s):
        cap.submit()
    for i in range(3):
        x.copy_(torch.from_numpy(synth.activations(rows, I, 8202 + i)))
        hidden.fill_(float("nan"))
        plan.submit()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(hidden.view(torch.int32), wide[:, :H].contiguous().view(torch.int32))
    for p in (plan, cap):
        p.destroy()
    for w in ws:
        w.destroy()


def test_swiglu_graph_outlives_its_plan(ctx):
    """Rows and state of a destroyed plan stay with the weights: a graph captured
    from it replays with the same bits, and touches nothing allocated since."""
    I, H, rows = 1024, 256, 3
    print(f"swiglu graph after destroy {I}->{H} R={rows}", flush=True)
    ws = [runtime.Weights(ctx, *synth.layer(I, H, 4, 8400 + i, bias=False), "mul1") for i in range(2)]
    x = torch.from_numpy(synth.activations(rows, I, 8401)).to(DEV)
    hidden, want = torch.empty((rows, H), device=DEV), torch.empty((rows, H), device=DEV)
    g, s = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    cap = runtime.TpSwigluPlan(*ws, x, hidden, stream=s)
    with torch.cuda.graph(g, stream=s):
        cap.submit()
    cap.destroy()
    others = [runtime.TpSwigluPlan(*ws, x, want) for _ in range(4)]   # the sizes a freed block would go to
    guards = [torch.full((n,), 7.0, device=DEV) for n in (2048, 4096, 65536)]
    for i in range(4):
        x.copy_(torch.from_numpy(synth.activations(rows, I, 8402 + i)).to(DEV))
        others[i].submit()
        hidden.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(hidden.view(torch.int32), want.view(torch.int32))
    assert all(bool((t == 7.0).all()) for t in guards)
    for p in others:
        p.destroy()
    for w in ws:
        w.destroy()
