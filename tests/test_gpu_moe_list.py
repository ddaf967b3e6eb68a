"""The routed-expert block's group list: against the oracle, and its down half
against the route resolution of a down launch of its own.

The input launch ahead of every gate/up lists the expert groups, which gate/up
and a submission's down read; a down launch of its own resolves the routes
itself.  For any routes (shared and distinct experts, zero scores, tokens that
are invalid by an id outside the bank, a repeated id, a negative or non-finite
score, one to 64 routes, a bank as small as one expert, routes rewritten between
submissions) hidden and the block output meet the block's bars against the staged
FP32 oracle, and both downs give the same bits.
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


def _draw(g, E, rows, k, case):
    ids = np.stack([g.choice(E, k, replace=False) for _ in range(rows)]).astype(np.int32)
    sc = g.uniform(0.1, 1.0, (rows, k)).astype(np.float32)
    if case == "same":
        ids[:] = ids[0]
    for r in range(rows):
        if case == "mixed" and r % 3 == 1:
            bad = r // 3 % 4
            if bad == 0:
                ids[r, k - 1] = E
            elif bad == 1 and k > 1:
                ids[r, 0] = ids[r, k - 1]
            elif bad == 2:
                sc[r, 0] = -1.0
            else:
                sc[r, k - 1] = np.inf
        elif case == "mixed":
            sc[r, g.integers(0, k)] = 0.0
        elif case == "invalid":
            ids[r, 0] = E + r
    return ids, sc


@pytest.mark.parametrize("E,rows,k", [(1, 1, 1), (6, 1, 4), (9, 8, 8), (8, 8, 3), (40, 5, 6)])
def test_list_matches_own_resolution(ctx, E, rows, k):
    I, H = 512, 256
    bank = synth.moe_bank(E, I, H, 2, 9100 + E)
    ws = [tuple(runtime.Weights(ctx, *e[n][:4], "mul1") for n in ("gate", "up", "down")) for e in bank]
    xh = synth.activations(rows, I, 9101)
    x = torch.from_numpy(xh).to(DEV)
    cache = {}
    ids = torch.zeros((rows, k), dtype=torch.int32, device=DEV)
    sc = torch.zeros((rows, k), device=DEV)
    y0, y1 = torch.empty((rows, I), device=DEV), torch.empty((rows, I), device=DEV)
    listed = runtime.MoePlan(ctx, ws, x, y0, device_ids=ids, device_scores=sc)
    own = runtime.MoePlan(ctx, ws, x, y1, device_ids=ids, device_scores=sc)
    g = synth.rng(9102)
    for case in ("plain", "mixed", "same", "invalid", "mixed"):
        i, s = _draw(g, E, rows, k, case)
        print(f"moe list E={E} rows={rows} k={k} {case}", flush=True)
        ids.copy_(torch.from_numpy(i))
        sc.copy_(torch.from_numpy(s))
        y0.fill_(7.0)
        y1.fill_(7.0)
        listed.hidden.fill_(7.0)
        listed.submit()
        own.gate_up()
        own.down()
        torch.cuda.synchronize()
        assert torch.equal(y0.view(torch.int32), y1.view(torch.int32)), case
        if case == "invalid":
            assert bool(torch.isnan(y0).all())
        got, hidden = y0.cpu().numpy(), listed.hidden.cpu().numpy().reshape(rows, k, H)
        ref, href = moe.moe_block(xh, bank, i, s, cache=cache)
        valid = moe.token_valid(i, s, E)
        assert np.isnan(got[~valid]).all()
        done = valid[:, None] & (s != 0)
        assert (hidden[~done] == 7.0).all()   # no route but these is written
        if done.any():
            # hidden = SwiGLU of two projections: twice the single-linear bar; the
            # down half from the device's own hidden: the single-linear gate; the
            # three projections in a row: 1e-3 of the largest value
            a, r = hidden[done].astype(np.float64), href[done].astype(np.float64)
            assert np.max(np.abs(a - r)) <= 5e-4 * max(1.0, np.max(np.abs(r)))
            assert np.sqrt(np.sum((a - r) ** 2) / np.sum(r ** 2)) <= 6e-5
            synth.gate(got[valid], moe.down_combine(hidden, bank, i, s, cache=cache)[valid])
            assert np.max(np.abs(got[valid] - ref[valid])) <= 1e-3 * np.max(np.abs(ref[valid]))
    for p in (listed, own):
        p.destroy()
    for e in ws:
        for w in e:
            w.destroy()
