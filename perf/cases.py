"""Performance cases of the trellis linear layers on one GPU.

Each case is one pass through a public entry point, on sizes of the
repository's benchmark, tests and tensor-parallel site table:

* decode: prepared GEMV plans of 1-8 rows, the output head, the grouped `o_a`
  plan, the shared expert's SwiGLU plan and the routed-expert block;
* batched decode and prefill: GEMM plans and `strix_gemm` calls of a few to a
  few thousand rows.

The inputs come from the seed alone.  `exact` restates a pass in plain torch
without the library: the format's own roundings (FP16 weights, FP16 core
inputs) are kept, every sum after them is taken in FP64.
"""
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "strix-trellis_amd"))

from strix_trellis import runtime  # noqa: E402

DEV = "cuda:0"

# ---------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------


def listed():
    return [
        # One token through a square projection: the smallest call, where the
        # launch and the two memory round trips count.
        {"name": "decode_r1", "kind": "gemv", "I": 4096, "N": 4096, "K": 4, "rows": 1,
         "codebook": "mul1", "bias": False},
        # Eight concurrent sequences through the hidden-size projection.
        {"name": "decode_r8", "kind": "gemv", "I": 5120, "N": 5120, "K": 5, "rows": 8,
         "codebook": "mul1", "bias": True},
        # One token through the output head, the largest layer of a model.
        {"name": "head_r1", "kind": "gemv", "I": 5120, "N": 129280, "K": 6, "rows": 1,
         "codebook": "mul1", "bias": False},
        # The attention output's grouped low-rank projection of a decode batch.
        {"name": "grouped_r4", "kind": "grouped", "G": 16, "I": 4096, "N": 1024, "K": 5, "rows": 4},
        # A tensor-parallel rank's half of the shared expert (gate, up, SwiGLU),
        # written into a wider activation.
        {"name": "swiglu_r6", "kind": "swiglu", "I": 5120, "N": 1152, "K": 4, "rows": 6},
        # Routed experts of one token: top-6 on a rank's half experts.
        {"name": "moe_r1", "kind": "moe", "E": 48, "I": 5120, "H": 1152, "K": 2, "rows": 1, "top": 6},
        # Routed experts of a decode batch: most of the bank is touched.
        {"name": "moe_r8", "kind": "moe", "E": 64, "I": 4096, "H": 1536, "K": 2, "rows": 8, "top": 8},
        # Decode of a batch past the GEMV's eight rows (a serving batch bucket).
        {"name": "batch_m24", "kind": "gemm_plan", "I": 5120, "N": 5120, "K": 5, "rows": 24,
         "codebook": "mul1", "bias": False},
        # A short prompt, odd length, the second codebook and a bias.
        {"name": "prefill_m200", "kind": "gemm", "I": 4096, "N": 12288, "K": 6, "rows": 200,
         "codebook": "mcg", "bias": True},
        # A medium prompt on a square layer: fewer tiles than compute units.
        {"name": "prefill_m512", "kind": "gemm", "I": 5120, "N": 5120, "K": 4, "rows": 512,
         "codebook": "mul1", "bias": False},
        # A prefill chunk through the widest dense layer.
        {"name": "prefill_m2048", "kind": "gemm", "I": 4096, "N": 12288, "K": 4, "rows": 2048,
         "codebook": "mul1", "bias": False},
        # A long ragged chunk through a rank's low-rank query expansion: a
        # short K, so outputs weigh as much as products.
        {"name": "prefill_m3000", "kind": "gemm", "I": 1280, "N": 16384, "K": 5, "rows": 3000,
         "codebook": "mul1", "bias": False},
    ]


# Dense layers of the benchmark and of the tensor-parallel sites (whole and per rank).
_DENSE = [(4096, 4096), (5120, 5120), (4096, 12288), (1280, 32768), (1280, 16384), (8192, 5120), (4096, 5120),
          (5120, 2304), (5120, 1152), (2304, 5120), (1152, 5120), (5120, 1280), (5120, 512), (2048, 2048)]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "grouped", "swiglu", "moe", "gemm_plan", "gemm", "gemm", "gemm"])
    codebook = rng.choice(["mul1", "mul1", "mul1", "mcg", "3inst"])
    if kind in ("gemv", "gemm", "gemm_plan"):
        I, N = rng.choice(_DENSE)
        if kind == "gemv":
            rows = rng.randint(1, 8)
        elif kind == "gemm_plan":
            rows = _log_int(rng, 9, 128)
        else:
            rows = _log_int(rng, 48, min(4096, 2048 * 4096 * 12288 // (I * N)))
        return {"kind": kind, "I": I, "N": N, "K": rng.choice([2, 3, 4, 4, 5, 5, 6, 8]), "rows": rows,
                "codebook": codebook, "bias": rng.random() < 0.3}
    if kind == "grouped":
        return {"kind": kind, "G": rng.choice([2, 4, 8, 16]), "I": rng.choice([2048, 4096]), "N": 1024,
                "K": rng.choice([4, 5]), "rows": rng.randint(1, 8)}
    if kind == "swiglu":
        return {"kind": kind, "I": rng.choice([4096, 5120]), "N": rng.choice([1152, 1536, 2304]),
                "K": rng.choice([4, 5]), "rows": rng.randint(1, 8)}
    I, H = rng.choice([(5120, 1152), (5120, 2304), (4096, 1536)])
    rows = rng.randint(1, 8)
    return {"kind": kind, "E": rng.randint(24, 64), "I": I, "H": H, "K": rng.choice([2, 2, 3]), "rows": rows,
            "top": rng.choice([2, 4, 6, 8])}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------


def _rng(case, seed, part=0):
    return np.random.Generator(np.random.SFC64([seed, part, case["I"], case["rows"]]))


def _layer(g, I, N, K, bias=False):
    """A packed layer: any bits are a valid trellis (decoded weights of order
    one); suh holds signs, svh signs with a per-column scale that keeps the
    outputs of order one."""
    trellis = np.frombuffer(g.bytes(I * N * K // 8), dtype=np.uint16).reshape(I // 16, N // 16, 16 * K)
    suh = (1.0 - 2.0 * g.integers(0, 2, I)).astype(np.float16)
    svh = ((1.0 - 2.0 * g.integers(0, 2, N)) * g.uniform(0.5, 1.5, N) / math.sqrt(I)).astype(np.float16)
    b = g.standard_normal(N, dtype=np.float32) if bias else None
    return trellis, suh, svh, b


def _activations(g, rows, width):
    """Normalised hidden states: a spread of channel scales."""
    scale = np.exp(0.5 * g.standard_normal(width, dtype=np.float32))
    return torch.from_numpy(g.standard_normal((rows, width), dtype=np.float32) * scale).to(DEV)


def _routes(g, case):
    rows, top, E = case["rows"], case["top"], case["E"]
    ids = np.stack([g.choice(E, top, replace=False) for _ in range(rows)]).astype(np.int32)
    logits = g.standard_normal((rows, top)).astype(np.float32)
    e = np.exp(logits - logits.max(axis=1, keepdims=True))
    return ids, (e / e.sum(axis=1, keepdims=True)).astype(np.float32)


_CONTEXT = []


def _context():
    if not _CONTEXT:
        _CONTEXT.append(runtime.Context(0))
    return _CONTEXT[0]


class _State:
    """Buffers, weights and plan of one case; the library's handles go with it."""

    def __init__(self):
        self.plan, self.weights = None, []

    def __del__(self):
        try:
            torch.cuda.synchronize()
            if self.plan is not None:
                self.plan.destroy()
            for w in self.weights:
                w.destroy()
        except Exception:
            pass


def prepare(case, seed):
    s, ctx, rows = _State(), _context(), case["rows"]
    s.kind = case["kind"]
    g = _rng(case, seed)

    def weights(g, I, N, K, bias=False, codebook="mul1"):
        w = runtime.Weights(ctx, *_layer(g, I, N, K, bias), codebook)
        w._keep = []   # preparation has copied the host arrays
        s.weights.append(w)
        return w

    if s.kind in ("gemv", "gemm", "gemm_plan"):
        w = weights(g, case["I"], case["N"], case["K"], case["bias"], case["codebook"])
        s.x = _activations(g, rows, case["I"])
        s.y = torch.zeros((rows, case["N"]), device=DEV)
        if s.kind == "gemm":
            s.workspace = runtime.alloc_workspace(runtime.workspace_bytes(w, s.x, s.y), DEV)
        else:
            s.plan = runtime.LinearPlan(w, s.x, s.y, operation="gemv" if s.kind == "gemv" else "gemm")
    elif s.kind == "grouped":
        G, I, N = case["G"], case["I"], case["N"]
        ws = [weights(g, I, N, case["K"]) for _ in range(G)]
        s.x = _activations(g, rows, G * I)
        s.y = torch.zeros((rows, G * N), device=DEV)
        s.plan = runtime.GroupedGemvPlan(ws, s.x, s.y, rows, I, N, G * I, G * N)
    elif s.kind == "swiglu":
        I, N = case["I"], case["N"]
        gate, up = weights(g, I, N, case["K"]), weights(g, I, N, case["K"])
        s.x = _activations(g, rows, I)
        s.wide = torch.zeros((rows, 2 * N), device=DEV)
        s.y = s.wide[:, :N]
        s.plan = runtime.TpSwigluPlan(gate, up, s.x, s.y)
    else:
        I, H, K = case["I"], case["H"], case["K"]
        s.x = _activations(g, rows, I)
        ids, scores = _routes(g, case)
        s.ids, s.scores = torch.from_numpy(ids).to(DEV), torch.from_numpy(scores).to(DEV)
        experts = []
        for e in range(case["E"]):
            ge = _rng(case, seed, 1 + e)
            experts.append((weights(ge, I, H, K), weights(ge, I, H, K), weights(ge, H, I, K)))
        s.y = torch.zeros((rows, I), device=DEV)
        s.plan = runtime.MoePlan(ctx, experts, s.x, s.y, device_ids=s.ids, device_scores=s.scores)
    torch.cuda.synchronize()
    return s


def run(state):
    if state.kind == "gemm":
        return runtime.gemm(state.weights[0], state.x, state.y, workspace=state.workspace)
    state.plan.submit()
    return state.y


def work(case):
    rows, K = case["rows"], case["K"]
    if case["kind"] == "moe":
        I, H, top = case["I"], case["H"], case["top"]
        # every distinct expert of the routes is read once (its count depends
        # on the routes: the expected one of uniform draws)
        E = case["E"]
        experts = E * (1.0 - (1.0 - top / E) ** rows)
        per = 3 * (I * H * K // 8 + 2 * (I + H))
        return {"bytes": int(experts * per + rows * (2 * I * 4 + 8 * top)), "flops": 6 * rows * top * I * H}
    I, N = case["I"], case["N"]
    n = case.get("G", 1) * (2 if case["kind"] == "swiglu" else 1)
    inputs = case.get("G", 1) * I
    outputs = case.get("G", 1) * N
    weights = n * (I * N * K // 8 + 2 * (I + N) + (4 * N if case.get("bias") else 0))
    return {"bytes": weights + 4 * rows * (inputs + outputs), "flops": 2 * rows * n * I * N}


def tolerance(case):
    # 32-bit sums of exact FP16 products: 1.3e-7 to 4.1e-7 from `exact` as
    # measured, four to eight times that allowed.  The routed experts round the
    # hidden vector to FP16 between two products, where the last bit of a sum
    # moves some elements by one FP16 step: 1.8e-5 to 6e-5 measured.
    if case["kind"] == "moe":
        return {"rel": 2.4e-4, "max": 2e-3}
    return {"rel": 2e-6, "max": 2e-5}


# ---------------------------------------------------------------------------
# The same passes in plain torch
# ---------------------------------------------------------------------------

_MULTIPLIER = {"mul1": 0x83DCD12D, "mcg": 0xCBAC1FED, "3inst": 89226354}


def _codebook(name):
    """FP16 value of each 16-bit state."""
    s = torch.arange(65536, dtype=torch.int64, device=DEV)
    p = (s * _MULTIPLIER[name] + (64248484 if name == "3inst" else 0)) & 0xFFFFFFFF
    half = lambda bits: torch.tensor([bits], dtype=torch.int16, device=DEV).view(torch.float16).double()
    if name == "mul1":
        b = sum((p >> k) & 0xFF for k in (0, 8, 16, 24))
        return ((1024 + b).double() * half(0x1EEE) + half(0xC931 - 65536)).half()
    q = (p & 0x8FFF8FFF) ^ 0x3B603B60
    as_half = lambda v: torch.where(v >= 32768, v - 65536, v).to(torch.int16).view(torch.float16).double()
    return (as_half(q & 0xFFFF) + as_half(q >> 16)).half()


def _decode(trellis, K, codebook):
    """FP16 weights [I][N] of a packed layer [I/16][N/16][16 K] (on the GPU)."""
    words = torch.from_numpy(trellis.view(np.int32)).to(DEV).to(torch.int64) & 0xFFFFFFFF   # 8K ring words
    ti, tn = words.shape[:2]
    n = 8 * K
    p = torch.arange(256, device=DEV)
    # the 16 bits ending at bit (p + 1) K of the ring, bit 31 of each word first
    start = ((p + 1) * K - 16) % (32 * n)
    i0, off = start // 32, start % 32
    table = _codebook(codebook)
    t, f = p // 8, p % 8
    row, col = 2 * (t % 4) + f % 2 + 8 * ((f // 2) % 2), t // 4 + 8 * (f // 4)
    out = torch.empty((ti, tn, 256), dtype=torch.float16, device=DEV)
    step = max(1, (1 << 25) // (tn * 256))
    for a in range(0, ti, step):
        w = words[a:a + step]
        pair = (w[..., i0] << 32) | w[..., (i0 + 1) % n]
        out[a:a + step, :, row * 16 + col] = table[(pair >> (48 - off)) & 0xFFFF]
    return out.view(ti, tn, 16, 16).permute(0, 2, 1, 3).reshape(ti * 16, tn * 16)


def _hadamard(v):
    """Butterflies of strides 1 .. 64 over each 128 channels, then 1/sqrt(128)."""
    shape = v.shape
    for k in range(7):
        s = 1 << k
        v = v.reshape(-1, 64 // s, 2, s)
        v = torch.stack((v[:, :, 0] + v[:, :, 1], v[:, :, 0] - v[:, :, 1]), dim=2)
    # the FP32 stage multiplies by the FP32 constant
    scale = torch.tensor(1.0 / math.sqrt(128.0), dtype=v.dtype, device=v.device)
    return v.reshape(shape) * scale


def _linear(x, layer, K, codebook="mul1"):
    """[rows][N] FP64 outputs of a packed layer on FP32 inputs x."""
    trellis, suh, svh, bias = layer
    a = (x * torch.from_numpy(suh).to(DEV).float()).half().float()
    a = _hadamard(a).half()
    N = len(svh)
    core = torch.empty((x.shape[0], N), dtype=torch.float64, device=DEV)
    cols = max(128, ((1 << 27) // len(suh)) // 128 * 128)
    for c in range(0, N, cols):
        part = np.ascontiguousarray(trellis[:, c // 16:min(N, c + cols) // 16])
        core[:, c:c + cols] = a.double() @ _decode(part, K, codebook).double()
    y = _hadamard(core) * torch.from_numpy(svh).to(DEV).double()
    return y if bias is None else y + torch.from_numpy(bias).to(DEV).double()


def _swiglu(g, u):
    return g * torch.sigmoid(g) * u


def exact(case, seed):
    rows, K = case["rows"], case["K"]
    g = _rng(case, seed)
    if case["kind"] in ("gemv", "gemm", "gemm_plan"):
        layer = _layer(g, case["I"], case["N"], K, case["bias"])
        return _linear(_activations(g, rows, case["I"]), layer, K, case["codebook"])
    if case["kind"] == "grouped":
        G, I = case["G"], case["I"]
        layers = [_layer(g, I, case["N"], K) for _ in range(G)]
        x = _activations(g, rows, G * I)
        return torch.cat([_linear(x[:, i * I:(i + 1) * I], layers[i], K) for i in range(G)], dim=1)
    if case["kind"] == "swiglu":
        gate, up = _layer(g, case["I"], case["N"], K), _layer(g, case["I"], case["N"], K)
        x = _activations(g, rows, case["I"])
        return _swiglu(_linear(x, gate, K), _linear(x, up, K))
    I, H = case["I"], case["H"]
    x = _activations(g, rows, I)
    ids, scores = _routes(g, case)
    y = torch.zeros((rows, I), dtype=torch.float64, device=DEV)
    for e in sorted(set(ids.reshape(-1).tolist())):
        ge = _rng(case, seed, 1 + e)
        gate, up, down = _layer(ge, I, H, K), _layer(ge, I, H, K), _layer(ge, H, I, K)
        r, slot = np.nonzero(ids == e)
        xe = x[torch.from_numpy(r).to(DEV)]
        hidden = _swiglu(_linear(xe, gate, K), _linear(xe, up, K)).float()
        out = _linear(hidden, down, K)
        y.index_add_(0, torch.from_numpy(r).to(DEV),
                     out * torch.from_numpy(scores[r, slot]).to(DEV).double()[:, None])
    return y
