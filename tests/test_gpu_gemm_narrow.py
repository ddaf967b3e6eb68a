"""GPU parity of the narrow GEMM core at the edges of its row blocks.

Every call of fewer than 256 rows, and any call on a layer whose width is not a
multiple of 256, runs workgroups of 16, 32, 64, 128 or 256 rows; blocks of 16
rows fold their K-split planes in the last workgroup to arrive, the others in a
second launch.  Checked here on both sides of every block size:
  * the full operator against the oracle's staged FP32 layer (reference GPU
    gate, docs/GPU_TESTS.md:124-143) on the first and last rows;
  * every row's bits equal those of the same row in the largest call (one
    accumulation order whatever the block);
  * a dirty workspace (stale arrival counts) and a second call on it give the
    same bits, and alpha / beta act on the same core.
"""
import numpy as np
import pytest

import synth
from oracle import codec, linear

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


def _bits(t):
    return t.view(torch.int32)


# (I, N, K, codebook, splits): one split, one stage per split, the most splits,
# and a layer wide enough for 256-row blocks.
@pytest.mark.parametrize("I,N,K,codebook,splits", [(384, 128, 4, "mul1", 1), (1024, 256, 5, "mcg", 8),
                                                    (2048, 384, 3, "3inst", 16), (512, 8192, 4, "mul1", 4)])
def test_narrow_row_blocks(ctx, I, N, K, codebook, splits):
    sizes = (1, 15, 16, 17, 31, 32, 33, 64, 65, 128, 129, 200, 255) + ((300, 520) if N % 256 else ())
    print(f"narrow gemm {I}x{N} K={K} {codebook} S={splits} M={sizes}", flush=True)
    tr, suh, svh, b = synth.layer(I, N, K, 7100 + I + N, bias=True)
    w = runtime.Weights(ctx, tr, suh, svh, b, codebook)
    assert w.gemm_splits(16) == splits
    top = max(sizes)
    x = torch.from_numpy(synth.activations(top, I, 7101)).to(DEV)
    y_top = torch.full((top, N), float("nan"), device=DEV)
    runtime.gemm(w, x, y_top)
    q = codec.dequantize_rotated(tr, K, codebook)
    sel = np.r_[0:4, 14:18, top - 4:top]
    ref = linear.matmul_fp32_stages(x.cpu().numpy()[sel], tr, suh, svh, K, codebook, b, rotated=q)["output_fp32"]
    synth.gate(y_top.cpu().numpy()[sel], ref)
    for m in sizes:
        xm = x[top - m:].contiguous()
        y = torch.full((m, N), float("nan"), device=DEV)
        ws = runtime.alloc_workspace(runtime.workspace_bytes(w, xm, y), DEV)
        ws.fill_(0xA5)
        for _ in range(2):
            y.fill_(float("nan"))
            runtime.gemm(w, xm, y, workspace=ws)
            assert torch.equal(_bits(y), _bits(y_top[top - m:])), m
        old = torch.from_numpy(synth.rng(7102 + m).standard_normal((m, N)).astype(np.float32)).to(DEV)
        y_ab = old.clone()
        runtime.gemm(w, xm, y_ab, alpha=-0.5, beta=2.0, workspace=ws)
        want = linear.apply_alpha_beta(y.cpu().numpy(), old.cpu().numpy(), -0.5, 2.0)
        np.testing.assert_array_equal(y_ab.cpu().numpy().view(np.uint32), want.view(np.uint32))
    w.destroy()


@pytest.mark.parametrize("I,N,K,codebook", [(1024, 1152, 6, "mcg"), (1024, 1152, 8, "mul1")])
def test_narrow_256_row_blocks(ctx, I, N, K, codebook):
    """Several 256-row blocks (2 (N / 128) S workgroups per block, at least 512 in
    all): whole, one row past a block, and a ragged last one, whose row tiles past
    the rows read out of range; more than 4 bits take two loads per chunk."""
    sizes = (769, 1024, 1025, 1300)
    print(f"narrow gemm 256-row blocks {I}x{N} K={K} {codebook} M={sizes}", flush=True)
    tr, suh, svh, b = synth.layer(I, N, K, 7200 + K, bias=True)
    w = runtime.Weights(ctx, tr, suh, svh, b, codebook)
    assert w.gemm_splits(16) == 8 and 2 * (N // 128) * 8 * ((769 + 255) // 256) >= 512
    top = max(sizes)
    x = torch.from_numpy(synth.activations(top, I, 7201)).to(DEV)
    small = torch.empty((top, N), device=DEV)
    for r in range(0, top, 128):   # 128-row blocks, one per call
        part = torch.empty((min(128, top - r), N), device=DEV)
        runtime.gemm(w, x[r:r + 128].contiguous(), part)
        small[r:r + 128] = part
    q = codec.dequantize_rotated(tr, K, codebook)
    sel = np.r_[0:2, 254:258, 510:514, 766:770, 1022:1026, top - 2:top]
    ref = linear.matmul_fp32_stages(x.cpu().numpy()[sel], tr, suh, svh, K, codebook, b, rotated=q)["output_fp32"]
    for m in sizes:
        y = torch.full((m + 1, N), float("nan"), device=DEV)   # one guard row
        runtime.gemm(w, x[:m].contiguous(), y[:m])
        assert torch.equal(_bits(y[:m]), _bits(small[:m])), m
        assert bool(torch.isnan(y[m]).all())
        rows = sel[sel < m]
        synth.gate(y.cpu().numpy()[rows], ref[:len(rows)])
    w.destroy()


def test_narrow_passes(ctx):
    """A call whose planes pass 1 GiB runs in several passes, each row with the
    bits of a call of its own rows."""
    I, N, K, M = 128, 32896, 2, 8200
    print(f"narrow gemm passes {I}x{N} K={K} M={M}", flush=True)
    tr, suh, svh, b = synth.layer(I, N, K, 7300, bias=True)
    w = runtime.Weights(ctx, tr, suh, svh, b, "mul1")
    x = torch.from_numpy(synth.activations(M, I, 7301)).to(DEV)
    y = torch.full((M, N), float("nan"), device=DEV)
    ws = runtime.workspace_bytes(w, x, y)
    assert ws < (1 << 30) + M * I * 2 + (1 << 20) < M * N * 4 + M * I * 2
    runtime.gemm(w, x, y)
    edge = (1 << 30) // (N * 4) // 256 * 256   # rows of the first pass
    for a, e in ((0, 40), (edge - 40, edge), (edge, edge + 40), (M - 40, M)):
        part = torch.empty((e - a, N), device=DEV)
        runtime.gemm(w, x[a:e].contiguous(), part)
        assert torch.equal(_bits(y[a:e]), _bits(part)), (a, e)
    w.destroy()
