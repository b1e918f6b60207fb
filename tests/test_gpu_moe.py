"""GPU parity of the MoE pieces: comm-quant (moe.py:79-143), its wire format,
and the grouped per-expert GEMM over a token-offset table."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from _gpu_util import assert_bits_equal, rel_fro_bf16, seeded, to_np32
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _ref_comm(x: torch.Tensor, granularity: str, rounding: int, bits: int, seed: int, offset: int):
    """Oracle dq with the reference's group choice, then the reference STE in torch CPU ops."""
    xn = to_np32(x).reshape(-1, x.shape[-1]) if x.dim() >= 2 else to_np32(x).reshape(1, -1)
    R, K = xn.shape
    if granularity in ("tile_1x128", "block_128x128"):
        gr, gc = R, 128
    elif granularity == "channel" and x.dim() >= 2:
        gr, gc = R, 1
    else:
        gr, gc = R, K
    _, _, _, dq = O.quant_grouped(xn, gr, gc, bits=bits, rounding=rounding, seed=seed, offset=offset,
                                  scale_rule=O.SCALE_BEFORE_DIVIDE)
    xc = x.detach().cpu()
    dqt = torch.from_numpy(dq).reshape(x.shape).to(x.dtype)
    return xc + (dqt - xc)


@pytest.mark.parametrize("granularity", ["block_128x128", "tile_1x128", "channel", "tensor"])
@pytest.mark.parametrize("rounding", ["nearest", "stochastic"])
@pytest.mark.parametrize("shape,dtype", [((7, 257), torch.float32), ((64, 1024), torch.bfloat16),
                                         ((3, 5, 300), torch.bfloat16), ((128, 2048), torch.float16)])
def test_comm_quant_dequant_parity(gpu_device, granularity, rounding, shape, dtype):
    """Every rounding step of the reference's straight-through expression in
    the input dtype, float16 included (dq = q*s rounded to fp32 and then to
    f16, not in one step)."""
    from lowbit import moe

    x = seeded(shape, seed=20260401, dtype=dtype, outliers=0.01).to(gpu_device).requires_grad_(True)
    out = moe.comm_quant_dequant(x, granularity=granularity, rounding_mode=rounding, bits=8, seed=9, offset=4)
    rc = O.ROUND_STOCHASTIC if rounding == "stochastic" else O.ROUND_NEAREST
    ref = _ref_comm(x, granularity, rc, 8, 9, 4)
    assert out.shape == x.shape and out.dtype == x.dtype
    assert_bits_equal(out.detach().float().cpu().numpy(), ref.float().numpy(), "comm dq")
    out.float().sum().backward()  # straight-through gradient
    assert x.grad is not None and torch.equal(x.grad, torch.ones_like(x))


# rows of one wave each, on both sides of the counts from which a workgroup
# takes a second, third and fourth row (3400 waves per row with a scale per
# chunk, 896 with one per element, 1792 of those where K is no multiple of 8)
@pytest.mark.parametrize("granularity,shape", [("tensor", (6799, 64)), ("tensor", (6801, 64)), ("tensor", (10201, 72)),
                                               ("tensor", (13605, 40)), ("tile_1x128", (6803, 129)),
                                               ("channel", (1793, 64)), ("channel", (2689, 72)), ("channel", (3587, 64)),
                                               ("channel", (3585, 65)), ("channel", (7171, 63))])
@pytest.mark.parametrize("rounding", ["nearest", "stochastic"])
def test_comm_quant_dequant_rows_per_workgroup(gpu_device, granularity, shape, rounding):
    from lowbit import moe

    x = seeded(shape, seed=20260403, outliers=0.01).to(gpu_device)
    out = moe.comm_quant_dequant(x, granularity=granularity, rounding_mode=rounding, seed=9, offset=4)
    rc = O.ROUND_STOCHASTIC if rounding == "stochastic" else O.ROUND_NEAREST
    assert_bits_equal(out.float().cpu().numpy(), _ref_comm(x, granularity, rc, 8, 9, 4).float().numpy(), "comm dq")


def test_comm_quant_dequant_special_values(gpu_device):
    from lowbit import moe

    x = torch.zeros(4, 256)
    x[0, 3] = float("inf")
    x[1, 130] = float("nan")
    x[2, :2] = torch.tensor([1e-45, -1e-45])
    x = x.to(gpu_device)
    for g in ("block_128x128", "tensor", "channel"):
        out = moe.comm_quant_dequant(x, granularity=g, rounding_mode="nearest", seed=1, offset=1)
        ref = _ref_comm(x, g, O.ROUND_NEAREST, 8, 1, 1)
        assert_bits_equal(out.float().cpu().numpy(), ref.float().numpy(), f"comm dq {g}")


@pytest.mark.parametrize("rounding", ["nearest", "stochastic"])
def test_comm_quant_dequant_subnormal_group_amax(gpu_device, rounding):
    """A group whose amax is subnormal: the reference divides it by qmax
    after the check (moe.py:94-98), the scale underflows to zero and the
    group's values become NaN (zeros) or +-qmax times zero (the rest); the
    other groups are ordinary."""
    from lowbit import moe

    x = torch.zeros(4, 384)
    x[0, :2] = torch.tensor([1e-45, -1e-45])
    x[1, 300] = 1e-42
    x[:, 128:256] = torch.randn(4, 128, generator=torch.Generator().manual_seed(20260403))
    x = x.to(gpu_device)
    rc = O.ROUND_STOCHASTIC if rounding == "stochastic" else O.ROUND_NEAREST
    for g in ("tile_1x128", "tensor", "channel"):
        out = moe.comm_quant_dequant(x, granularity=g, rounding_mode=rounding, seed=1, offset=1)
        ref = _ref_comm(x, g, rc, 8, 1, 1)
        assert_bits_equal(out.float().cpu().numpy(), ref.float().numpy(), f"comm dq {g}")
    # the strips' scales: the first and last underflow
    assert torch.isnan(moe.comm_quant_dequant(x, granularity="tile_1x128", rounding_mode=rounding)[2, 5]).item()


@pytest.mark.parametrize("fmt,grid", [("e4m3", O.GRID_E4M3), ("int_grid", O.GRID_INT)])
def test_comm_wire_format_round_trip(gpu_device, fmt, grid):
    from lowbit import moe

    x = seeded((300, 7168 // 4), seed=20260402, outliers=0.01).to(gpu_device)
    payload = moe.comm_quant(x, fmt=fmt)
    y = moe.comm_dequant(payload)
    codes, scales, _, dq = O.quant_tile_1x128(to_np32(x), grid=grid)
    assert_bits_equal(payload.q.codes.cpu().numpy(), codes, "wire codes")
    assert_bits_equal(payload.q.scales.cpu().numpy(), scales, "wire scales")
    expect = torch.from_numpy(dq).to(x.dtype).float().numpy()
    if grid == O.GRID_E4M3:
        assert_bits_equal(to_np32(y), expect, "received tokens")
    else:
        # int8 codes have no -0: a negative value that rounds to zero arrives as +0
        got = to_np32(y)
        assert np.array_equal(got, expect)
        nz = expect != 0
        assert_bits_equal(got[nz], expect[nz], "received tokens (nonzero)")
    assert payload.nbytes == x.numel() + scales.size * 4


def _routing(T, E, k, seed, device):
    from lowbit import workloads

    return workloads.zipf_topk_routing(T, E, k, seed=seed, device=device)


@pytest.mark.parametrize("fmt,grid", [("e4m3", O.GRID_E4M3), ("int_grid", O.GRID_INT)])
@pytest.mark.parametrize("T,E,k,H,I", [(64, 4, 2, 256, 256), (300, 8, 3, 384, 128), (5, 16, 2, 128, 256)])
def test_grouped_linear_matches_per_expert_oracle(gpu_device, fmt, grid, T, E, k, H, I):
    from lowbit import moe

    tokens = seeded((T, H), seed=20260403).to(gpu_device)
    routing = _routing(T, E, k, 20260404, gpu_device)
    w = seeded((E, I, H), seed=20260405, std=0.02).to(gpu_device)
    order, tok_idx, offsets = moe.sort_by_expert(routing, E)
    xs = tokens[tok_idx]
    wc, ws, wn = moe.quantize_expert_weights(w, fmt=fmt)
    y = moe.grouped_linear(xs, offsets, wc, ws, fmt=fmt, w_nan_rows=wn)
    torch.cuda.synchronize()
    off = offsets.cpu().numpy()
    xs_n = to_np32(xs)
    _, _, _, xdq = O.quant_tile_1x128(xs_n, grid=grid)
    ref = np.zeros((xs_n.shape[0], I))
    for e in range(E):
        lo, hi = off[e], off[e + 1]
        if hi == lo:
            continue
        _, _, _, wdq = O.quant_block_128x128(to_np32(w[e]), grid=grid)
        ref[lo:hi] = O.gemm_ref(xdq[lo:hi], wdq)
    assert rel_fro_bf16(y, ref) <= 1e-3


def test_sort_by_expert_offsets(gpu_device):
    from lowbit import moe

    routing = _routing(1000, 32, 8, 7, gpu_device)
    order, tok_idx, offsets = moe.sort_by_expert(routing, 32)
    flat = routing.reshape(-1).cpu()
    off = offsets.cpu()
    assert off[0] == 0 and off[-1] == flat.numel()
    sorted_ids = flat[order.cpu()]
    for e in range(32):
        assert (sorted_ids[off[e]:off[e + 1]] == e).all()
    # distinct experts per token (top-k without replacement)
    assert all(len(set(r.tolist())) == 8 for r in routing.cpu())


def test_c4_grouped_up_projection_full_size_sampled(gpu_device):
    """benchmark config 4: 4096 tokens, top-8 of 32 experts, W_up [2048, 7168]."""
    from lowbit import moe, workloads

    tokens, routing, w_up, _ = workloads.c4_inputs(device="cpu")
    tokens, routing = tokens.to(gpu_device), routing.to(gpu_device)
    w_up = w_up.to(gpu_device)
    order, tok_idx, offsets = moe.sort_by_expert(routing, 32)
    xs = tokens[tok_idx]
    wc, ws, wn = moe.quantize_expert_weights(w_up, fmt="e4m3")
    y = moe.grouped_linear(xs, offsets, wc, ws, fmt="e4m3", w_nan_rows=wn)
    torch.cuda.synchronize()
    assert y.shape == (32768, 2048)
    off = offsets.cpu().numpy()
    rng = np.random.default_rng(3)
    for e in rng.choice(32, 4, replace=False):
        lo, hi = off[e], off[e + 1]
        if hi == lo:
            continue
        rows = np.arange(lo, hi)[:64]
        _, _, _, xdq = O.quant_tile_1x128(to_np32(xs[rows]), grid=O.GRID_E4M3)
        _, _, _, wdq = O.quant_block_128x128(to_np32(w_up[e]), grid=O.GRID_E4M3)
        assert rel_fro_bf16(y[rows], O.gemm_ref(xdq, wdq)) <= 1e-3


def _offsets(counts, device):
    return torch.tensor(np.concatenate([[0], np.cumsum(counts)]), dtype=torch.int32, device=device)


@pytest.mark.parametrize("grouped", [False, True])
@pytest.mark.parametrize("fmt", ["e4m3", "int_grid"])
@pytest.mark.parametrize("rounding", ["nearest", "stochastic"])
def test_swiglu_quant_matches_unfused(gpu_device, grouped, fmt, rounding):
    """The gate/up GEMM with the SwiGLU + 1x128 epilogue equals, bit for bit,
    two separate GEMMs, torch's F.silu(gate) * up on their bf16 outputs
    (moe.py:191) and the 1x128 quantizer on that h: same accumulation order,
    same exp and division, same roundings."""
    import torch.nn.functional as F

    from lowbit import moe, ops

    H, I = 384, 256
    counts = [300, 0, 17, 260, 129] if grouped else [300]
    E, T = len(counts), sum(counts)
    x = seeded((T, H), seed=20260601, outliers=0.01).to(gpu_device)
    x[5, 7] = float("nan")
    wg = seeded((E, I, H), seed=20260602, std=0.03).to(gpu_device)
    wu = seeded((E, I, H), seed=20260603, std=0.03).to(gpu_device)
    gc, gs, gn = moe.quantize_expert_weights(wg, fmt=fmt)
    uc, us_, un = moe.quantize_expert_weights(wu, fmt=fmt)
    codes, scales, nan = moe.interleave_gate_up(gc, gs, uc, us_, gn, un)
    qx = ops.quant_tile_1x128(x, fmt=fmt, want_nan_rows=True)
    kw = dict(fmt=fmt, rounding=rounding, seed=41, offset=9)
    if grouped:
        offs = _offsets(counts, gpu_device)
        h, qh = ops.gemm_swiglu_quant(qx, codes, scales, offsets=offs, want_nan_rows=True, b_nan_rows=nan, **kw)
        g_out = ops.gemm_grouped_blockscaled(qx, gc, gs, offs, N=I, b_nan_rows=gn)
        u_out = ops.gemm_grouped_blockscaled(qx, uc, us_, offs, N=I, b_nan_rows=un)
    else:
        h, qh = ops.gemm_swiglu_quant(qx, codes[0], scales[0], want_nan_rows=True, b_nan_rows=nan[0], **kw)
        qg = ops.QTensor(gc[0], gs[0].contiguous(), gs.shape[2], 1, 7, qx.grid, I, H, gn[0], None)
        qu = ops.QTensor(uc[0], us_[0].contiguous(), us_.shape[2], 1, 7, qx.grid, I, H, un[0], None)
        g_out = ops.gemm_blockscaled(qx, qg)
        u_out = ops.gemm_blockscaled(qx, qu)
    h_ref = F.silu(g_out) * u_out
    q_ref = ops.quant_tile_1x128(h_ref, want_nan_rows=True, **kw)
    torch.cuda.synchronize()
    assert torch.equal(h.view(torch.int16), h_ref.view(torch.int16)), "h differs from the unfused path"
    assert torch.equal(qh.codes, q_ref.codes)
    assert torch.equal(qh.scales[:, :T], q_ref.scales[:, :T])
    assert torch.equal(qh.nan_rows, q_ref.nan_rows)


def test_expert_mlp_matches_oracle(gpu_device):
    """ExpertMLP.forward (moe.py:190-193) for all experts, three kernels, against
    the oracle pipeline (1x128 x, 128x128 weights, float64 GEMMs, bf16
    projections, F.silu's formula, 1x128 h).  Checked in stages, each at the
    1e-3 relative-Frobenius bar of one GEMM: h against the oracle's h, and the
    output against the oracle's down projection of the GPU's h.  End to end
    the bar is 5e-3: about 1% of the bf16 projections land one ulp away from
    the float64 result (fp32 accumulation order), and re-quantizing h to 8-bit
    codes turns a few of those into whole-code steps."""
    from lowbit import moe

    H, I = 512, 256
    counts = [200, 64, 0, 311]
    E, T = len(counts), sum(counts)
    x = seeded((T, H), seed=20260611).to(gpu_device)
    wg = seeded((E, I, H), seed=20260612, std=0.03).to(gpu_device)
    wu = seeded((E, I, H), seed=20260613, std=0.03).to(gpu_device)
    wd = seeded((E, H, I), seed=20260614, std=0.03).to(gpu_device)
    gu = moe.interleave_gate_up(*moe.quantize_expert_weights(wg)[:2], *moe.quantize_expert_weights(wu)[:2])
    dn = moe.quantize_expert_weights(wd)
    offs = _offsets(counts, gpu_device)
    out, h = moe.expert_mlp(x, offs, gu, dn, want_h=True)
    torch.cuda.synchronize()

    xn = to_np32(x)
    hg = to_np32(h)
    _, _, _, xdq = O.quant_tile_1x128(xn, grid=O.GRID_E4M3)
    h_ref = np.zeros((T, I), dtype=np.float64)
    out_from_gpu_h = np.zeros((T, H), dtype=np.float64)
    out_ref = np.zeros((T, H), dtype=np.float64)
    bounds = np.concatenate([[0], np.cumsum(counts)])
    for e in range(E):
        lo, hi = bounds[e], bounds[e + 1]
        if hi == lo:
            continue
        dq = lambda w: O.quant_block_128x128(to_np32(w[e]), grid=O.GRID_E4M3)[3]  # noqa: E731
        g = O.round_bf16(O.gemm_ref(xdq[lo:hi], dq(wg)).astype(np.float32))
        u = O.round_bf16(O.gemm_ref(xdq[lo:hi], dq(wu)).astype(np.float32))
        sg = O.round_bf16((g / (np.float32(1) + np.exp(-g))).astype(np.float32))
        hh = O.round_bf16((sg * u).astype(np.float32))
        h_ref[lo:hi] = hh
        out_ref[lo:hi] = O.gemm_ref(O.quant_tile_1x128(hh, grid=O.GRID_E4M3)[3], dq(wd))
        out_from_gpu_h[lo:hi] = O.gemm_ref(O.quant_tile_1x128(hg[lo:hi], grid=O.GRID_E4M3)[3], dq(wd))
    assert rel_fro_bf16(h, h_ref) <= 1e-3
    assert rel_fro_bf16(out, out_from_gpu_h) <= 1e-3
    assert rel_fro_bf16(out, out_ref) <= 5e-3


@pytest.mark.parametrize("fmt,grid", [("e4m3", O.GRID_E4M3), ("int_grid", O.GRID_INT)])
def test_grouped_gemm_tile_boundaries(gpu_device, fmt, grid):
    """Experts whose last 256-row tile has exactly 128 rows (its second half
    is all padding), 129 rows (one row in the second half), 1 row, a whole
    tile, none, and one and a half tiles, against the per-expert oracle."""
    from lowbit import moe, ops

    counts = [128, 129, 1, 256, 0, 384]
    E, T, H, N = len(counts), sum(counts), 256, 384
    x = seeded((T, H), seed=20261310, outliers=0.01).to(gpu_device)
    w = seeded((E, N, H), seed=20261311, std=0.02).to(gpu_device)
    wc, ws, wn = moe.quantize_expert_weights(w, fmt=fmt)
    qx = ops.quant_tile_1x128(x, fmt=fmt, want_nan_rows=True)
    offs = _offsets(counts, gpu_device)
    y = ops.gemm_grouped_blockscaled(qx, wc, ws, offs, N=N, b_nan_rows=wn)
    torch.cuda.synchronize()
    _, _, _, xdq = O.quant_tile_1x128(to_np32(x), grid=grid)
    ref = np.zeros((T, N))
    lo = 0
    for e, c in enumerate(counts):
        if c:
            _, _, _, wdq = O.quant_block_128x128(to_np32(w[e]), grid=grid)
            ref[lo:lo + c] = O.gemm_ref(xdq[lo:lo + c], wdq)
        lo += c
    assert rel_fro_bf16(y, ref) <= 1e-3
    for e, c in enumerate(counts):  # every expert on its own, so none hides in the total
        lo = sum(counts[:e])
        if c:
            assert rel_fro_bf16(y[lo:lo + c], ref[lo:lo + c]) <= 1e-3, f"expert {e} ({c} rows)"


@pytest.mark.parametrize("fmt", ["e4m3", "int_grid"])
@pytest.mark.parametrize("E,counts", [
    (70, {0: 1, 3: 16, 64: 17, 69: 40}),  # 16-row tiles; the expert search passes its first 64
    (6, {0: 33, 2: 32, 3: 1, 5: 130}),  # 32-row tiles, one expert with a lot more than the average
])
def test_few_rows_per_expert_match_single_expert_calls(gpu_device, fmt, E, counts):
    """The few-row expert tiles against the 256x256 tiles, which the same rows
    take when each expert is called on its own (more than 64 rows for the one
    expert): both sum the K blocks in order, so every output bit agrees."""
    from lowbit import moe, ops

    H, I, N = 384, 256, 384
    counts = [counts.get(e, 0) for e in range(E)]
    T = sum(counts) + 3  # rows past the last expert belong to nobody
    x = seeded((T, H), seed=20262401, outliers=0.01).to(gpu_device)
    x[0, 7] = float("nan")
    qx = ops.quant_tile_1x128(x, fmt=fmt, want_nan_rows=True)
    wc, ws, wn = moe.quantize_expert_weights(seeded((E, N, H), seed=20262402, std=0.03).to(gpu_device), fmt=fmt)
    gc, gs, gn = moe.quantize_expert_weights(seeded((E, 2 * I, H), seed=20262403, std=0.03).to(gpu_device), fmt=fmt)
    wn[:, 5] = gn[:, 130] = 1
    bounds = np.concatenate([[0], np.cumsum(counts)])
    offs = torch.tensor(bounds, dtype=torch.int32, device=gpu_device)
    kw = dict(fmt=fmt, rounding="stochastic", seed=43, offset=5, want_nan_rows=True)
    gu = torch.zeros((T, 2 * I), dtype=torch.bfloat16, device=gpu_device)
    y = ops.gemm_grouped_blockscaled(qx, wc, ws, offs, N=N, b_nan_rows=wn)
    h, qh = ops.gemm_swiglu_quant(qx, gc, gs, offsets=offs, b_nan_rows=gn, gu_out=gu, **kw)
    bits = lambda t: t.view(torch.int16)  # noqa: E731
    for e in np.flatnonzero(counts):
        r = slice(int(bounds[e]), int(bounds[e + 1]))
        one = torch.tensor([r.start, r.stop], dtype=torch.int32, device=gpu_device)
        gu1 = torch.zeros_like(gu)
        y1 = ops.gemm_grouped_blockscaled(qx, wc[e:e + 1], ws[e:e + 1], one, N=N, b_nan_rows=wn[e:e + 1])
        h1, qh1 = ops.gemm_swiglu_quant(qx, gc[e:e + 1], gs[e:e + 1], offsets=one, b_nan_rows=gn[e:e + 1],
                                        gu_out=gu1, **kw)
        assert torch.equal(bits(y[r]), bits(y1[r])), f"expert {e}"
        assert torch.equal(bits(h[r]), bits(h1[r])) and torch.equal(bits(gu[r]), bits(gu1[r])), f"expert {e}"
        assert torch.equal(qh.codes[r], qh1.codes[r]) and torch.equal(qh.scales[:, r], qh1.scales[:, r])
        assert torch.equal(qh.nan_rows[r], qh1.nan_rows[r])
    assert int(gu[T - 3:].count_nonzero()) == 0
