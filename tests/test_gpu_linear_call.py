"""The one-call linear (ntlb_linear_forward and its two backwards) against the
general path of HipLowBitBackend, which issues the same quantizers and GEMMs
one by one: outputs and gradients bit for bit, over the dtypes, code formats,
roundings and backward rules the one-call route accepts, ragged and strided
operands, a dY whose rows need the padded copy, gradients of a subset of the
inputs, and NaN and infinite values.  e4m3 runs without NaN row flags there, so
the NaN cases compare its products with the flagged ones.

The straight-through gradients are the exception to bit for bit: small ones run
on other tiles than the separate calls and sum the contraction in ranges.  Both
routes round an fp32 sum of the same bf16 products to bf16; the sums differ by
less than 1e-5 of the result's norm (fp32 reassociation), which moves a bf16
rounding of a few values by one step of 2^-8: below 1e-3 of the norm."""

from __future__ import annotations

import pytest
import torch

from _gpu_util import seeded

pytestmark = pytest.mark.gpu


def _backend(fmt, rounding, recipe, K, N):
    from lowbit.backend import HipLowBitBackend
    from lowbit.contracts import LowBitKernelSpec

    spec = LowBitKernelSpec("linear", K, N, True, "tile_1x128", "block_128x128", rounding)
    return HipLowBitBackend(mode="fp8", kernel_spec=spec, code_format=fmt, backward=recipe, seed=77)


def _same(a, b):
    if a is None or b is None:
        return a is None and b is None
    a, b = a.detach(), b.detach()
    if a.shape != b.shape or a.dtype != b.dtype:
        return False
    nan = torch.isnan(a)
    return torch.equal(nan, torch.isnan(b)) and torch.equal(a[~nan], b[~nan])


def _close(a, b):
    """_same up to the reassociation of an fp32 sum"""
    if a is None or b is None:
        return a is None and b is None
    a, b = a.detach(), b.detach()
    fin = torch.isfinite(a)
    if a.shape != b.shape or a.dtype != b.dtype or not torch.equal(fin, torch.isfinite(b)):
        return False
    if not torch.equal(torch.isnan(a), torch.isnan(b)):
        return False
    d = (a[fin].double() - b[fin].double()).norm()
    return float(d) <= 1e-3 * float(b[fin].double().norm()) + 1e-30


def _agree(recipe, one, gen):
    """y bit for bit; gradients too, except the straight-through dX and dW"""
    near = _close if recipe == "ste" else _same
    return _same(one[0], gen[0]) and near(one[1], gen[1]) and near(one[2], gen[2]) and _close(one[3], gen[3])


def _both(fmt, rounding, recipe, x, w, b, dy, grads=(True, True, True), general_dy=None):
    """[y, dx, dw, db] through the one-call route and through the general one"""
    out = []
    for general in (False, True):
        be = _backend(fmt, rounding, recipe, w.shape[1], w.shape[0])
        calls = []
        if general:
            be._one_call = lambda *a: False
        else:
            orig = be._one_call
            be._one_call = lambda *a: calls.append(orig(*a)) or calls[-1]
        t = [None if v is None else v.detach().requires_grad_(g) for v, g in zip((x, w, b), grads)]
        y = be.linear(*t)
        wanted = [v for v in t if v is not None and v.requires_grad]
        up = general_dy if general and general_dy is not None else dy
        g = list(torch.autograd.grad(y, wanted, up)) if wanted else []
        out.append([y] + [g.pop(0) if v is not None and v.requires_grad else None for v in t])
        if not general:
            assert calls == [True], "the case should take the one-call route"
    return out


@pytest.mark.parametrize("fmt", ["e4m3", "int_grid"])
@pytest.mark.parametrize("recipe,rounding", [("ste", "nearest"), ("fp8", "nearest"), ("fp8", "stochastic")])
@pytest.mark.parametrize("mnk", [(1, 64, 128), (37, 129, 257), (130, 320, 200), (300, 1541, 1000)])
def test_one_call_equals_the_general_path(gpu_device, mnk, fmt, recipe, rounding):
    M, N, K = mnk
    x = seeded((M, K), seed=20262101, outliers=0.01).to(gpu_device)
    w = seeded((N, K), seed=20262102, std=0.02).to(gpu_device)
    b = seeded((N,), seed=20262103).to(gpu_device)
    dy = seeded((M, N), seed=20262104, std=1e-3).to(gpu_device)
    one, gen = _both(fmt, rounding, recipe, x, w, b, dy)
    assert _agree(recipe, one, gen)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_other_dtypes(gpu_device, dtype):
    """forward without gradients for every rounding, and the fp32 recipe backward"""
    x = seeded((2, 35, 300), seed=20262111, dtype=dtype).to(gpu_device)
    w = seeded((200, 300), seed=20262112, std=0.02, dtype=dtype).to(gpu_device)
    b = seeded((200,), seed=20262113, dtype=dtype).to(gpu_device)
    for rounding in ("nearest", "stochastic"):
        one, gen = _both("e4m3", rounding, "ste", x, w, b, None, grads=(False, False, False))
        assert _same(one[0], gen[0])
    dy = seeded((2, 35, 200), seed=20262114, std=1e-3, dtype=dtype).to(gpu_device)
    one, gen = _both("int_grid", "nearest", "fp8", x, w, b, dy)
    assert all(_same(p, q) for p, q in zip(one, gen))


@pytest.mark.parametrize("recipe", ["ste", "fp8"])
@pytest.mark.parametrize("grads", [(True, False, False), (False, True, False), (False, False, True)])
def test_gradient_subsets_and_strides(gpu_device, recipe, grads):
    """3-D input, a column-sliced x and weight (row pitch above K), a dY that is
    a slice at an odd column, and one whose rows are one expanded row"""
    M, N, K = 66, 192, 256
    x = seeded((M, K + 24), seed=20262121).to(gpu_device)[:, :K].reshape(2, M // 2, K)
    w = seeded((N, K + 8), seed=20262122, std=0.02).to(gpu_device)[:, :K]
    b = seeded((N,), seed=20262123).to(gpu_device)
    big = seeded((2, M // 2, N + 3), seed=20262124, std=1e-3).to(gpu_device)
    for dy in (big[..., :N], big[..., 3:], big[:1, :1, :N].expand(2, M // 2, N)):
        one, gen = _both("e4m3", "nearest", recipe, x, w, b, dy, grads, general_dy=dy.contiguous())
        assert _agree(recipe, one, gen)


@pytest.mark.parametrize("fmt", ["e4m3", "int_grid"])
@pytest.mark.parametrize("recipe,rounding", [("ste", "nearest"), ("fp8", "nearest"), ("fp8", "stochastic")])
@pytest.mark.parametrize("mnk", [(20, 72, 200), (300, 700, 1500), (1100, 2100, 700)])
def test_nan_and_inf_operands(gpu_device, mnk, fmt, recipe, rounding):
    """NaN and infinities in x, the weight and dY: NaN exactly where the flagged
    products of the general path have it, every other value the same"""
    M, N, K = mnk
    x = seeded((M, K), seed=20262131).to(gpu_device)
    w = seeded((N, K), seed=20262132, std=0.02).to(gpu_device)
    dy = seeded((M, N), seed=20262133, std=1e-3).to(gpu_device)
    x[3, 17], x[5, K - 1], x[M - 1, 4] = float("nan"), float("inf"), float("-inf")
    w[7, 100], w[N - 1, 5] = float("nan"), float("inf")
    dy[9, 11], dy[2, N - 1] = float("nan"), float("inf")
    one, gen = _both(fmt, rounding, recipe, x, w, None, dy)
    assert torch.isnan(one[0][3]).all() and torch.isnan(one[0][:, 7]).all() and not torch.isnan(one[0][0, 0])
    assert _agree(recipe, one, gen)


# M, N, K of the layer: dX is M x K over N, dW N x K over M; together each tile
# of the rule (16x16 to 128x128) and the 256x256 kernels beyond it
@pytest.mark.parametrize("mnk", [(70, 200, 90), (150, 700, 1000), (500, 900, 1900), (700, 3000, 1100),
                                 (2100, 2000, 2200)])
def test_small_straight_through_gradients_match_float64(gpu_device, mnk):
    """dX and dW of a bf16 layer against float64 products of the decoded
    operands: one bf16 rounding (2^-9 relative at most, 2^-9 / sqrt(3) in the
    mean) of an fp32 sum"""
    M, N, K = mnk
    x = seeded((M, K), seed=20262141, outliers=0.01).to(gpu_device).requires_grad_(True)
    w = seeded((N, K), seed=20262142, std=0.02).to(gpu_device).requires_grad_(True)
    dy = seeded((M, N), seed=20262143, std=1e-3).to(gpu_device)
    from lowbit import ops

    be = _backend("e4m3", "nearest", "ste", K, N)
    dx, dw = torch.autograd.grad(be.linear(x, w, None), (x, w), dy)
    wq = ops.dequant(ops.quant_block_128x128(w.detach(), fmt="e4m3")[0], out_dtype=torch.bfloat16).double()
    xq = ops.dequant(ops.quant_tile_1x128(x.detach(), fmt="e4m3"), out_dtype=torch.bfloat16).double()
    for got, ref in ((dx, dy.double() @ wq), (dw, dy.double().T @ xq)):
        assert float((got.double() - ref).norm() / ref.norm()) <= 2.0 ** -9
        assert float(((got.double() - ref).abs() / ref.abs().clamp(min=float(ref.abs().max()) * 1e-3)).max()) <= 2.0 ** -7


@pytest.mark.parametrize("shape", [(1, 1), (63, 130), (64, 128), (1003, 1541), (300, 70), (70000, 3), (191, 1024),
                                   (193, 1024), (3073, 512), (2049, 8192), (8193, 768), (16385, 64)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
def test_colsum_of_few_columns_or_rows(gpu_device, shape, dtype):
    """column sums on the 64-row and the 256-row chunks, at both sides of the
    rule's lines (odd columns and pitches, one row, many rows) against float64;
    M fp32 additions"""
    from lowbit import ops

    M, N = shape
    x = seeded((M, N), seed=20262151 + N, dtype=dtype).to(gpu_device)
    for t in (x, torch.nn.functional.pad(x, (1, 2))[:, 1:1 + N]):
        got = ops.colsum(t, out_dtype=torch.float32).double()
        ref = x.double().sum(0)
        assert float(((got - ref).abs() / x.double().abs().sum(0)).max()) <= M * 2.0 ** -24


@pytest.mark.parametrize("recipe", ["ste", "fp8"])
@pytest.mark.parametrize("attr,value", [("seed", 78), ("code_format", "e4m3"), ("bits", 4), ("_rounding_mode", "nearest")])
def test_backend_attributes_are_read_at_every_call(gpu_device, attr, value, recipe):
    """seed, code format, bits and rounding changed between two calls of one
    shape: the later call's outputs and gradients are those of the general path
    after the same change (the straight-through rule draws only in its forward)"""
    M, N, K = 40, 192, 300
    x = seeded((M, K), seed=20262161).to(gpu_device)
    w = seeded((N, K), seed=20262162, std=0.02).to(gpu_device)
    dy = seeded((M, N), seed=20262163, std=1e-3).to(gpu_device)
    grads = recipe == "fp8"
    out = []
    for general in (False, True):
        be = _backend("int_grid", "stochastic", recipe, K, N)
        if general:
            be._one_call = lambda *a: False
        before = getattr(be, attr)
        for change in (False, True):
            if change:
                setattr(be, attr, value)
            t = [v.clone().requires_grad_(grads) for v in (x, w)]
            y = be.linear(*t, None)
            out.append([y, *(torch.autograd.grad(y, t, dy) if grads else ())])
        if grads:  # changed back between a forward and its backward, which quantizes dY, W and X anew
            t = [v.clone().requires_grad_(True) for v in (x, w)]
            y = be.linear(*t, None)
            setattr(be, attr, before)
            out.append([y, *torch.autograd.grad(y, t, dy)])
    half = len(out) // 2
    assert not _same(out[0][0], out[1][0]), "the change should show in the output"
    for one, gen in zip(out[:half], out[half:]):
        assert all(_same(p, q) for p, q in zip(one, gen))


@pytest.mark.parametrize("recipe", ["ste", "fp8"])
def test_one_row_with_a_short_pitch(gpu_device, recipe):
    """One token: a [1, N] gradient and a [1, K] input that are transposes of
    columns have strides (1, 1), which torch counts as contiguous"""
    N, K = 192, 256
    x = seeded((1, K), seed=20262171).to(gpu_device)
    w = seeded((N, K), seed=20262172, std=0.02).to(gpu_device)
    b = seeded((N,), seed=20262173).to(gpu_device)
    dy = seeded((1, N), seed=20262174, std=1e-3).to(gpu_device)
    up = dy.reshape(N, 1).clone().t()
    assert up.stride() == (1, 1)
    one, gen = _both("e4m3", "nearest", recipe, x, w, b, up, general_dy=dy)
    assert _agree(recipe, one, gen)
    xt = x.reshape(K, 1).clone().t()
    assert xt.stride() == (1, 1)
    be = _backend("e4m3", "nearest", recipe, K, N)
    t = [xt.requires_grad_(True), w.clone().requires_grad_(True), b.clone().requires_grad_(True)]
    y = be.linear(*t)
    assert _agree(recipe, [y, *torch.autograd.grad(y, t, dy)], gen)


@pytest.mark.parametrize("recipe", ["ste", "fp8"])
def test_saved_tensor_hooks(gpu_device, recipe):
    """what was kept for the backward may go through host memory, or come back
    in another layout; left in host memory, or cut short, it is an error
    before any launch"""
    M, N, K = 40, 192, 320
    x = seeded((M, K), seed=20262191).to(gpu_device)
    w = seeded((N, K), seed=20262192, std=0.02).to(gpu_device)
    dy = seeded((M, N), seed=20262193, std=1e-3).to(gpu_device)

    def grads(pack, unpack):
        be = _backend("e4m3", "nearest", recipe, K, N)
        t = [v.clone().requires_grad_(True) for v in (x, w)]
        with torch.autograd.graph.saved_tensors_hooks(pack, unpack):
            y = be.linear(*t, None)
        return torch.autograd.grad(y, t, dy)

    plain = grads(lambda s: s, lambda s: s)
    layouts = [lambda s: s.cpu(), lambda s: s.t().contiguous().t() if s.dim() == 2 else s.clone()]
    for pack in layouts:
        assert all(_same(p, q) for p, q in zip(plain, grads(pack, lambda s: s.to(gpu_device))))
    with pytest.raises(RuntimeError, match="ROCm device"):
        grads(lambda s: s.cpu(), lambda s: s)
    with pytest.raises(RuntimeError, match="saved codes" if recipe == "ste" else "another size"):
        grads(lambda s: s, lambda s: s[:-256] if recipe == "ste" else s[:-1])


@pytest.mark.parametrize("grads", [(True, True, True), (True, False, True), (False, True, False), (False, False, True)])
def test_saved_memory_follows_the_wanted_gradients(gpu_device, grads):
    """the storage kept for a straight-through backward: W's codes for dX, X's
    codes for dW, neither for db, as the general path keeps them (plus the
    alignment of the parts and the int grid's row flags)"""
    M, N, K = 500, 700, 1000
    x = seeded((M, K), seed=20262181).to(gpu_device)
    w = seeded((N, K), seed=20262182, std=0.02).to(gpu_device)
    b = seeded((N,), seed=20262183).to(gpu_device)
    held = []
    for general in (False, True):
        be = _backend("int_grid", "nearest", "ste", K, N)
        if general:
            be._one_call = lambda *a: False
        t = [v.clone().requires_grad_(g) for v, g in zip((x, w, b), grads)]
        storages = {}

        def pack(s):
            storages[s.untyped_storage().data_ptr()] = s.untyped_storage().nbytes()
            return s

        with torch.autograd.graph.saved_tensors_hooks(pack, lambda s: s):
            be.linear(*t)
        held.append(sum(storages.values()))
    assert held[0] <= held[1] + 6 * 256 + 4 * (M + N), held


@pytest.mark.parametrize("grads", [(True, True), (True, False), (False, True)])
def test_gradient_of_another_dtype(gpu_device, grads):
    """an fp32 dY handed to the backward: the dequantized operands, rebuilt from
    the parts that were kept"""
    M, N, K = 70, 200, 300
    x = seeded((M, K), seed=20262195).to(gpu_device)
    w = seeded((N, K), seed=20262196, std=0.02).to(gpu_device)
    dy = seeded((M, N), seed=20262197, std=1e-3, dtype=torch.float32).to(gpu_device)
    from lowbit.backend import _HipLowBitLinear

    out = []
    for general in (False, True):
        be = _backend("int_grid", "nearest", "ste", K, N)
        if general:
            be._one_call = lambda *a: False
        t = [v.clone().requires_grad_(g) for v, g in zip((x, w), grads)]
        y = be.linear(*t, None)
        out.append(_HipLowBitLinear.backward(y.grad_fn, dy))
    assert all(_same(p, q) for p, q in zip(*out))
    assert [v is not None for v in out[0]] == [*grads, False, False]


@pytest.mark.parametrize("mnk", [(64, 256, 320), (500, 1536, 4600)])
def test_wide_gradient_rows(gpu_device, mnk):
    """a dY whose row pitch is past the one the small dX and dW tiles take (the
    last columns of a wider gradient): the 256x256 tiles, dX with its split tail"""
    M, N, K = mnk
    x = seeded((M, K), seed=20262201).to(gpu_device)
    w = seeded((N, K), seed=20262202, std=0.02).to(gpu_device)
    big = seeded((M, 2 * N), seed=20262203, std=1e-3).to(gpu_device)
    one, gen = _both("e4m3", "nearest", "ste", x, w, None, big[:, N:], general_dy=big[:, N:].contiguous())
    assert _agree("ste", one, gen)
