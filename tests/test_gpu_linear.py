"""The one-launch FP8 rollout linear (``ops.fp8_linear``) against a float64
product of the same codes, scales and activations, and the calls that
``_FP8W8A8Linear`` must still hand to the library product."""

from __future__ import annotations

import threading

import numpy as np
import pytest
import torch
import torch.nn as nn

from lumenrl_amd.quantization import FP8Config, WeightQuantizer, fp8_linear, ops
from lumenrl_amd.quantization import fp8_rollout
from lumenrl_amd.quantization.fp8_rollout import _FP8W8A8Linear

pytestmark = pytest.mark.gpu
DEV = "cuda"


def operands(m, n, k, dtype, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(m, k, generator=g, device=DEV)
    x[:, k // 3] *= 40.0
    codes = torch.randint(0, 256, (n, k), generator=g, device=DEV, dtype=torch.uint8)
    codes[(codes & 0x7F) == 0x7F] = 0x30  # every code but the NaNs
    scales = (torch.rand(n, k // 128, generator=g, device=DEV) + 0.5) * 1e-4
    return x.to(dtype), codes.view(torch.float8_e4m3fn), scales.to(torch.bfloat16)


def wide(codes, scales):
    n, k = codes.shape
    return (codes.to(torch.float64).view(n, -1, 128) * scales.to(torch.float64)[..., None]).view(n, k)


def check(y, x, codes, scales, bias=None, subnormal=2.0 ** -24):
    """|y - exact| within the result's own rounding and the float32 sums' bound:
    no sum is longer than 128 products, K/128 blocks and 16 waves or parts, each
    rounding (or truncating) by at most 2^-23 of the terms' magnitude; x_dq moves
    a term by at most 2^-23 of itself.  ``subnormal``: one unit of the type's
    subnormals, twice their rounding."""
    k = x.shape[-1]
    w = wide(codes, scales)
    xd = x.double().reshape(-1, k)
    want, size = xd @ w.T, xd.abs() @ w.abs().T
    if bias is not None:
        want, size = want + bias.double(), size + bias.double().abs()
    half_ulp = 2.0 ** -9 if y.dtype == torch.bfloat16 else 2.0 ** -12
    bound = 2 * half_ulp * want.abs() + (128 + k // 128 + 20) * 2.0 ** -23 * size + subnormal
    off = (y.double() - want).abs()
    assert bool((off <= bound).all()), float((off / bound).max())


# one shape for each kernel there is, its last rows and columns cut
EVERY_KERNEL = [(15, 300), (15, 4099), (15, 8200), (31, 2170), (17, 4099), (30, 8200), (30, 12410), (40, 5510), (40, 8200),
                (40, 1410), (60, 6275), (8200, 15), (70, 5510), (150, 4100), (200, 4100), (129, 12289), (390, 9364),
                (1030, 6999)]


# K of one block, an odd number above the waves' eight, and two per wave
@pytest.mark.parametrize("m,n", EVERY_KERNEL)
@pytest.mark.parametrize("dtype,k", [(torch.bfloat16, 128), (torch.float16, 1152), (torch.bfloat16, 2048)])
def test_linear_every_kernel_vs_float64(m, n, dtype, k):
    x, codes, scales = operands(m, n, k, dtype, seed=m * 3 + n)
    bias = torch.randn(n, device=DEV)
    check(fp8_linear(x, codes, scales, bias), x, codes, scales, bias)


@pytest.mark.parametrize("m,n", [(2, 4096), (48, 8200), (200, 4100), (1030, 6999)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_linear_rounds_its_sums_only(dtype, m, n):
    """The share of results that are not the exact product's rounding.  Float32 sums over
    K = 4096 are off by about 2e-6 of the result, which crosses a rounding boundary in 4e-6 of
    a unit in the last place (2^-7 to 2^-8 of it in bf16, 2^-10 to 2^-11 in fp16): 0.1 % and
    0.6 % at most, a few times that where terms cancel.  An operand rounded to bf16 is off by
    1e-3: a third of the bf16 results, nearly all of the fp16 ones."""
    k = 4096
    x, codes, scales = operands(m, n, k, dtype, seed=11)
    x[:, k // 3] /= 40.0
    want = x.double() @ wide(codes, scales).T
    assert (fp8_linear(x, codes, scales) != want.to(dtype)).double().mean() < 0.02


# tokens at the edges of the 16-row groups; weight rows at the edges of 16 and 32
# row tiles and where the tile's shape changes; K of fewer blocks than waves,
# an odd number of blocks and several per wave
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m", [1, 2, 16, 17, 33, 48, 49, 64])
@pytest.mark.parametrize("n,k", [(1, 128), (15, 384), (17, 1152), (1000, 1024), (4099, 256), (12288, 256), (8200, 640)])
def test_linear_vs_float64(dtype, m, n, k):
    x, codes, scales = operands(m, n, k, dtype, seed=m * 7 + n)
    y = fp8_linear(x, codes, scales)
    assert y.dtype == dtype and y.shape == (m, n)
    check(y, x, codes, scales)


# many tokens: every size of tile, with whole and cut last rows and
# columns (also widths that 8 does not divide, stored one by one), one block of K,
# an odd number and an even one; grids of one round and of several
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", [(65, 4096, 256), (129, 12289, 128), (200, 1003, 1024), (512, 4096, 128),
                                   (500, 4090, 384), (700, 4097, 256), (1024, 7168, 128), (1030, 6999, 256),
                                   (1025, 6992, 384), (2049, 4095, 640), (4100, 8192, 128)])
def test_linear_many_tokens_vs_float64(dtype, m, n, k):
    x, codes, scales = operands(m, n, k, dtype, seed=m + n)
    bias = torch.randn(n, device=DEV) if m % 2 else None
    check(fp8_linear(x, codes, scales, bias), x, codes, scales, bias)


@pytest.mark.parametrize("bias_dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_linear_bias_strides_and_alignment(bias_dtype):
    n, k = 264, 512
    big, codes, scales = operands(40, n, 1600, torch.bfloat16, seed=3)
    codes, scales = codes[:, :k].contiguous(), scales[:, :4].contiguous()
    bias = torch.randn(n, device=DEV).to(bias_dtype)
    tall = torch.randn(1100, 2 * k + 5, device=DEV).to(torch.bfloat16)
    for x in (tall[:, 3:3 + k], tall[:600, :2 * k:2], big[:, :k], big[1:20, 3:3 + k], big[:, :2 * k:2], big[None, :6, :k].expand(1, 6, k), big[5, 7:7 + k]):
        y = fp8_linear(x, codes, scales, bias)
        check(y, x, codes, scales, bias)
    with pytest.raises(ValueError):  # rows that share memory are refused, as by act_qdq
        fp8_linear(big[:1, :k].expand(3, k), codes, scales)
    with pytest.raises(ValueError):
        fp8_linear(big[:, :k], codes[:, :384], scales)


@pytest.mark.parametrize("m,n", EVERY_KERNEL)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_linear_over_the_whole_exponent_range(dtype, m, n):
    """Tokens from subnormal to near the type's maximum, in the same tiles: block sums that
    overflow before the weight's scale is applied, results that are subnormal, and both in one
    launch.  No token's result depends on another's size, or on another being inf or NaN."""
    k = 384
    _, codes, scales = operands(1, n, k, dtype, seed=m)
    exps = [0, -112, 118, -118, 0, -124, 114, -130] if dtype == torch.bfloat16 else [0, -14, 10, -18, 0, -20, 11, -22]
    g = torch.Generator(device=DEV).manual_seed(n)
    x = torch.randn(m, k, generator=g, device=DEV).clamp(-4, 4).double()
    x = (x * torch.tensor([2.0 ** exps[i % 8] for i in range(m)], device=DEV, dtype=torch.float64)[:, None]).to(dtype)
    y = fp8_linear(x, codes, scales)
    check(y, x, codes, scales, subnormal=2.0 ** -133 if dtype == torch.bfloat16 else 2.0 ** -24)
    for bad in (float("inf"), float("nan")):
        v = x.clone()
        v[m // 2, 7] = bad
        z = fp8_linear(v, codes, scales)
        assert bool(z[m // 2].isnan().all())
        z[m // 2] = y[m // 2]
        assert torch.equal(z, y)


@pytest.mark.parametrize("m,n", EVERY_KERNEL)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_linear_non_finite_and_extreme_values(dtype, m, n):
    k = 512
    x, codes, scales = operands(m, n, k, dtype, seed=9)
    x[3, 100], x[4, 200], x[5, 300] = float("inf"), float("nan"), float("-inf")
    x[6], x[7] = 0.0, torch.finfo(dtype).max / 2
    x[8] = x[8].sign() * torch.finfo(dtype).tiny * 4
    y = fp8_linear(x, codes, scales)
    keep = [r for r in range(m) if r not in (3, 4, 5, 7)]
    assert bool(y[3:6].isnan().all())  # s is inf or NaN: the whole block, so the whole row, is NaN
    assert bool((y[6] == 0).all())
    check(y[keep], x[keep], codes, scales)
    # finite operands never overflow on the way: only where the result does
    want = x[7].double() @ wide(codes, scales).T
    fits = want.abs() < torch.finfo(dtype).max * 0.99
    check(y[7:8][:, fits], x[7:8], codes[fits], scales[fits])
    over = want.abs() > torch.finfo(dtype).max * 1.01
    assert bool((y[7][over] == torch.where(want[over] > 0, float("inf"), float("-inf")).to(dtype)).all())
    bad = codes.view(torch.uint8).clone()
    bad[5, 40] = 0x7F  # a NaN code: that row of the weight, for every token
    y = fp8_linear(x[8:12], bad.view(torch.float8_e4m3fn), scales)
    assert bool(y[:, 5].isnan().all()) and not bool(y[:, 6:].isnan().any())


@pytest.mark.parametrize("shape", [(0,), (3, 0), (2, 0, 0), (2, 5, 0)])
def test_linear_of_no_columns(shape):
    """K = 0: a row of the bias, or of zeros, for each token there is."""
    x = torch.empty(shape, device=DEV, dtype=torch.bfloat16)
    codes, scales = torch.empty(24, 0, device=DEV, dtype=torch.float8_e4m3fn), torch.empty(24, 0, device=DEV, dtype=torch.bfloat16)
    bias = torch.randn(24, device=DEV)
    rows = int(np.prod(shape[:-1]))
    assert torch.equal(fp8_linear(x, codes, scales), torch.zeros(rows, 24, device=DEV, dtype=torch.bfloat16))
    assert torch.equal(fp8_linear(x, codes, scales, bias), bias.bfloat16().expand(rows, 24))


def module(out, cols, dtype, bias=True, blk=128):
    lin = nn.Linear(cols, out, bias=bias).to(DEV, dtype)
    cfg = FP8Config(precision="fp8")
    return _FP8W8A8Linear(lin, WeightQuantizer(cfg), cfg, blk)


def test_module_routes(monkeypatch):
    """The one-launch path where it applies; F.linear where autocast, the bias's
    gradient, another block, type or device need it, with the results it gives."""
    calls = []
    real = ops.fp8_linear_checked
    monkeypatch.setattr(ops, "fp8_linear_checked", lambda *a: calls.append(1) or real(*a))
    torch.manual_seed(1)
    mod, x = module(1024, 512, torch.bfloat16), torch.randn(2, 9, 512, device=DEV, dtype=torch.bfloat16)

    def taken(m, v):
        calls.clear()
        y = m(v)
        return y, bool(calls)

    y_grad, fused = taken(mod, x)  # the bias wants a gradient
    assert not fused and y_grad.requires_grad
    with torch.no_grad():
        y, fused = taken(mod, x)
        assert fused and y.shape == (18, 1024) and y.dtype == torch.bfloat16
        check(y, x, mod.weight_fp8, mod.weight_scale, mod.bias)
        monkeypatch.setattr(fp8_rollout, "_ONE_LAUNCH_MIN_WEIGHT", 1 << 30)
        y_lib, fused = taken(mod, x)
        monkeypatch.setattr(fp8_rollout, "_ONE_LAUNCH_MIN_WEIGHT", 1 << 18)
        # the same sums in another order: one unit of the last place where they round apart
        assert not fused
        assert bool(((y.double() - y_lib.double()).abs() <= 2.0 ** -7 * y_lib.double().abs() + 1e-5).all())
        with torch.autocast("cuda", torch.bfloat16):
            assert not taken(mod, x)[1]
        assert not taken(mod, x.float())[1] and not taken(mod, x.double())[1] and not taken(mod, x.cpu())[1]
        assert not taken(mod, x[:0])[1]
        assert not taken(module(1024, 384, torch.bfloat16, blk=96), x[..., :384])[1]
        assert not taken(module(384, 512, torch.bfloat16), x)[1]  # a small weight
        with pytest.raises(RuntimeError):  # F.linear's own error for a width that is not the weight's
            mod(x[..., :256])
        half = module(1024, 512, torch.float16, bias=False)
        y, fused = taken(half, x[0, 0].half())
        assert fused and y.shape == (1, 1024)
        check(y, x[0, :1].half(), half.weight_fp8, half.weight_scale)


class _Watched(torch.Tensor):
    seen = []

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        cls.seen.append(func)
        return super().__torch_function__(func, types, args, kwargs or {})


@pytest.mark.filterwarnings("ignore::torch.jit.TracerWarning")
def test_module_shows_its_linear_to_whoever_watches(monkeypatch):
    """A function mode, a dispatch mode, a subclass of Tensor and the tracer see F.linear, as with
    the library product; a default device, which is a function mode too, changes nothing."""
    calls = []
    real = ops.fp8_linear_checked
    monkeypatch.setattr(ops, "fp8_linear_checked", lambda *a: calls.append(1) or real(*a))
    torch.manual_seed(4)
    mod, x = module(1024, 512, torch.bfloat16), torch.randn(5, 512, device=DEV, dtype=torch.bfloat16)
    bias = mod.bias.detach()

    class Functions(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            self.seen.append(func)
            return func(*args, **(kwargs or {}))

    class Operators(torch.utils._python_dispatch.TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.seen.append(func)
            return func(*args, **(kwargs or {}))

    with torch.no_grad():
        y = mod(x)
        assert calls == [1]
        for mode in (Functions(), Operators()):
            mode.seen = []
            with mode:
                check(mod(x), x, mod.weight_fp8, mod.weight_scale, bias)
            assert any("linear" in str(f) or "addmm" in str(f) for f in mode.seen) and calls == [1]
        with torch.device(DEV):
            assert torch.equal(mod(x), y) and calls == [1, 1]
        del mod.bias
        mod.bias = bias.as_subclass(_Watched)
        _Watched.seen.clear()
        check(mod(x), x, mod.weight_fp8, mod.weight_scale, bias)
        assert nn.functional.linear in _Watched.seen and calls == [1, 1]
        mod.bias = bias
        traced = torch.jit.trace(mod, (x,), check_trace=False)
        assert "aten::linear" in str(traced.inlined_graph) and calls == [1, 1]


def test_module_with_replaced_buffers():
    """A bias or scales that do not have one value per row (or block) of the weight
    go to the ops that check them: F.linear broadcasts one bias for all, and refuses
    other lengths; the dequantization refuses scales that are too few.  A bias under
    vmap is a batch of them."""
    torch.manual_seed(2)
    mod, x = module(1024, 512, torch.bfloat16), torch.randn(6, 512, device=DEV, dtype=torch.bfloat16)
    codes, scales = mod.weight_fp8, mod.weight_scale
    with torch.no_grad():
        mod.bias = nn.Parameter(torch.full((1,), 0.5, device=DEV, dtype=torch.bfloat16))
        check(mod(x), x, codes, scales, mod.bias.expand(1024))
        mod.bias = nn.Parameter(torch.zeros(1000, device=DEV, dtype=torch.bfloat16))
        with pytest.raises(RuntimeError):
            mod(x)
        mod.bias = None
        mod.weight_scale = scales[:1000].contiguous()
        with pytest.raises(ValueError):
            mod(x)
        mod.weight_scale = scales
        batch = torch.randn(3, 1024, device=DEV, dtype=torch.bfloat16)

        def with_bias(b):
            mod.__dict__["bias"] = b
            return mod(x)

        del mod.bias
        y = torch.vmap(with_bias)(batch)
        for i in range(3):
            check(y[i], x, codes, scales, batch[i])


def test_linear_on_side_streams_from_two_threads():
    """Each thread on a stream of its own, with inputs made there, many calls in flight."""
    done = [None, None]

    def work(i):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            ops_ = [operands(m, 1100, 512, torch.bfloat16, seed=50 * i + m) for m in (1, 40, 200, 600)]
            ys = [[fp8_linear(*o) for o in ops_] for _ in range(20)]
        stream.synchronize()
        done[i] = ops_, ys

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for ops_, ys in done:
        for i, o in enumerate(ops_):
            check(ys[0][i], *o)
            assert all(torch.equal(y[i], ys[0][i]) for y in ys)


def test_linear_in_a_graph():
    """Captured and replayed with new inputs and eager work between the replays."""
    x, codes, scales = operands(8, 1024, 512, torch.bfloat16)
    fp8_linear(x, codes, scales)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = fp8_linear(x, codes, scales)
    for seed in range(3):
        x.copy_(operands(8, 1024, 512, torch.bfloat16, seed=seed + 20)[0])
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(y.view(torch.int16).cpu().numpy(), fp8_linear(x, codes, scales).view(torch.int16).cpu().numpy())
