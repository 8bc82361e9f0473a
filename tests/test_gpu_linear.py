"""The few-row projection kernel (``kda_linear_fwd``) against float64, and what it leaves to the library."""

from __future__ import annotations

import importlib

import pytest
import torch

DEV = "cuda:0"


@pytest.fixture(scope="module")
def host(kda_pkg):
    return importlib.import_module("kimi_linear_amd._native").host()


def data(M, K, N, dtype, seed=0):
    gen = torch.Generator().manual_seed(seed)
    x = torch.randn(M, K, generator=gen).to(dtype).to(DEV)
    w = (torch.randn(N, K, generator=gen) * K ** -0.5).to(dtype).to(DEV)
    return x, w


def check(y, x, w):
    """|y - x w^T| within the result's rounding (half an ulp, 2^-11 or 2^-8 of
    it) and that of K fp32 additions (K 2^-24 of the sum of magnitudes; fp16
    results below 2^-14 round to multiples of 2^-24)."""
    x, w = x.double(), w.double()
    ref, mag = x @ w.t(), x.abs() @ w.abs().t()
    ulp = 2.0 ** (-11 if y.dtype == torch.float16 else -8)
    bound = ulp * ref.abs() + x.shape[-1] * 2.0 ** -24 * mag + 2.0 ** -24
    assert bool(((y.double() - ref).abs() <= bound).all())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M", [1, 15, 16, 17, 33, 64])
@pytest.mark.parametrize("K,N", [(2048, 6416), (128, 2048), (32, 16), (96, 48), (512, 32), (544, 64), (1024, 16),
                                 (1152, 6160), (3328, 16), (64, 6144)])
def test_few_rows(host, M, K, N, dtype):
    """Tile edges of the rows, one and several waves a tile, steps left over by every depth."""
    x, w = data(M, K, N, dtype)
    big = torch.full((M, 1, K + 24), float("nan"), dtype=dtype, device=DEV)     # strided rows
    big[:, 0, 8:K + 8] = x
    if M > 16 and K > (1024 if M <= 32 else 512):
        assert host.linear(x.view(M, 1, K), w, None, None) is None              # the library's
        return
    res = torch.randn(M, 1, N, device=DEV).to(dtype)
    y = host.linear(big[..., 8:K + 8], w, None, None)
    check(y[:, 0], x, w)
    out = torch.full((M, 1, N), float("nan"), dtype=dtype, device=DEV)
    assert host.linear(x.view(M, 1, K), w, res, out).data_ptr() == out.data_ptr()
    assert torch.equal(out, res + y)
    w2 = data(M, K, N + 32, dtype, seed=1)[1]
    y0, y1 = host.linear2(x.view(M, 1, K), w, big[..., 8:K + 8], w2)
    assert torch.equal(y0, y)
    check(y1[:, 0], x, w2)


@pytest.mark.gpu
def test_left_to_the_library(host):
    x, w = data(4, 64, 32, torch.float16)
    x = x.view(2, 2, 64)
    assert host.linear(x, w, None, None) is not None
    assert host.linear(x.float(), w.float(), None, None) is None
    assert host.linear(x, w.bfloat16(), None, None) is None
    assert host.linear(x, w[:24], None, None) is None                     # N not a multiple of 16
    assert host.linear(x[..., :48], w[:, :48], None, None) is None        # w not contiguous, K no multiple of 32
    assert host.linear(x[..., :32], w[:, :32].contiguous(), None, None) is not None
    odd = torch.zeros(2, 2, 68, dtype=x.dtype, device=DEV)
    assert host.linear(odd[..., 1:33], w[:, :32].contiguous(), None, None) is None      # rows not 16-byte aligned
    assert host.linear(x.expand(2, 2, 64).repeat(33, 1, 1), w, None, None) is None      # 132 rows
    assert host.linear(x.transpose(0, 1), w, None, None) is None          # rows of two strides
    assert host.linear(x, w, None, x[..., :32]) is None                   # an output that overlaps an input
    assert host.linear(x[:0], w, None, None) is None
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert host.linear(x, w, None, None) is None
    assert host.linear(x, w.clone().requires_grad_(), None, None) is None


@pytest.mark.gpu
def test_modules_with_a_behaviour_of_their_own_are_called(kda_pkg):
    """A hook or a replaced projection takes part in a decode step as in any other call."""
    layer = importlib.import_module("kimi_linear_amd.layer")
    mod = torch.nn.Linear(64, 32, bias=False, device=DEV, dtype=torch.float16)
    x = torch.randn(1, 1, 64, device=DEV, dtype=torch.float16)
    with torch.no_grad():
        assert layer._plain_weight(mod) is mod.weight
        hook = mod.register_forward_hook(lambda m, a, y: y * 0)
        assert layer._plain_weight(mod) is None and not layer._project(mod, x).any()
        hook.remove()
        mod.forward = lambda a: a.new_ones(1, 1, 32)
        assert torch.equal(layer._project(mod, x), torch.ones_like(x[..., :32]))
    assert layer._plain_weight(torch.nn.Linear(64, 32)) is None           # a bias


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", [(512, 64, 128), (513, 2048, 128), (545, 64, 256), (1000, 1024, 128),
                                   (8192, 2048, 128), (8225, 64, 128)])
def test_weight_gradient(host, M, N, K, dtype):
    """dy^T x: rows left over by a step, by the waves and by the splits, strided
    rows.  Bound: the result's rounding and M fp32 additions."""
    gen = torch.Generator().manual_seed(M)
    dy = torch.randn(M, N, generator=gen).to(dtype).to(DEV)
    big = torch.full((1, M, K + 24), float("nan"), dtype=dtype, device=DEV)
    big[0, :, 8:K + 8] = torch.randn(M, K, generator=gen).to(dtype)
    x = big[..., 8:K + 8]
    dw = host.linear_wgrad(dy.view(1, M, N), x)
    assert torch.equal(dw, host.linear_wgrad(dy.view(1, M, N), x))
    check_bound = dy.double().t() @ x[0].double()
    mag = dy.double().abs().t() @ x[0].double().abs()
    ulp = 2.0 ** (-11 if dtype == torch.float16 else -8)
    assert bool(((dw.double() - check_bound).abs() <= ulp * check_bound.abs() + M * 2.0 ** -24 * mag + 2.0 ** -24).all())


@pytest.mark.gpu
def test_weight_gradient_left_to_the_library(host):
    dy = torch.zeros(2, 300, 64, device=DEV, dtype=torch.float16)
    x = torch.zeros(2, 300, 128, device=DEV, dtype=torch.float16)
    assert host.linear_wgrad(dy, x) is not None
    assert host.linear_wgrad(dy[..., :32], x[..., :32]) is None
    assert host.linear_wgrad(dy.float(), x.float()) is None
    assert host.linear_wgrad(dy, x.bfloat16()) is None
    assert host.linear_wgrad(dy[:, :280], x[:, :280]) is None             # rows of two strides
    assert host.linear_wgrad(dy[:1], x[:1]) is None                       # 300 tokens
    assert host.linear_wgrad(dy[:, :0], x[:, :0]) is None
    odd = torch.zeros(2, 300, 130, device=DEV, dtype=torch.float16)
    assert host.linear_wgrad(dy, odd[..., 1:129]) is None                 # rows not 8-byte aligned


@pytest.mark.gpu
def test_linear_function_gradients(kda_pkg):
    """The training path's up-projection against autograd's own linear layer."""
    layer = importlib.import_module("kimi_linear_amd.layer")
    mod = torch.nn.Linear(128, 256, bias=False, device=DEV, dtype=torch.float16)
    x = torch.randn(2, 400, 128, device=DEV, dtype=torch.float16, requires_grad=True)
    dy = torch.randn(2, 400, 256, device=DEV, dtype=torch.float16)
    y, ref = layer._project_train(mod, x), mod(x)
    assert torch.equal(y, ref) and type(y.grad_fn).__name__ == "_LinearFnBackward"
    dx, dw = torch.autograd.grad(y, (x, mod.weight), dy)
    rx, rw = torch.autograd.grad(ref, (x, mod.weight), dy)
    for a, b in ((dx, rx), (dw, rw)):       # two roundings of sums of 800 products, a few tens in size
        assert bool(((a.double() - b.double()).abs() <= 2.0 ** -10 * b.double().abs() + 800 * 2.0 ** -23 * 60).all())
    mod.register_full_backward_hook(lambda *a: None)
    assert type(layer._project_train(mod, x).grad_fn).__name__ != "_LinearFnBackward"


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 16])
@pytest.mark.parametrize("K,N", [(512, 4096), (512, 4112), (1024, 4112), (544, 6160), (96, 4128)])
def test_rows_of_w_per_workgroup(host, M, K, N):
    """Around 4096 outputs: 16 or 32 rows of W a workgroup, a last one half empty, one wave a workgroup."""
    x, w = data(M, K, N, torch.float16, seed=N)
    y = host.linear(x.view(M, 1, K), w, None, None)
    check(y[:, 0], x, w)
    part = host.linear(x.view(M, 1, K), w[:2048], None, None)       # 16 rows a workgroup: the same sums
    assert torch.equal(y[..., :2048], part)
