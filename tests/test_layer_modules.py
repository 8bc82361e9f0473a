"""CPU tests of the layer's callable helper modules -- ``ShortConv``,
``HeadwiseRMSNorm`` and ``l2norm`` (``kimi_linear/kda.py:258-325``) -- for
reference-side code that calls them directly.  The checkers are the layer
oracle's pieces, which tests/test_layer_oracle.py pins against
``F.conv1d`` with history, ``F.rms_norm`` and ``F.normalize``."""

from __future__ import annotations

import pytest
import torch

from oracle.kda_layer_oracle import head_rmsnorm_ref, l2norm_ref, short_conv_ref


def _rel(a, b):
    a, b = a.double(), b.double()
    return ((a - b).norm() / b.norm()).item()


@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("cs", [4, 2])
def test_short_conv_forward_and_cached_step(kda_pkg, bias, cs):
    torch.manual_seed(cs + bias)
    B, T, D = 2, 21, 48
    m = kda_pkg.ShortConv(D, cs, bias=bias)
    x = torch.randn(B, T, D)
    with torch.no_grad():
        y = m(x)
        ref = short_conv_ref(x, m.conv.weight, m.conv.bias)
        assert y.shape == (B, T, D) and _rel(y, ref) <= 1e-6
        # one cached token continues the sequence: the window is the last cs - 1 inputs + x_t
        state = x[:, T - cs:T - 1] if cs > 1 else x[:, :0]
        yt, new_state = m(x[:, T - 1:T], state, use_cache=True)
        assert yt.shape == (B, 1, D) and _rel(yt[:, 0], ref[:, T - 1]) <= 1e-6
        assert torch.equal(new_state, x[:, T - cs + 1:T])
        # fp16 inputs keep their dtype, the cached sum runs in fp32
        yh, _ = m.half()(x[:, :1].half(), state[:, :cs - 1].half(), use_cache=True)
        assert yh.dtype == torch.float16


def test_headwise_rmsnorm_forward(kda_pkg):
    torch.manual_seed(3)
    B, T, H, D = 2, 5, 3, 32
    m = kda_pkg.HeadwiseRMSNorm(H, D, 1e-6)
    with torch.no_grad():
        m.weight.normal_(1.0, 0.1)
    x = torch.randn(B, T, H, D)
    with torch.no_grad():
        assert _rel(m(x), head_rmsnorm_ref(x, m.weight, 1e-6)) <= 1e-6
        assert m(x.half()).dtype == torch.float16


def test_l2norm(kda_pkg):
    torch.manual_seed(4)
    x = torch.randn(3, 7, 2, 64)
    assert _rel(kda_pkg.l2norm(x, 1e-6), l2norm_ref(x, 1e-6)) <= 1e-6
    tiny = torch.full((1, 64), 1e-9)                      # rsqrt clamped to 1 / eps
    assert torch.allclose(kda_pkg.l2norm(tiny, 1e-6), tiny * 1e6)
    assert kda_pkg.l2norm(x.half(), 1e-6).dtype == torch.float16


def test_a_function_mode_or_subclass_sees_the_projections(kda_pkg):
    """A torch function mode or a tensor subclass may change ``F.linear``: the
    projections are then the module's own call."""
    import importlib
    from torch.overrides import TorchFunctionMode
    layer = importlib.import_module("kimi_linear_amd.layer")

    class Mode(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Sub(torch.Tensor):
        pass

    mod, x = torch.nn.Linear(8, 4, bias=False), torch.randn(1, 1, 8)
    assert layer._plain_weight(mod, x) is mod.weight
    assert layer._plain_weight(mod, x.as_subclass(Sub)) is None
    with Mode():
        assert layer._plain_weight(mod, x) is None
    mod.weight = torch.nn.Parameter(mod.weight.detach().as_subclass(Sub))
    assert layer._plain_weight(mod, x) is None


@pytest.mark.parametrize("rows,k,n,own", [
    (1, 2048, 6416, True), (16, 2048, 2048, True), (17, 2048, 2048, False), (32, 1024, 4096, True), (33, 1024, 4096, False),
    (64, 512, 2048, True), (65, 128, 2048, False), (64, 128, 2048, True),
    (1, 2048, 12576, False), (32, 512, 12576, True), (33, 512, 12576, False), (1, 2048, 8192, True),
    (4, 2304, 4096, True), (5, 2304, 4096, False), (1, 2304, 6416, False), (1, 2304, 512, False), (1, 4096, 2304, True),
    (1, 4128, 4096, False), (1, 3104, 4096, False), (1, 1568, 2048, False), (16, 1568, 4096, True), (1, 1056, 2048, True), (17, 1056, 4096, False),
    (1, 544, 2048, True), (1, 48, 2048, False)])
def test_few_row_projections_where_they_are_faster(kda_pkg, rows, k, n, own):
    import importlib
    layer = importlib.import_module("kimi_linear_amd.layer")
    assert layer._few_rows(rows, k, n) is own
    if own:       # nothing that the kernel refuses
        assert k % 32 == 0 and (rows <= 16 or k <= (1024 if rows <= 32 else 512))


def test_gate_projections_may_hold_further_modules(kda_pkg, monkeypatch):
    """The gates' projections are the first and second module of theirs, whatever follows."""
    import importlib
    layer = importlib.import_module("kimi_linear_amd.layer")
    monkeypatch.setattr(layer, "kda_prep", lambda *a, **kw: (None,) * 6)
    m = kda_pkg.KimiDeltaAttention(kda_pkg.linear_attn_config(hidden_size=64, num_heads=1, head_dim=64,
                                                              value_head_dim=64))
    x = torch.randn(1, 5, 64)
    with torch.no_grad():
        want = m._projections(x)
        for proj in (m.gk_proj, m.og_proj):
            proj.append(torch.nn.ReLU())
        got = m._projections(x)
    assert torch.equal(got[3], want[3]) and torch.equal(got[6], want[6])
