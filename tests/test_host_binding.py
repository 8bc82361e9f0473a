"""The wrapper's native side (``csrc/host_binding.cpp``) against its general
path: the same bits for every call it answers, and None -- the general path's
case -- for every call with something to convert, copy, differentiate, trace
or refuse."""

from __future__ import annotations

import importlib

import pytest
import torch

DEV = "cuda:0"


@pytest.fixture(scope="module")
def kda(kda_pkg):
    return importlib.import_module("kimi_linear_amd.kda")


@pytest.fixture(scope="module")
def host(kda_pkg):
    return importlib.import_module("kimi_linear_amd._native").host()


def inputs(dtype, B=2, T=64, H=2, K=64, V=64, gate=torch.float32, device=DEV):
    wl = importlib.import_module("kimi_linear_amd.workloads")
    i = wl.make_inputs(B, T, H, K, V, device=device, seed=5, qkv_dtype=dtype, gate_dtype=gate, state_std=0.05)
    return [i[n] for n in ("q", "k", "v", "g", "beta")], i["state"]


def call(host, args, state=None, recurrent=False, chunk=32, state_dtype=torch.float32, state_out=None,
         gate=(None, None), epilogue=(None, None, 0.0), segments=1):
    return host.core(recurrent, *args, state, chunk, state_dtype, state_out, *gate, *epilogue, segments)


def test_declines_what_is_not_a_plain_device_tensor(host):
    args, state = inputs(torch.float16, device="cpu")
    assert call(host, args) is None                                       # no HIP device
    assert call(host, [x.to("meta") for x in args]) is None
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode():
        fake = [torch.empty(x.shape, dtype=x.dtype, device="cuda") for x in args]
        assert call(host, fake) is None                                   # a dispatch mode is active
    assert call(host, fake) is None                                       # a tensor subclass outside it
    with pytest.raises(TypeError):
        call(host, [None, *args[1:]])
    seen = []

    def f(x):
        seen.append(call(host, [x, *args[1:]]))
        return x.sum()
    torch.vmap(f)(torch.stack([args[0]] * 2))
    assert seen == [None]


def test_params_key_follows_every_change(host):
    a, b = torch.zeros(4), torch.zeros(4)
    k0 = host.params_key([a, b])
    assert host.params_key([a, b]) == k0
    a.add_(1)
    assert host.params_key([a, b]) != k0
    k1 = host.params_key([a, b])
    assert host.params_key([a, b.clone()]) != k1 and host.params_key([b, a]) != k1
    assert host.params_key([a, a.view(torch.int32)]) != host.params_key([a, a])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,gate", [(torch.float16, torch.float32), (torch.bfloat16, torch.float32),
                                        (torch.float32, torch.float32), (torch.float16, torch.float16)])
@pytest.mark.parametrize("kind", ["chunkwise", "recurrent"])
def test_same_bits_as_the_general_path(kda, host, dtype, gate, kind):
    args, state = inputs(dtype, gate=gate)
    rec = kind == "recurrent"
    forms = {
        "plain": args,
        "body": [x[:, :32] for x in args],                                # token rows of a longer buffer
        "heads": [x.transpose(1, 2).contiguous().transpose(1, 2) for x in args],   # head-major memory
        "batch": [x[1:] for x in args],
    }
    with torch.no_grad():
        for name, a in forms.items():
            B = a[0].shape[0]
            for st in (None, state[:B].contiguous(), state[:B].half()):
                for sd in (torch.float32, torch.bfloat16, None):
                    got = call(host, a, st, rec, state_dtype=sd)
                    if not rec and gate is not torch.float32:
                        assert got is None                                # the chunk pipeline reads fp32 gates
                        continue
                    want = kda._forward(kind, *a, st, 32, sd)
                    assert got is not None, name
                    assert got[0].dtype == want[0].dtype and got[1].dtype == want[1].dtype
                    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]), name


@pytest.mark.gpu
def test_declines_what_needs_the_general_path(kda, host):
    args, state = inputs(torch.float16)
    q, k, v, g, beta = args
    none = lambda *a, **kw: call(host, *a, **kw) is None                  # noqa: E731
    with torch.no_grad():
        assert none([q.float(), k, v, g, beta])                           # q in another type
        assert none([q.double(), k.double(), v.double(), g, beta])
        assert none([q, k, v, g.half(), beta])                            # the chunk pipeline reads fp32 gates
        assert none([q[..., ::2], k[..., ::2], v, g[..., ::2], beta])     # strided channels
        assert none([q[:, :1].expand(-1, 64, -1, -1), k, v, g, beta])     # broadcast token rows
        assert none([q, k, v, g, beta[:, :1].expand(-1, 64, -1)])
        assert none(args, state.transpose(2, 3))                          # a state of other strides
        assert none(args, state.double())
        assert none(args, chunk=48) and none(args, chunk=0)               # T % chunk != 0
        assert none(args, state_dtype=torch.float64)
        assert none([q, k[:, :32], v, g, beta]) and none([q, k, v, g, beta[..., :1]])
        assert none([q, k, v.cpu(), g, beta])
        assert none(args, state, state_out=state)                         # in place is the recurrence's
        assert not none(args, state, recurrent=True, state_out=state.clone())
        assert none(args, state, recurrent=True, state_out=state.half())
        both = torch.empty(state.numel() + 8, device=DEV)
        a, b = both[:-8].view(state.shape), both[8:].view(state.shape)
        assert none(args, a, recurrent=True, state_out=b)                 # partial overlap
        assert none([x[:0] for x in args]) and none([x[..., :48] for x in (q, k)] + [v, g[..., :48], beta])
        assert not none(args)
    qg = q.clone().requires_grad_()
    assert none([qg, k, v, g, beta])
    with torch.no_grad():
        assert not none([qg, k, v, g, beta])
    import torch.autograd.forward_ad as fwad
    with fwad.dual_level():
        assert none([fwad.make_dual(q, torch.ones_like(q)), k, v, g, beta])


@pytest.mark.gpu
def test_layer_kernels_match_their_general_path(kda_pkg, monkeypatch):
    """kda_prep and kda_output through the native side and with it turned off."""
    ops = importlib.import_module("kimi_linear_amd.layer_ops")
    B, T, H, K, V = 2, 21, 2, 64, 128
    gen = torch.Generator().manual_seed(1)
    rn = lambda *s: torch.randn(*s, generator=gen).half().to(DEV)          # noqa: E731
    big = rn(B, T, 3 * H * K + H * V + H)
    x = big.split((H * K, H * K, H * V, H * K, H), -1)
    w = [rn(D, 1, 4) for D in (H * K, H * K, H * V)]
    bias = [rn(H * K), None, rn(H * V)]
    al, dt = rn(H, K).float(), rn(H, K).float()
    hist = dict(zip("qkv", (rn(B, 3, D) for D in (H * K, H * K, H * V))))
    o, wn = rn(B, T, H, V), rn(H, V)

    def run():
        with torch.no_grad():
            out = [ops.kda_prep(*x[:3], w, bias, gk, al, dt, x[4], num_heads=H, head_dim=K, value_head_dim=V,
                                l2_eps=1e-6, hist=h, want_hist=wh)
                   for gk in (None, x[3]) for h in (None, hist) for wh in (False, True)]
            return out, ops.kda_output(o, big[..., :H * V], wn, 1e-6)

    got, y = run()

    class Off:
        prep = output = staticmethod(lambda *a: None)
    monkeypatch.setattr(ops._native, "host", lambda: Off)
    want, y2 = run()
    assert torch.equal(y, y2)
    for a, b in zip(got, want):
        for p, r in zip(a, b):
            if isinstance(r, dict):
                assert all(torch.equal(p[n], r[n]) for n in "qkv")
            else:
                assert (p is None and r is None) or torch.equal(p, r)


# ---- the native side on CPU tensors, bound to stand-ins for the library's entry points
@pytest.fixture
def stand_in(kda_pkg, tmp_path):
    """``bind(**entries)``: a copy of the native module of its own whose library
    consists of the given callables (args, stream, ..) -> status."""
    import ctypes
    import importlib.util
    import shutil
    native = importlib.import_module("kimi_linear_amd._native")
    error = importlib.import_module("kimi_linear_amd.kda").KdaError
    path = shutil.copy(native.HOST_PATH, tmp_path / "_kda_host.so")
    spec = importlib.util.spec_from_file_location("_kda_host", str(path))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    keep, lib = [], native.load()

    def bind(**entries):
        addr = {n: ctypes.cast(getattr(lib, n), ctypes.c_void_p).value for n in native.EXPORTED_SYMBOLS}
        for n, f in entries.items():
            if not isinstance(f, int):
                keep.append(ctypes.CFUNCTYPE(ctypes.c_int, *[ctypes.c_void_p] * 4)(f))
                f = ctypes.cast(keep[-1], ctypes.c_void_p).value
            addr[n] = f
        mod.bind(addr, lambda index: 0, error, "cpu")
        return mod
    yield bind
    keep.clear()


def host_calls(mod):
    """entry point -> a call of the native side that ends in it"""
    args, state = inputs(torch.float16, device="cpu")
    B, T, H, K = args[0].shape
    V = args[2].shape[-1]
    ga = (torch.rand(H, K), torch.rand(H, K))
    gated = [*args[:3], args[3].half(), args[4].half()]
    og, wn = torch.rand(B, T, H * V).half(), torch.rand(H, V)
    long = [x[:1, :1].expand(1, 4096, *x.shape[2:]).contiguous() for x in args]
    x = torch.rand(B, T, H * K).half()
    w = [torch.rand(H * D, 1, 4).half() for D in (K, K, V)]
    hist = [torch.rand(B, 3, H * D).half() for D in (K, K, V)]
    few, wl = torch.rand(2, 1, 64).half(), torch.rand(32, 64).half()
    none = (None, None, None)
    return {
        "kda_recurrent_fwd": lambda: call(mod, args, state, True, state_out=state),
        "kda_recurrent_gated_fwd": lambda: call(mod, gated, state, True, state_out=state, gate=ga),
        "kda_chunkwise_fwd": lambda: call(mod, args),
        "kda_chunkwise_gated_fwd": lambda: call(mod, gated, gate=ga),
        "kda_chunkwise_fused_fwd": lambda: call(mod, gated, gate=ga, epilogue=(og, wn, 1e-6)),
        "kda_chunkwise_long_fwd": lambda: call(mod, long, segments=2),
        "kda_prep_fwd": lambda: mod.prep((x, x, x), w, none, None, None, None, None, H, K, V, 1e-6, hist, hist, False),
        "kda_output_fwd": lambda: mod.output(args[2], og, wn.half(), 1e-6),
        "kda_linear_fwd": lambda: mod.linear(few, wl, None, None),
        "kda_linear_wgrad": lambda: mod.linear_wgrad(torch.rand(1, 512, 64).half(), torch.rand(1, 512, 128).half()),
    }


@pytest.mark.parametrize("status", ["launch", "refused", "ok"])
def test_a_failed_launch_is_not_run_again(stand_in, kda, status):
    """A launch error raises after one call (its kernels may have run, on a state
    in place); only a refusal, which launches nothing, is the general path's."""
    code = {"launch": 6, "refused": 4, "ok": 0}[status]
    seen = []
    names = list(host_calls(None))
    entry = {n: (lambda *a, n=n: seen.append(n) or code) for n in names}
    # (the segmented call in its one-launch form: no split workspace)
    mod = stand_in(**entry, kda_chunkwise_split_workspace_size=lambda *a: 0)
    for n, f in host_calls(mod).items():
        with torch.no_grad():
            if status == "launch":
                with pytest.raises(kda.KdaError, match="launch failed"):
                    f()
            else:
                assert (f() is None) == (status == "refused")
        assert seen == [n]
        seen.clear()


def test_launches_run_without_the_interpreter_lock(stand_in):
    """Other Python threads run while a launch waits for a full queue: the entry
    points are called without the lock (PyGILState_Check is 0, their KDA_OK)."""
    import ctypes
    check = ctypes.cast(ctypes.pythonapi.PyGILState_Check, ctypes.c_void_p).value
    mod = stand_in(**{n: check for n in host_calls(None)}, kda_chunkwise_split_workspace_size=lambda *a: 0)
    for n, f in host_calls(mod).items():
        with torch.no_grad():
            assert f() is not None, n


def test_another_torch_than_it_was_compiled_against(kda_pkg, monkeypatch):
    """torch's C++ interface changes between releases: the native side refuses to run under another one."""
    native = importlib.import_module("kimi_linear_amd._native")
    monkeypatch.setattr(native, "_host", None)
    assert native.host().torch_version == torch.__version__
    monkeypatch.setattr(native, "_host", None)
    monkeypatch.setattr(torch, "__version__", "0.0.1")
    with pytest.raises(native.NativeLibraryError, match="torch 0.0.1; rebuild"):
        native.host()


def test_an_output_among_the_rows_of_an_input_is_the_general_paths(stand_in):
    """x or the residual as every other row of a buffer whose last row is the output:
    it lies past as many bytes as they hold, before their end."""
    mod = stand_in(kda_linear_fwd=lambda *a: 0)
    w = torch.rand(64, 64).half()
    buf = torch.rand(8, 1, 64).half()
    rows, out = buf[:7:2], buf[5:6]                       # rows 0, 2, 4, 6
    with torch.no_grad():
        assert mod.linear(rows[:3], w, None, buf[5:8]) is not None
        assert mod.linear(rows, w, None, buf[4:8]) is None
        assert mod.linear(buf[:1].expand(1, 1, 64), w, rows[:1], out) is not None
        x = torch.rand(4, 1, 64).half()
        assert mod.linear(x, w, rows, buf[4:8]) is None and mod.linear(x, w, rows, None) is not None
        assert mod.linear(x, w[:16], None, x.view(-1)[64:128].view(4, 1, 16)) is None


@pytest.mark.parametrize("T,segments,first", [(32768, 8, True), (16384, 8, False), (32768, 16, False), (32704, 8, False),
                                              (65536, 8, True)])
def test_the_split_form_is_for_long_segments(stand_in, kda, monkeypatch, T, segments, first):
    """Transition columns before V columns only in segments of at least 2048
    tokens, from the native side and from the general path."""
    assert kda._transitions_first(T, segments) is first
    seen = []

    class Host:
        @staticmethod
        def core(*a):
            seen.append(a[-2:])
    q = torch.empty(1, T, 2, 128, device="meta")
    monkeypatch.setattr(kda._native, "host", lambda: Host)
    monkeypatch.setattr(kda, "long_segments", lambda *a: segments)
    kda._common("chunkwise", q, q, q, q, q[..., 0], None, 64, None, split=True)
    assert seen == [(segments, first)]
    calls = []
    entry = {n: (lambda *a, n=n: calls.append(n) or 0) for n in ("kda_chunkwise_split_fwd", "kda_chunkwise_long_fwd")}
    mod = stand_in(**entry, kda_chunkwise_split_workspace_size=lambda *a: 256)
    args, _ = inputs(torch.float16, device="cpu")
    one = [x[:1].repeat(1, 4, *[1] * (x.dim() - 2)) for x in args]
    with torch.no_grad():
        assert mod.core(False, *one, None, 64, None, None, None, None, None, None, 0.0, 2, first) is not None
    assert calls == ["kda_chunkwise_split_fwd" if first else "kda_chunkwise_long_fwd"]
