"""The split of a long sequence whose transition columns end once they are
zero (``kda_chunkwise_split_fwd``), against one pass and against the split in
one launch (``kda_chunkwise_long_fwd``) at the same number of segments.

Bounds: as the one-launch split's against one pass, 1e-3 (fp16) or 4e-3 (bf16)
of the outputs and 1e-3 of the state.  Against that split: outputs past the
coefficients' end are the same sum rounded once, so equal; before it they are
the same products.
"""

from __future__ import annotations

import ctypes
import importlib

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def native(kda_pkg):
    return importlib.import_module("kimi_linear_amd._native")


def call(native, inp, segments, form):
    kda = importlib.import_module("kimi_linear_amd.kda")
    lib = native.load()
    q, k, v, g, beta, state = (inp[n] for n in ("q", "k", "v", "g", "beta", "state"))
    B, T, H, K = q.shape
    V = v.shape[-1]
    o = torch.full((B, T, H, V), float("nan"), device=DEV, dtype=v.dtype)
    s = torch.full((B, H, K, V), float("nan"), device=DEV)
    a = native.KdaFwdArgs()
    a.B, a.T, a.H, a.K, a.V = B, T, H, K, V
    for n in ("q", "k", "v", "g", "beta"):
        setattr(a, n, inp[n].data_ptr())
        setattr(a, f"{n}_stride", (ctypes.c_int64 * 3)(*inp[n].stride()[:3]))
    a.qkv_dtype, a.g_dtype, a.beta_dtype = kda._DTYPE_CODE[v.dtype], native.DTYPE_F32, native.DTYPE_F32
    a.state_in, a.state_in_dtype = (state.data_ptr() if state is not None else None), native.DTYPE_F32
    a.state_out, a.state_out_dtype, a.o = s.data_ptr(), native.DTYPE_F32, o.data_ptr()
    a.scale, a.chunk_size = K ** -0.5, T
    if form == "one":
        assert lib.kda_chunkwise_fwd(ctypes.byref(a), None) == 0
    else:
        size = getattr(lib, f"kda_chunkwise_{form}_workspace_size")(B, T, H, K, V, segments)
        assert size > 0
        ws = torch.full((size,), 255, device=DEV, dtype=torch.uint8)      # NaN wherever it is read unwritten
        status = getattr(lib, f"kda_chunkwise_{form}_fwd")(ctypes.byref(a), segments, ctypes.c_void_p(ws.data_ptr()),
                                                           None)
        assert status == 0
    torch.cuda.synchronize()
    return o, s


def inputs(B, T, H, K, V, dtype, decay, state=True):
    wl = importlib.import_module("kimi_linear_amd.workloads")
    inp = wl.make_inputs(B, T, H, K, V, device=DEV, seed=K + V, qkv_dtype=dtype, state_std=0.05 if state else None)
    inp["g"] = inp["g"] * decay
    return inp


def rel(a, b):
    return ((a.double() - b.double()).norm() / b.double().norm()).item()


@pytest.mark.parametrize("B,T,H,K,V,dtype,decay,state", [
    (1, 4096, 2, 128, 128, torch.float16, 1.0, True),       # ends after a few chunks
    (1, 4096, 2, 128, 128, torch.float16, 1.0, False),      # no initial state: segment 0 needs no correction
    (1, 4176, 3, 128, 128, torch.float16, 0.05, True),      # ends part-way; segments end inside a chunk
    (1, 4096, 2, 128, 128, torch.bfloat16, 1e-3, True),     # never ends
    (2, 4096, 1, 64, 64, torch.float16, 1.0, True),
    (1, 4240, 2, 64, 192, torch.bfloat16, 0.1, True),
    (1, 4096, 1, 128, 256, torch.float16, 0.3, False),
])
def test_split_matches_one_pass(native, B, T, H, K, V, dtype, decay, state):
    inp = inputs(B, T, H, K, V, dtype, decay, state)
    o, s = call(native, inp, 2, "split")                    # 2 segments, doubled to 4
    ol, sl = call(native, inp, 4, "long")
    o1, s1 = call(native, inp, 1, "one")
    d_o, d_s = rel(o, o1), rel(s, s1)
    print(f"split B{B} T{T} H{H} K{K} V{V} {dtype} x{decay}: vs one pass o {d_o:.2e} s {d_s:.2e}", flush=True)
    assert d_o <= (1e-3 if dtype == torch.float16 else 4e-3) and d_s <= 1e-3
    assert torch.equal(s, sl)
    assert torch.equal(o, ol)


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_split_keeps_what_is_not_finite(native, bad):
    """An infinity or a NaN in the initial state: the same entries are NaN or
    infinite as in the one-launch split, past the coefficients' end too."""
    inp = inputs(1, 4096, 2, 128, 128, torch.float16, 1.0)
    inp["state"][0, 1, 17, 40] = bad
    o, s = call(native, inp, 2, "split")
    ol, sl = call(native, inp, 4, "long")
    assert not torch.isfinite(o[0, :, 1, 40]).any()
    assert torch.equal(torch.isfinite(o), torch.isfinite(ol)) and torch.equal(torch.isfinite(s), torch.isfinite(sl))
    ok = torch.isfinite(ol)
    assert torch.equal(o[ok], ol[ok])


def test_split_form_and_its_limits(native):
    lib = native.load()
    size = lib.kda_chunkwise_split_workspace_size
    assert size(1, 32768, 16, 128, 128, 8) > lib.kda_chunkwise_long_workspace_size(1, 32768, 16, 128, 128, 8)
    assert size(1, 4096, 16, 128, 128, 8) == 0              # segments of 512 are not halved
    assert size(1, 32768, 16, 128, 64, 16) == 0             # V + K = 192
    assert size(1, 32768, 16, 128, 128, 16) == 0            # the one-launch form would take two rounds
    assert size(1, 32768, 16, 32, 32, 8) == 0
    assert size(1, 4096, 1, 64, 64, 3) == 0
