"""The recurrence over several tokens (``recurrent_seq_kernel``) against the
float64 recurrence: edges of its 16-token groups (8 at K = 256) and of the
four tokens a loop step takes, every number of columns a workgroup can own,
rows that may and may not be fetched 16 bytes at a time, and the states it
stores for the backward of fp32 activations.

Bounds.  fp32: a token rounds each state entry about four times and each sum
over K = 256 entries at most log2(16) + 16 times on its longest path, all
relative to values the recurrence keeps at the size of its inputs, so errors
stay within a few 2^-24 per token and are damped by the decay: 1e-6 relative.
16-bit: one rounding of the output, 2^-11 (fp16) or 2^-8 (bf16) of its value.
"""

from __future__ import annotations

import importlib

import pytest
import torch

from oracle import kda_recurrent_f64

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
O_TOL = {torch.float32: 1e-6, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}
S_TOL = 1e-6


def rel(a, b):
    a, b = a.detach().double().cpu(), b.detach().double().cpu()
    return ((a - b).norm() / b.norm()).item()


def inputs(B, T, H, K, V, dtype, gate_dtype=torch.float32, state=True):
    wl = importlib.import_module("kimi_linear_amd.workloads")
    inp = wl.make_inputs(B, T, H, K, V, seed=B + 7 * T + K + V, qkv_dtype=dtype, gate_dtype=gate_dtype,
                         state_std=0.05 if state else None)
    return inp, {n: (x.to(DEV) if x is not None else None) for n, x in inp.items()}


def reference(inp):
    o, s = kda_recurrent_f64(inp["q"], inp["k"], inp["v"], inp["g"], inp["beta"], inp["state"])
    return torch.from_numpy(o), torch.from_numpy(s)


def check(tag, o, s, ref, dtype):
    eo, es = rel(o, ref[0]), rel(s, ref[1])
    print(f"[{tag}] o rel {eo:.2e}  state rel {es:.2e}", flush=True)
    assert eo <= O_TOL[dtype] and es <= S_TOL


@pytest.mark.parametrize("B,T,H,K,V,dtype", [
    (1, 2, 2, 128, 128, torch.float32),      # T below one loop step
    (2, 3, 3, 64, 48, torch.float32),        # 16-column workgroups (V = 48)
    (1, 15, 2, 128, 16, torch.float16),
    (1, 16, 2, 32, 32, torch.bfloat16),      # one whole group
    (2, 17, 2, 128, 64, torch.float32),      # a second group of one token
    (1, 39, 1, 256, 32, torch.float32),      # groups of 8
    (1, 8, 2, 256, 64, torch.float16),
    (9, 21, 4, 64, 128, torch.float32),      # 288 column tiles of 16: 32-column workgroups
    (9, 34, 16, 32, 128, torch.float16),     # 1152: 64-column workgroups
    (5, 9, 16, 128, 256, torch.bfloat16),    # 1280, K = 128
    (40, 8, 8, 64, 128, torch.float16),      # a state above the wide bound, at T = 8
    (40, 7, 8, 64, 128, torch.float16),      # and just below it (the per-token kernel)
    (257, 2, 1, 64, 64, torch.float32),      # smaller states whose tokens are faster one at a time
    (65, 2, 1, 128, 128, torch.float16),
    (65, 2, 1, 256, 64, torch.float32),
    (129, 4, 1, 256, 64, torch.bfloat16),
    (129, 7, 1, 256, 128, torch.float32),
    (769, 4, 1, 64, 32, torch.float16),
    (1025, 3, 1, 128, 16, torch.float32),
])
def test_span_matches_float64(kda_pkg, B, T, H, K, V, dtype):
    inp, dev = inputs(B, T, H, K, V, dtype)
    with torch.no_grad():
        o, s = kda_pkg.kda_recurrent(dev["q"], dev["k"], dev["v"], dev["g"], dev["beta"], state=dev["state"],
                                     state_dtype=torch.float32)
    check(f"B{B} T{T} H{H} K{K} V{V} {dtype}", o, s, reference(inp), dtype)


@pytest.mark.parametrize("dtype,gate_dtype", [(torch.float16, torch.float16), (torch.bfloat16, torch.float32),
                                              (torch.float32, torch.float32), (torch.float32, torch.bfloat16)])
@pytest.mark.parametrize("shift", [0, 1])
def test_span_row_alignment(kda_pkg, dtype, gate_dtype, shift):
    """Rows cut out of wider ones, from an aligned and from an odd element:
    the same results, and no state given is a zero state."""
    B, T, H, K, V = 2, 19, 3, 64, 32
    inp, dev = inputs(B, T, H, K, V, dtype, gate_dtype, state=False)

    def cut(x):
        wide = torch.full((*x.shape[:-1], x.shape[-1] + 8), float("nan"), device=DEV, dtype=x.dtype)
        wide[..., shift:shift + x.shape[-1]] = x
        return wide[..., shift:shift + x.shape[-1]]

    with torch.no_grad():
        plain = kda_pkg.kda_recurrent(dev["q"], dev["k"], dev["v"], dev["g"], dev["beta"], state_dtype=torch.float32)
        o, s = kda_pkg.kda_recurrent(cut(dev["q"]), cut(dev["k"]), cut(dev["v"]), cut(dev["g"]), dev["beta"],
                                     state_dtype=torch.float32)
    inp["state"] = torch.zeros(B, H, K, V)
    check(f"{dtype} {gate_dtype} shift {shift}", o, s, reference(inp), dtype)
    assert torch.equal(o, plain[0]) and torch.equal(s, plain[1])


def test_span_state_types_and_in_place(kda_pkg):
    inp, dev = inputs(2, 11, 2, 128, 32, torch.float32)
    args = [dev[n] for n in ("q", "k", "v", "g", "beta")]
    with torch.no_grad():
        o, s = kda_pkg.kda_recurrent(*args, state=dev["state"], state_dtype=torch.float32)
        st = dev["state"].clone()
        o2, s2 = kda_pkg.kda_recurrent(*args, state=st, state_dtype=torch.float32, state_out=st)
        half = dev["state"].half()
        o3, s3 = kda_pkg.kda_recurrent(*args, state=half, state_dtype=torch.float16)
        o4, s4 = kda_pkg.kda_recurrent(*args, state=half.float(), state_dtype=torch.float32)
    assert s2 is st and torch.equal(o, o2) and torch.equal(s, s2)
    assert torch.equal(o3, o4) and torch.equal(s3, s4.half())


def test_span_values_past_t_do_not_count(kda_pkg):
    """A view of the first tokens of a longer buffer whose rest is NaN."""
    _, dev = inputs(2, 18, 2, 128, 32, torch.float32)
    long = {}
    for n in ("q", "k", "v", "g", "beta"):
        x = dev[n]
        buf = torch.full((x.shape[0], 40, *x.shape[2:]), float("nan"), device=DEV, dtype=x.dtype)
        buf[:, :18] = x
        long[n] = buf[:, :18]
    with torch.no_grad():
        a = kda_pkg.kda_recurrent(*(dev[n] for n in ("q", "k", "v", "g", "beta")), state=dev["state"])
        b = kda_pkg.kda_recurrent(*(long[n] for n in ("q", "k", "v", "g", "beta")), state=dev["state"])
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


@pytest.mark.parametrize("T", [31, 32, 65])
def test_fp32_checkpoints_hold_the_states(kda_pkg, T):
    """The record of every 32-token chunk starts with the state before it."""
    kda = importlib.import_module("kimi_linear_amd.kda")
    B, H, K, V = 1, 2, 64, 64
    _, dev = inputs(B, T, H, K, V, torch.float32)
    args = [dev[n] for n in ("q", "k", "v", "g", "beta")]
    with torch.no_grad():
        o, s, ck = kda._forward("chunkwise", *args, dev["state"], 1, torch.float32, ckpt=True)
        for c in range((T + 31) // 32):
            if c == 0:
                want = dev["state"]
            else:
                want = kda_pkg.kda_recurrent(*(x[:, :32 * c] for x in args), state=dev["state"])[1]
            got = ck[:, :, c, :K * V].reshape(B, H, K, V)
            assert torch.equal(got, want)


def test_bf16_rounding_is_nearest_even(kda_pkg):
    """Stored bf16 values (here the state of a call without tokens) are torch's
    rounding of the fp32 ones bit for bit: any exponent, ties, denormals,
    infinities; a NaN stays one."""
    gen = torch.Generator().manual_seed(3)
    x = torch.randint(-2 ** 31, 2 ** 31 - 1, (4, 1, 128, 128), generator=gen).to(torch.int32)
    edge = [0x7f800000, 0x7f7fffff, 0x7f7f8000, 1, 0x7fffff, 0x8000, 0x18000, 0x3f808000, 0x3f818000, 0x7f800001,
            0x7fc00000, 0x7fffffff]
    x.view(-1)[:len(edge)] = torch.tensor(edge, dtype=torch.int64).to(torch.int32)
    f = x.view(torch.float32).to(DEV)
    e = torch.zeros(4, 0, 1, 128, device=DEV, dtype=torch.bfloat16)
    with torch.no_grad():
        _, s = kda_pkg.kda_recurrent(e, e, e, e.float(), torch.zeros(4, 0, 1, device=DEV), state=f,
                                     state_dtype=torch.bfloat16)
    nan = torch.isnan(f)
    assert torch.isnan(s[nan]).all()
    assert torch.equal(s[~nan].view(torch.int16), f[~nan].to(torch.bfloat16).view(torch.int16))
