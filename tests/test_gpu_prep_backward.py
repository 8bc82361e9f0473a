"""The pre-processing's backward at the edges of its units (tokens per tile,
channels per wave, conv sizes), and its gradients as slices of one tensor."""

from __future__ import annotations

import importlib

import pytest
import torch

from test_gpu_layer_train import DEV, TOL_K, _prep_inputs, _prep_ref, rel


@pytest.fixture(scope="module")
def ops(kda_pkg):
    return importlib.import_module("kimi_linear_amd.layer_ops")


def run(ops, inp, up, dtype, H, K, V, row=None):
    dev = lambda t: t.to(DEV) if t is not None else None  # noqa: E731
    return ops.kda_prep_backward(
        *(dev(x) for x in inp["x"]), [dev(w.to(dtype)) for w in inp["w"]],
        [dev(b.to(dtype)) if b is not None else None for b in inp["b"]], dev(inp["gk"]), dev(inp["a_log"]),
        dev(inp["dt_bias"]), dev(inp["logit"]), *(dev(up[n]) for n in ("dq", "dk", "dv", "dg", "dbeta")),
        num_heads=H, head_dim=K, value_head_dim=V, l2_eps=1e-6, row=row)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,T,H,K,V,cs", [(1, 1, 1, 64, 64, 4), (2, 3, 3, 64, 128, 4), (1, 61, 5, 128, 64, 1),
                                          (2, 65, 9, 64, 64, 3), (1, 33, 5, 128, 128, 4), (3, 132, 2, 128, 64, 4),
                                          (2, 67, 1, 64, 64, 2), (1, 128, 1, 64, 64, 4)])
def test_unit_edges(ops, dtype, B, T, H, K, V, cs):
    """Tiles with 1 to 4 rows left and one row into the next, channel runs that end
    inside a wave.  Bounds as for the same kernels elsewhere."""
    inp, up = _prep_inputs(B, T, H, K, V, cs, dtype, seed=T + cs)
    got = run(ops, inp, up, dtype, H, K, V)
    ref_in = dict(inp, w=[w.to(dtype) for w in inp["w"]], b=[b.to(dtype) for b in inp["b"]])
    outs, leaves = _prep_ref(ref_in, H, K, V, 1e-6)
    ups = [up[n].to(dtype if i < 3 else torch.float32).double() for i, n in enumerate(("dq", "dk", "dv", "dg", "dbeta"))]
    torch.autograd.backward(outs, ups)
    ref = ([x.grad for x in leaves["x"]], [w.grad for w in leaves["w"]], [b.grad for b in leaves["b"]],
           leaves["gk"].grad, leaves["logit"].grad, leaves["a_log"].grad, leaves["dt_bias"].grad)
    pairs = [*zip(got[:3], ref[0]), *zip(got[3], ref[1]), *zip(got[4], ref[2]), *zip(got[5:], ref[3:])]
    for i, (a, b) in enumerate(pairs):
        assert a.shape == b.shape and rel(a, b) <= TOL_K[dtype], i
    # the same as slices of one tensor's rows
    width = H * (2 * K + V) + H
    row = run(ops, inp, up, dtype, H, K, V, row=width + 19 * (K // 64) * (V // 64) + width % 2)
    for a, b in zip([*got[:3], *got[3], *got[4], *got[5:]], [*row[:3], *row[3], *row[4], *row[5:]]):
        assert torch.equal(a, b)
    assert row[0]._base is row[6]._base and row[0]._base.shape[-1] >= width


class Halves(torch.autograd.Function):
    """a and b as they are; their gradients as slices of one [.., row] tensor."""

    @staticmethod
    def forward(ctx, a, b, row):
        ctx.row = row
        return a.clone(), b.clone()

    @staticmethod
    def backward(ctx, da, db):
        n, m = da.shape[-1], db.shape[-1]
        with torch.no_grad():
            a, b = da.new_full((*da.shape[:-1], ctx.row), float("nan"))[..., :n + m].split((n, m), -1)
            a.copy_(da)
            b.copy_(db)
        return a, b, None


@pytest.mark.parametrize("case", ["joined", "missing", "narrower", "foreign", "create_graph", "twice"])
def test_split_gradient(ops, case):
    """split_joined's gradient is torch.split's, whatever the parts' gradients are made of."""
    gen = torch.Generator().manual_seed(0)
    y = torch.randn(2, 3, 10, generator=gen, requires_grad=True)
    w = torch.randn(2, 3, 10, generator=gen)
    sizes = (3, 4, 2, 1)

    def loss(parts):
        a, b, c, d = parts
        if case != "foreign":
            a, b = Halves.apply(a, b, 9 if case == "narrower" else 10)
        terms = [a * w[..., :3], b * w[..., 3:7], c * w[..., 7:9]] + ([] if case == "missing" else [d * w[..., 9:]])
        return sum((t ** 2).sum() for t in terms)

    graph = case in ("create_graph", "twice")
    out = loss(ops.split_joined(y, sizes))
    ref = torch.autograd.grad(loss(y.split(sizes, -1)), y)[0]
    got = torch.autograd.grad(out, y, create_graph=case == "create_graph", retain_graph=graph)[0]
    assert torch.equal(got, ref)
    if case == "twice":
        again = torch.autograd.grad(out, y)[0]
        assert torch.equal(again, ref) and torch.equal(got, ref)


class Parts(torch.autograd.Function):
    """a and b as they are; their gradients as the caller's own tensors."""

    @staticmethod
    def forward(ctx, a, b, grads):
        ctx.grads = grads
        return a.clone(), b.clone()

    @staticmethod
    def backward(ctx, da, db):
        return (*ctx.grads, None)


def test_split_gradient_leaves_the_callers_tensors(ops):
    """Gradients that are slices of a tensor of the caller's, in the split's very
    layout: it is neither written to nor returned."""
    y = torch.randn(2, 3, 10, requires_grad=True)
    own = torch.randn(2, 3, 10)
    before = own.clone()
    a, b, c, d = ops.split_joined(y, (3, 4, 2, 1))
    a, b = Parts.apply(a, b, own.split((3, 4, 2, 1), -1)[:2])
    got = torch.autograd.grad((a.sum(), b.sum(), (2 * c).sum()), y, [torch.tensor(1.)] * 3)[0]
    assert torch.equal(own, before)
    assert got.data_ptr() != own.data_ptr()
    assert torch.equal(got, torch.cat([before[..., :7], torch.full((2, 3, 2), 2.), torch.zeros(2, 3, 1)], -1))


def test_split_gradient_of_two_splits(ops):
    """The parts of one joined gradient that belong to two splits: each gets its own."""
    y, z = torch.randn(2, 3, 10, requires_grad=True), torch.randn(2, 3, 10, requires_grad=True)
    sizes = (3, 4, 2, 1)
    joined = ops.joined_gradient((2, 3, 10), sizes[:2], torch.float32, y.device)
    want = [torch.randn_like(p) for p in joined]
    for p, w in zip(joined, want):
        p.copy_(w)
    a, b = Parts.apply(ops.split_joined(y, sizes)[0], ops.split_joined(z, sizes)[1], joined)
    gy, gz = torch.autograd.grad((a.sum(), b.sum()), (y, z))
    assert torch.equal(gy, torch.cat([want[0], torch.zeros(2, 3, 7)], -1))
    assert torch.equal(gz, torch.cat([torch.zeros(2, 3, 3), want[1], torch.zeros(2, 3, 3)], -1))


@pytest.mark.parametrize("case", ["joined", "missing", "narrower", "create_graph"])
def test_split_gradient_in_place(ops, case):
    """Parts of a joined gradient stay where they are, beside the others."""
    sizes, row = (3, 4, 2, 1), 9 if case == "narrower" else 10
    y = torch.randn(2, 3, 10, requires_grad=True)
    joined = ops.joined_gradient((2, 3, row), sizes[:2], torch.float32, y.device)
    for p in joined:
        p.normal_()
    want = [p.clone() for p in joined]
    a, b, c, d = ops.split_joined(y, sizes)
    a, b = Parts.apply(a, b, joined)
    out = a.sum() + b.sum() + (2 * c).sum() + (0 if case == "missing" else (3 * d).sum())
    got = torch.autograd.grad(out, y, create_graph=case == "create_graph")[0]
    want += [torch.full((2, 3, 2), 2.), torch.full((2, 3, 1), 0. if case == "missing" else 3.)]
    assert torch.equal(got, torch.cat(want, -1))
    assert (got.data_ptr() == joined[0].data_ptr()) == (case in ("joined", "missing"))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,H,K,V,cs", [(70, 8, 64, 64, 4), (19, 4, 128, 128, 3), (5, 4, 128, 128, 2), (33, 6, 128, 64, 1)])
def test_bits_do_not_depend_on_the_other_heads(ops, dtype, T, H, K, V, cs):
    """A head's gradients are the same bits in a wide call and alone (eight or four channels a lane)."""
    B = 2
    inp, up = _prep_inputs(B, T, H, K, V, cs, dtype, seed=T)
    want = run(ops, inp, up, dtype, H, K, V)
    dims = (K, K, V)
    for h in range(H):
        ch = [slice(h * D, (h + 1) * D) for D in dims]
        one_in = dict(inp, x=[x[..., c].contiguous() for x, c in zip(inp["x"], ch)], w=[w[c] for w, c in zip(inp["w"], ch)],
                      b=[b[c] for b, c in zip(inp["b"], ch)], gk=inp["gk"][..., ch[0]].contiguous(),
                      logit=inp["logit"][..., h:h + 1].contiguous(), a_log=inp["a_log"][h:h + 1],
                      dt_bias=inp["dt_bias"][h:h + 1])
        one_up = {n: u[:, :, h:h + 1].contiguous() for n, u in up.items()}
        got = run(ops, one_in, one_up, dtype, 1, K, V)
        for i in range(3):
            assert torch.equal(want[i][..., ch[i]], got[i]), i
            assert torch.equal(want[3][i][ch[i]], got[3][i]) and torch.equal(want[4][i][ch[i]], got[4][i]), i
        assert torch.equal(want[5][..., ch[0]], got[5]) and torch.equal(want[6][..., h:h + 1], got[6])
        assert torch.equal(want[7][h:h + 1], got[7]) and torch.equal(want[8][h:h + 1], got[8])
