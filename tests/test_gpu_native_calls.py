"""The native call path against the registered ops: the same outputs and
gradients for every form of call it takes, and the ops' own behaviour (results
and errors) for every form it leaves alone."""

import pytest
import torch
from torch.utils.checkpoint import checkpoint

import kotodama_amd
from kotodama_amd import ops
from kotodama_amd._native import native

from ._tiny_model import TinyModel

pytestmark = pytest.mark.gpu
BF, F32 = torch.bfloat16, torch.float32
OP = torch.ops.attnres_hip


class Norm:
    def __init__(self, weight):
        self.weight = weight
        self.eps = 1e-5


def _tensors(gpu, dtype=BF, pdt=None, s=3, batch=(2, 9), d=264, q=0, seed=0):
    g = torch.Generator(device=gpu).manual_seed(seed)
    buf = torch.randn((s, *batch, d), generator=g, device=gpu).to(dtype)
    query = (torch.randn((q, d) if q else (d,), generator=g, device=gpu) * 0.1).to(pdt or dtype)
    gain = (1 + 0.1 * torch.randn(d, generator=g, device=gpu)).to(pdt or dtype)
    return buf, query, gain


def _same(a, b):
    for x, y in zip(a, b):
        if x is None or y is None:
            assert x is None or x.numel() == 0
            assert y is None or y.numel() == 0
        else:
            assert x.shape == y.shape and x.dtype == y.dtype and torch.equal(x, y)


FORMS = [dict(), dict(dtype=F32), dict(pdt=F32), dict(batch=(7,)), dict(batch=()), dict(q=1), dict(q=5),
         dict(dtype=F32, q=3), dict(s=1), dict(s=16)]


@pytest.mark.parametrize("form", FORMS, ids=[",".join(f"{k}={v}" for k, v in f.items()) or "plain" for f in FORMS])
@pytest.mark.parametrize("with_gain", [True, False])
def test_forward_forms_equal_the_ops(gpu, form, with_gain):
    buf, query, gain = _tensors(gpu, **form)
    gain = gain if with_gain else None
    n, dt = buf.shape[0], buf.dtype
    for weights in (False, True):
        for aux in (False, True):
            want = OP.route(buf, n, query, gain, 1e-5, dt, weights, aux)
            got = native.route(buf, n, query, gain, 1e-5, dt, weights, weights, aux, ops._TUPLE, None)
            assert got is not None
            _same(got, want)
            _same(native.route_list(list(buf), query, gain, 1e-5, dt, weights, weights, aux, ops._TUPLE, False), want)
            _same(ops.route(buf, n, query, gain, 1e-5, dt, weights, aux), want)
    if buf.dim() > 2 and query.dim() == 1:
        arena, ref = buf.clone(), buf.clone()
        delta = torch.randn_like(buf[0])
        for commit in (False, True):
            if n + int(commit) > 16 or (commit and n < 2):
                continue
            nc = n - 1 - int(commit)
            got = native.block_step(arena, nc, commit, delta, query, gain, 1e-5, True)
            _same(got, OP.block_step(ref, nc, commit, delta, query, gain, 1e-5, True))
            assert torch.equal(arena, ref)


@pytest.mark.parametrize("form", FORMS, ids=[",".join(f"{k}={v}" for k, v in f.items()) or "plain" for f in FORMS])
@pytest.mark.parametrize("stacked", [True, False], ids=["stacked", "list"])
@pytest.mark.parametrize("used", ["rows", "lse", "both", "rows of both"])
def test_gradients_equal_the_ops(gpu, form, stacked, used):
    want_lse = used != "rows"
    weights = [False, True] if stacked and want_lse else [False]  # a recorded list call with weights is the op's
    res = []
    for direct in [*weights, None]:  # native, and last the op
        buf, query, gain = _tensors(gpu, **form)
        leaves = [t.requires_grad_() for t in ([buf] if stacked else [b.clone() for b in buf])]
        query.requires_grad_(), gain.requires_grad_()
        # one inactive slot where the buffer has more than one
        n = max(1, buf.shape[0] - 1)
        args = (leaves[0], n) if stacked else (leaves[:n],)
        if direct is None:
            call = OP.route if stacked else OP.route_list
            out, _, lse, _, _ = call(*args, query, gain, 1e-5, buf.dtype, want_lse, False)
        else:
            call = native.route if stacked else native.route_list
            got = call(*args, query, gain, 1e-5, buf.dtype, direct, want_lse, False, ops._TUPLE, True)
            assert got is not None, "the native path left the call alone"
            out, w, lse, _, _ = got
            assert ("RouteStacked" if stacked else "RouteList") in out.grad_fn.name()
            assert w is None or not w.requires_grad
        g = torch.Generator(device=gpu).manual_seed(5)
        loss = 0
        if used != "lse":
            loss = (out.float() * torch.randn(out.shape, generator=g, device=gpu)).sum()
        if used in ("lse", "both"):
            loss = loss + lse.sum()
        res.append(torch.autograd.grad(loss, [*leaves[:n], query, gain]))
    for got in res[:-1]:
        _same(got, res[-1])


@pytest.mark.parametrize("dtypes", [(BF, BF, BF), (F32, F32, F32), (BF, F32, BF), (F32, BF, F32)])
def test_merge_equals_the_op(gpu, dtypes):
    res = []
    for direct in (True, False):
        g = torch.Generator(device=gpu).manual_seed(3)
        p, q, inter = (torch.randn(s, generator=g, device=gpu).to(dt).requires_grad_()
                       for s, dt in zip(((2, 7, 264), (264,), (2, 7, 264)), dtypes))
        lse = torch.randn((2, 7), generator=g, device=gpu).requires_grad_()
        out = ops.merge_call(p, q, inter, lse, 1e-5) if direct else OP.merge(p, q, inter, lse, 1e-5)[0]
        go = torch.randn(out.shape, generator=g, device=gpu).to(out.dtype)
        res.append([out.detach(), *torch.autograd.grad(out, [p, q, inter, lse], go)])
    _same(*res)


def test_calls_left_to_the_ops(gpu):
    buf, query, gain = _tensors(gpu, d=512)

    def taken(b, q=query, g=gain, n=2):
        return native.route(b, n, q, g, 1e-5, None, False, False, False, ops._ROWS, None) is not None

    class Sub(torch.Tensor):
        pass

    assert taken(buf)
    assert not taken(buf, n=4) and not taken(buf, n=-1)  # outside the buffer
    assert not taken(buf.transpose(1, 2)) and not taken(buf[..., ::2], query[::2].contiguous(), gain[::2].contiguous())
    assert not taken(buf, query[:256].repeat_interleave(2)[::1].expand(512).as_strided((512,), (0,)))
    assert not taken(buf.half(), query.half(), gain.half()) and not taken(buf, query, gain.float())
    assert not taken(buf.cpu()) and not taken(buf, query.cpu()) and not taken(buf.as_subclass(Sub))
    assert not taken(buf.to_sparse()) and not taken(buf, query[:256])
    assert not taken(buf.requires_grad_())  # recorded, and the caller did not ask for that
    with torch.no_grad():
        assert taken(buf)
    # a flag that is true but not True is not read as False
    with torch.no_grad():
        assert native.route(buf, 2, query, gain, 1e-5, BF, 1, 1, False, ops._TUPLE, None) is None
        assert ops.route_call(buf, 2, query, gain, 1e-5, BF, want_weights=1)[1].shape == (1, 2, 2, 9)
        assert ops.block_step_call(buf.clone(), 1, 0, None, query, gain, 1e-5, 1)[1].shape == (2, 2, 9)
    # ... and the drop-in's result for them is the op's
    with torch.no_grad():
        strided = buf.transpose(1, 2)
        want = OP.route(strided.contiguous(), 2, query, gain, 1e-5, BF, False, False)[0][0]
        assert torch.equal(kotodama_amd.route_static(strided, query, Norm(gain), None, 2), want)
        with pytest.raises(ValueError, match="outside"):
            kotodama_amd.route_static(buf, query, Norm(gain), None, 4)
        with pytest.raises(TypeError, match="float32 and bfloat16"):
            kotodama_amd.route_static(buf.half(), query.half(), Norm(gain.half()), None, 2)
        with pytest.raises(RuntimeError, match="num_sources"):
            ops.route(torch.zeros(17, 2, 512, device=gpu), 17, query.float(), None, 1e-5, F32, False, False)


def test_recorded_calls_keep_autograds_contract(gpu):
    buf, query, gain = _tensors(gpu, d=512)
    buf.requires_grad_()
    norm = Norm(gain)
    plain = torch.autograd.grad(kotodama_amd.route_static(buf, query, norm, None, 3).float().square().sum(), buf)[0]
    # saved tensors go through the hooks (checkpointing recomputes them)
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append(t.shape) or t, lambda t: t):
        out = kotodama_amd.route_static(buf, query, norm, None, 3)
    assert buf.shape in seen
    again = checkpoint(lambda b: kotodama_amd.route_static(b, query, norm, None, 3), buf, use_reentrant=False)
    for o in (out, again):
        assert torch.equal(torch.autograd.grad(o.float().square().sum(), buf)[0], plain)
    # a saved tensor changed in place is reported
    work = buf.detach().clone().requires_grad_()
    out = kotodama_amd.route_static(work, query, norm, None, 3)
    with torch.no_grad():
        work.add_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.float().sum().backward()
    # the gradient has no derivative of its own, and says so
    out = kotodama_amd.route_static(buf, query, norm, None, 3)
    (first,) = torch.autograd.grad(out.float().square().sum(), buf, create_graph=True)
    assert torch.equal(first.detach(), plain)
    with pytest.raises(RuntimeError):
        torch.autograd.grad(first.float().sum(), buf)
    # no forward-mode rule
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(buf.detach().clone().requires_grad_(), torch.ones_like(buf))
        with pytest.raises((RuntimeError, NotImplementedError)):
            kotodama_amd.route_static(dual, query, norm, None, 3)


def test_calls_on_a_side_stream(gpu):
    buf, query, gain = _tensors(gpu, d=512, batch=(64, 33))
    want = kotodama_amd.route_static(buf, query, Norm(gain), None, 3)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        got = kotodama_amd.route_static(buf, query, Norm(gain), None, 3) + 0
    side.synchronize()
    assert torch.equal(got, want)


def _merge_args(gpu):
    g = torch.Generator(device=gpu).manual_seed(1)
    return [torch.randn(s, generator=g, device=gpu).to(t).requires_grad_()
            for s, t in (((2, 9, 264), BF), ((264,), BF), ((2, 9, 264), BF), ((2, 9), F32))]


# name -> (tensors, the differentiable output of one recorded call on them)
RECORDED = {
    "rows": lambda b, q, g: kotodama_amd.route_static(b, q, Norm(g), None, 2),
    "all-slots": lambda b, q, g: kotodama_amd.route_static(b, q, Norm(g), None, 3),
    "weights": lambda b, q, g: ops.route(b, 2, q, g, 1e-5, BF, True, False)[0],
    "aux": lambda b, q, g: ops.route(b, 2, q, g, 1e-5, BF, False, True)[0],
    "no-gain": lambda b, q, g: ops.route(b, 2, q, None, 1e-5, BF, False, False)[0] * g,
    "lse": lambda b, q, g: ops.route_call(b, 2, q, g, 1e-5, BF, want_lse=True)[2],
    "list": lambda b, q, g: kotodama_amd.block_attn_res_from_list(list(b.unbind(0)), q, Norm(g)),
    "list-lse": lambda b, q, g: ops.route_list_call(list(b.unbind(0)), q, g, 1e-5, BF, want_lse=True)[2],
}


@pytest.mark.parametrize("name", [*RECORDED, "merge"])
def test_backward_under_compiled_autograd(gpu, name):
    # the whole backward is traced (no graph break), once per set of inputs that need gradients
    def compiler(graph):
        return torch.compile(graph, backend="aot_eager", fullgraph=True)

    torch._dynamo.reset()
    for needed in ((0, 1, 2), (0,), (1, 2)):
        leaves = _merge_args(gpu) if name == "merge" else list(_tensors(gpu))
        leaves = [t.requires_grad_(i in needed) for i, t in enumerate(leaves)]
        wanted = [t for t in leaves if t.requires_grad]

        def loss():
            out = ops.merge_call(*leaves, 1e-5) if name == "merge" else RECORDED[name](*leaves)
            return out.float().square().sum()

        want = torch.autograd.grad(loss(), wanted)
        for _ in range(2):
            for t in wanted:
                t.grad = None
            total = loss()
            with torch._dynamo.compiled_autograd._enable(compiler):
                total.backward()
            _same([t.grad for t in wanted], want)


def test_recorded_calls_appear_in_a_profile(gpu):
    buf, query, gain = (t.requires_grad_() for t in _tensors(gpu))
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        RECORDED["rows"](buf, query, gain).float().sum().backward()
        RECORDED["list"](buf, query, gain).float().sum().backward()
        ops.merge_call(*_merge_args(gpu), 1e-5).float().sum().backward()
        with torch.no_grad():
            ops.route(buf, 3, query, gain, 1e-5, BF, True, False)
    seen = {e.key: e.count for e in prof.key_averages() if e.key.startswith("attnres_hip::")}
    names = {f"attnres_hip::{n}{d}": 1 for n in ("route", "route_list", "merge") for d in ("", "_bwd")}
    assert seen == {**names, "attnres_hip::route": 2}


class _Recorder:
    """The native functions, counting the calls taken; with ``off`` none is."""

    def __init__(self, off):
        self.off, self.taken = off, {}

    def __getattr__(self, name):
        def call(*args):
            res = None if self.off else getattr(native, name)(*args)
            if res is not None:
                self.taken[name] = self.taken.get(name, 0) + 1
            return res

        return call


# (hidden, dtype, the training points' native functions that the loop must reach)
LOOPS = [(512, BF, {"step", "bwd_rows", "bwd_defer", "gather_seg"}), (1024, BF, {"step", "bwd_defer", "gather_seg"}),
         (264, BF, {"step", "bwd_rows"}), (512, F32, {"step", "bwd_rows"})]


@pytest.mark.parametrize("d,dtype,reached", LOOPS, ids=[f"d{c[0]}-{str(c[1])[6:]}" for c in LOOPS])
def test_training_loop_equals_the_python_launches(gpu, monkeypatch, d, dtype, reached):
    model = TinyModel(d=d, num_layers=6, boundaries=(0, 2, 4), elementwise=True).to(gpu).to(dtype)
    g = torch.Generator(device=gpu).manual_seed(d)
    embed = torch.randn((2, 33, d), generator=g, device=gpu).to(dtype).requires_grad_()
    grad = torch.randn((2, 33, d), generator=g, device=gpu).to(dtype)
    params = [p for p in model.parameters() if p.requires_grad]
    res = []
    for off in (False, True):
        rec = _Recorder(off)
        monkeypatch.setattr(ops, "native", rec)
        out = kotodama_amd.forward_attn_res(model, embed)
        res.append([out.detach(), *torch.autograd.grad(out, [embed, *params], grad, allow_unused=True)])
        assert off or reached <= set(rec.taken), rec.taken
        assert not off or not rec.taken
    _same(*res)


def test_calls_the_ops_refuse_stay_refused(gpu):
    buf, query, gain = _tensors(gpu)
    rows, blocks = lambda g: kotodama_amd.route_static(buf, query, Norm(g), None, 3), list(buf)
    for leaves in (False, True):
        query.requires_grad_(leaves)
        # no output dtype: only the drop-ins promote one
        with pytest.raises(RuntimeError, match="out_dtype"):
            ops.route(buf, 3, query, gain, 1e-5, None, False, False)
        with pytest.raises(RuntimeError, match="out_dtype"):
            ops.route_list(blocks, query, gain, 1e-5, None, False, False)
        for call, src in ((lambda *a: ops.route_call(a[0], 3, *a[1:]), buf), (ops.route_list_call, blocks)):
            with pytest.raises((TypeError, RuntimeError)):
                call(src, query, gain, 1e-5, None)
        # the drop-ins need a gain and a sequence
        with pytest.raises(AttributeError, match="dtype"):
            rows(None)
        with pytest.raises(AttributeError, match="dtype"):
            kotodama_amd.block_attn_res_from_list(blocks, query, Norm(None))
        with pytest.raises(TypeError, match="subscriptable"):
            kotodama_amd.block_attn_res_from_list((b for b in buf), query, Norm(gain))
    want = rows(gain)
    for seq in (tuple(blocks), type("Blocks", (list,), {})(blocks)):
        assert torch.equal(kotodama_amd.block_attn_res_from_list(seq, query, Norm(gain)), want)
