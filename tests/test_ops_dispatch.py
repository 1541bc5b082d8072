"""Which calls skip the dispatcher: ordinary eager ones on ordinary tensors,
and no call that a mode, transform, trace, subclass or autograd could
interpose on.  On the GPU, a direct call and the op give the same bits and
advance the same version counters."""
import pytest
import torch

from vllm_neuron_amd import ops
from vllm_neuron_amd import workloads as W


def _contexts():
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.autograd import forward_ad
    from torch.overrides import TorchFunctionMode

    class Sub(torch.Tensor):
        pass

    x = torch.zeros(4)
    seen = {}

    def note(name, *a):
        seen[name] = ops._plain(*a)
        return a[0] * 1

    with FakeTensorMode():
        seen["fake mode"] = ops._plain(x)
    with TorchFunctionMode():
        seen["function mode"] = ops._plain(x)
    with forward_ad.dual_level():
        note("forward AD", x)
    with torch.profiler.profile():
        note("profiler", x)
    torch.func.vmap(lambda t: note("vmap", t))(torch.zeros(2, 4))
    torch.func.grad(lambda t: note("func.grad", t).sum())(x)
    torch.func.functionalize(lambda t: note("functionalize", t))(x)
    torch.jit.trace(lambda t: note("jit trace", t), x, check_trace=False)
    torch.fx.experimental.proxy_tensor.make_fx(lambda t: note("make_fx", t))(x)
    note("requires grad", x.clone().requires_grad_())
    note("subclass", x.as_subclass(Sub))
    note("neg view", torch._neg_view(x))
    with torch.inference_mode():
        y = torch.zeros(4)
    note("inference tensor", y)
    return seen


def test_interposed_calls_take_the_op():
    import torch.fx.experimental.proxy_tensor  # noqa: F401

    assert {k: v for k, v in _contexts().items() if v} == {}


def test_plain_calls_go_direct():
    x = torch.zeros(4)
    assert ops._plain(x, None, torch.nn.Parameter(x, requires_grad=False))
    with torch.no_grad():
        assert ops._plain(x.clone().requires_grad_())
    with torch.inference_mode():
        assert ops._plain(x, torch.zeros(4))


def _project(x, w):
    """The decode block's choice between the few-row kernel and the library."""
    return ops.skinny_linear(x, w) if ops.skinny_linear_ok(x, w) else x @ w


def test_few_row_projection_keeps_the_library_products_transforms(monkeypatch):
    """Tangents, batching, gradients, subclasses and autocast are those of
    ``x @ w``; ordinary calls take the kernel (stubbed here by the product)."""
    calls = []

    def launch(x, w, *a):
        calls.append(type(w))
        return torch.mm(x.detach(), w.detach())

    monkeypatch.setattr(ops.K, "skinny_linear", launch)
    g = torch.Generator().manual_seed(0)
    x, w, t = (torch.randn(s, generator=g).to(torch.bfloat16) for s in ((4, 64), (64, 32), (64, 32)))

    assert torch.equal(_project(x, w), x @ w) and len(calls) == 1
    out, tangent = torch.func.jvp(lambda a: _project(x, a), (w,), (t,))
    assert torch.equal(out, x @ w) and torch.equal(tangent, x @ t)
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(w, t)
        assert torch.equal(torch.autograd.forward_ad.unpack_dual(_project(x, dual)).tangent, x @ t)
    ws = torch.stack((w, t))
    assert torch.equal(torch.func.vmap(lambda a: _project(x, a))(ws), torch.matmul(x, ws))
    assert _project(x, w.clone().requires_grad_()).requires_grad

    class Sub(torch.Tensor):
        seen = []

        @classmethod
        def __torch_function__(cls, func, types, args=(), kwargs=None):
            cls.seen.append(func.__name__)
            return super().__torch_function__(func, types, args, kwargs or {})

    _project(x, w.as_subclass(Sub))
    assert any("matmul" in n for n in Sub.seen)
    assert len(calls) == 1  # none of these took the kernel
    with torch.autocast("cpu", dtype=torch.float16):
        assert not ops.skinny_linear_ok(x, w)
    with torch.autocast("cpu", dtype=torch.bfloat16):
        assert ops.skinny_linear_ok(x, w)
    compiled = torch.compile(lambda a: ops.skinny_linear_ok(x, a), backend="eager", fullgraph=True)
    assert compiled(w)


@pytest.mark.parametrize("k, n, few", [
    (256, 32, True), (2880, 32, True), (2880, 8192, True), (2048, 8224, False), (2048, 48, False),
    (2912, 3040, False), (2912, 3072, True), (4096, 3072, True), (4096, 2880, False),
    (4096, 6144, True), (4096, 8192, False), (4128, 3072, False), (8192, 1024, False),
    (8192, 4096, True), (8192, 4064, False), (16384, 32, False), (16384, 6144, True),
    (16384, 6176, False),
])
def test_few_row_projection_sizes(k, n, few):
    """The kernel where it measured faster: few rows of K, or columns enough
    for every CU and fewer than the library streams as fast."""
    w = torch.empty(k, n, dtype=torch.bfloat16, device="meta")
    for T in (1, 16):
        x = torch.empty(T, k, dtype=torch.bfloat16, device="meta")
        assert ops.K.skinny_linear_ok(x, w) == few
    assert not ops.K.skinny_linear_ok(torch.empty(17, k, dtype=torch.bfloat16, device="meta"), w)


@pytest.mark.gpu
@pytest.mark.parametrize("inference", [False, True])
def test_direct_calls_equal_the_ops(gpu, monkeypatch, inference):
    cfg = W.DecodeConfig("t", 3, 8, 2, 128, 32, 50, 500, sink=True, seed=3)
    pcfg = W.PrefillConfig("t", 1, 8, 2, 128, 32, 70, 96, 96, seed=4)
    got = []
    for direct in (True, False):
        monkeypatch.setattr(ops, "_plain", ops._plain if direct else lambda *t: False)
        b, p = W.make_decode_batch(cfg, gpu), W.make_prefill_batch(pcfg, gpu)
        qkv = torch.randn(5, 12 * 128, generator=torch.Generator().manual_seed(1)).to(
            torch.bfloat16).to(gpu)
        with torch.inference_mode(inference):
            out = torch.empty_like(b.q)
            o = ops.paged_decode(b.q, b.k_new, b.v_new, b.k_cache, b.v_cache, b.block_table,
                                 softmax_scale=0.1, pos_ids=b.pos, sink=b.sink, out=out,
                                 write_slots=b.slots)
            o2 = ops.paged_prefill(p.q, p.cu_seqlens, p.prior, 70, p.k_cache, p.v_cache,
                                   p.block_table, scale=0.1)
            ops.kv_write(p.k_new, p.v_new, p.slots, p.k_cache, p.v_cache)
            q, _, _ = ops.qkv_epilogue(qkv, 8, 2, 128)
            n = ops.row_norm(qkv, ops.NORM_RMS, 1e-5)
        tensors = [o, o2, q, n, b.k_cache, b.v_cache, p.k_cache, p.v_cache]
        versions = [] if inference else [t._version for t in (out, b.k_cache, b.v_cache, p.k_cache,
                                                              b.q, qkv, n)]
        versions += [t._version for t in (b.k_cache, p.v_cache, b.block_table)]
        got.append((tensors, versions))
    for x, y in zip(got[0][0], got[1][0]):
        assert torch.equal(x.view(torch.int16), y.view(torch.int16))
    assert got[0][1] == got[1][1]
