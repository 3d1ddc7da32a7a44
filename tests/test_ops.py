"""The ``torch.library`` registration of the operators (``torch.ops.sfl``).

CPU: the schemas (which arguments the ops write) and shape-only dispatch on
meta and fake tensors, which is what tracing (``torch.compile``, export) runs.
GPU: the ops called directly, and through a ``torch.compile`` graph, match the
CPU oracle.
"""

import pytest
import torch

import systems_for_llms_amd.attention  # noqa: F401  (registers the ops)
import systems_for_llms_amd.decode  # noqa: F401


def test_schemas_declare_the_written_arguments():
    decode = str(torch.ops.sfl.decode_attention.default._schema)
    masked = str(torch.ops.sfl.masked_attention.default._schema)
    for name in ("partial_max", "partial_sum", "partial_output", "out"):
        assert f"!) {name}" in decode
    assert "Tensor q," in decode and "Tensor k," in decode and "Tensor lengths" in decode
    assert "!) out" in masked and "!)? lse" in masked
    assert "Tensor? row_ptr" in masked and "Tensor? document_ids" in masked


def _decode_args(device):
    q = torch.empty(2, 8, 64, device=device, dtype=torch.bfloat16)
    k = torch.empty(2, 2, 128, 64, device=device, dtype=torch.bfloat16)
    lengths = torch.empty(2, device=device, dtype=torch.int32)
    pm = torch.empty(2, 8, 3, device=device)
    po = torch.empty(2, 8, 3, 64, device=device)
    return q, k, k, lengths, pm, pm.clone(), po, torch.empty_like(q), 3, 0.125


def test_meta_and_fake_dispatch_launch_nothing():
    torch.ops.sfl.decode_attention(*_decode_args("meta"))
    q = torch.empty(1, 2, 128, 64, device="meta", dtype=torch.bfloat16)
    torch.ops.sfl.masked_attention(q, q, q, torch.empty_like(q), None, 0.125, True, -1, -1, 0, None, None,
                                   None, None, True)
    from torch._subclasses.fake_tensor import FakeTensorMode

    with FakeTensorMode():
        torch.ops.sfl.decode_attention(*_decode_args("cpu"))


def _prepared(*tensors):
    from systems_for_llms_amd.decode import PreparedDecode

    return PreparedDecode(*tensors, 3, 0.125, "token")


def _masked(q):
    from systems_for_llms_amd.attention import _launch_masked

    out = torch.empty_like(q)
    _launch_masked(q, q, q, out, None, 0.125, True, -1, -1, 0, None, None, None, None, True)
    return out


def _seen_by_mode(call):
    from torch.utils._python_dispatch import TorchDispatchMode

    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    seen = []
    with Watch():
        call()
    return seen


def _seen_by_function_mode(call):
    class Watch(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    seen = []
    with Watch():
        call()
    return seen


def _seen_by_profiler(call):
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as profile:
        call()
    return [event.key.replace("::", ".") for event in profile.key_averages()]


def _seen_by_observer(call):
    import json
    import tempfile
    from pathlib import Path

    with tempfile.TemporaryDirectory() as folder:
        path = Path(folder) / "trace.json"
        observer = torch.profiler.ExecutionTraceObserver()
        observer.register_callback(str(path))
        observer.start()
        call()
        observer.stop()
        observer.unregister_callback()
        return [node["name"].replace("::", ".") for node in json.loads(path.read_text())["nodes"]]


def _seen_by_make_fx(call):
    from torch.fx.experimental.proxy_tensor import make_fx

    return [make_fx(lambda x: (call(), x)[1])(torch.zeros(1)).code]


@pytest.mark.parametrize("watch", [_seen_by_mode, _seen_by_function_mode, _seen_by_profiler, _seen_by_observer,
                                   _seen_by_make_fx])
def test_operator_apis_launch_in_sight_of_whatever_watches(watch):
    prepared = _prepared(*_decode_args("meta")[:8])
    q = torch.empty(1, 2, 128, 64, device="meta", dtype=torch.bfloat16)
    assert any("sfl.decode_attention" in name for name in watch(prepared))
    assert any("sfl.masked_attention" in name for name in watch(lambda: _masked(q)))


def test_operator_apis_are_traced_by_jit():
    args = _decode_args("meta")[:8]
    graph = torch.jit.trace(lambda *tensors: _prepared(*tensors)(), args, check_trace=False).graph
    assert "sfl::decode_attention" in str(graph)
    q = torch.empty(1, 2, 128, 64, device="meta", dtype=torch.bfloat16)
    assert "sfl::masked_attention" in str(torch.jit.trace(_masked, (q,), check_trace=False).graph)


def test_operator_apis_count_versions_and_leave_transforms_to_the_op(monkeypatch):
    from systems_for_llms_amd import ops

    tensors = _decode_args("meta")[:8]
    args = tuple(t.clone() for t in tensors)
    for guard in (ops._below_autograd, None):
        monkeypatch.setattr(ops, "_below_autograd", guard)  # None: as in a torch without it
        before = [t._version for t in args]
        _prepared(*args)()
        assert [t._version for t in args] == [v + (i >= 4) for i, v in enumerate(before)]
        with torch.inference_mode():
            _prepared(*[t.clone() for t in tensors])()  # inference tensors have no counter
        with pytest.raises(RuntimeError, match="Batching rule not implemented"):
            torch.func.vmap(lambda q: (_prepared(q, *args[1:])(), q)[1])(torch.stack([args[0]] * 2))
        with pytest.raises(RuntimeError, match="functorch transforms"):
            torch.func.grad(lambda q: (_prepared(q, *args[1:])(), q.sum())[1])(torch.zeros_like(args[0]))
        torch.func.vmap(lambda row: (_prepared(*args)(), row)[1])(torch.zeros(2))


def test_mark_written_bumps_versions_like_the_op():
    from systems_for_llms_amd.ops import mark_written

    x, y = torch.zeros(2), torch.zeros(2)
    mark_written(x, None, y)
    assert x._version == 1 and y._version == 1
    with torch.inference_mode():
        mark_written(torch.zeros(2))  # inference tensors have no counter


@pytest.mark.gpu
def test_prepared_decode_bumps_the_output_version():
    from systems_for_llms_amd.decode import prepare

    q, k = torch.randn(1, 4, 64, device="cuda"), torch.randn(1, 4, 32, 64, device="cuda")
    op = prepare(q, k, k.clone())
    weight = torch.ones_like(q, requires_grad=True)
    product = op() * weight  # saves the output for the backward
    op()
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        product.sum().backward()


@pytest.mark.gpu
def test_lazily_negated_tensors_are_resolved():
    from systems_for_llms_amd.attention import attention, causal_prefill
    from systems_for_llms_amd.decode import decode
    from systems_for_llms_amd.masks import MaskSpec, compile_mask

    g = torch.Generator(device="cuda").manual_seed(1)
    k, v = (torch.randn((2, 2, 70, 64), device="cuda", generator=g).bfloat16() for _ in range(2))
    q = torch.randn((2, 4, 64), device="cuda", generator=g).bfloat16()
    assert torch.equal(decode(q, k, torch._neg_view(v)), decode(q, k, -v))
    spec = MaskSpec(causal=True)
    schedule = compile_mask(70, spec)
    assert torch.equal(attention(torch._neg_view(k), k, v, schedule, spec), attention(-k, k, v, schedule, spec))
    want, got = (torch.empty_like(k) for _ in range(2))
    assert torch.equal(causal_prefill(k, torch._neg_view(k), v, got), causal_prefill(k, -k, v, want))


@pytest.mark.gpu
def test_decode_op_and_compiled_graph_match_oracle():
    from oracle.attention import decode_reference

    g = torch.Generator().manual_seed(3)
    q = torch.randn(3, 8, 64, generator=g).bfloat16()
    k = torch.randn(3, 2, 100, 64, generator=g).bfloat16()
    v = torch.randn(3, 2, 100, 64, generator=g).bfloat16()
    lengths = torch.tensor([100, 0, 37], dtype=torch.int32)
    expected = decode_reference(q, k, v, lengths)
    qd, kd, vd, ld = q.cuda(), k.cuda(), v.cuda(), lengths.cuda()
    pm = torch.empty(3, 8, 4, device="cuda")
    ps = torch.empty_like(pm)
    po = torch.empty(3, 8, 4, 64, device="cuda")
    out = torch.empty_like(qd)
    torch.ops.sfl.decode_attention(qd, kd, vd, ld, pm, ps, po, out, 4, 0.125)
    torch.testing.assert_close(out.float().cpu(), expected, atol=0.02, rtol=0.02)

    def step(q_, k_, v_, l_):
        o = torch.empty_like(q_)
        torch.ops.sfl.decode_attention(q_, k_, v_, l_, torch.empty(3, 8, 4, device=q_.device),
                                       torch.empty(3, 8, 4, device=q_.device),
                                       torch.empty(3, 8, 4, 64, device=q_.device), o, 4, 0.125)
        return o * 2

    compiled = torch.compile(step, backend="aot_eager", fullgraph=True)
    torch.testing.assert_close(compiled(qd, kd, vd, ld).float().cpu(), 2 * expected, atol=0.04, rtol=0.02)


@pytest.mark.gpu
def test_masked_op_matches_oracle_with_lse():
    from oracle.attention import dense_mask, masked_attention

    g = torch.Generator().manual_seed(5)
    q, k, v = (torch.randn(1, 2, 130, 64, generator=g).bfloat16() for _ in range(3))
    out, lse = masked_attention(q, k, v, dense_mask(130, causal=True, window_left=40))
    out, lse = out.float(), lse.float()
    qd, kd, vd = q.cuda(), k.cuda(), v.cuda()
    o = torch.empty_like(qd)
    lse_d = torch.empty(1, 2, 130, device="cuda")
    torch.ops.sfl.masked_attention(qd, kd, vd, o, lse_d, 0.125, True, 40, -1, 0, None, None, None, None, True)
    torch.testing.assert_close(o.float().cpu(), out, atol=0.02, rtol=0.02)
    # The row sums come from the bf16-rounded probabilities: the masked-attention tests' bf16 tolerance.
    torch.testing.assert_close(lse_d.cpu(), lse, atol=1e-2, rtol=1e-2)
