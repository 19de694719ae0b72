"""The native host path (csrc/host.cpp) against the Python route of the same calls: equal bit for bit where it
serves a call, None -- and the Python route -- where something is not what it recognises (needs an MI355X)."""
import copy
import gc

import pytest
import torch

from tests.gpu_util import DEV, e8_table_f16, say

pytestmark = pytest.mark.gpu


def _bits(g, *shape):
    return torch.randint(-32768, 32768, shape, generator=g, device=DEV, dtype=torch.int16)


def _signs(g, n):
    return (torch.randint(0, 2, (n,), generator=g, device=DEV) * 2 - 1).half()


def _layer(kind, out_f, in_f, bias):
    from glq_amd.quantized_linear import E8RHTLinear
    g = torch.Generator(device=DEV).manual_seed(out_f + in_f)
    if kind.startswith("trellis"):
        lin = E8RHTLinear(in_f, out_f, bias=bias, codebook_type="trellis").to(DEV)
        tiles = (out_f // 16) * (in_f // 16)
        lin.trellis_packed = _bits(g, tiles, 64)
        if kind == "trellis2":
            lin.trellis_packed2, lin.inv_resid_scale2 = _bits(g, tiles, 32), torch.tensor(0.3, device=DEV)
    else:
        lin = E8RHTLinear(in_f, out_f, bias=bias, block_diagonal=kind != "shell_pow2").to(DEV)
        for s in range(int(kind == "shell2") + 1):
            setattr(lin, ("Qidxs", "Qidxs2")[s], _bits(g, lin.m_pad, lin.n_pad // 8))
        if kind == "shell2":
            lin.inv_resid_scale = torch.tensor(1 / 3.0, device=DEV)
        lin.set_codebook(e8_table_f16(), e8_table_f16())
    lin.SU, lin.SV, lin.Wscale = _signs(g, lin.m_pad), _signs(g, lin.n_pad), torch.tensor(0.02, device=DEV)
    if bias:
        lin.bias = torch.randn(out_f, generator=g, device=DEV).half()
    return lin


@pytest.mark.parametrize("kind,out_f,in_f,bias,dtype,shape", [
    ("trellis", 512, 2048, False, torch.bfloat16, (1,)), ("trellis", 96, 192, True, torch.float16, (2, 3)),
    ("trellis2", 160, 128, True, torch.bfloat16, (37,)), ("shell", 960, 960, True, torch.float16, (5,)),
    ("shell2", 2048, 2304, False, torch.bfloat16, (1, 4)), ("shell2", 2048, 2304, False, torch.bfloat16, (65,)),
    ("shell_pow2", 100, 200, True, torch.float16, (3,))])
def test_native_forward_equals_the_python_route(kind, out_f, in_f, bias, dtype, shape):
    say("native forward", kind, out_f, in_f, bias, dtype, shape)
    lin = _layer(kind, out_f, in_f, bias)
    lin.prepare()
    x = torch.randn(*shape, in_f, generator=torch.Generator().manual_seed(3)).to(DEV, dtype)
    assert lin._fast is not None                                 # made by the load-time step
    y = lin(x)
    lin._fast = None
    ref = lin(x)                                                 # the Python route, which makes the native form again
    assert torch.equal(y, ref)
    y = lin._fast(lin.__dict__, x)
    assert y is not None and y.shape == ref.shape and y.dtype == ref.dtype and torch.equal(y, ref)
    assert torch.equal(lin(x), ref)
    # what it leaves to the Python route
    assert lin._fast(lin.__dict__, x.float()) is None and lin._fast(lin.__dict__, x.cpu()) is None
    assert lin._fast(lin.__dict__, x[..., :0]) is None and lin._fast(lin.__dict__, x[:0]) is None
    if x.numel() > in_f:
        assert lin._fast(lin.__dict__, x.transpose(0, -1)) is None
    assert lin(x.float()).dtype == torch.float32
    # buffers are read on every call, copies make their own plan
    if not bias:
        su = lin.SU
        lin.SU = -su
        assert torch.equal(lin(x), -ref)
        lin.SU = su
    twin = copy.deepcopy(lin)
    assert twin._fast is None and torch.equal(twin(x), ref)


def test_native_shell_forward_notices_changed_indices_and_released_streams():
    from glq_amd import ext
    say("native shell forward, changed buffers")
    lin = _layer("shell2", 2048, 2304, False)
    lin.prepare()
    x = torch.randn(2, 2304, generator=torch.Generator().manual_seed(1)).to(DEV, torch.bfloat16)
    lin(x)
    assert lin._fast(lin.__dict__, x) is not None
    ext.e8_release(lin.Qidxs, lin.Qidxs2)                        # the plan does not keep the streams alive
    assert lin._fast(lin.__dict__, x) is None
    lin.prepare()
    y = lin(x)
    lin.Qidxs.add_(1)
    assert lin._fast(lin.__dict__, x) is None
    assert not torch.equal(lin(x), y)


@pytest.mark.parametrize("bpw,B", [(4, 1), (4, 9), (4, 100), (6, 1), (6, 40)])
def test_native_merged_forward_equals_the_python_route(bpw, B):
    from glq_amd import linear_method as LM
    say("native merged", bpw, B)
    lins = [_layer("trellis2" if bpw == 6 else "trellis", m, 192, False) for m in (96, 64, 64)]
    ml = LM.MergedTrellisLinear.from_linears(lins, bpw=bpw).process_weights_after_loading(DEV)
    x = torch.randn(B, 192, generator=torch.Generator().manual_seed(B)).to(DEV, torch.bfloat16)
    assert ml._fast is not None                                  # made by the load-time step
    ml._fast = None
    ref = ml.apply(x)                                            # the Python route, which makes it again
    y = ml._fast(ml.__dict__, x)
    assert y is not None and torch.equal(y, ref)
    bias = torch.randn(224, generator=torch.Generator().manual_seed(0)).to(DEV)
    assert torch.equal(ml.apply(x, bias), ref + bias.to(ref.dtype))
    ml.trellis_packed._shard_data[1] = torch.zeros(0, dtype=torch.int16, device=DEV)    # an unloaded shard
    assert ml._fast(ml.__dict__, x) is None


def test_dispatch_modes_take_the_python_route():
    from torch.utils._python_dispatch import TorchDispatchMode
    say("native forward under a dispatch mode")

    class Count(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))
    lin = _layer("trellis", 64, 64, False)
    x = torch.randn(1, 64, generator=torch.Generator().manual_seed(0)).to(DEV, torch.bfloat16)
    ref = lin(x)
    with Count():
        assert lin._fast(lin.__dict__, x) is None
        assert torch.equal(lin(x), ref)


@pytest.mark.parametrize("kind", ["trellis2", "shell2", "merged"])
def test_buffers_replaced_by_another_thread_during_calls(kind):
    """A thread that keeps replacing a layer's sign vector (and writing over memory of its size) while another one
    calls the layer: every result is the one of a sign vector that the layer has had."""
    import threading

    from glq_amd import linear_method as LM
    say("native forward, buffers replaced by another thread", kind)
    x = torch.randn(3, 2304, generator=torch.Generator().manual_seed(2)).to(DEV, torch.bfloat16)
    if kind == "merged":
        lins = [_layer("trellis", m, 2304, False) for m in (512, 64)]
        layer = LM.MergedTrellisLinear.from_linears(lins).process_weights_after_loading(DEV)
        call, put = (lambda: layer.apply(x)), (lambda su: layer.SU._shard_data.__setitem__(0, su))
        su = layer.SU.get_shard(0)
    else:
        layer = _layer(kind, 512, 2304, True)
        layer.prepare()
        call, put, su = (lambda: layer(x)), (lambda s: setattr(layer, "SU", s)), layer.SU
    two = [su, -su]
    refs = []
    for s in two:
        put(s)
        call()                                                   # the first makes the native form
        assert layer._fast(layer.__dict__, x) is not None
        refs.append(call())
    assert not torch.equal(*refs)
    stop, failed = threading.Event(), []

    def replace():
        try:
            i = 0
            while not stop.is_set():
                put(two[i & 1].clone())                          # the only reference: the one before it is freed
                torch.full_like(su, float("nan"))
                i += 1
        except BaseException as e:                               # noqa: BLE001 - reported by the main thread
            failed.append(e)
    worker = threading.Thread(target=replace)
    worker.start()
    try:
        got = [call() for _ in range(300)]
    finally:
        stop.set()
        worker.join()
    assert not failed, failed
    assert all(torch.equal(y, refs[0]) or torch.equal(y, refs[1]) for y in got)


@pytest.mark.parametrize("kind", ["trellis", "trellis2"])
def test_tracing_and_gradients_see_the_operator(kind):
    """torch.jit.trace records the operator, not its result, and an input that wants a gradient gets an output with the
    autograd node that says that the operator has no derivative, instead of one that silently needs none."""
    from glq_amd import custom_ops
    say("native forward under tracing", kind)
    custom_ops.register()
    lin = _layer(kind, 64, 128, False)
    g = torch.Generator().manual_seed(0)
    x, other = (torch.randn(2, 128, generator=g).to(DEV, torch.bfloat16) for _ in range(2))
    lin(x)
    assert lin._fast(lin.__dict__, x) is not None
    traced = torch.jit.trace(lin, x)
    assert torch.equal(traced(other), lin(other))
    assert any(n.kind().startswith("glq::") for n in traced.graph.nodes())
    w = x.clone().requires_grad_()
    assert lin._fast(lin.__dict__, w) is None
    y = lin(w)
    assert y.requires_grad and y.grad_fn is not None and torch.equal(y, lin(x))
    with torch.no_grad():
        assert lin._fast(lin.__dict__, w) is not None and not lin(w).requires_grad


def test_a_failing_bias_addition_keeps_no_output():
    say("native forward, bias of a wrong length")
    lin = _layer("trellis", 512, 2048, True)
    x = torch.randn(64, 2048, generator=torch.Generator().manual_seed(0)).to(DEV, torch.bfloat16)
    lin(x)
    lin.bias = torch.zeros(511, device=DEV).half()
    gc.collect()                                                 # what earlier tests left in reference cycles
    held = []
    for _ in range(3):
        with pytest.raises(RuntimeError, match="size"):
            lin._fast(lin.__dict__, x)
        held.append(torch.cuda.memory_allocated())
    assert held[0] == held[1] == held[2]


@pytest.mark.parametrize("kind", ["trellis", "shell2", "merged"])
def test_block_tables_on_another_device_are_declined(kind):
    """A plan made while the block tables were elsewhere (here: on the host) does not hand their addresses to the GPU."""
    from glq_amd import ext, linear_method as LM
    say("native forward, block tables on another device", kind)
    x = torch.randn(2, 192, generator=torch.Generator().manual_seed(0)).to(DEV, torch.bfloat16)
    if kind == "merged":
        layer = LM.MergedTrellisLinear.from_linears([_layer("trellis", m, 192, False) for m in (96, 64)])
        layer.process_weights_after_loading(DEV)
        layer._glq_trellis_meta[0]["_bnm"] = layer._glq_trellis_meta[0]["_bnm"].cpu()
        layer._fast = None
        layer._make_native(ext, False)
        assert layer._fast(layer.__dict__, x) is None
        return
    lin = _layer(kind, 96, 192, False)
    lin.prepare()
    ref, sc = lin(x), lin._scalars
    h = ext.host()
    for which in ("_blocks_n_meta_gpu", "_blocks_m_meta_gpu"):
        kept = getattr(lin, which)
        setattr(lin, which, kept.cpu())
        assert lin._native(ext, sc)(lin.__dict__, x) is None
        if kind == "trellis":
            assert h.trellis_linear(x, lin.SV, lin.SU, lin.trellis_packed, None, lin._blocks_n_tensor, lin._blocks_m_tensor,
                                    lin._blocks_n_meta_gpu, lin._blocks_m_meta_gpu, 0.02, 0.0, 192, 96, 192, 96, None) is None
        setattr(lin, which, kept)
    # a layer that goes away and comes back has its native form again after one call
    lin.to("cpu")
    assert lin._fast is None
    lin.to(DEV)
    assert torch.equal(lin(x), ref)
    y = lin._fast(lin.__dict__, x)
    assert y is not None and torch.equal(y, ref)
    # a form made for another device (a layer whose buffers were assigned one by one) is replaced, not kept
    lin._fast_device = torch.device("cpu")
    old = lin._fast
    lin(x.float())                                               # the Python route
    assert lin._fast is not old and lin._fast_device == x.device


def test_calls_without_the_native_host_path(monkeypatch):
    """The same results where the host path cannot be loaded: layers, merged layers and codewords through Python."""
    from glq_amd import ext, linear_method as LM
    say("without the native host path")
    x = torch.randn(3, 192, generator=torch.Generator().manual_seed(0)).to(DEV, torch.bfloat16)
    lins = [_layer("trellis", m, 192, True) for m in (96, 64)] + [_layer("shell2", 96, 192, False)]
    merged = LM.MergedTrellisLinear.from_linears([_layer("trellis", m, 192, False) for m in (96, 64)])
    calls = [lambda l=l: l(x) for l in lins] + [lambda: merged.process_weights_after_loading(DEV).apply(x)]
    table, v = e8_table_f16().float(), torch.randn(99, 8, generator=torch.Generator().manual_seed(1)).to(DEV)
    calls.append(lambda: ext.e8_quantize(v, table)[1])
    refs = [f() for f in calls for _ in range(2)][1::2]
    monkeypatch.setattr(ext, "_host", ext._NoHost)
    for l in lins:
        l._fast = None
    for f, ref in zip(calls, refs):
        assert torch.equal(f(), ref) and torch.equal(f(), ref)


def test_load_time_steps_make_no_native_form_for_what_forward_refuses():
    from glq_amd import linear_method as LM
    say("native form of layers that are refused")
    lin = _layer("trellis", 64, 128, False)
    lin.set_codebook(type("natural", (), {"has_kernel": False})())
    lin.prepare()
    x = torch.zeros(1, 128, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(RuntimeError, match="natural-layout"):
        lin(x)
    lins = [_layer("trellis", 64, 128, False), _layer("trellis2", 32, 128, False)]
    mixed = LM.MergedTrellisLinear.from_linears(lins, bpw=4)
    mixed.trellis_packed2._shard_data[1] = torch.zeros(0, dtype=torch.int16, device=DEV)
    mixed.trellis_packed._shard_data[1] = torch.zeros(0, dtype=torch.int16, device=DEV)       # never loaded
    mixed.process_weights_after_loading(DEV)
    assert mixed._fast is None and float(mixed.apply(x)[:, 64:].abs().max()) == 0.0
