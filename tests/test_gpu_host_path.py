"""The native host path (csrc/bw_host.cpp) against the C ABI call it stands for: every layout, dtype and leading shape of x that
the module forward accepts, the autograd node, and the calls it leaves to the general path."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _layer(k, n, bits, g, bias=True, seed=0):
    from bitween_amd import QuantizedLinear
    torch.manual_seed(seed)
    return QuantizedLinear.from_float(torch.nn.Linear(k, n, bias=bias, device="cuda", dtype=torch.float16), bits, g)


def _w16(q):
    from bitween_amd.kernels import hip_loader as hip
    return hip.dequantize(q.qweight, q.scale, q.zero_point, q.group_size, q.bits, torch.float16)


def _close(y, x16, q):
    """2^-10 of the value (two float16 roundings) and float32 accumulation on sum |x| |w|, as the sweep's bound."""
    w = _w16(q).double()
    x64 = x16.double()
    ref = x64 @ w.T + (0 if q.bias is None else q.bias.double())
    return ((y.double() - ref).abs() <= 2.0 ** -10 * ref.abs() + 2.0 ** -12 * (x64.abs() @ w.abs().T) + 1e-6).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows", [1, 16, 17, 49, 130])         # the decode kernels, the batch kernel
def test_layouts_of_x(dtype, rows):
    q = _layer(256, 97, 4, 64)
    base = torch.randn(rows, 3, 2 * 256 + 8, device="cuda").to(dtype)
    views = [base[:, 0, :256],                                  # padded rows
             base[:, :, 8:264],                                 # 3-D, padded
             base[:, 1, 4:260],                                 # rows that start off a 16-byte boundary
             base[:, 2, :512:2],                                # strided columns
             base[:1, 0, :256].expand(rows, 256),               # one row repeated
             base[:, 0, :256].contiguous().view(1, rows, 1, 256)]
    for x in views:
        y = q(x)
        assert y.shape == x.shape[:-1] + (97,) and y.dtype is torch.float16
        assert _close(y.reshape(-1, 97), x.reshape(-1, 256).to(torch.float16), q)
    assert q(base[:0, 0, :256]).shape == (0, 97)                # no rows: the general path


@pytest.mark.parametrize("bits,g,k,n", [(4, 128, 256, 96), (4, 64, 192, 61), (8, 32, 128, 33)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_gradient_matches_the_autograd_function(bits, g, k, n, dtype):
    """module(x).backward against QuantizedLinearFunction (the Python node with the reference's interface): same kernels, same bits."""
    from bitween_amd import QuantizedLinearFunction
    q = _layer(k, n, bits, g, seed=n)
    x = torch.randn(2, 5, k, device="cuda").to(dtype).requires_grad_(True)
    x2 = x.detach().clone().requires_grad_(True)
    y, y2 = q(x), QuantizedLinearFunction.apply(x2, q.qweight, q.scale, q.zero_point, q.bias, q.bits, q.group_size)
    assert torch.equal(y, y2) and y.requires_grad
    go = torch.randn_like(y)
    y.backward(go)
    y2.backward(go)
    assert x.grad.dtype is dtype and torch.equal(x.grad, x2.grad)
    with pytest.raises(RuntimeError):                           # the node's buffers are released
        y.backward(go)
    with torch.no_grad():
        assert not q(x).requires_grad


def test_gradient_of_a_recorded_backward_and_of_a_changed_layer():
    q = _layer(128, 64, 4, 64)
    x = torch.randn(3, 128, device="cuda", dtype=torch.float16, requires_grad=True)
    go = torch.randn(3, 64, device="cuda", dtype=torch.float16, requires_grad=True)
    gx, = torch.autograd.grad(q(x), x, go, create_graph=True)
    v = torch.randn_like(gx)
    gg, = torch.autograd.grad(gx, go, v)                        # d(go W)/d(go) applied to v = v W^T
    ref = v.float() @ _w16(q).float().T
    assert (gg.float() - ref).abs().max() <= 2.0 ** -9 * ref.abs().max()
    y = q(x)
    q.scale.mul_(2.0)                                           # the weights of a recorded forward changed in place
    with pytest.raises(RuntimeError, match="modified by an inplace"):
        y.sum().backward()


def test_subclasses_and_parameters_as_inputs():
    class Sub(torch.Tensor):
        pass

    q = _layer(128, 64, 4, 64)
    x = torch.randn(3, 128, device="cuda", dtype=torch.float16)
    want = q(x)
    assert torch.equal(q(x.as_subclass(Sub)).as_subclass(torch.Tensor), want)
    assert torch.equal(q(torch.nn.Parameter(x)), want)
    with torch.inference_mode():
        y = q(x)
    assert y.is_inference() and torch.equal(y, want)


def test_quantize_copies_what_it_does_not_replace():
    """The copy that Bitween.quantize returns shares nothing with the model: containers, hooks, plain attributes."""
    import bitween_amd
    model = torch.nn.Sequential(torch.nn.Linear(128, 64, device="cuda", dtype=torch.float16), torch.nn.LayerNorm(64, device="cuda"))
    model.notes, model.empty = {"a": [1]}, {}
    calls = []
    model[1].register_forward_hook(lambda *a: calls.append(1))
    out = bitween_amd.Bitween(model, bits=4, group_size=64).quantize(rtn=True, verbose=False)
    assert isinstance(out[0], bitween_amd.QuantizedLinear) and isinstance(model[0], torch.nn.Linear)
    assert out.notes == {"a": [1]} and out.notes["a"] is not model.notes["a"] and out.empty == {} and out.empty is not model.empty
    assert out[1].weight is not model[1].weight and torch.equal(out[1].weight, model[1].weight)
    for name, value in model[1].__dict__.items():
        if isinstance(value, (dict, set)):
            assert out[1].__dict__[name] is not value and type(out[1].__dict__[name]) is type(value) and len(out[1].__dict__[name]) == len(value)
    assert len(out[1]._forward_hooks) == 1


def test_buffers_are_looked_at_on_every_call():
    """A buffer whose tensor object and address stay but whose layout or type does not, and a changed group size, are seen by the next call."""
    q = _layer(128, 64, 4, 64)
    x = torch.randn(3, 128, device="cuda", dtype=torch.float16)
    want = q(x)
    scale, dt = q.scale.data, q.scale.data.clone().t().contiguous().t()
    q.scale.data = dt                                           # same values, column-major
    assert torch.equal(q(x), want)
    q.scale.data = scale
    q.scale.data = scale.view(torch.bfloat16)                   # same address, another type
    with pytest.raises(TypeError):
        q(x)
    q.scale.data = scale
    assert torch.equal(q(x), want)
    q.group_size = 32                                           # the buffers do not belong to this one
    with pytest.raises(ValueError):
        q(x)


def test_transforms_that_the_python_function_refuses_stay_refused():
    q = _layer(128, 64, 4, 64)
    x = torch.randn(3, 128, device="cuda", dtype=torch.float16)
    with pytest.raises(RuntimeError):                           # no vmap rule
        torch.func.vmap(q)(x)
    with pytest.raises(RuntimeError):                           # no setup_context
        torch.func.grad(lambda t: q(t).float().sum())(x)
    import torch.autograd.forward_ad as fwd
    with fwd.dual_level(), pytest.raises(RuntimeError):         # no jvp
        q(fwd.make_dual(x.clone().requires_grad_(True), torch.ones_like(x)))


SLOW_LIBRARY = r"""
#include <stddef.h>
#include <stdint.h>
#include <unistd.h>
#define SLOW(name) int name() { usleep(300000); return 0; }
SLOW(bw_qlinear_ws) SLOW(bw_qdgrad) SLOW(bw_quantize_pack_add) SLOW(bw_dequantize) SLOW(bw_cast_bf16_f16)
size_t bw_qlinear_workspace_bytes() { return 0; }
size_t bw_qdgrad_workspace_bytes() { return 0; }
int bw_qdgrad_tile_rows() { return 128; }
"""


def test_other_threads_run_while_a_call_is_under_way(tmp_path):
    """A launch that blocks (a full queue) must not hold the interpreter lock: a second copy of the native module, bound to a library whose
    entry points sleep for 0.3 s, leaves another Python thread running in every function."""
    import ctypes
    import importlib.util
    import shutil
    import subprocess
    import threading
    import time
    from bitween_amd.kernels import hip_loader as hip
    q = _layer(128, 64, 4, 64)
    x = torch.randn(3, 128, device="cuda", dtype=torch.float16)
    go = torch.randn(3, 64, device="cuda", dtype=torch.float16)
    (tmp_path / "slow.c").write_text(SLOW_LIBRARY)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(tmp_path / "slow.so"), str(tmp_path / "slow.c")], check=True)
    slow = ctypes.CDLL(str(tmp_path / "slow.so"))
    shutil.copy(hip._HOST_PATH, tmp_path / "_bw_host.so")
    spec = importlib.util.spec_from_file_location("slow_copy._bw_host", tmp_path / "_bw_host.so")
    host = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(host)
    names = [n for n in hip.ENTRY_POINTS if hasattr(slow, n)]
    _bind(host, {n: ctypes.cast(getattr(slow, n), ctypes.c_void_p).value for n in names})
    ticks, stop = [0], threading.Event()

    def count():
        while not stop.is_set():
            time.sleep(0.001)
            ticks[0] += 1

    thread = threading.Thread(target=count)
    thread.start()
    try:
        buffers = (q.qweight, q.scale, q.zero_point)
        calls = {"forward": lambda: host.forward(q.__dict__, x), "matmul": lambda: host.matmul(x, *buffers, q.bias, 4, 64),
                 "recorded forward": lambda: host.forward(q.__dict__, x.clone().requires_grad_(True)),
                 "input_grad": lambda: host.input_grad(go, *buffers, 4, 64),
                 "quantize": lambda: host.quantize(x, None, 4, 64, hip.BW_F32, hip.BW_F16, hip.BW_F16),
                 "dequantize": lambda: host.dequantize(*buffers, 64, 4, hip.BW_F16)}
        for name, call in calls.items():
            call()                                              # (allocator warm: the second call only sleeps)
            before, start = ticks[0], time.perf_counter()
            assert call() is not None, name
            seconds = time.perf_counter() - start
            assert seconds > 0.25 and ticks[0] - before > 20, (name, seconds, ticks[0] - before)
    finally:
        stop.set()
        thread.join()


def _bind(host, table):
    from bitween_amd import modules
    from bitween_amd.kernels import hip_loader as hip
    host.bind(table, hip._check, vars(modules))


def test_from_float_runs_the_constructor_where_someone_looks_on(monkeypatch):
    """Global buffer registration hooks are called for every buffer, a subclass's and a replaced constructor run; the layers are those of the
    short way, and a bias that does not fit its layer is refused."""
    from torch.nn.modules.module import register_module_buffer_registration_hook
    import bitween_amd
    from bitween_amd.modules import BitweenShapeError
    lin = torch.nn.Linear(128, 64, device="cuda", dtype=torch.float16)
    plain = bitween_amd.QuantizedLinear.from_float(lin, 4, 64)
    seen = []
    handle = register_module_buffer_registration_hook(lambda module, name, buffer: seen.append((type(module).__name__, name)))
    try:
        hooked = bitween_amd.QuantizedLinear.from_float(lin, 4, 64)
    finally:
        handle.remove()
    assert seen == [("QuantizedLinear", n) for n in ("qweight", "scale", "zero_point", "bias")]

    class Sub(bitween_amd.QuantizedLinear):
        def __setattr__(self, name, value):
            seen.append(name)
            super().__setattr__(name, value)

    sub = Sub.from_float(lin, 4, 64)
    assert "in_features" in seen and "group_size" in seen
    calls, init = [], bitween_amd.QuantizedLinear.__init__
    monkeypatch.setattr(bitween_amd.QuantizedLinear, "__init__", lambda self, *a, **k: (calls.append(a), init(self, *a, **k))[1])
    replaced = bitween_amd.QuantizedLinear.from_float(lin, 4, 64)
    monkeypatch.undo()
    assert len(calls) == 1
    for layer in (hooked, sub, replaced):
        assert set(layer.__dict__) == set(plain.__dict__) and repr(layer) == repr(plain)
        for name, value in plain._buffers.items():
            assert torch.equal(layer._buffers[name], value) and layer._buffers[name].device == value.device
    bad = torch.nn.Linear(128, 64, device="cuda", dtype=torch.float16)
    bad.bias = torch.nn.Parameter(torch.zeros(63, device="cuda", dtype=torch.float16))
    with pytest.raises(BitweenShapeError):
        bitween_amd.QuantizedLinear.from_float(bad, 4, 64)


@pytest.mark.parametrize("bias", [True, False])
def test_node_looks_like_that_of_the_autograd_function(bias):
    """The node of q(x) against that of QuantizedLinearFunction.apply: name, saved tensors, edges, hooks; x changed in place is noticed, and
    saved-tensor hooks see the same tensors."""
    from bitween_amd import QuantizedLinearFunction
    q = _layer(128, 64, 4, 64, bias=bias)
    leaf = torch.randn(3, 128, device="cuda", dtype=torch.float16, requires_grad=True)

    def make(module, x):
        return q(x) if module else QuantizedLinearFunction.apply(x, q.qweight, q.scale, q.zero_point, q.bias, q.bits, q.group_size)

    looks = []
    for module in (True, False):
        packed, x = [], leaf * 1
        with torch.autograd.graph.saved_tensors_hooks(lambda t: (packed.append(tuple(t.shape)), t)[1], lambda t: t):
            y = make(module, x)
        node, fired = y.grad_fn, []
        node.register_hook(lambda grad_in, grad_out: fired.append((len(grad_in), grad_in[0].shape, len(grad_out))))
        saved = node.saved_tensors
        assert saved[0].data_ptr() == x.data_ptr() and (saved[4] is None) == (not bias)
        look = [node.name(), type(node).__name__, len(node.next_functions), node.next_functions[0][0].name(), node.bits, node.group_size,
                packed, [None if t is None else (t.dtype, tuple(t.shape), t.requires_grad) for t in saved], node.needs_input_grad[0]]
        y.sum().backward()
        looks.append(look + [fired])
        with pytest.raises(RuntimeError, match="second time"):
            node.saved_tensors
        x = leaf * 1
        y = make(module, x)
        x.mul_(2)
        with pytest.raises(RuntimeError, match="modified by an inplace"):
            y.sum().backward()
    assert looks[0] == looks[1]


def test_gradient_that_does_not_arrive_counts_as_zero():
    from bitween_amd import QuantizedLinearFunction

    class Nothing(torch.autograd.Function):
        @staticmethod
        def forward(ctx, y):
            return y.clone()

        @staticmethod
        def backward(ctx, grad):
            return None

    q = _layer(128, 64, 4, 64)
    for module in (True, False):
        x = torch.randn(3, 128, device="cuda", dtype=torch.float16, requires_grad=True)
        y = q(x) if module else QuantizedLinearFunction.apply(x, q.qweight, q.scale, q.zero_point, q.bias, q.bits, q.group_size)
        Nothing.apply(y).sum().backward()
        assert x.grad is not None and not x.grad.any()


def test_row_limits_of_the_fused_gradient_are_looked_at_by_every_backward(monkeypatch):
    """modules.FUSED_DGRAD_MAX_ROWS and _LARGE_MAX_ROWS, changed between forward and backward, decide which way the gradient takes: the
    dequantised weight has to be in memory on one way only."""
    from bitween_amd import QuantizedLinearFunction, modules
    q = _layer(4096, 4096, 4, 64)
    go = torch.randn(8, 4096, device="cuda", dtype=torch.float16)

    def memory(module):
        x = torch.randn(8, 4096, device="cuda", dtype=torch.float16, requires_grad=True)
        y = q(x) if module else QuantizedLinearFunction.apply(x, q.qweight, q.scale, q.zero_point, q.bias, q.bits, q.group_size)
        monkeypatch.setattr(modules, "FUSED_DGRAD_MAX_ROWS", rows)
        monkeypatch.setattr(modules, "FUSED_DGRAD_LARGE_MAX_ROWS", rows)
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        y.backward(go)
        return torch.cuda.max_memory_allocated() - before

    for module in (True, False):
        for rows, unfused in ((512, False), (7, True), (8, False), (0, True), (512, False)):
            assert (memory(module) >= 2 * 4096 * 4096) == unfused, (module, rows)
