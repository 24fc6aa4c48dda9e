"""The native host half of qlinear.py (csrc/ttq_torch.cpp): what it hands back to Python, that a call through it is
the call through the C ABI, and the Python code that serves the calls where it is not built."""
import sys
import threading
import time

import pytest
import torch

import tattletale_amd
from tattletale_amd import QuantGatedMLP, QuantLinear, TtqError, _lib, build, formats as F, qlinear, quantize as Q


@pytest.fixture
def python_host(monkeypatch):
    """The program of a user who built libttq_hip.so only."""
    monkeypatch.delattr(tattletale_amd, "_ttq_torch", raising=False)
    monkeypatch.setitem(sys.modules, "tattletale_amd._ttq_torch", None)         # importing it raises ImportError
    monkeypatch.setattr(qlinear, "_native_module", None)


def test_tensors_it_does_not_take_go_back_to_python():
    n = qlinear._native()
    x, g = torch.zeros(2, 256), torch.ones(256)
    assert n.silu_and_mul(x) == 1 and n.rmsnorm(x, g, 1e-5, None) == 1          # not on a GPU
    assert n.silu_and_mul(None) == 1 and n.linear_forward() == 1
    layer = QuantLinear(torch.zeros(144, dtype=torch.uint8), F.Q4_K, 256, 1)
    for bad, status in ((x, _lib.ERR_UNSUPPORTED), (x[0, 0], _lib.ERR_SHAPE), (x[:, 1:], _lib.ERR_SHAPE)):
        with pytest.raises(TtqError) as e:
            layer.forward(bad)
        assert e.value.status == status


def test_calls_are_served_where_the_extension_is_not_built(python_host):
    layer = QuantLinear(torch.zeros(144, dtype=torch.uint8), F.Q4_K, 256, 1)
    with pytest.warns(RuntimeWarning, match="_ttq_torch is not used"):
        with pytest.raises(TtqError) as e:                      # the operator's own answer to a CPU tensor
            layer.forward(torch.zeros(2, 256))
    assert e.value.status == _lib.ERR_UNSUPPORTED and qlinear._native() is qlinear._PythonHost


def test_an_extension_of_another_torch_is_not_used(monkeypatch):
    assert qlinear._native().torch_version == torch.__version__                 # it is built here
    monkeypatch.setattr(qlinear, "_native_module", None)
    monkeypatch.setattr(torch, "__version__", "0.0.0")
    with pytest.warns(RuntimeWarning, match="this is 0.0.0"):
        assert qlinear._native() is qlinear._PythonHost


def test_the_extension_is_built_again_for_another_torch(monkeypatch, tmp_path):
    runs = []

    def gxx(cmd, **kw):
        runs.append(cmd)
        (tmp_path / "ext.so").write_bytes(b"")
        return type("Done", (), {"returncode": 0, "stdout": "", "stderr": ""})
    monkeypatch.setattr(build.subprocess, "run", gxx)
    monkeypatch.setattr(build, "TORCH_EXT", str(tmp_path / "ext.so"))
    monkeypatch.setattr(build, "TORCH_EXT_COMMAND", str(tmp_path / "build" / "ext.command"))
    build.build_torch_ext(force=False)
    build.build_torch_ext(force=False)
    assert len(runs) == 1
    monkeypatch.setattr(torch, "__version__", "0.0.0")
    build.build_torch_ext(force=False)
    assert len(runs) == 2


def _every_call():
    """Results of each entry point with a native half, by name."""
    def packed(fmt, n_out, n_in, seed):
        return torch.from_numpy(Q.quantize(fmt, Q.fill_normal(seed, 0, 0.02, n_out * n_in).reshape(n_out, n_in))).cuda()
    gen = torch.Generator(device="cuda").manual_seed(1)
    n_in, n_ff, out = 2048, 2048, {}
    gu = QuantLinear.init(packed(F.Q4_K, 2 * n_ff, n_in, 1), F.Q4_K, n_in, 2 * n_ff)
    down = QuantLinear.init(packed(F.Q6_K, n_in, n_ff, 2), F.Q6_K, n_ff, n_in, bias=torch.ones(n_in, device="cuda"))
    mlp = QuantGatedMLP.init(gu, down)
    for dtype in (torch.float32, torch.float16, torch.bfloat16):
        gamma = torch.randn(n_in, generator=gen, device="cuda").to(dtype)
        for m in (1, 3, 20):
            x = torch.randn(m, n_in, generator=gen, device="cuda").to(dtype)
            ws = torch.zeros(max(16, down.workspace_bytes(m, dtype)), dtype=torch.uint8, device="cuda")
            key = (m, dtype)
            out["linear", key] = down.forward(x, out_dtype=torch.float32)
            out["workspace", key] = down.forward(x, workspace=ws)
            out["silu", key] = qlinear.silu_and_mul(x)
            out["mlp", key] = mlp.forward(x.view(1, m, n_in))
            out["norm", key], none = qlinear.rmsnorm(x, gamma, 1e-5)
            out["norm + residual", key], out["residual", key] = qlinear.rmsnorm(x, gamma, 1e-5, x)
            assert none is None
    return out


@pytest.mark.gpu
def test_both_host_halves_give_the_same_results(request):
    assert qlinear._native().torch_version == torch.__version__
    native = _every_call()
    request.getfixturevalue("python_host")
    with pytest.warns(RuntimeWarning):
        python = _every_call()
    assert native.keys() == python.keys()
    for k in native:
        a, b = native[k], python[k]
        assert a.shape == b.shape and a.dtype == b.dtype and torch.equal(a, b), k


@pytest.mark.gpu
def test_forward_is_the_c_abi_call_and_errors_keep_their_status():
    n_out, n_in = 48, 512
    packed = torch.from_numpy(Q.quantize(F.Q4_K, Q.fill_normal(3, 0, 0.02, n_out * n_in).reshape(n_out, n_in))).cuda()
    layer = QuantLinear.init(packed, F.Q4_K, n_in, n_out, bias=torch.ones(n_out, device="cuda"))
    x = torch.randn(2, 3, n_in, device="cuda", dtype=torch.bfloat16)
    y = layer.forward(x, out_dtype=torch.float32)
    st, want = layer._struct(), torch.empty(6, n_out, device="cuda")
    import ctypes as C
    _lib.check(_lib.lib().ttq_linear_forward(C.byref(st), x.data_ptr(), F.BF16, 6, want.data_ptr(), F.F32,
                                             torch.cuda.current_stream().cuda_stream), "abi")
    assert y.shape == (2, 3, n_out) and torch.equal(y.view(6, n_out), want)
    ws = torch.zeros(max(16, layer.workspace_bytes(6, x.dtype)), dtype=torch.uint8, device="cuda")
    assert torch.equal(layer.forward(x, torch.float32, ws), y)
    assert layer.forward(x[:0]).shape == (0, 3, n_out)
    for bad, status in ((x[..., ::2], _lib.ERR_SHAPE), (x.transpose(0, 1), _lib.ERR_SHAPE), (x.cpu(), _lib.ERR_UNSUPPORTED),
                        (x.double(), _lib.ERR_DTYPE)):
        with pytest.raises(TtqError) as e:
            layer.forward(bad)
        assert e.value.status == status
    with pytest.raises(TtqError) as e:                          # a status of the library itself
        layer.forward(x, torch.float32, ws[1:])
    assert e.value.status == _lib.ERR_WORKSPACE
    out, res = qlinear.rmsnorm(x, torch.ones(n_in, device="cuda", dtype=x.dtype), 1e-5, x)
    assert torch.equal(res, x + x) and out.shape == x.shape


@pytest.mark.gpu
@pytest.mark.parametrize("x_dtype,r_dtype", [(torch.float32, torch.bfloat16), (torch.float32, torch.float16),
                                             (torch.bfloat16, torch.float32), (torch.bfloat16, torch.float16)])
@pytest.mark.parametrize("host", ["native", "python"])
def test_rmsnorm_refuses_a_residual_of_another_type(x_dtype, r_dtype, host, monkeypatch):
    """The kernel reads the residual as x's type: one of half the size would be read beyond its end."""
    monkeypatch.setattr(qlinear, "_native_module", qlinear._PythonHost if host == "python" else qlinear._native())
    x, gamma = torch.ones(3, 256, device="cuda", dtype=x_dtype), torch.ones(256, device="cuda", dtype=x_dtype)
    with pytest.raises(TtqError) as e:
        qlinear.rmsnorm(x, gamma, 1e-5, torch.ones(3, 256, device="cuda", dtype=r_dtype))
    assert e.value.status == _lib.ERR_SHAPE


@pytest.mark.gpu
@pytest.mark.parametrize("host", ["native", "python"])
def test_no_rows_give_outputs_of_no_rows(host, monkeypatch):
    monkeypatch.setattr(qlinear, "_native_module", qlinear._PythonHost if host == "python" else qlinear._native())
    x = torch.zeros(2, 0, 256, device="cuda", dtype=torch.bfloat16)
    gamma = torch.ones(256, device="cuda", dtype=x.dtype)
    layer = QuantLinear.init(torch.zeros(16 * 144, dtype=torch.uint8, device="cuda"), F.Q4_K, 256, 16)
    normed, residual = qlinear.rmsnorm(x, gamma, 1e-5, x)
    assert normed.shape == residual.shape == x.shape and qlinear.rmsnorm(x, gamma, 1e-5)[1] is None
    assert layer.forward(x).shape == (2, 0, 16) and qlinear.silu_and_mul(x).shape == (2, 0, 128)


@pytest.mark.gpu
@pytest.mark.parametrize("host", ["native", "python"])
@pytest.mark.parametrize("shape", [(), (3, 0), (0,)])
def test_rows_of_no_elements_are_refused_as_a_shape(shape, host, monkeypatch):
    monkeypatch.setattr(qlinear, "_native_module", qlinear._PythonHost if host == "python" else qlinear._native())
    x, empty = torch.zeros(shape, device="cuda"), torch.zeros(0, device="cuda")
    for call in (lambda: qlinear.silu_and_mul(x), lambda: qlinear.rmsnorm(x, empty, 1e-5), lambda: qlinear.rmsnorm(x, empty, 1e-5, x)):
        with pytest.raises(TtqError) as e:
            call()
        assert e.value.status == _lib.ERR_SHAPE


def _calls(seed):
    """Small inputs of their own, and the four calls on them in sequence."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    n_in, n_ff = 1024, 2048
    gu, down = (QuantLinear.init(torch.from_numpy(Q.quantize(F.Q4_K, Q.fill_normal(seed, i, 0.03, a * b).reshape(a, b))).cuda(),
                                 F.Q4_K, b, a) for i, (a, b) in enumerate(((2 * n_ff, n_in), (n_in, n_ff))))
    mlp, gamma = QuantGatedMLP.init(gu, down), torch.ones(n_in, device="cuda", dtype=torch.bfloat16)

    def run(x):
        normed, residual = qlinear.rmsnorm(x, gamma, 1e-5, x)
        return normed, residual, mlp.forward(normed), qlinear.silu_and_mul(gu.forward(normed))
    return torch.randn(5, n_in, generator=gen, device="cuda").bfloat16(), run


@pytest.mark.gpu
def test_calls_run_on_the_callers_stream():
    """The input is filled on a side stream, behind work that holds it up: a call on another stream would read it empty."""
    x, run = _calls(1)
    want = run(x)
    a = torch.ones(8192, 8192, device="cuda", dtype=torch.bfloat16)
    b, late, side = torch.mm(a, a), torch.zeros_like(x), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        for _ in range(20):
            torch.mm(a, a, out=b)
        late.copy_(x)
        got = run(late)
    side.synchronize()
    assert all(torch.equal(g, w) for g, w in zip(got, want))


@pytest.mark.gpu
def test_threads_on_streams_of_their_own():
    work = [_calls(10 + i) for i in range(4)]
    want = [run(x) for x, run in work]
    torch.cuda.synchronize()
    wrong = []

    def go(i):
        x, run = work[i]
        try:
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                got = [run(x) for _ in range(25)]
            stream.synchronize()
            wrong.extend((i, k) for k, g in enumerate(got) if not all(torch.equal(p, q) for p, q in zip(g, want[i])))
        except Exception as e:
            wrong.append((i, e))
    threads = [threading.Thread(target=go, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


@pytest.mark.gpu
def test_an_input_that_requires_grad():
    x, run = _calls(2)
    got = run(x.clone().requires_grad_())
    assert all(torch.equal(g, w) and not g.requires_grad for g, w in zip(got, run(x)))


@pytest.mark.gpu
@pytest.mark.parametrize("call", ["linear", "rmsnorm", "silu_and_mul", "gate_up_silu"])
def test_other_threads_run_while_an_output_is_allocated(call):
    """An allocation that waits for the GPU (at the memory limit, for a block that another stream still uses) stops the
    calling thread only: here for as long as 300 matrix products take, while a second thread ticks every half
    millisecond.  Bound: no two ticks are half of the wait apart."""
    x = torch.randn(32768, 1024, device="cuda").bfloat16()
    packed = torch.from_numpy(Q.quantize(F.Q4_K, Q.fill_normal(3, 0, 0.02, 1024 * 1024).reshape(1024, 1024))).cuda()
    layer = QuantLinear.init(packed, F.Q4_K, 1024, 1024)
    gamma = torch.ones(1024, device="cuda", dtype=x.dtype)
    run = {"linear": lambda: layer.forward(x), "silu_and_mul": lambda: qlinear.silu_and_mul(x),
           "rmsnorm": lambda: qlinear.rmsnorm(x, gamma, 1e-5),
           "gate_up_silu": lambda: qlinear._native().q4_k_silu_mul(packed, x, 512, 1024, True)}[call]
    a = torch.ones(8192, 8192, device="cuda", dtype=torch.bfloat16)
    b, side = torch.empty_like(a), torch.cuda.Stream()
    run()                                                       # kernels loaded, workspaces made
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        torch.mm(a, a, out=b)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    reserved, fill = torch.cuda.memory_reserved(), []
    while torch.cuda.memory_reserved() == reserved:             # until no free block is left that could hold the output
        fill.append(torch.empty(32 << 20, dtype=torch.uint8, device="cuda"))
    fill.pop()
    torch.cuda.empty_cache()
    held = torch.empty(1 << 30, dtype=torch.uint8, device="cuda")
    gaps, stop = [], threading.Event()

    def ticks():
        last = time.perf_counter()
        while not stop.is_set():
            time.sleep(0.0005)
            now = time.perf_counter()
            gaps.append(now - last)
            last = now

    thread = threading.Thread(target=ticks)
    thread.start()
    total = torch.cuda.get_device_properties(0).total_memory
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (8 << 20)) / total)
        with torch.cuda.stream(side):
            for _ in range(300):
                torch.mm(a, a, out=b)
        held.record_stream(side)
        del held                                                # free again once the side stream is through
        start = time.perf_counter()
        run()
        took = time.perf_counter() - start
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
        stop.set()
        thread.join()
    assert took > 0.05, "the allocation did not wait"
    assert max(gaps) < took / 2


@pytest.mark.gpu
def test_an_output_that_does_not_fit_raises_and_leaves_the_program_usable():
    """The exception leaves the stretch without the interpreter lock with the lock taken again."""
    x = torch.randn(32768, 1024, device="cuda").bfloat16()
    want = qlinear.silu_and_mul(x).clone()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (1 << 30)) / total)
        layer = QuantLinear.init(torch.zeros(65536 * 4 * 144, dtype=torch.uint8, device="cuda"), F.Q4_K, 1024, 65536)
        with pytest.raises(torch.OutOfMemoryError):
            layer.forward(x)                                    # 4 GiB
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(qlinear.silu_and_mul(x), want)
