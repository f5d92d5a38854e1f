"""What torch's public registration and tracing APIs see of the operators, on the CPU."""
import concurrent.futures
import inspect
import subprocess
import sys
import textwrap
from pathlib import Path

import pytest
import torch

from mindpipe_amd import ops

ROOT = Path(__file__).resolve().parent.parent
OPS = [n for n in dir(ops) if isinstance(getattr(ops, n), torch.library.CustomOpDef)]


def test_every_registered_op_is_a_custom_op_def():
    assert {"w4a16_gemm", "quant_per_token_i8", "w8a8_gemm", "w8a8_linear", "w8a8_linear_fake", "moe_w8a8_forward",
            "dense_mlp_w8a8"} <= set(OPS)


@pytest.mark.parametrize("name", ["register_kernel", "register_fake", "register_autograd", "register_vmap",
                                  "register_torch_dispatch", "set_kernel_enabled"])
def test_custom_op_def_methods(name):
    method = getattr(ops.w4a16_gemm, name)
    assert callable(method) and inspect.signature(method)


def _python(code):
    """Runs ``code`` in a process of its own: registrations and reloads outlive a test."""
    head = "import importlib, torch\nfrom mindpipe_amd import ops\nx = torch.randn(2, 64).half()\n"
    subprocess.run([sys.executable, "-c", head + textwrap.dedent(code)], check=True, cwd=ROOT, timeout=120)


@pytest.mark.parametrize("register", [
    'torch.library.register_kernel("mindpipe_amd::quant_per_token_i8", "cpu", mine)',
    'ops.quant_per_token_i8.register_kernel("cpu")(mine)',
    'lib = torch.library.Library("mindpipe_amd", "IMPL"); lib.impl("quant_per_token_i8", mine, "CPU")',
])
def test_a_registered_kernel_is_used(register):
    _python(f"""
        mine = lambda v, fake_rule=False: (torch.zeros_like(v, dtype=torch.int8), torch.full((len(v),), 3.0))
        {register}
        for got in (ops.quant_per_token_i8(x), torch.ops.mindpipe_amd.quant_per_token_i8(x)):
            assert got[1].tolist() == [3.0, 3.0]
    """)


def test_reload():
    _python("""
        for _ in range(2):
            importlib.reload(ops)
        for op in (ops.quant_per_token_i8, torch.ops.mindpipe_amd.quant_per_token_i8):
            try:
                op(x)
            except RuntimeError as e:
                assert "must be on the GPU" in str(e)
            else:
                raise AssertionError("no CPU path")
        y = torch.ops.mindpipe_amd_light.quant_per_token_i8(x.to("meta"), False)
        assert y[0].shape == x.shape and y[0].is_meta
    """)


@pytest.mark.gpu
@pytest.mark.parametrize("register", [
    'torch.library.register_kernel("mindpipe_amd::quant_per_token_i8", "cuda", mine)',
    'lib = torch.library.Library("mindpipe_amd", "IMPL"); lib.impl("quant_per_token_i8", mine, "CUDA")',
])
def test_a_registered_gpu_kernel_is_used(register):
    _python(f"""
        x = x.cuda()
        assert ops.quant_per_token_i8(x)[1].tolist() != [3.0, 3.0]
        mine = lambda v, fake_rule=False: (torch.zeros_like(v, dtype=torch.int8), v.new_full((len(v),), 3.0))
        {register}
        assert ops.quant_per_token_i8(x)[1].tolist() == [3.0, 3.0]
    """)


@pytest.mark.gpu
def test_traces_and_modes_see_the_custom_op():
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode
    x = torch.randn(2, 64, device="cuda").half()
    graph = make_fx(lambda v: ops.quant_per_token_i8(v))(x).graph
    assert torch.ops.mindpipe_amd.quant_per_token_i8.default in [n.target for n in graph.nodes]
    seen = []

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    for mode in (Dispatch, Function):
        seen.clear()
        with mode():
            ops.quant_per_token_i8(x)
        assert torch.ops.mindpipe_amd.quant_per_token_i8.default in seen


def _outcome(f):
    try:
        return f()
    except Exception as e:
        return type(e)


@pytest.mark.gpu
def test_vmap_and_forward_ad_do_what_the_custom_op_does():
    x = torch.randn(3, 2, 64, device="cuda").half()
    direct, custom = ops.quant_per_token_i8, torch.ops.mindpipe_amd.quant_per_token_i8.default
    got, want = (_outcome(lambda: torch.vmap(lambda v: op(v)[0])(x)) for op in (direct, custom))
    assert torch.equal(got, want) if isinstance(want, torch.Tensor) else got == want
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(x, torch.ones_like(x))
        got, want = (_outcome(lambda: torch.autograd.forward_ad.unpack_dual(op(dual)[1]).tangent is None)
                     for op in (direct, custom))
        assert got == want


@pytest.mark.gpu
def test_other_streams_and_threads():
    """Each stream and each thread's calls read and write on their own current stream."""
    w = torch.randint(-127, 128, (512, 1024), device="cuda", dtype=torch.int8)
    sc = torch.rand(512, device="cuda") * 0.01
    xs = [torch.randn(64, 1024, device="cuda").half() for _ in range(4)]
    want = [ops.w8a8_linear(x, w, sc, None, torch.float16, False) for x in xs]
    torch.cuda.synchronize()

    def work(x):
        side = torch.cuda.Stream()
        with torch.cuda.stream(side):
            out = [ops.w8a8_linear(x, w, sc, None, torch.float16, False) for _ in range(20)]
        side.synchronize()
        return out
    with concurrent.futures.ThreadPoolExecutor(4) as pool:
        for got, ref in zip(pool.map(work, xs), want):
            assert all(torch.equal(g, ref) for g in got)
