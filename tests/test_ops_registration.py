"""What torch's public registration and tracing APIs see of the operators, on the CPU."""
import inspect

import pytest
import torch

from mindpipe_amd import ops

OPS = [n for n in dir(ops) if isinstance(getattr(ops, n), torch.library.CustomOpDef)]


def test_every_registered_op_is_a_custom_op_def():
    assert {"w4a16_gemm", "quant_per_token_i8", "w8a8_gemm", "w8a8_linear", "w8a8_linear_fake", "moe_w8a8_forward",
            "dense_mlp_w8a8"} <= set(OPS)


@pytest.mark.parametrize("name", ["register_kernel", "register_fake", "register_autograd", "register_vmap",
                                  "register_torch_dispatch", "set_kernel_enabled"])
def test_custom_op_def_methods(name):
    method = getattr(ops.w4a16_gemm, name)
    assert callable(method) and inspect.signature(method)
