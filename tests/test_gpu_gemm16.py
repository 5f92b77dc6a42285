"""GPU parity of the 16-bit matrix-core GEMM (activations and weights both fp16 or both
bf16): every tile shape of its choice, at sizes with ragged rows, columns and K.

Small integers make every fp32 partial sum exact, so any summation order gives the exact
product: the outputs are compared bit for bit with the float64 product rounded once to
the output type.  The non-finite case checks that infinities and NaN land where IEEE
products and sums of the same operands put them."""
from __future__ import annotations

import pytest
import torch

from nano_vllm_cpp_amd import ops

pytestmark = pytest.mark.gpu

W = {torch.float16: ops.W_F16, torch.bfloat16: ops.W_BF16}
TYPES = [torch.float16, torch.bfloat16]
# (m, n, k): the tile that the choice takes is named beside each
SIZES = [
    (3, 40, 8),            # 32 x 32, one partial stage
    (31, 1001, 1000),      # 32 x 32, odd columns (element stores), K groups past the end
    (32, 24580, 136),      # 32 x 64
    (17, 65601, 72),       # 64 x 128 on an LM head's width
    (129, 6000, 264),      # 64 x 64
    (200, 3590, 520),      # 64 x 64, 2 K groups
    (300, 1500, 328),      # 64 x 32, 4 K groups
    (700, 4001, 200),      # 64 x 128
    (513, 9730, 192),      # 128 x 128
    (1021, 3584, 136),     # 128 x 128, 2 K groups
    (1021, 37890, 64),     # 256 x 256
    (4097, 24577, 72),     # 256 x 256, one row and one column in the last tiles
]


def ints(shape, dtype, device, seed):
    g = torch.Generator(device=device)
    g.manual_seed(seed)
    return torch.randint(-4, 5, shape, generator=g, device=device).to(dtype)


@pytest.mark.parametrize("dtype", TYPES, ids=["f16", "bf16"])
@pytest.mark.parametrize("m,n,k", SIZES)
def test_exact_on_integers(gpu, dtype, m, n, k):
    print(f"[case] gemm16 {m}x{n}x{k} {dtype}", flush=True)
    x, w = ints((m, k), dtype, gpu, 1), ints((n, k), dtype, gpu, 2)
    want = x.double() @ w.double().T
    for out_dtype in (torch.float32, dtype):
        guard = torch.full((m * n + 64,), 7.0, dtype=out_dtype, device=gpu)
        out = ops.matmul(x, w, n, W[dtype], out=guard[32:32 + m * n].view(m, n), out_dtype=out_dtype)
        assert torch.equal(out, want.to(out_dtype)), (m, n, k, out_dtype)
        assert bool((guard[:32] == 7).all()) and bool((guard[32 + m * n:] == 7).all()), "wrote outside the output"


@pytest.mark.parametrize("dtype", TYPES, ids=["f16", "bf16"])
@pytest.mark.parametrize("m,n,k", [(40, 96, 3584), (300, 4100, 4096)])
def test_within_fp32_sum_bound(gpu, dtype, m, n, k):
    g = torch.Generator(device=gpu)
    g.manual_seed(3)
    x = torch.randn(m, k, generator=g, device=gpu).to(dtype)
    w = (torch.randn(n, k, generator=g, device=gpu) * 0.03).to(dtype)
    out = ops.matmul(x, w, n, W[dtype], out_dtype=torch.float32).double()
    # exact products summed in fp32 in any order: (k + 2) 2^-24 sum |x w|
    bound = (k + 2) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert bool(((out - x.double() @ w.double().T).abs() <= bound).all())


@pytest.mark.parametrize("dtype", TYPES, ids=["f16", "bf16"])
def test_non_finite_operands(gpu, dtype):
    m, n, k = 70, 200, 136
    x, w = ints((m, k), dtype, gpu, 4), ints((n, k), dtype, gpu, 5)
    x[3, 7], x[9, 100], x[20, 0] = float("inf"), float("-inf"), float("nan")
    w[11, 50], w[13, 135] = float("inf"), float("nan")
    want = (x.double()[:, None, :] * w.double()[None]).sum(-1)
    out = ops.matmul(x, w, n, W[dtype], out_dtype=torch.float32).double()
    assert torch.equal(torch.isnan(out), torch.isnan(want))
    assert torch.equal(out[~torch.isnan(want)], want[~torch.isnan(want)])
