"""GPU parity of the products on the 16-bit matrix cores: activations and weights both fp16
or both bf16, and K-quant weights with 16-bit activations.  Every tile shape of the
choices, at sizes with ragged rows, columns and K.

Small integers make every fp32 partial sum exact, so any summation order gives the exact
product: the outputs are compared bit for bit with the float64 product rounded once to
the output type.  The non-finite case checks that infinities and NaN land where IEEE
products and sums of the same operands put them."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from nano_vllm_cpp_amd import ops
from tests import harness as H

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


# ---------------------------------------------------------------------------
# K-quant weights (kq_gemm.hip, and kq_gemv.hip up to 16 rows), whole superblocks per row
# ---------------------------------------------------------------------------
KQ = [(12, H.GGML), (12, H.HIP_LEGACY), (13, H.GGML), (14, H.GGML)]
KQ_IDS = ["q4k", "q4k_legacy", "q5k", "q6k"]
# the workgroup's rows beside each
KQ_SIZES = [
    (1, 16400, 256),     # decode: one row, one superblock, 16 of 64 columns in the last workgroup
    (3, 100, 512),       # 8 K groups, most of them without a superblock
    (5, 33, 2304),       # two results per lane, one column past whole wave groups
    (8, 16390, 768),     # x in one stage
    (13, 16400, 2304),   # x in several stages, all four results per lane
    (2, 40, 8192),       # narrow and deep
    (17, 130, 256),      # 32: one superblock, two columns in the last tile
    (33, 129, 2304),     # 32, a second row of tiles
    (300, 3500, 256),    # 64
    (65, 24577, 256),    # 128 (Q6_K: 256)
    (129, 24580, 512),   # 256, one row in the last tile
]


def kq_case(seed, m, n, k, dt, kind):
    r = H.rng(seed)
    return H.gen_act(r, (m, k), dt), H.gen_weights(r, n, k, kind)


def kq_oracle(x, dt, w, kind, layout, m, n, k):
    want, err = np.empty((m, n), np.float64), np.empty((m, n), np.float64)
    H.oracle().orc_matmul_w(H.ptr(x), dt, H.ptr(w), kind, layout, m, n, k, H.ptr(want), H.ptr(err))
    return want, err


@pytest.mark.parametrize("kind,layout", KQ, ids=KQ_IDS)
@pytest.mark.parametrize("dt", [H.F16, H.BF16, H.F32], ids=["f16", "bf16", "f32"])
@pytest.mark.parametrize("m,n,k", KQ_SIZES)
def test_kquant_within_fp32_sum_bound(gpu, kind, layout, dt, m, n, k):
    if dt == H.F32 and m > 16:
        pytest.skip("fp32 rows beyond the decode product take the tile kernel of test_gpu_dense_gemm.py")
    print(f"[case] kq {kind}/{layout} {m}x{n}x{k} dt={dt}", flush=True)
    x, w = kq_case(100 * kind + m, m, n, k, dt, kind)
    want, err = kq_oracle(x, dt, w, kind, layout, m, n, k)
    for out_dtype in (torch.float32, H.torch_dtype(dt)):
        guard = torch.full((m * n + 64,), 7.0, dtype=out_dtype, device=gpu)
        out = ops.matmul(H.to_dev(x, gpu, dt), H.to_dev(w, gpu), n, kind, qk_layout=layout, out_dtype=out_dtype,
                         out=guard[32:32 + m * n].view(m, n))
        got = out.double().cpu().numpy()
        # the bound of fp32 sums of the decoded products, plus half an ulp of a 16-bit output
        tol = err + (0.0 if out_dtype == torch.float32 else 0.5 * H.ulp(want, dt))
        assert (np.abs(got - want) <= tol).all(), float((np.abs(got - want) / tol).max())
        assert bool((guard[:32] == 7).all()) and bool((guard[32 + m * n:] == 7).all()), "wrote outside the output"


@pytest.mark.parametrize("kind,layout", KQ, ids=KQ_IDS)
@pytest.mark.parametrize("dt", [H.F16, H.BF16], ids=["f16", "bf16"])
@pytest.mark.parametrize("m", [40, 7], ids=["prefill", "decode"])
def test_kquant_non_finite_operands(gpu, kind, layout, dt, m):
    n, k = 150, 512
    x, w = kq_case(7 * kind, m, n, k, dt, kind)
    xt = H.to_dev(x, gpu, dt)
    xt[3, 7], xt[5, 300], xt[1, 0] = float("inf"), float("-inf"), float("nan")
    if dt == H.BF16:
        xt[6, 5] = 3.0e38  # finite, but not times a sub-block's whole-number scale
    blk = w.reshape(n * k // 256, -1)
    d_at = 208 if kind == 14 else 0
    blk[4 * 2 + 1, d_at:d_at + 2] = np.array([np.inf], np.float16).view(np.uint8)  # column 4's second superblock
    want, _ = kq_oracle(H.to_host(xt), dt, w, kind, layout, m, n, k)
    got = ops.matmul(xt, H.to_dev(w, gpu), n, kind, qk_layout=layout, out_dtype=torch.float32).double().cpu().numpy()
    with np.errstate(over="ignore"):
        want32 = want.astype(np.float32).astype(np.float64)
    assert (np.isnan(got) == np.isnan(want32)).all()
    assert (np.isposinf(got) == np.isposinf(want32)).all() and (np.isneginf(got) == np.isneginf(want32)).all()
    fin = np.isfinite(want32)
    assert np.allclose(got[fin], want32[fin], rtol=1e-4, atol=1e-3 * np.abs(want32[fin & (np.abs(want32) < 1e6)]).max())


def cancelling_weights(r, n, k, kind, layout):
    """Q4_K / Q5_K superblocks whose scale and offset parts cancel: in every sub-block one quant
    q0 gives exactly 0 (every second superblock: almost 0), and all weights but one in every
    third superblock hold it."""
    nb = n * k // 256
    sc = r.integers(1, 13, (nb, 8))
    q0 = r.integers(1, np.minimum(16 if kind == 12 else 32, 63 // sc + 1))
    q = np.repeat(q0[..., None], 32, 2)
    some = np.arange(0, nb, 3)
    q[some, r.integers(0, 8, some.size), r.integers(0, 32, some.size)] = r.integers(0, 16 if kind == 12 else 32, some.size)
    d = r.uniform(1e-3, 1e-2, nb).astype(np.float16)
    dmin = np.where(np.arange(nb) % 2, np.nextafter(d, np.float16(1)), d)
    lo = (q & 15).astype(np.uint8)
    if layout == H.GGML:
        ql = (lo[:, 0::2] | lo[:, 1::2] << 4).reshape(nb, 128)
    else:
        ql = (lo[..., :16] | lo[..., 16:] << 4).reshape(nb, 128)
    parts = [d.view(np.uint8).reshape(nb, 2), dmin.view(np.uint8).reshape(nb, 2), H.pack_q4k_scales(sc, sc * q0)]
    if kind == 13:
        parts.append(((q >> 4) << np.arange(8)[:, None]).sum(1).astype(np.uint8))
    return np.concatenate(parts + [ql], 1).reshape(-1)


@pytest.mark.parametrize("kind,layout", KQ[:3], ids=KQ_IDS[:3])
@pytest.mark.parametrize("dt", [H.F16, H.BF16, H.F32], ids=["f16", "bf16", "f32"])
@pytest.mark.parametrize("m,n,k", [(1, 16400, 512), (4, 24, 8192), (13, 16400, 256), (70, 300, 768), (200, 130, 2048)])
def test_kquant_scale_and_offset_cancel(gpu, kind, layout, dt, m, n, k):
    """x of one sign on weights that are differences of large parts.  Around the quant q0
    nearest to dmin m / (d sc) a weight is w = d sc (q - q0) + r with |d sc (q - q0)| <= 2 |w| and
    |r| <= |w|, so sums of the two parts stay within three times the bound of sums of x w."""
    if dt == H.F32 and m > 16:
        pytest.skip("fp32 rows beyond the decode product take the tile kernel of test_gpu_dense_gemm.py")
    r = H.rng(31 * kind + m)
    x, w = H.gen_act(r, (m, k), dt, 1.0, 0.1), cancelling_weights(r, n, k, kind, layout)
    want, err = kq_oracle(x, dt, w, kind, layout, m, n, k)
    print(f"[case] kq cancel {kind}/{layout} {m}x{n}x{k} dt={dt}", flush=True)
    got = ops.matmul(H.to_dev(x, gpu, dt), H.to_dev(w, gpu), n, kind, qk_layout=layout, out_dtype=torch.float32)
    off = np.abs(got.double().cpu().numpy() - want)
    assert (off <= 3 * err).all(), float((off / err).max())


@pytest.mark.parametrize("m,n,k", [(1021, 4096, 3584), (8, 37888, 3584), (2, 3584, 18944)], ids=["prefill", "wide", "deep"])
def test_kquant_time_on_nan_activations(gpu, m, n, k):
    """Every output non-finite: they are made again on the fp32 matrix cores, at most 16 times (their
    rate to the 16-bit ones') the work of the product, and not one after the other."""
    w = H.to_dev(H.gen_weights(H.rng(5), n, k, 12), gpu)
    x = torch.ones(m, k, dtype=torch.float16, device=gpu)

    def time(v):
        best = float("inf")
        for _ in range(4):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            ops.matmul(v, w, n, 12)
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b))
        return best

    t0, t1 = time(x), time(torch.full_like(x, float("nan")))
    print(f"[case] NaN {m}x{n}x{k}: {1e3 * t0:.1f} us finite, {1e3 * t1:.1f} us NaN", flush=True)
    assert t1 < 16 * t0
