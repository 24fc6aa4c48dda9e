"""The decode kernels on shapes that the kernel for matrices of a few MB leaves to them: every call says by ``ttq_route_detail`` that the
kernel it is about runs.

Reference: the float64 product over the library's dense copy of the weights (bit-exact against the oracle, test_gpu_dequant.py).  Bounds:
fp32 arithmetic and packed dots, partial sums of at most 2^12 products before they are added up, 2^-24 * sqrt(2^12) = 4e-6; Q4_K dots
with fp16 rows, whose quants enter as 1024 + q and are 128 times themselves (7.5 in the mean) until the sums of x are taken off, 16
roundings to a sub-block: 2^-25 * 128 * sqrt(16) = 1.5e-5; 15-bit block fixed point, whose step is 2^-15 of a block's largest value (up
to four times its root mean square): 2^-15 * 4 = 1.2e-4."""
import pytest
import torch

from tattletale_amd import QuantLinear, formats as F
from tattletale_amd import qlinear as QL

from util import DEV, packed_to_dev, random_blocks

pytestmark = pytest.mark.gpu
DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
BLOCK = {F.Q8_0: 32, F.Q4_K: 256, F.Q6_K: 256}
EXACT, OFFSET, FIXED = 4e-6, 1.5e-5, 1.2e-4

CALLS = [
    # kernel, format, x, rows, n_out, n_in, bound
    ("gemv_generic", F.Q4_K, "f32", 1, 1999, 11008, EXACT), ("gemv_generic", F.Q4_K, "f32", 3, 16, 8448, EXACT),
    ("gemv_generic", F.Q4_K, "f32", 9, 40, 256, EXACT), ("gemv_generic", F.Q6_K, "f32", 4, 16, 8448, EXACT),
    ("gemv_generic", F.Q6_K, "f32", 9, 41, 768, EXACT), ("gemv_generic", F.Q8_0, "bf16", 1, 1000, 16384, EXACT),
    ("gemv_generic", F.Q8_0, "f32", 3, 40, 8448, EXACT), ("gemv_generic", F.Q8_0, "f16", 9, 41, 288, EXACT),
    ("gemv_dot2", F.Q4_K, "bf16", 1, 1536, 5120, EXACT), ("gemv_dot2", F.Q4_K, "f16", 1, 201, 53248, OFFSET),
    ("gemv_dot2", F.Q6_K, "bf16", 1, 1999, 11008, EXACT), ("gemv_dot2", F.Q6_K, "f16", 1, 10000, 2304, EXACT),
    ("gemv_dot2_multi", F.Q4_K, "bf16", 2, 16, 8448, EXACT), ("gemv_dot2_multi", F.Q4_K, "f16", 5, 17, 256, OFFSET),
    ("gemv_dot2_multi", F.Q6_K, "bf16", 4, 16, 8448, EXACT), ("gemv_dot2_multi", F.Q6_K, "f16", 9, 41, 1024, EXACT),
    ("gemv_q8_win", F.Q8_0, "f32", 1, 10000, 256, FIXED), ("gemv_q8_win", F.Q8_0, "bf16", 3, 20000, 256, FIXED),
    ("gemv_q8_win", F.Q8_0, "f32", 9, 1024, 256, FIXED), ("gemv_q4k_mfma", F.Q4_K, "bf16", 1, 10000, 256, FIXED),
    ("gemv_q4k_mfma", F.Q4_K, "f32", 2, 10000, 256, FIXED), ("gemv_q4k_mfma", F.Q4_K, "f32", 9, 2048, 256, FIXED),
    ("gemv_q4k_batch4", F.Q4_K, "bf16", 3, 6000, 256, FIXED), ("gemv_q4k_batch4", F.Q4_K, "f16", 5, 2048, 8448, FIXED),
    ("gemv_q4k_batch", F.Q4_K, "bf16", 5, 2048, 256, FIXED),
]


@pytest.mark.parametrize("kernel,fmt,xk,m,n_out,n_in,bound", CALLS, ids=["-".join(map(str, c[:6])) for c in CALLS])
def test_kernel(kernel, fmt, xk, m, n_out, n_in, bound):
    w = packed_to_dev(random_blocks(fmt, n_out * (n_in // BLOCK[fmt]), seed=n_out + n_in))
    lay = QuantLinear.init(w, fmt, n_in, n_out, precision=F.PRECISION_F32_SCALES)
    assert lay.route_detail(m, DT[xk], torch.float32) == kernel
    x = torch.randn(m, n_in, device=DEV, generator=torch.Generator(DEV).manual_seed(m)).to(DT[xk])
    wd = QL.dequantize(fmt, w, n_out, n_in).double()
    size = ((x.double() ** 2) @ (wd ** 2).T).sqrt()          # (a single output can cancel)
    y = lay.forward(x, out_dtype=torch.float32).double()
    assert ((y - x.double() @ wd.T).norm(dim=-1) / size.norm(dim=-1)).max().item() <= bound
