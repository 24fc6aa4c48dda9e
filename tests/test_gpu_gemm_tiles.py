"""The prefill GEMM's tiles at their edges: an identity activation returns the dequantized weights, rounded once to the type of x, bit for
bit, whatever tile and division along K the launch takes.  Row counts and outputs around 64 and 112 columns and 64, 128 and 256
rows, one and several blocks of 256 values to a row."""
import pytest
import torch

from tattletale_amd import QuantLinear, formats as F
from tattletale_amd import qlinear as QL

from util import DEV, packed_to_dev, random_blocks

pytestmark = pytest.mark.gpu
NAMES = {F.Q8_0: "q8_0", F.Q4_K: "q4_k", F.Q6_K: "q6_k"}
BLOCK = {F.Q8_0: 32, F.Q4_K: 256, F.Q6_K: 256}


@pytest.mark.parametrize("n_out,n_in,m", [(64, 256, 256), (72, 256, 129), (1144, 512, 128), (4096, 768, 200), (4160, 1024, 1000),
                                          (264, 2048, 333), (512, 4096, 65), (16392, 256, 300)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("fmt", list(NAMES), ids=list(NAMES.values()))
def test_identity_rows(fmt, dtype, n_out, n_in, m):
    w = packed_to_dev(random_blocks(fmt, n_out * (n_in // BLOCK[fmt]), seed=n_out + n_in))
    lay = QuantLinear.init(w, fmt, n_in, n_out)
    wd = QL.dequantize(fmt, w, n_out, n_in)
    assert wd.abs().amax().item() < 65504
    cols = (torch.arange(m, device=DEV) * 37 + 5) % n_in
    x = torch.zeros(m, n_in, device=DEV, dtype=dtype)
    x[torch.arange(m, device=DEV), cols] = 1.0
    y = lay.forward(x, out_dtype=dtype)
    assert torch.equal(y + 0.0, wd[:, cols].t().to(dtype) + 0.0)
    # rows do not depend on their neighbours: the same rows with others around them
    x[m // 2:] = torch.randn(m - m // 2, n_in, device=DEV, generator=torch.Generator(DEV).manual_seed(m)).to(dtype)
    assert torch.equal(lay.forward(x, out_dtype=dtype)[: m // 2], y[: m // 2])
