"""The prefill GEMM's tiles.  At their edges: an identity activation returns the dequantized weights, rounded once to the type of x, bit for
bit; row counts and outputs around 64 and 112 columns and 64, 128 and 256 rows, one and several blocks of 256 values to a row (these
shapes take 64x64, 128x112 and 256x112 tiles).  Then one call at least of every tile, number of copies along K and way to the
activations that the chooser takes over a grid of shapes, by what ``ttq_route_detail`` says of it."""
import ctypes as C

import pytest
import torch

from tattletale_amd import QuantLinear, _lib, formats as F
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


DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
BYTES = {F.Q8_0: 34, F.Q4_K: 144, F.Q6_K: 210}
TILES = ("256x112", "256x64", "128x112", "128x64", "64x64")
# what the grid has to reach: every tile (64x112 only where K is divided), two, four, seven and eight copies, and for bf16 both ways to
# the activations (Q8_0: 128x112 tiles read them as they are)
PACKED = {t + " packed" for t in TILES} | {"256x112 k/2 packed", "256x112 k/4 packed", "256x64 k/2 packed", "256x64 k/4 packed", "256x64 k/7 packed"}
WANTED = {
    "bf16": PACKED | set(TILES) | {"128x112 k/2", "128x112 k/4", "128x112 k/7", "128x64 k/2", "128x64 k/4", "128x64 k/7", "128x64 k/8",
                                   "64x64 k/2", "64x64 k/4", "64x64 k/7", "64x64 k/8", "64x112 k/4"},
    "f16": PACKED | {"128x112 k/2 packed", "128x112 k/4 packed", "128x64 k/2 packed", "128x64 k/4 packed", "128x64 k/7 packed",
                     "64x64 k/2 packed", "64x64 k/4 packed", "64x64 k/7 packed", "64x64 k/8 packed", "64x112 k/4 packed"},
}
WANTED["f32"] = WANTED["f16"]


def blocks(fmt, n_out, n_in, gen):
    """Random packed rows, their scales below 2."""
    b = torch.randint(0, 256, (n_out * (n_in // BLOCK[fmt]), BYTES[fmt]), dtype=torch.uint8, device=DEV, generator=gen)
    for at in {F.Q8_0: [1], F.Q4_K: [1, 3], F.Q6_K: [209]}[fmt]:
        b[:, at] &= 0x3F
    return b.view(-1)


def forms(fmt, xk):
    """What the tiled kernel launches -> the smallest shape of a grid that has it."""
    L, text, code, found = _lib.lib(), C.create_string_buffer(64), QL._code(DT[xk]), {}
    for n_in in (256, 512, 768, 1024, 2048, 4096, 5376, 14336):
        for n_out in (64, 72, 264, 512, 1000, 1144, 2048, 2304, 4096, 4160, 8192, 16392, 20000):
            for m in (65, 100, 129, 200, 256, 257, 300, 512, 513, 600, 1000, 1500, 2049):
                if n_out * n_in > 6e7:
                    continue
                st = _lib.QLinearStruct(format=fmt, n_out=n_out, n_in=n_in)
                assert L.ttq_route_detail(C.byref(st), m, code, _lib.F32, text, 64) > 0
                kernel, _, form = text.value.decode().partition(" ")
                if kernel == "gemm_pc" and m * n_out * n_in < found.get(form, (1 << 62,))[0]:
                    found[form] = (m * n_out * n_in, m, n_out, n_in)
    return {form: shape[1:] for form, shape in found.items()}


@pytest.mark.parametrize("xk", list(DT))
@pytest.mark.parametrize("fmt", list(NAMES), ids=list(NAMES.values()))
def test_every_form_that_is_chosen(fmt, xk):
    """Against the float64 product with the weights as the kernel rounds them (to bf16, or to fp16 for fp16 and fp32 rows; the fp32 rows
    hold fp16 values, which their scaling by powers of two keeps): what is left is the fp32 sums, 2^-24 * sqrt(14336) = 7e-6."""
    gen = torch.Generator(DEV).manual_seed(11)
    found = forms(fmt, xk)
    wanted = WANTED[xk] - ({"128x112 packed"} if (fmt, xk) == (F.Q8_0, "bf16") else set())
    assert wanted <= set(found), wanted - set(found)
    for form, (m, n_out, n_in) in found.items():
        lay = QuantLinear.init(blocks(fmt, n_out, n_in, gen), fmt, n_in, n_out)
        assert lay.route_detail(m, DT[xk], torch.float32) == "gemm_pc " + form
        x = torch.randn(m, n_in, device=DEV, generator=gen).half().to(DT[xk])
        w = QL.dequantize(fmt, lay.qweight, n_out, n_in)
        ref = x.double() @ w.to(torch.bfloat16 if xk == "bf16" else torch.float16).double().T
        y = lay.forward(x, out_dtype=torch.float32).double()
        assert ((y - ref).norm(dim=-1) / ref.norm(dim=-1)).max().item() <= 1e-5, (form, m, n_out, n_in)


def test_every_form_of_the_fused_gate_up_kernel_that_is_chosen():
    """silu(gate) * up from fp32 sums, rounded once to bf16: 2^-9 of every value at most."""
    L, text, found = _lib.lib(), C.create_string_buffer(64), {}
    for n_ff in (64, 200, 1000, 1536, 2048, 3072, 4096, 8192):
        for n_in in (256, 512, 1024, 2048):
            for m in (65, 129, 200, 300, 600, 1000, 1500, 2048):
                assert L.ttq_gemm_q4_k_silu_mul_detail(m, n_ff, n_in, text, 64) >= 0
                kernel, _, form = text.value.decode().partition(" ")
                if kernel == "gemm_pc_silu_mul" and m * n_ff * n_in < found.get(form, (1 << 62,))[0]:
                    found[form] = (m * n_ff * n_in, m, n_ff, n_in)
    assert set(TILES) <= set(found)
    gen = torch.Generator(DEV).manual_seed(12)
    for form, (_, m, n_ff, n_in) in found.items():
        q = blocks(F.Q4_K, 2 * n_ff, n_in, gen)
        x = torch.randn(m, n_in, device=DEV, generator=gen).bfloat16()
        s = x.double() @ QL.dequantize(F.Q4_K, q, 2 * n_ff, n_in).bfloat16().double().T
        ref = torch.nn.functional.silu(s[:, :n_ff]) * s[:, n_ff:]
        y = QL.gemm_q4_k_silu_mul(q, x, n_ff, n_in).double()
        assert ((y - ref).norm() / ref.norm()).item() <= 2.2e-3, (form, m, n_ff, n_in)
