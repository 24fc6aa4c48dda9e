"""The decode kernel for matrices of a few MB (ttq_gemv_short.hip): rows that do and do not fill its wavefronts (1024 values each), one
and several wavefronts to a row, row counts around its groups, one to eight activation rows.

The float64 product over the library's own dense copy of the weights (bit-exact against the oracle, test_gpu_dequant.py) is the
reference.  Bound, of the root of the sum of the products' squares (a single output can cancel): fp32 chains of up to 32 products,
whose rounding errors, 2^-25 of a growing partial sum each, add as squares to 2^-25 * sqrt(32 / 2) of the sub-block's, three roundings for
scales and result, all else in fp64; the mins of Q4_K, sums of their own, double it: 2 * 2^-25 * 7 = 4e-7."""
import pytest
import torch

from tattletale_amd import QuantLinear, formats as F
from tattletale_amd import qlinear as QL

from util import DEV, packed_to_dev, random_blocks

pytestmark = pytest.mark.gpu
DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
BLOCK = {F.Q8_0: 32, F.Q4_K: 256, F.Q6_K: 256}
NAMES = {F.Q8_0: "q8_0", F.Q4_K: "q4_k", F.Q6_K: "q6_k"}
TOL = 4e-7

# rows shorter than a wavefront's 1024 values, exactly one, one block more, two and several wavefronts, the longest; outputs around
# the groups of two, four and eight rows
SHAPES = [(1, 256), (3, 768), (255, 1024), (513, 1280), (777, 2048), (130, 3072), (17, 5120), (66, 8192), (9, 16384)]


def layer(fmt, n_out, n_in, bias=None):
    w = packed_to_dev(random_blocks(fmt, n_out * (n_in // BLOCK[fmt]), seed=n_out + n_in))
    return QuantLinear.init(w, fmt, n_in, n_out, bias=bias, precision=F.PRECISION_F32_SCALES)


def dense(lay):
    return QL.dequantize(lay.format, lay.qweight, lay.out_features, lay.in_features).double()


def rows(fmt, xk, n_in):
    """Activation rows that the kernel takes on small matrices."""
    if n_in > 8192:
        return [1]
    if fmt == F.Q8_0 or (xk == "f32" and n_in <= 4096):
        return [1, 2, 3, 4, 5, 8]
    return [1, 2, 3, 4]


@pytest.mark.parametrize("xk", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("fmt,n_out,n_in", [(f, o, i) for f in BLOCK for o, i in SHAPES] + [(F.Q8_0, 70, 96), (F.Q8_0, 70, 1056)])
def test_edges(fmt, n_out, n_in, xk):
    gen = torch.Generator(DEV).manual_seed(n_out)
    bias = torch.randn(n_out, device=DEV, generator=gen).to(DT[xk])
    lay = layer(fmt, n_out, n_in, bias)
    plain = QuantLinear.init(lay.qweight, fmt, n_in, n_out, precision=F.PRECISION_F32_SCALES)
    wd = dense(lay)
    for m in rows(fmt, xk, n_in):
        family = "gemv_generic" if fmt == F.Q8_0 or xk == "f32" else ("gemv_dot2" if m == 1 else "gemv_dot2_multi")
        assert lay.route(m, DT[xk], torch.float32) == family
        assert lay.route_detail(m, DT[xk], torch.float32) == "gemv_short"
        x = torch.randn(m, n_in, device=DEV, generator=gen).to(DT[xk])
        ref = x.double() @ wd.T + bias.double()
        y = lay.forward(x, out_dtype=torch.float32)
        size = ((x.double() ** 2) @ (wd ** 2).T + bias.double() ** 2).sqrt()
        assert ((y.double() - ref).norm(dim=-1) / size.norm(dim=-1)).max().item() <= TOL, m
        if xk != "f32":      # 16-bit outputs are the same sums, rounded once
            assert torch.equal(lay.forward(x), y.to(DT[xk]))
        # unit vectors: the dequantized columns, bit for bit (up to the sign of a zero)
        cols = ([n_in - 1, 0, 15, 16, 17, n_in - 16, n_in // 2, n_in - 31])[:m]
        e = torch.zeros(m, n_in, device=DEV, dtype=DT[xk])
        e[torch.arange(m), torch.tensor(cols)] = 1.0
        assert torch.equal(plain.forward(e, out_dtype=torch.float32) + 0.0, wd[:, cols].T.float() + 0.0), m


@pytest.mark.parametrize("n_out,n_in", [(6144, 1024), (2304, 768), (4096, 1024), (1536, 5120)])
@pytest.mark.parametrize("fmt,xk,m", [(F.Q8_0, "f32", 1), (F.Q8_0, "bf16", 4), (F.Q4_K, "bf16", 1), (F.Q6_K, "f16", 1), (F.Q6_K, "bf16", 2), (F.Q4_K, "f32", 2)])
def test_more_wavefronts_than_two_rows_each(fmt, xk, m, n_out, n_in):
    lay = layer(fmt, n_out, n_in)
    x = torch.randn(m, n_in, device=DEV, generator=torch.Generator(DEV).manual_seed(n_out)).to(DT[xk])
    ref = x.double() @ dense(lay).T
    y = lay.forward(x, out_dtype=torch.float32)
    bound = TOL if (fmt, n_out) != (F.Q4_K, 1536) else 2e-6     # (that one has the packed-dot kernel for 16-bit rows)
    # (16-bit rows of 1536 x 5120 stay with the packed-dot kernels)
    other = {(F.Q4_K, 1): "gemv_dot2", (F.Q6_K, 2): "gemv_dot2_multi"}.get((fmt, m)) if n_out == 1536 else None
    assert lay.route_detail(m, DT[xk], torch.float32) == ("gemv_short" if other is None or xk == "f32" else other)
    assert ((y.double() - ref).norm(dim=-1) / ref.norm(dim=-1)).max().item() <= bound


@pytest.mark.parametrize("fmt", list(BLOCK), ids=list(NAMES.values()))
@pytest.mark.parametrize("xk", ["f32", "bf16"])
def test_non_finite_rows_stay_alone_and_large_values_are_exact(fmt, xk):
    n_out, n_in, m = 300, 1280, 4
    lay = layer(fmt, n_out, n_in)
    x = torch.randn(m, n_in, device=DEV, generator=torch.Generator(DEV).manual_seed(3)).to(DT[xk])
    want = lay.forward(x, out_dtype=torch.float32)
    for bad in (float("inf"), float("nan")):
        z = x.clone()
        z[2, 700] = bad
        y = lay.forward(z, out_dtype=torch.float32)
        assert not torch.isfinite(y[2]).any() and torch.equal(y[[0, 1, 3]], want[[0, 1, 3]])
    # one value whose products with scale and quant stay finite, whatever its own size: the column, bit for bit
    z = torch.zeros_like(x)
    z[:, 513] = 2.0 ** 112
    assert torch.equal(lay.forward(z, out_dtype=torch.float32) + 0.0, (dense(lay)[:, 513] * 2.0 ** 112).float().expand(m, -1) + 0.0)


def positive_rows(fmt, n_out, n_in):
    """Packed rows whose weights are all above zero, and the byte range of a block's scale."""
    blocks = n_out * (n_in // BLOCK[fmt])
    one = torch.tensor([0.01], dtype=torch.float16).view(torch.uint8)
    if fmt == F.Q8_0:
        b = torch.full((blocks, 34), 3, dtype=torch.uint8)
        b[:, :2] = one
        return b, slice(0, 2)
    if fmt == F.Q4_K:
        b = torch.full((blocks, 144), 0x11, dtype=torch.uint8)       # scales and quants above zero, d_min zero
        b[:, :2], b[:, 2:4] = one, 0
        return b, slice(0, 2)
    b = torch.full((blocks, 210), 0xFF, dtype=torch.uint8)           # q - 32 = 31
    b[:, 192:208], b[:, 208:210] = 5, one
    return b, slice(208, 210)


@pytest.mark.parametrize("n_in", [256, 1024, 1280, 3072, 4352])
@pytest.mark.parametrize("m", [1, 2, 3])
@pytest.mark.parametrize("xk", ["f32", "bf16"])
@pytest.mark.parametrize("fmt", list(BLOCK), ids=list(NAMES.values()))
def test_infinite_block_scale_gives_infinity(fmt, xk, m, n_in):
    """Lanes past the end of a row read its first block: its scale may be anything."""
    n_out, row = 24, 5
    b, scale = positive_rows(fmt, n_out, n_in)
    b[row * (n_in // BLOCK[fmt]), scale] = torch.tensor([float("inf")], dtype=torch.float16).view(torch.uint8)
    lay = QuantLinear.init(b.to(DEV).view(-1), fmt, n_in, n_out, precision=F.PRECISION_F32_SCALES)
    x = torch.ones(m, n_in, device=DEV, dtype=DT[xk])
    y = lay.forward(x, out_dtype=torch.float32)
    assert torch.equal(torch.isposinf(y), torch.isposinf(x.double() @ dense(lay).T))
    assert torch.isposinf(y[:, row]).all() and torch.isfinite(y).sum().item() == m * (n_out - 1)
