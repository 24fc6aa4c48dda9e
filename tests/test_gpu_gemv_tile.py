"""The Q6_K decode kernel for one to eight rows (route ``gemv_tile``): edges of its tiles (4, 8 and 16 weight
rows by 4, 2 and 1 blocks), of the workgroups' shares, of the rows' ends and of the matrix's end.

The float64 product over the library's own dense copy of the weights (bit-exact against the oracle, test_gpu_dequant.py) is
the reference.  Bound: products are exact, a sum over a sub-block of 16 in fp32 carries the offset 256 + 63 of the quants beside
weights of up to 32 in magnitude, so its rounding is 2^-24 * 320 / 32 per addition at worst, 6e-7 of the largest term; over
random signs and many sub-blocks the relative 2-norm stays below 2e-6 (3e-7 measured)."""
import numpy as np
import pytest
import torch

from tattletale_amd import QuantLinear, formats as F
from tattletale_amd import qlinear as QL

from util import DEV, packed_to_dev, random_blocks

pytestmark = pytest.mark.gpu
DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def layer(n_out, n_in, bias=None):
    w = packed_to_dev(random_blocks(F.Q6_K, n_out * (n_in // 256), seed=n_out + n_in))
    return QuantLinear.init(w, F.Q6_K, n_in, n_out, bias=bias, precision=F.PRECISION_F32_SCALES)


def dense(lay):
    return QL.dequantize(F.Q6_K, lay.qweight, lay.out_features, lay.in_features).double()


# rows of 1, 2, 3, 5, 9 and 27 blocks (an odd and an even number of blocks in all: where the matrix ends inside a dword),
# row counts that are and are not whole tiles
SHAPES = [(33337, 256), (33344, 256), (66700, 512), (11115, 768), (45003, 768), (6671, 1280), (30006, 1280), (3709, 2304), (1237, 6912),
          (2451, 6912), (3001, 6912), (48001, 1024)]
ROWS = [("f32", 1), ("bf16", 1), ("f16", 1), ("bf16", 2), ("f16", 2), ("f16", 3), ("bf16", 4), ("f16", 5), ("bf16", 8)]


def another_kernel(n_out, n_in, xk, m):
    """Calls of the lists above that another decode kernel serves faster: small matrices, few rows of weights, rows of weights too
    long for eight rows of activations."""
    if xk == "f32":
        return False
    if m == 1:
        return n_out * n_in < 14_000_000 or n_out == 1237
    return n_in == 6912 and (n_out == 1237 or m > 4)


@pytest.mark.parametrize("n_out,n_in,xk,m", [(o, i, x, m) for o, i in SHAPES for x, m in ROWS if not another_kernel(o, i, x, m)])
def test_tile_edges(n_out, n_in, xk, m):
    gen = torch.Generator(DEV).manual_seed(n_out)
    bias = torch.randn(n_out, device=DEV, generator=gen).to(DT[xk])
    lay = layer(n_out, n_in, bias)
    assert lay.route(m, DT[xk], torch.float32) == "gemv_tile"
    x = torch.randn(m, n_in, device=DEV, generator=gen).to(DT[xk])
    wd = dense(lay)
    ref = x.double() @ wd.T + bias.double()
    y = lay.forward(x, out_dtype=torch.float32)
    assert ((y.double() - ref).norm(dim=-1) / ref.norm(dim=-1)).max().item() <= 2e-6
    if xk != "f32":      # 16-bit outputs are the same sums, rounded once
        assert torch.equal(lay.forward(x), y.to(DT[xk]))
    # unit vectors: the dequantized columns, bit for bit (without the bias)
    lay = QuantLinear.init(lay.qweight, F.Q6_K, n_in, n_out, precision=F.PRECISION_F32_SCALES)
    cols = [0, n_in - 1, 15, 16, 127, 128, n_in - 256, n_in - 17][:m] if m > 1 else [n_in - 1]
    e = torch.zeros(m, n_in, device=DEV, dtype=DT[xk])
    e[torch.arange(m), torch.tensor(cols)] = 1.0
    assert torch.equal(lay.forward(e, out_dtype=torch.float32), wd[:, cols].T.float() + 0.0)


@pytest.mark.parametrize("n_out,n_in,xk", [(1024, 40960, "bf16"), (1024, 41216, "f16"), (1027, 41472, "bf16"), (777, 44800, "f16")])
def test_rows_that_leave_little_lds(n_out, n_in, xk):
    """Rows on both sides of the length where a tile of two blocks along K no longer fits beside the activations.  Bound: the sums
    of 2^-24 * 320 / 32 per addition of the module's docstring, over more sub-blocks: the same 2e-6."""
    lay = layer(n_out, n_in)
    assert lay.route(1, DT[xk], torch.float32) == "gemv_tile"
    x = torch.randn(1, n_in, device=DEV, generator=torch.Generator(DEV).manual_seed(n_out)).to(DT[xk])
    ref = x.double() @ dense(lay).T
    y = lay.forward(x, out_dtype=torch.float32)
    assert ((y.double() - ref).norm() / ref.norm()).item() <= 2e-6


@pytest.mark.parametrize("n_out,n_in", [(30006, 1280), (5120, 5120), (4096, 7680)])
@pytest.mark.parametrize("m", [1, 2])
def test_fp32_rows_whose_mean_is_not_zero(n_out, n_in, m):
    """fp32 activations meet q - 32 itself, so their mean leaves nothing behind.  Bound: a product's first terms are whole
    multiples of a common power of two and their sums exact, what is rounded are the running sums, once a tile and lane: at
    most 40 additions of a growing sum (in the square mean a third of its end), each off by 0.29 ulp, 0.29 * 2^-23 * sqrt(40 / 3) =
    1.3e-7 (with an offset in the sums: 1.5e-7 to 2.0e-7)."""
    lay = layer(n_out, n_in)
    assert lay.route(m, torch.float32, torch.float32) == "gemv_tile"
    x = torch.randn(m, n_in, device=DEV, generator=torch.Generator(DEV).manual_seed(n_in)) + 1
    ref = x.double() @ dense(lay).T
    y = lay.forward(x)
    assert ((y.double() - ref).norm(dim=-1) / ref.norm(dim=-1)).max().item() <= 1.3e-7


def test_an_infinite_fp32_value_gives_infinities():
    n_out, n_in = 30006, 1280
    lay = layer(n_out, n_in)
    wd = dense(lay)
    x = torch.randn(2, n_in, device=DEV, generator=torch.Generator(DEV).manual_seed(7))
    x[0, 300], x[1, 1279] = float("inf"), float("-inf")
    assert lay.route(2, torch.float32, torch.float32) == "gemv_tile"
    for y, z in ((lay.forward(x), x), (lay.forward(x[:1]), x[:1])):
        want = (z.double() @ wd.T).float()                     # infinite times zero: not a number
        assert torch.equal(torch.nan_to_num(y, nan=0.0, posinf=1.0, neginf=-1.0), torch.nan_to_num(want, nan=0.0, posinf=1.0, neginf=-1.0))
        assert torch.equal(y.isnan(), want.isnan()) and want.isinf().float().mean() > 0.9


@pytest.mark.parametrize("m", [1, 2, 4, 8])
@pytest.mark.parametrize("size", [3e38, 1e36, 1e-34])
def test_bf16_activations_at_both_ends_of_the_range(m, size):
    """Whole rows of activations of one magnitude, signs at random: finite results, as exact as others.  The block scales are
    turned down (up for small ones), so that the results lie inside of the type.  Bound: the module's; for 1e-34 the products,
    divided by 4096, end at 2^-149 and are 2^-126 and larger: 23 bits."""
    n_out, n_in = 30006, 1280
    raw = random_blocks(F.Q6_K, n_out * (n_in // 256), seed=1).reshape(-1, 210)
    raw[:, 208:210] = np.frombuffer(np.float16(1e-6 if size > 1 else 1e3).tobytes(), np.uint8)
    lay = QuantLinear.init(packed_to_dev(raw.reshape(-1)), F.Q6_K, n_in, n_out, precision=F.PRECISION_F32_SCALES)
    assert lay.route(m, torch.bfloat16, torch.float32) == "gemv_tile"
    sign = torch.randint(0, 2, (m, n_in), device=DEV, generator=torch.Generator(DEV).manual_seed(m)) * 2.0 - 1
    x = (sign * size).to(torch.bfloat16)
    x[0] = x[0].abs()
    ref = x.double() @ dense(lay).T
    y = lay.forward(x, out_dtype=torch.float32)
    assert torch.isfinite(ref.float()).all() and torch.isfinite(y).all()
    assert ((y.double() - ref).norm(dim=-1) / ref.norm(dim=-1)).max().item() <= 2e-6


def test_every_size_of_route_is_reached():
    """Each of the kernel's forms runs at least on these (16-bit one row by four and by two blocks, two, four and eight rows; one and
    two fp32 rows)."""
    for n_out, n_in, m, dt in [(33337, 256, 1, "f32"), (48001, 1024, 1, "bf16"), (66700, 512, 1, "bf16"), (2451, 6912, 1, "bf16"),
                               (66700, 512, 2, "f16"), (33337, 256, 4, "bf16"), (6671, 1280, 8, "bf16"), (30006, 1280, 2, "f32")]:
        assert layer(n_out, n_in).route(m, DT[dt], torch.float32) == "gemv_tile", (n_out, n_in, m, dt)


@pytest.mark.parametrize("xk,m", [("f32", 1), ("bf16", 1), ("f16", 2), ("bf16", 4), ("f16", 8)])
def test_non_finite_rows_and_large_values(xk, m):
    n_out, n_in = 30006, 1280
    lay = layer(n_out, n_in)
    assert lay.route(m, DT[xk], torch.float32) == "gemv_tile"
    x = torch.randn(m, n_in, device=DEV, generator=torch.Generator(DEV).manual_seed(3)).to(DT[xk])
    want = lay.forward(x, out_dtype=torch.float32)
    for bad in (float("inf"), float("nan")):
        z = x.clone()
        z[m - 1, 700] = bad
        y = lay.forward(z, out_dtype=torch.float32)
        assert not torch.isfinite(y[m - 1]).any()
        assert torch.equal(y[: m - 1], want[: m - 1])
    if xk == "f32":      # one value near the top of the range: its products with quants of up to 63 stay finite
        z = torch.zeros_like(x)
        z[0, 700] = 5e36
        ref = z.double() @ dense(lay).T
        fits = ref.abs() < 3e38
        y = lay.forward(z)
        assert fits.float().mean() > 0.5 and torch.isfinite(y[fits]).all()
        assert ((y.double() - ref)[fits].norm() / ref[fits].norm()).item() <= 1e-6
