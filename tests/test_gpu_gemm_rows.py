"""The few-row GEMM over many weight rows, and over any number of them (ttq_gemm_rows.hip): edges of its blocks of 16 weight rows
and 16 tokens, of the shares of workgroups and passes, rows of one block, the end of the matrix inside a dword.

Reference: the float64 product over the library's own dense copy of the weights.  Bound: every weight is rounded once to the
activation type, by at most u = 2^-8 (bf16, 8 significant bits) or 2^-11 (fp16, 11 bits) of its size, fp32 activations to fp16 as well; the roundings are
independent and their standard deviation is below 0.6 u |x w| (0.6 sqrt(2) u for fp32), so that of an output is below
0.6 u sqrt(sum (x w)^2); five of them, 3 u (4.2 u), hold for the 10^7 outputs here."""
import pytest
import torch

from tattletale_amd import QuantLinear, formats as F
from tattletale_amd import qlinear as QL

from util import DEV, packed_to_dev, random_blocks

pytestmark = pytest.mark.gpu
DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
TOL = {"bf16": 3 * 2.0 ** -8, "f16": 3 * 2.0 ** -11, "f32": 4.2 * 2.0 ** -11}


def run(fmt, n_out, n_in, m, xk, bias=True, route=None):
    gen = torch.Generator(DEV).manual_seed(n_out + m)
    w = packed_to_dev(random_blocks(fmt, n_out * (n_in // 256), seed=n_out + n_in))
    b = torch.randn(n_out, device=DEV, generator=gen).to(DT[xk]) if bias else None
    lay = QuantLinear.init(w, fmt, n_in, n_out, bias=b)
    if route is not None:
        assert lay.route(m, DT[xk], torch.float32) == route
    x = torch.randn(m, n_in, device=DEV, generator=gen).to(DT[xk])
    wd = QL.dequantize(fmt, w, n_out, n_in).double()
    ref = x.double() @ wd.T + (b.double() if bias else 0)
    y = lay.forward(x, out_dtype=torch.float32)
    size = ((x.double() ** 2) @ (wd ** 2).T).sqrt()
    err = ((y.double() - ref).abs() / size.clamp_min(1e-30)).max().item()
    assert err <= TOL[xk], err
    if xk != "f32":
        assert torch.equal(lay.forward(x), y.to(DT[xk]))      # 16-bit outputs: the same sums, rounded once
    return lay, x, y


# (fp32 activations: the kernel runs on their scaled fp16 copy wherever the matrix has five blocks of rows to a compute unit, or an
# odd number of them; the route names the copy)
ROUTE = {"bf16": "gemm_rows", "f16": "gemm_rows", "f32": "gemm_skinny_f32_scaled_f16"}
ROWS = [(9, "f16"), (16, "bf16"), (17, "f16"), (33, "bf16"), (48, "f16"), (49, "bf16"), (64, "f16"), (64, "bf16"), (12, "f32"), (50, "f32")]
LARGE = [(20480, 256), (20488, 768), (65544, 512), (33000, 1280), (20488, 2304)]


def decodes(fmt, n_out, n_in, m, xk):
    """Calls of the lists above that passes of the decode kernels serve faster."""
    if fmt == F.Q4_K:
        return xk != "f32" and (m <= 16 or (n_out == 65544 and xk == "f16" and m < 64))
    return (n_out, n_in, m) == (20480, 256, 9)


@pytest.mark.parametrize("fmt,n_out,n_in,m,xk", [(f, o, i, m, x) for f in (F.Q4_K, F.Q6_K) for o, i in LARGE for m, x in ROWS
                                                 if not decodes(f, o, i, m, x)])
def test_many_weight_rows(fmt, n_out, n_in, m, xk):
    run(fmt, n_out, n_in, m, xk, route=ROUTE[xk])


@pytest.mark.parametrize("fmt,n_out,n_in,m", [(F.Q6_K, o, i, m) for o, i in [(20487, 768), (65537, 512), (20481, 2304)] for m in (9, 17, 33, 64)] +
                         [(F.Q4_K, o, i, m) for o, i in [(20487, 768), (65537, 512), (20481, 2304)] for m in (33, 64)] +
                         [(f, o, i, m) for o in (1, 3, 15, 17, 100, 255, 1003, 4097) for f, i, m in
                          [(F.Q4_K, 256, 17), (F.Q4_K, 768, 40), (F.Q4_K, 1024, 64), (F.Q6_K, 256, 32), (F.Q6_K, 768, 48), (F.Q6_K, 1024, 64)]])
def test_any_number_of_outputs(fmt, n_out, n_in, m):
    run(fmt, n_out, n_in, m, "bf16", route="gemm_rows")


@pytest.mark.parametrize("fmt,n_out,m", [(F.Q4_K, 15, 64), (F.Q4_K, 1003, 64), (F.Q4_K, 4097, 31), (F.Q6_K, 1003, 64), (F.Q6_K, 4097, 31)])
def test_any_number_of_outputs_fp32(fmt, n_out, m):
    run(fmt, n_out, 1024, m, "f32", route=ROUTE["f32"])


@pytest.mark.parametrize("fmt", [F.Q4_K, F.Q6_K])
@pytest.mark.parametrize("n_out", [1, 3, 15, 17, 100, 255, 1003, 4097])
@pytest.mark.parametrize("m,xk", [(5, "f16"), (16, "f16"), (31, "f32"), (64, "f16"), (7, "bf16"), (40, "bf16")])
def test_outputs_that_are_not_whole_groups_of_eight(fmt, n_out, m, xk):
    """The same bounds for the calls around them, most of which the decode kernels take: fp16 ones with such a number of outputs
    decode at every row count."""
    run(fmt, n_out, 1024, m, xk)


@pytest.mark.parametrize("fmt", [F.Q4_K, F.Q6_K])
def test_non_finite_rows_stay_alone_and_rows_do_not_depend_on_their_neighbours(fmt):
    lay, x, y = run(fmt, 20488, 1280, 21, "f16", bias=False, route="gemm_rows")
    z = x.clone()
    z[20, 1279] = float("inf")
    got = lay.forward(z, out_dtype=torch.float32)
    assert not torch.isfinite(got[20]).any() and torch.equal(got[:20], y[:20])
    assert lay.route(18, torch.float16, torch.float32) == "gemm_rows"
    assert torch.equal(lay.forward(x[:18], out_dtype=torch.float32), y[:18])


@pytest.mark.parametrize("n_out,n_in", [(20487, 1280), (33337, 256), (3001, 5120)])
@pytest.mark.parametrize("m", [9, 16, 33, 48, 64, 70])
def test_exact_form(n_out, n_in, m):
    """fp16 rows that decode (an odd number of outputs): nothing is rounded before the fp32 sums.  Bound: a group's sum starts at
    -288 sum(x) and adds (256 + q) x, so a rounding is at most 2^-24 of 288 scale |x| sqrt(16) for random x, some eight of them to a
    group (its sum of x, the start, the products' tree, the scale, the row's sum); the groups' errors add as squares.  Times 4 for
    the worst of up to 2 million outputs."""
    gen = torch.Generator(DEV).manual_seed(m)
    raw = random_blocks(F.Q6_K, n_out * (n_in // 256), seed=n_out)
    w = packed_to_dev(raw)
    lay = QuantLinear.init(w, F.Q6_K, n_in, n_out, precision=F.PRECISION_F32_SCALES)
    assert lay.route(m, torch.float16, torch.float32) == ("gemv_tile" if (n_out, m) == (3001, 9) else "gemm_rows_exact")
    x = torch.randn(m, n_in, device=DEV, generator=gen).half()
    wd = QL.dequantize(F.Q6_K, w, n_out, n_in).double()
    blk = w.view(-1, 210)
    scale = blk[:, 192:208].contiguous().view(torch.int8).double() * blk[:, 208:210].contiguous().view(torch.float16).double()
    scale = scale.view(n_out, n_in // 16).repeat_interleave(16, dim=1)
    bound = 4 * 8 ** 0.5 * 2.0 ** -24 * 288 * ((x.double() ** 2) @ (scale ** 2).T).sqrt()
    y = lay.forward(x, out_dtype=torch.float32)
    assert bool(((y.double() - x.double() @ wd.T).abs() <= bound).all())
    e = torch.zeros(m, n_in, device=DEV, dtype=torch.float16)
    cols = torch.randint(0, n_in, (m,), device=DEV, generator=gen)
    e[torch.arange(m, device=DEV), cols] = 1.0
    assert torch.equal(lay.forward(e, out_dtype=torch.float32), wd[:, cols].T.float() + 0.0)


@pytest.mark.parametrize("m", [2, 3, 4])
def test_a_few_fp32_rows_of_any_number_of_outputs(m):
    """Two fp32 rows to a pass of the integer decode kernel, as six bf16 ones."""
    n_out, n_in = 11115, 768
    w = packed_to_dev(random_blocks(F.Q6_K, n_out * (n_in // 256), seed=5))
    lay = QuantLinear.init(w, F.Q6_K, n_in, n_out)
    assert lay.route(m, torch.float32) == "gemv_tile"
    x = torch.randn(m, n_in, device=DEV, generator=torch.Generator(DEV).manual_seed(m))
    ref = x.double() @ QL.dequantize(F.Q6_K, w, n_out, n_in).double().T
    y = lay.forward(x)
    assert ((y.double() - ref).norm(dim=-1) / ref.norm(dim=-1)).max().item() <= 2e-6
    assert torch.equal(y[:1], lay.forward(x[:2])[:1])
