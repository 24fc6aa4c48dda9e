"""Which kernel family the dispatcher picks (``ttq_route``): the benchmark configurations, the gate||up shape and
the attention projections reach the kernels built for them.  A pure host query: no GPU is needed (without a visible
device the dispatcher assumes 256 compute units, the MI355X count)."""
import ctypes as C

import pytest

from tattletale_amd import _lib
from tattletale_amd._lib import QLinearStruct, F32, F16, BF16, Q8_0, Q4_K, Q6_K, EXL3


def route(fmt, n_out, n_in, m, x_dtype, y_dtype, bits=0, precision=_lib.PRECISION_AUTO):
    L = _lib.lib()
    st = QLinearStruct(format=fmt, n_out=n_out, n_in=n_in, bits=bits, codebook=_lib.CB_MCG, precision=precision)
    r = L.ttq_route(C.byref(st), m, x_dtype, y_dtype)
    assert r >= 0, r
    name = L.ttq_route_name(r).decode()
    assert _lib.ROUTE[name] == r
    return name


# (what, format, n_out, n_in, m, x dtype, y dtype, bits, kernel family)
PINNED = [
    ("config 1: Q8_0 GEMV 4096x4096, fp32 x", Q8_0, 4096, 4096, 1, F32, F32, 0, "gemv_q8_stream"),
    ("config 2: Q4_K GEMV 14336x4096 (headline)", Q4_K, 14336, 4096, 1, BF16, F32, 0, "gemv_q4k_stream"),
    ("config 3: Q6_K GEMV 128256x4096 (LM head)", Q6_K, 128256, 4096, 1, BF16, F32, 0, "gemv_q6k_stream"),
    ("config 4: Q4_K GEMM M=64", Q4_K, 14336, 4096, 64, BF16, BF16, 0, "gemm_skinny"),
    ("config 4: Q4_K GEMM M=512 (headline)", Q4_K, 14336, 4096, 512, BF16, BF16, 0, "gemm_pc_packed"),
    ("config 4: Q4_K GEMM M=2048", Q4_K, 14336, 4096, 2048, BF16, BF16, 0, "gemm_pc_packed"),
    ("config 5: EXL3 3-bit GEMV 4096x4096", EXL3, 4096, 4096, 1, F16, F32, 3, "exl3_gemv_sliced"),
    ("gate||up 28672x4096, decode", Q4_K, 28672, 4096, 1, BF16, F32, 0, "gemv_q4k_stream"),
    ("q / o projection 4096x4096, decode", Q4_K, 4096, 4096, 1, BF16, F32, 0, "gemv_q4k_stream"),
    ("k / v projection 1024x4096, decode", Q4_K, 1024, 4096, 1, BF16, F32, 0, "gemv_dot2"),
    ("down projection 4096x14336, decode", Q4_K, 4096, 14336, 1, BF16, F32, 0, "gemv_q4k_slice"),
    ("q / o projection, prefill 512 rows", Q4_K, 4096, 4096, 512, BF16, BF16, 0, "gemm_pc"),
    ("down projection, prefill 512 rows", Q4_K, 4096, 14336, 512, BF16, BF16, 0, "gemm_pc_packed_split_k"),
    ("gate||up weight as a plain GEMM, 2048 rows (eight full rounds of tiles)", Q4_K, 28672, 4096, 2048, BF16, BF16, 0, "gemm_pc_packed"),
    ("headline shape, 4096 rows", Q4_K, 14336, 4096, 4096, BF16, BF16, 0, "gemm_pc_packed"),
    ("down projection, prefill 1024 rows", Q4_K, 4096, 14336, 1024, BF16, BF16, 0, "gemm_pc_packed"),
    ("two rows of the headline shape", Q4_K, 14336, 4096, 2, BF16, F32, 0, "gemv_q4k_stream4"),
    ("three rows of the LM head", Q6_K, 128256, 4096, 3, BF16, F32, 0, "gemv_q6k_stream4"),
    ("trellis layer, prefill 512 rows", EXL3, 4096, 4096, 512, F16, F32, 3, "exl3_gemm"),
    ("fp16 activations, prefill 512 rows of the headline shape", Q4_K, 14336, 4096, 512, F16, F16, 0, "gemm_pc_f16"),
    ("fp32 activations, prefill 512 rows of the headline shape", Q4_K, 14336, 4096, 512, F32, F32, 0, "gemm_pc_f32_scaled_f16"),
    ("fp16 activations, 64 rows", Q4_K, 14336, 4096, 64, F16, F16, 0, "gemm_skinny_chunked"),
    ("fp32 activations, 8 rows of the headline shape", Q4_K, 14336, 4096, 8, F32, F32, 0, "gemm_skinny_f32_scaled_f16"),
    ("fp32 activations, 64 rows of the down projection", Q6_K, 4096, 14336, 64, F32, F32, 0, "gemm_skinny_f32_scaled_f16"),
    ("down projection of a 53248-wide MLP, decode", Q4_K, 16384, 53248, 1, BF16, F32, 0, "gemv_dot2"),
    ("rows beyond 65536 values", Q4_K, 4096, 65536 + 256, 1, BF16, F32, 0, "gemv_long"),
    ("fp32 activations beyond 16384 values", Q8_0, 4096, 16384 + 32, 1, F32, F32, 0, "gemv_long"),
    ("6-bit projection 5120x5120, decode", Q6_K, 5120, 5120, 1, F16, F16, 0, "gemv_tile"),
    ("LM head of an odd vocabulary, decode", Q6_K, 32003, 5120, 1, F16, F32, 0, "gemv_tile"),
    ("LM head, eight rows", Q6_K, 128256, 4096, 8, BF16, F32, 0, "gemv_tile"),
    ("6-bit projection, one fp32 row", Q6_K, 5120, 5120, 1, F32, F32, 0, "gemv_tile"),
    ("LM head of an odd vocabulary, 43 fp16 rows", Q6_K, 32003, 5120, 43, F16, F32, 0, "gemm_rows_exact"),
    ("LM head, 43 fp16 rows", Q6_K, 152064, 3584, 43, F16, F32, 0, "gemm_rows"),
    ("gate||up of a wide MLP, 43 fp16 rows", Q4_K, 37888, 3584, 43, F16, F16, 0, "gemm_rows"),
    ("LM head of an odd vocabulary, 33 bf16 rows", Q6_K, 32003, 5120, 33, BF16, F32, 0, "gemm_rows"),
    # few rows of weights: the kernels that give a wavefront a row of its own, or the tiled one
    ("short 6-bit matrix, four rows", Q6_K, 1536, 4096, 4, BF16, BF16, 0, "gemv_dot2_multi"),
    ("short 6-bit matrix, two rows", Q6_K, 758, 8192, 2, F16, F16, 0, "gemv_dot2_multi"),
    ("short 6-bit matrix, long rows, decode", Q6_K, 1280, 13568, 1, BF16, BF16, 0, "gemv_dot2"),
    ("short 6-bit matrix, long rows, one fp32 row", Q6_K, 896, 14336, 1, F32, F32, 0, "gemv_generic"),
    ("short 6-bit matrix, three fp32 rows", Q6_K, 2560, 2560, 3, F32, F32, 0, "gemv_generic"),
    ("6-bit projection 3072x4096, one fp32 row", Q6_K, 3072, 4096, 1, F32, F32, 0, "gemv_generic"),
    ("odd number of outputs, 37 rows", Q4_K, 1145, 4096, 37, BF16, BF16, 0, "gemm_pc_split_k"),
    ("odd number of outputs, 100 rows", Q6_K, 638, 768, 100, BF16, BF16, 0, "gemm_pc"),
    ("many rows of weights, 278 fp16 rows", Q6_K, 26816, 256, 278, F16, F16, 0, "gemm_pc_f16"),
]


@pytest.mark.parametrize("what,fmt,n_out,n_in,m,xd,yd,bits,want", PINNED, ids=[p[0] for p in PINNED])
def test_benchmark_and_model_shapes_reach_their_kernels(what, fmt, n_out, n_in, m, xd, yd, bits, want):
    assert route(fmt, n_out, n_in, m, xd, yd, bits) == want


def test_many_exact_rows_of_a_small_matrix_take_one_launch():
    for n_out, n_in, m, xd in ((960, 6656, 267, F32), (1024, 6144, 8, F32), (2560, 4096, 64, F32), (1024, 6144, 2, F32)):
        assert route(Q6_K, n_out, n_in, m, xd, F32, precision=_lib.PRECISION_F32_SCALES) == "gemv_generic"
    assert route(Q6_K, 1536, 4096, 32, BF16, BF16, precision=_lib.PRECISION_F32_SCALES) == "gemv_dot2_multi"
    for n_out, n_in, m, xd in ((131071, 512, 221, F32), (5120, 5120, 64, F32), (5120, 5120, 64, BF16), (3072, 4096, 32, BF16)):
        assert route(Q6_K, n_out, n_in, m, xd, F32, precision=_lib.PRECISION_F32_SCALES) == "gemv_tile"


def test_precision_flags_steer_the_route():
    # fp32 activations: decode kernels for a handful of rows, then the fp16 matrix-core kernels over a copy scaled
    # row by row -- the few-row kernel, then the prefill GEMM -- (the 1e-3 class either way), never a bf16 copy by default
    for m in (1, 2):
        assert route(Q4_K, 14336, 4096, m, F32, F32).startswith("gemv_")
    assert route(Q6_K, 14336, 4096, 1, F32, F32).startswith("gemv_")             # a single row always decodes
    assert route(Q6_K, 14336, 4096, 2, F32, F32) == "gemm_skinny_f32_scaled_f16"  # no decode kernel of several fp32 rows
    for m in (4, 5, 16, 64):
        assert route(Q4_K, 14336, 4096, m, F32, F32) == "gemm_skinny_f32_scaled_f16"
        assert route(Q4_K, 14336, 4096, m, F32, F32, precision=_lib.PRECISION_F32_SCALES).startswith("gemv_")
    for m in (65, 255, 256, 600, 4096):
        assert route(Q4_K, 14336, 4096, m, F32, F32) == "gemm_pc_f32_scaled_f16"
        assert route(Q4_K, 14336, 4096, m, F32, F32, precision=_lib.PRECISION_F32_SCALES).startswith("gemv_")
    # fp16 activations: their own matrix-core kernels (few rows; the fp16 form of the prefill GEMM), never a bf16
    # copy, whatever the layer allows
    assert route(Q4_K, 14336, 4096, 40, F16, F16) == "gemm_skinny_chunked"
    for prec in (_lib.PRECISION_AUTO, _lib.PRECISION_BF16_OK):
        assert route(Q4_K, 14336, 4096, 256, F16, F16, precision=prec) == "gemm_pc_f16"
    assert route(Q4_K, 14336, 4096, 256, F16, F16, precision=_lib.PRECISION_F32_SCALES).startswith("gemv_")
    # only a layer that allows it rounds fp32 activations to bf16
    assert route(Q4_K, 14336, 4096, 256, F32, F32, precision=_lib.PRECISION_BF16_OK) == "gemm_pc_bf16_copy"
    assert route(Q4_K, 14336, 4096, 255, F32, F32, precision=_lib.PRECISION_BF16_OK) != "gemm_pc_bf16_copy"
    # F32_SCALES pins the decode kernels for bf16 activations too
    assert route(Q4_K, 14336, 4096, 512, BF16, BF16, precision=_lib.PRECISION_F32_SCALES).startswith("gemv_")
    assert route(EXL3, 4096, 4096, 512, F16, F32, bits=3, precision=_lib.PRECISION_F32_SCALES).startswith("exl3_gemv")


def test_the_single_role_gemm_serves_only_activations_beyond_4_gib():
    # every row count of every shape below reaches the few-row or the producer/consumer kernels
    for n_out, n_in in ((28672, 4096), (14336, 4096), (4096, 14336), (128256, 4096), (16384, 256)):
        for m in (65, 300, 1024, 2048, 4096, 8192, 8200, 100000):
            if m * n_in * 2 < (1 << 32):
                assert route(Q4_K, n_out, n_in, m, BF16, BF16) != "gemm_q4k_tiles", (n_out, n_in, m)
    assert route(Q4_K, 48, 256, (1 << 32) // 512, BF16, BF16) == "gemm_q4k_tiles"


def test_every_form_of_the_tile_kernel_that_is_chosen_fits_a_compute_unit():
    """The form of a call (blocks along K to a tile) decides how much LDS it takes; the route query fails for a form that needs more
    than a compute unit has.  Every row length the staged kernels take, matrices on both sides of the forms' rule."""
    L = _lib.lib()
    tile = 0
    for x_dtype, longest in ((F32, 64), (F16, 256), (BF16, 256)):
        for blocks in range(1, longest + 1):
            for n_out in (745, 2600, 8192, 32003):
                for m in (1, 2, 3, 5, 8, 17):
                    st = QLinearStruct(format=Q6_K, n_out=n_out, n_in=256 * blocks, precision=_lib.PRECISION_F32_SCALES)
                    r = L.ttq_route(C.byref(st), m, x_dtype, F32)
                    assert r > 0, (x_dtype, n_out, 256 * blocks, m, r)
                    tile += r == _lib.ROUTE["gemv_tile"]
    assert tile > 1000
    assert route(Q6_K, 1024, 41472, 1, BF16, F32) == route(Q6_K, 8192, 44800, 1, F16, F32) == "gemv_tile"


def test_route_is_a_pure_query():
    L = _lib.lib()
    st = QLinearStruct(format=Q4_K, n_out=14336, n_in=4096)
    assert L.ttq_route(None, 1, BF16, F32) == _lib.ERR_NULL
    assert L.ttq_route(C.byref(st), 1, 9, F32) == _lib.ERR_DTYPE
    assert L.ttq_route(C.byref(st), -1, BF16, F32) == _lib.ERR_SHAPE
    assert L.ttq_route(C.byref(st), 0, BF16, F32) == _lib.ROUTE["none"]         # an empty batch launches nothing
    st.n_in = 100
    assert L.ttq_route(C.byref(st), 1, BF16, F32) == _lib.ERR_SHAPE
    assert L.ttq_route_name(12345) == b"unknown route"
    # the same answer every time, with no buffer behind the layer
    st.n_in = 4096
    assert len({L.ttq_route(C.byref(st), 512, BF16, BF16) for _ in range(5)}) == 1


def detail(fmt, n_out, n_in, m, x_dtype, y_dtype, precision=_lib.PRECISION_AUTO):
    text = C.create_string_buffer(128)
    st = QLinearStruct(format=fmt, n_out=n_out, n_in=n_in, precision=precision)
    r = _lib.lib().ttq_route_detail(C.byref(st), m, x_dtype, y_dtype, text, len(text))
    assert r == _lib.lib().ttq_route(C.byref(st), m, x_dtype, y_dtype) >= 0
    return text.value.decode()


def test_route_detail_names_the_kernel_and_the_tile():
    """Calls of one family that go to different kernels, and the tiled GEMM's launches, told apart."""
    assert detail(Q4_K, 14336, 4096, 1, BF16, F32) == "gemv_q4k_stream"         # a family of one kernel: its name
    assert detail(Q4_K, 1024, 4096, 1, BF16, BF16) == detail(Q8_0, 2048, 1024, 1, F32, F32) == "gemv_short"
    assert detail(Q6_K, 2560, 2560, 3, F32, F32) == detail(Q6_K, 1024, 1024, 2, F16, F16) == "gemv_short"
    assert detail(Q4_K, 16384, 53248, 1, BF16, F32) == "gemv_dot2"
    assert detail(Q6_K, 1536, 4096, 4, BF16, BF16) == "gemv_dot2_multi"
    assert detail(Q4_K, 14336, 4096, 512, BF16, BF16) == "gemm_pc 256x112 packed"
    assert detail(Q4_K, 4096, 4096, 512, BF16, BF16) == "gemm_pc 128x64"
    assert detail(Q4_K, 4096, 14336, 512, BF16, BF16) == "gemm_pc 256x64 k/2 packed"
    assert detail(Q4_K, 14336, 4096, 0, BF16, BF16) == "none (empty call)"


def test_calls_that_are_faster_in_chunks_of_64_rows_stay_there():
    """65 to 184 rows where the tiled kernel's fitted time is too low, and neighbours that do go to tiles."""
    for fmt, n_out, n_in, m, xd, chunks in ((Q6_K, 5440, 6400, 68, F16, True), (Q6_K, 192, 6400, 141, BF16, True), (Q6_K, 864, 9984, 139, BF16, True),
                                            (Q6_K, 4112, 6400, 79, F32, True), (Q8_0, 2608, 6400, 122, F16, True), (Q6_K, 1408, 2560, 102, BF16, False),
                                            (Q6_K, 1008, 7168, 77, BF16, False), (Q8_0, 928, 5376, 72, BF16, False), (Q8_0, 1424, 2048, 160, BF16, False)):
        want = "gemm_skinny_f32_scaled_f16" if xd == F32 else "gemm_skinny_chunked"
        assert (route(fmt, n_out, n_in, m, xd, xd) == want) is chunks, (fmt, n_out, n_in, m)


def test_long_fp32_rows_of_q8_0_at_five_to_eight_rows():
    """The windowed kernel is the faster one from some 7 million weights (rows rounded up to 1024 values) on; bf16 rows are not concerned."""
    exact = _lib.PRECISION_F32_SCALES
    for n_out, n_in, m in ((1289, 5632, 8), (1536, 4608, 7), (1281, 5376, 5)):
        assert detail(Q8_0, n_out, n_in, m, F32, F32, exact) == "gemv_q8_win"
        assert detail(Q8_0, n_out, n_in, m, BF16, F32, exact) == "gemv_short"
    assert detail(Q8_0, 1100, 5632, 8, F32, F32, exact) == detail(Q8_0, 2560, 2560, 8, F32, F32, exact) == "gemv_short"


def test_matrices_that_the_packed_dots_are_faster_on_stay_with_them():
    """bf16 rows with fp32 outputs, whose stores cost the packed dots less; two rows of Q6_K with more than 1024 outputs."""
    for n_out, n_in in ((1536, 4096), (1999, 2560), (1200, 3584)):
        assert detail(Q4_K, n_out, n_in, 1, BF16, F32) == "gemv_dot2"
        assert detail(Q4_K, n_out, n_in, 1, BF16, BF16) == detail(Q4_K, n_out, n_in, 1, F16, F32) == "gemv_short"
    assert detail(Q4_K, 800, 4096, 1, BF16, F32) == detail(Q4_K, 1536, 2048, 1, BF16, F32) == "gemv_short"
    for n_out, n_in in ((1312, 2560), (1090, 4096)):
        assert detail(Q6_K, n_out, n_in, 2, F16, F16) == detail(Q6_K, n_out, n_in, 2, BF16, F32) == "gemv_dot2_multi"
    assert detail(Q6_K, 1000, 2560, 2, F16, F16) == detail(Q6_K, 1312, 2048, 2, F16, F16) == "gemv_short"
    assert detail(Q4_K, 1145, 2816, 4, F16, F16) == "gemv_dot2_multi" and detail(Q4_K, 1145, 2816, 4, F16, F32) == "gemv_short"


def test_long_launches_keep_the_tile_that_was_measured_for_them():
    """Beyond the rows that the fitted times have seen: Q8_0 with more than a few columns reads a packed copy, and another tile than the
    earlier model's has to be a fifth ahead for 16-bit rows."""
    for n_out, n_in, m in ((5184, 512, 16871), (9136, 256, 5868), (4096, 2048, 12000)):
        assert route(Q8_0, n_out, n_in, m, BF16, BF16) == "gemm_pc_packed"
    assert route(Q8_0, 512, 4096, 20000, BF16, BF16) == route(Q8_0, 256, 4096, 16384, BF16, BF16) == "gemm_pc"
    assert detail(Q4_K, 34944, 1024, 5993, BF16, BF16) == detail(Q4_K, 2304, 1536, 3648, BF16, BF16) == "gemm_pc 256x112 packed"
    assert detail(Q4_K, 12288, 1024, 3905, F16, F16) == "gemm_pc 256x112 packed"
    assert detail(Q8_0, 512, 4096, 6338, F16, F16) == "gemm_pc 128x112 packed"
    # and the shortest: two copies along K are kept against one of smaller tiles
    assert detail(Q4_K, 14048, 8192, 62, BF16, BF16) == "gemm_pc 64x112 k/2"


@pytest.mark.parametrize("fmt,n_out,n_in,m", [(Q8_0, 8317, 3072, 25463), (Q8_0, 7773, 256, 18290), (Q4_K, 116, 7168, 13668), (Q4_K, 512, 14336, 8300),
                                              (Q6_K, 258, 5376, 12071), (Q6_K, 9481, 512, 25813), (Q4_K, 3676, 256, 13139)])
def test_blocks_of_a_packed_launch_are_chosen_among_packed_forms(fmt, n_out, n_in, m):
    """More than 8192 rows are packed and multiplied a block at a time: a block's copy is there already, so its tile and copies along K
    are those of the packed kernel's times alone, whatever type the copy was made from."""
    plan = detail(fmt, n_out, n_in, m, BF16, BF16)
    assert plan == detail(fmt, n_out, n_in, m, F16, F16)
    assert [form.endswith(" packed") for form in plan.split("; ")] == [True, True]


def test_route_detail_checks_its_arguments():
    L, text = _lib.lib(), C.create_string_buffer(b"x" * 15, 16)
    st = QLinearStruct(format=Q4_K, n_out=4096, n_in=14336)
    assert L.ttq_route_detail(C.byref(st), 512, BF16, BF16, None, 16) == _lib.ERR_NULL
    assert L.ttq_route_detail(C.byref(st), 512, BF16, BF16, text, 0) == _lib.ERR_NULL
    assert L.ttq_route_detail(None, 512, BF16, BF16, text, 16) == _lib.ERR_NULL and text.value == b""
    assert L.ttq_route_detail(C.byref(st), 512, BF16, BF16, text, 16) == _lib.ROUTE["gemm_pc_packed_split_k"]
    assert text.value == b"gemm_pc 256x64 "                                     # cut, and zero-terminated
    assert L.ttq_gemm_q4_k_silu_mul_detail(512, 14336, 4096, None, 16) == _lib.ERR_NULL
    assert L.ttq_gemm_q4_k_silu_mul_detail(512, 14336, 100, text, 16) == _lib.ERR_SHAPE
    big = C.create_string_buffer(64)
    assert L.ttq_gemm_q4_k_silu_mul_detail(2048, 14336, 4096, big, 64) >= 0 and big.value == b"gemm_pc_silu_mul 256x112"
    assert L.ttq_gemm_q4_k_silu_mul_detail(32, 3072, 1024, big, 64) >= 0 and big.value == b"gemm_skinny_silu_mul"
    assert L.ttq_gemm_q4_k_silu_mul_detail(0, 3072, 1024, big, 64) == _lib.ROUTE["none"] and big.value == b""


def test_workspace_size_query_and_argument_checks():
    L = _lib.lib()
    q = QLinearStruct(format=Q4_K, n_out=4096, n_in=14336)
    assert L.ttq_workspace_bytes(C.byref(q), 1, BF16) == 0                       # decode kernels take none
    split = L.ttq_workspace_bytes(C.byref(q), 512, BF16)
    assert split > (4 << 20)                                                     # header + partial sums
    small = QLinearStruct(format=Q4_K, n_out=1024, n_in=1024)                    # a short GEMM reads X itself ...
    ok = QLinearStruct(format=Q4_K, n_out=1024, n_in=1024, precision=_lib.PRECISION_BF16_OK)
    assert (L.ttq_workspace_bytes(C.byref(ok), 512, F32) >=                      # ... unless its rows must be rounded
            L.ttq_workspace_bytes(C.byref(small), 512, BF16) + 512 * 1024 * 2)
    assert L.ttq_workspace_bytes(C.byref(q), 0, BF16) == 0
    # two to four rows decode without a workspace, except fp32 ones, which may take the few-row kernel over a scaled
    # fp16 copy (the copy and a factor per row)
    for m in (2, 3, 4):
        assert L.ttq_workspace_bytes(C.byref(q), m, BF16) == 0 and L.ttq_workspace_bytes(C.byref(q), m, F16) == 0
        assert L.ttq_workspace_bytes(C.byref(q), m, F32) >= m * 14336 * 2 + 4 * m
    assert L.ttq_workspace_bytes(C.byref(q), 1, F32) == 0
    assert L.ttq_workspace_bytes(None, 1, BF16) == _lib.ERR_NULL
    assert L.ttq_workspace_bytes(C.byref(q), 1, 5) == _lib.ERR_DTYPE
    t = QLinearStruct(format=EXL3, n_out=4096, n_in=4096, bits=3, codebook=_lib.CB_MCG)
    assert L.ttq_workspace_bytes(C.byref(t), 1, F16) > (4 << 20)                 # hand-off words
    # a workspace that cannot be one is refused before anything else happens
    assert L.ttq_linear_forward_ws(C.byref(q), None, BF16, 512, None, BF16, None, 1024, None) == _lib.ERR_WORKSPACE
    assert L.ttq_linear_forward_ws(C.byref(q), None, BF16, 512, None, BF16, 8, 1024, None) == _lib.ERR_WORKSPACE
    assert L.ttq_linear_forward_ws(C.byref(q), None, BF16, 512, None, BF16, None, -1, None) == _lib.ERR_WORKSPACE
    assert L.ttq_linear_forward_ws(C.byref(q), None, BF16, 0, None, BF16, None, 0, None) == _lib.OK
    assert L.ttq_strerror(_lib.ERR_WORKSPACE) not in (b"unknown status", b"ok")


def test_fitted_time_moves_no_exact_call():
    """A long fp32 matrix of few rows decodes exactly (its estimate as tiles or few-row chunks is above the decode's), although
    the tiled kernel's fitted time is below: the fitted time decides between kernels that round the weights only."""
    assert route(Q4_K, 48, 14848, 170, F32, F32) == "gemv_generic"
    assert route(Q4_K, 2816, 2816, 191, F32, F32) == "gemm_pc_f32_scaled_f16"
