"""The tiled product (tile_gemm.h) at the sizes where it can go wrong: rows and columns around the edges of every tile shape,
fewer K steps than the prefetch distance or than the wave groups along K, K parts with a short last part, strided
activations, odd output widths."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

# (M, N, K): every tile shape of the int8 table, with and without K parts (checked below)
CASES = [
    (17, 4100, 8320), (33, 4096, 8192), (64, 3072, 4224), (65, 5121, 6528), (96, 8200, 4096), (97, 16400, 4096), (129, 1100, 4096),
    (191, 16400, 2048), (192, 24600, 2048), (193, 15000, 2176), (255, 14336, 1024), (256, 14336, 1024), (257, 21000, 1024), (384, 12416, 2048),
    (769, 130, 128), (770, 127, 256), (1000, 600, 1024), (1025, 14336, 512), (513, 28672, 640),
    (70, 1028, 4096), (24, 4100, 4096), (160, 1001, 2048), (640, 14337, 512),
    (1, 300, 64), (5, 2000, 192), (40, 4096, 8256),  # in_features not a multiple of 128: any row count
]


def _plan(M, N, K):
    from ao_amd import _lib

    out = ctypes.create_string_buffer(64)
    _lib.check(_lib.lib().ao_amd_int8wo_linear_plan(M, K, N, out, 64))
    return out.value.decode()


def _run(M, N, K, bias=False, pad=0):
    from ao_amd import ops

    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    w = torch.randint(-128, 128, (N, K), device="cuda", dtype=torch.int8, generator=g)
    x = torch.randn(M, K + pad, device="cuda", generator=g).bfloat16()[:, :K]
    s = (torch.rand(N, device="cuda", generator=g) * 0.01 + 0.001).bfloat16()
    b = torch.randn(N, device="cuda", generator=g).bfloat16() if bias else None
    y = ops.int8wo_linear(x, w, s, b)
    acc = x.float() @ w.float().t()
    want = (acc.bfloat16().float() * s.float()).bfloat16()
    if bias:
        want = (want.float() + b.float()).bfloat16()
    rel = ((y.float() - want.float()).norm() / want.float().norm()).item()
    # exact products; sums of K <= 8320 of them in fp32 differ by their order in about 1e-6 relative, which moves a rounding
    # of the result (relative step 2^-8) now and then: few elements, by one step of the value (or of the sum before the
    # bias, which can cancel)
    assert (y != want).float().mean() <= 0.01 and rel <= 1e-3, (M, N, K, rel)


def test_cases_cover_every_tile_shape():
    plans = {c: _plan(*c) for c in CASES}
    shapes = {p.split()[1] for p in plans.values() if p != "streaming"}
    assert shapes == {"64x64", "64x128", "96x128", "128x128", "192x128", "128x256", "192x256"}, plans
    assert any(p.endswith("parts=1") for p in plans.values()) and any(not p.endswith("parts=1") for p in plans.values())


@pytest.mark.parametrize("case", CASES)
def test_int8_tiles(case):
    _run(*case)


# weights that come in two steps at a time: one pair, one more or fewer than the ring and the groups hold, K parts of
# different lengths, a last row of the weight that ends the buffer, and the widths that end within a pair
@pytest.mark.parametrize("case,plan", [
    ((390, 14336, 128), "tile 128x256 parts=1"), ((390, 14336, 384), "tile 128x256 parts=1"), ((391, 14330, 640), "tile 128x256 parts=1"),
    ((390, 14336, 576), "tile 128x256 parts=1"), ((131, 8192, 256), "tile 64x128 parts=1"), ((257, 4096, 384), "tile 64x128 parts=1"),
    ((257, 4096, 640), "tile 64x128 parts=1"), ((516, 2048, 1152), "tile 64x128 parts=1"), ((257, 4096, 704), "tile 64x128 parts=1"),
    ((40, 14336, 6400), "tile 64x128 parts=2"), ((257, 1024, 6400), "tile 64x128 parts=4"), ((131, 1024, 9088), "tile 64x128 parts=8"),
])
def test_int8_weights_in_pairs_of_steps(case, plan):
    assert _plan(*case) == plan
    _run(*case)   # (the bound of _run: at most 9088 exact products a sum)


# two waves share a column block, each with 96 rows: the second one with one, two or all of its rows, K shorter than the ring of
# buffers and just past it, columns that end within a block
@pytest.mark.parametrize("M,N,K", [(290, 14336, 64), (289, 14290, 128), (380, 11008, 320), (384, 14290, 192), (300, 14336, 1088)])
def test_tiles_of_two_waves_a_column_block(M, N, K):
    assert _plan(M, N, K) == "tile 192x128 parts=1"
    _run(M, N, K)
    N = N // 64 * 64
    assert _tiled_plan("fp6", M, N, K) == "tile 192x128 parts=1"
    _fp6_tiles(M, N, K, 3, 2)


@pytest.mark.parametrize("case", [(65, 5121, 6528), (257, 21000, 1024), (129, 1100, 4096)])
def test_int8_tiles_bias_and_row_stride(case):
    _run(*case, bias=True, pad=72)


@pytest.mark.parametrize("case,plan", [
    ((3, 4096, 14336), "streaming"), ((5, 4090, 14336), "streaming"), ((6, 2064, 11008), "streaming"), ((2, 4096, 28672), "streaming"),  # rows staged in 65 to 140 KB
    ((6, 4096, 14336), "streaming"),                                                                                                     # just past that
    ((3, 2048, 16512), "streaming parts=8"), ((9, 4104, 8320), "streaming parts=3"), ((8, 4104, 8320), "streaming parts=3"), ((8, 5128, 13824), "streaming parts=3"),
    ((9, 24592, 8192), "tile 64x128 parts=1"), ((8, 10240, 8192), "tile 64x128 parts=3"), ((12, 4104, 14336), "tile 64x128 parts=7"),
    ((3, 8192, 28672), "tile 64x128 parts=4"), ((5, 11010, 17408), "tile 64x128 parts=2"),
])
def test_int8_few_rows(case, plan):
    assert _plan(*case) == plan
    # the bound of _run holds here too: the sums are at most 3.5 times as long, and their order moves them by about
    # sqrt(K) 2^-24 of their size, 1e-5 at most, against the 2^-8 steps of the result
    _run(*case)


def _tiled_plan(fmt, M, N, K):
    from ao_amd import _lib

    out = ctypes.create_string_buffer(64)
    _lib.check(getattr(_lib.lib(), f"ao_amd_{fmt}_linear_tiled_plan")(M, K, N, out, 64))
    return out.value.decode()


def _tiled_bytes(fmt, M, N, K, *group):
    from ao_amd import _lib

    need = ctypes.c_int64(0)
    _lib.check(getattr(_lib.lib(), f"ao_amd_{fmt}_linear_tiled_bytes")(M, K, N, *group, ctypes.byref(need)))
    return need.value


# (M, N, K): every tile shape of the FP6 table, with and without K parts, K a multiple of 64 but not of 128, one K step
FP6_TILES = [
    (1, 64, 64), (33, 4160, 4096), (65, 1088, 192), (65, 14336, 1024), (96, 4096, 8192), (97, 14400, 512), (129, 14336, 1024), (200, 14336, 1024),
    (257, 14336, 1024), (192, 24640, 512), (512, 14336, 512), (640, 14400, 512), (769, 4096, 2112), (1000, 4096, 3072), (100, 8192, 8192),
]


def _fp6_tiles(M, N, K, ebits, mbits):
    from ao_amd import _lib, ops

    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    w = (torch.randn(N, K, device="cuda", generator=g) * 0.05).half()
    tc, scale = ops.fp6_quantize_pack(w, ebits, mbits)
    native = ops.fp6_repack(tc, 1 + ebits + mbits)
    x = torch.randn(M, K, device="cuda", generator=g).half()
    wd = ops.fp6_dequantize(tc, scale, ebits, mbits).half()    # the kernels multiply fp16(value * scale)
    want = (x.float() @ wd.float().t()).half()
    ws = torch.empty(8 * M * N, device="cuda")
    for size in (ws.numel() * 4, 0):                           # with the plan's K parts, and without room for them
        y = torch.full((M, N), float("nan"), device="cuda").half()
        _lib.check(_lib.lib().ao_amd_fp6_linear_tiled(x.data_ptr(), M, K, native.data_ptr(), scale.data_ptr(), N, ebits, mbits, y.data_ptr(),
                                                      ws.data_ptr() if size else None, size, torch.cuda.current_stream().cuda_stream))
        # the products are exact in fp32 and sums of K <= 8192 of them differ by their order in about 1e-6 relative, which moves
        # a rounding of the result (relative step 2^-11) now and then
        rel = ((y.float() - want.float()).norm() / want.float().norm()).item()
        assert rel <= 1e-4, (M, N, K, rel)
    return x, native, scale, y


@pytest.mark.parametrize("case", FP6_TILES)
def test_fp6_tiles(case):
    _fp6_tiles(*case, 3, 2)


@pytest.mark.parametrize("ebits,mbits", [(2, 3), (2, 2), (3, 1)])
def test_fp6_tiles_other_formats(ebits, mbits):
    _fp6_tiles(129, 4160, 1088, ebits, mbits)


def test_fp6_tiles_cover_every_shape_and_the_operator_takes_them():
    from ao_amd import ops

    plans = {c: _tiled_plan("fp6", *c) for c in FP6_TILES}
    assert {p.split()[1] for p in plans.values()} == {"64x64", "64x128", "96x128", "128x128", "192x128", "128x256", "192x256"}, plans
    assert any(p.endswith("parts=1") for p in plans.values()) and any(not p.endswith("parts=1") for p in plans.values())
    assert _tiled_bytes("fp6", 65, 14336, 4096) >= 0 and _tiled_bytes("fp6", 65, 1024, 4096) == -1
    assert _tiled_bytes("fp6", 33, 28672, 8192) >= 0 and _tiled_bytes("fp6", 512, 2112, 2112) == 0
    for M, N, K in ((160, 4096, 8192), (129, 14336, 1024), (512, 2112, 2112)):
        x, native, scale, _ = _fp6_tiles(M, N, K, 3, 2)
        eager = ops.fp6_linear_native(3, 2, x, native, scale)
        assert torch.equal(eager, torch.ops.torchao.fp6_linear_native.default(3, 2, x, native, scale))   # both host paths


@pytest.mark.parametrize("M,N,K,tiled", [
    (32, 14336, 2048, False), (33, 14336, 2048, True), (48, 14336, 2048, True), (63, 14336, 2048, True), (64, 14336, 2048, True),
    (64, 14336, 4224, True), (48, 8192, 2048, False),
    # one line for 33 to 64 rows, by what the two routes take (us, tiles / the others): 14336 x 4096 at 63 / 64 rows 17.7 / 19.1, 17.6 / 19.0; at 33
    # rows 8448 x 4096 11.8 / 16.9, 8192 x 4096 13.1 / 12.2, 6400 x 5120 and 5120 x 5632 0.85 to 0.9 of them, 7168 x 6144 at 64 rows 17.7 / 16.9
    (33, 14336, 4096, True), (64, 14336, 4096, True), (33, 8448, 4096, True), (64, 8448, 4096, True), (33, 8192, 4096, False), (48, 8192, 4096, False),
    (64, 8192, 4096, False), (64, 6400, 5120, True), (40, 5120, 5632, True), (64, 7168, 6144, False), (64, 8192, 5632, False),
    (64, 4096, 14336, False), (65, 4096, 14336, True), (96, 4096, 14336, True), (97, 4096, 14336, False), (80, 4096, 8192, False),
])
def test_fp6_tiles_at_33_to_96_rows(M, N, K, tiled):
    """Both sides of the rule on rows and weight size, operator against the fp32 product (the tolerance of _fp6_tiles: the
    order of at most 14336 exact products' fp32 sums)."""
    from ao_amd import ops

    assert (_tiled_bytes("fp6", M, N, K) >= 0) == tiled
    x, native, scale, y = _fp6_tiles(M, N, K, 3, 2)
    rel = ((ops.fp6_linear_native(3, 2, x, native, scale).float() - y.float()).norm() / y.float().norm()).item()
    assert rel <= 1e-4, rel


# (M, N, K, group): every tile shape of the int4 table, groups below, at and beyond a K step, widths with part of a row block,
# in_features that the packed layout pads (to a multiple of 128 or of the group)
INT4_TILES = [
    (1, 20, 128, 32), (33, 4100, 4096, 64), (65, 1040, 256, 256), (65, 14330, 1024, 128), (96, 4096, 8192, 32), (97, 14336, 512, 64),
    (129, 14336, 1024, 128), (200, 14337, 1024, 256), (257, 14336, 1024, 64), (512, 14336, 512, 32), (640, 4096, 14336, 64), (769, 4096, 2048, 128),
    (1000, 4099, 2048, 64), (100, 8192, 4096, 256),
    # the prefill kernel's tiles with K parts: two and four of them, part lengths rounded up to an even number of steps, short last part
    (400, 4096, 9984, 256), (400, 4090, 12544, 32), (512, 6144, 12544, 128), (200, 11008, 8192, 64), (400, 11000, 14336, 64), (900, 4096, 14336, 64),
    (34, 1030, 64, 128), (70, 4096, 4032, 256), (130, 4099, 1088, 64), (40, 2048, 8256, 32),
]


def _int4_tiles(M, N, K, group, bias=False, pad=0):
    from ao_amd import _lib, ops

    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    packed, qp = ops.int4wo_quantize_pack((torch.randn(N, K, device="cuda", generator=g) * 0.02).bfloat16(), group)
    dq = ops.int4wo_dequantize(packed, qp, N, K, group)
    x = torch.randn(M, K + pad, device="cuda", generator=g).bfloat16()[:, :K]
    b = torch.randn(N, device="cuda", generator=g).bfloat16() if bias else None
    want = x.float() @ dq.float().t()
    want = (want + b.float() if bias else want).bfloat16()
    ws = torch.empty(8 * M * N, device="cuda")
    for size in (ws.numel() * 4, 0):
        y = torch.full((M, N), float("nan"), device="cuda").bfloat16()
        _lib.check(_lib.lib().ao_amd_int4wo_linear_tiled(x.data_ptr(), M, K, x.stride(0), packed.data_ptr(), qp.data_ptr(), N, group,
                                                         b.data_ptr() if bias else None, y.data_ptr(), N, ws.data_ptr() if size else None, size,
                                                         torch.cuda.current_stream().cuda_stream))
        # as above; the result's step is 2^-8
        rel = ((y.float() - want.float()).norm() / want.float().norm()).item()
        assert rel <= 1e-3 and (y != want).float().mean() <= 0.01, (M, N, K, rel)
    return x, packed, qp, b


@pytest.mark.parametrize("case", INT4_TILES)
def test_int4_tiles(case):
    _int4_tiles(*case)


@pytest.mark.parametrize("case", [(97, 4099, 1024, 64), (129, 4100, 8192, 32)])
def test_int4_tiles_bias_and_row_stride(case):
    _int4_tiles(*case, bias=True, pad=72)


def test_int4_tiles_read_the_weight_bit_for_bit():
    """One-hot rows return columns of the dequantized weight."""
    from ao_amd import _lib, ops

    M, N, K, group = 200, 1030, 1024, 32
    packed, qp = ops.int4wo_quantize_pack((torch.randn(N, K, device="cuda") * 0.02).bfloat16(), group)
    at = torch.arange(M, device="cuda") * 5 + 3
    x = torch.zeros(M, K, device="cuda").bfloat16()
    x[torch.arange(M, device="cuda"), at] = 1.0
    y = torch.empty(M, N, device="cuda").bfloat16()
    _lib.check(_lib.lib().ao_amd_int4wo_linear_tiled(x.data_ptr(), M, K, K, packed.data_ptr(), qp.data_ptr(), N, group, None, y.data_ptr(), N, None,
                                                     0, torch.cuda.current_stream().cuda_stream))
    assert torch.equal(y, ops.int4wo_dequantize(packed, qp, N, K, group)[:, at].t())


def test_int4_tiles_cover_every_shape_and_the_operator_takes_them():
    from ao_amd import ops

    plans = {c: _tiled_plan("int4wo", *c[:3]) for c in INT4_TILES}
    assert {p.split()[1] for p in plans.values()} == {"64x64", "64x128", "96x128", "128x128", "192x128", "256x128", "256x256"}, plans
    assert {f"tile 256x{n} parts={z}" for n, z in ((128, 2), (128, 4), (256, 2), (256, 4))} <= set(plans.values()), plans
    assert any(p.endswith("parts=1") for p in plans.values()) and any(not p.endswith("parts=1") for p in plans.values())
    # (us streamed / tiled at 33 / 48 rows 18.9 / 17.2, 19.3 / 17.3)
    for rows, taken in ((32, False), (33, True), (48, True), (128, False), (160, True), (256, True), (384, True), (768, False)):
        assert (_tiled_bytes("int4wo", rows, 14336, 4096, 64) >= 0) == taken, rows
    for case in ((160, 14336, 1024, 64), (96, 4096, 14336, 128), (130, 4099, 1088, 64)):
        for bias in (False, True):
            x, packed, qp, b = _int4_tiles(*case, bias=bias, pad=8)
            eager = ops.int4wo_linear(x, packed, qp, case[3], case[1], b)
            assert torch.equal(eager, torch.ops.torchao.int4wo_linear.default(x, packed, qp, case[3], case[1], b, False))


@pytest.mark.parametrize("M,N,K,group,shift", [
    (1, 14336, 4032, 64, 0), (1, 8192, 4100, 128, 0), (3, 4099, 4160, 32, 0), (16, 4096, 4041, 256, 0), (17, 4096, 4032, 256, 0), (33, 4100, 4160, 64, 0),
    (300, 4096, 4100, 64, 0), (600, 14336, 1090, 128, 0), (1703, 5088, 700, 64, 0),   # rows that end before the packed width
    (1, 14336, 4096, 64, 1), (9, 4096, 4096, 128, 3), (200, 4096, 4096, 64, 1),  # rows that are not 16-byte aligned
    (2, 64, 192, 64, 0), (1, 1024, 704, 64, 1),                              # too small for the copy to pay
])
def test_int4_rows_that_are_copied_to_the_packed_width(M, N, K, group, shift):
    from ao_amd import ops

    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    packed, qp = ops.int4wo_quantize_pack((torch.randn(N, K, device="cuda", generator=g) * 0.02).bfloat16(), group)
    dq = ops.int4wo_dequantize(packed, qp, N, K, group)
    x = torch.randn(M, K + 2 * shift, device="cuda", generator=g).bfloat16()[:, shift:K + shift]
    want = (x.float() @ dq.float().t()).bfloat16()
    for y in (ops.int4wo_linear(x, packed, qp, group, N), torch.ops.torchao.int4wo_linear.default(x, packed, qp, group, N, None, False)):
        rel = ((y.float() - want.float()).norm() / want.float().norm()).item()   # as for the tiles
        assert rel <= 1e-3, (M, N, K, rel)
    y32 = ops.int4wo_linear(x, packed, qp, group, N, fp32_out=True)
    want = x.double() @ dq.double().t()
    # sums of K <= 4160 exact products in fp32: sqrt(K) roundings of 2^-24 of the partial sum, about 4e-6, times the cancellation in it
    assert ((y32.double() - want).norm() / want.norm()).item() <= 2e-5


@pytest.mark.parametrize("M,N,K,group", [(65, 12300, 1024, 64), (96, 12288, 1152, 32), (97, 12288, 1152, 64), (130, 6150, 1280, 256), (192, 6144, 2176, 128),
                                         (257, 4100, 1024, 64), (288, 4096, 1408, 128), (289, 4096, 1024, 64)])
def test_int4_kwave_tiles_of_96_and_128_rows(M, N, K, group):
    """Edges of the 96-row tiles (up to 96, 192 and 288 rows; one more takes 128-row ones), K steps that leave the waves unequal and
    odd counts, against the fp32 product and, one-hot, the weight bit for bit."""
    from ao_amd import _lib, ops

    assert _lib.int4wo_linear_plan(M, K, N, group).startswith("int4wo_gemm_kwave_kernel")
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    packed, qp = ops.int4wo_quantize_pack((torch.randn(N, K, device="cuda", generator=g) * 0.02).bfloat16(), group)
    dq = ops.int4wo_dequantize(packed, qp, N, K, group)
    x = torch.randn(M, K, device="cuda", generator=g).bfloat16()
    hot = torch.zeros(M, K, device="cuda").bfloat16()
    at = (torch.arange(M, device="cuda") * 37 + 5) % K
    hot[torch.arange(M, device="cuda"), at] = 1.0
    for rows, want in ((x, (x.float() @ dq.float().t()).bfloat16()), (hot, dq[:, at].t())):
        y = torch.full((M, N), float("nan"), device="cuda").bfloat16()
        _lib.check(_lib.lib().ao_amd_int4wo_linear(rows.data_ptr(), M, K, K, packed.data_ptr(), qp.data_ptr(), N, group, None, y.data_ptr(),
                                                   _lib.BF16, N, torch.cuda.current_stream().cuda_stream))
        rel = ((y.float() - want.float()).norm() / want.float().norm()).item()   # as for the tiles; one-hot rows are exact
        assert rel <= (1e-3 if rows is x else 0.0), (M, N, K, rel)


@pytest.mark.parametrize("M,N,K,group,name", [
    (1, 14336, 4032, 64, "int4wo_gemv1_short_kernel"), (1, 560, 1856, 64, "int4wo_gemv1_short_kernel"), (1, 9316, 5312, 128, "int4wo_gemv1_short_kernel"),
    (1, 2288, 9736, 256, "int4wo_gemv1_short_kernel"), (1, 4096, 16136, 256, "int4wo_gemv1_short_kernel"), (1, 30000, 1032, 128, "int4wo_gemv1_short_kernel"),
    (2, 4099, 4160, 32, "int4wo_linear_kernel"), (15, 4096, 8072, 256, "int4wo_linear_kernel"), (3, 70, 136, 64, "int4wo_linear_kernel"),
    (4, 12290, 1096, 64, "int4wo_linear_rb4_kernel"), (16, 12336, 7552, 256, "int4wo_linear_rb4_kernel"), (17, 14344, 4040, 128, "int4wo_linear_rb4_kernel"),
    (48, 12300, 1160, 32, "int4wo_linear_rb4_kernel"), (64, 65552, 264, 64, "int4wo_linear_rb4_kernel"),
    (5, 12304, 1024, 64, "int4wo_linear_rb4_kernel"), (33, 14360, 2048, 128, "int4wo_linear_rb4_kernel"),   # row blocks that are no multiple of four
])
def test_int4_rows_that_are_read_as_they_end(M, N, K, group, name):
    """Rows of a multiple of 8 elements that end before the packed width, and row blocks that are no multiple of four, on the kernels that
    take them without a copy: the fp32 product (as for the tiles), single weights bit for bit, and nothing of what lies behind a row's
    end (NaN here) in the result."""
    from ao_amd import _lib, ops

    assert _lib.int4wo_linear_plan(M, K, N, group).startswith(name)
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    packed, qp = ops.int4wo_quantize_pack((torch.randn(N, K, device="cuda", generator=g) * 0.02).bfloat16(), group)
    dq = ops.int4wo_dequantize(packed, qp, N, K, group)
    rows = torch.full((M + 1, K + 264), float("nan"), device="cuda").bfloat16()
    x = rows[:M, :K]
    x.copy_(torch.randn(M, K, device="cuda", generator=g))
    y = ops.int4wo_linear(x, packed, qp, group, N)
    want = (x.float() @ dq.float().t()).bfloat16()
    rel = ((y.float() - want.float()).norm() / want.float().norm()).item()
    assert rel <= 1e-3 and (y != want).float().mean() <= 0.01, rel
    at = torch.arange(M, device="cuda") * 37 % K
    at[-1] = K - 1
    x.zero_()
    x[torch.arange(M, device="cuda"), at] = 1.0
    assert torch.equal(ops.int4wo_linear(x, packed, qp, group, N), dq[:, at].t())


@pytest.mark.parametrize("M,N,K,group,tiled", [
    (32, 12304, 1088, 128, False), (33, 12304, 1088, 128, True), (48, 12304, 1024, 64, True), (33, 12288, 1088, 32, True),
    (33, 12288, 1024, 64, True), (48, 12288, 1024, 64, True),       # us streamed / tiled 8.6 / 8.4, 9.1 / 8.3
    (33, 12290, 1032, 64, False),                                   # a width that the tiles do not take
    (48, 65552, 192, 64, False), (49, 65552, 192, 64, True), (64, 65540, 256, 32, True),
])
def test_int4_ragged_weights_at_33_to_64_rows(M, N, K, group, tiled):
    """Rows that end before the packed width, and row blocks that are no multiple of four: from 33 rows on the tiles are ahead of the
    streaming kernel that could read them (18837 x 1088 at 33 rows 12.0 / 14.9 us, 12304 x 4096 at 48 17.0 / 19.6).  The operator against the fp32
    product (as for the tiles); what lies behind a row's end is NaN."""
    from ao_amd import ops

    assert (_tiled_bytes("int4wo", M, N, K, group) >= 0) == tiled
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    packed, qp = ops.int4wo_quantize_pack((torch.randn(N, K, device="cuda", generator=g) * 0.02).bfloat16(), group)
    rows = torch.full((M, K + 8), float("nan"), device="cuda").bfloat16()
    x = rows[:, :K]
    x.copy_(torch.randn(M, K, device="cuda", generator=g))
    y, want = ops.int4wo_linear(x, packed, qp, group, N), (x.float() @ ops.int4wo_dequantize(packed, qp, N, K, group).float().t()).bfloat16()
    rel = ((y.float() - want.float()).norm() / want.float().norm()).item()
    assert rel <= 1e-3 and (y != want).float().mean() <= 0.01, rel


def test_int4_tiles_where_their_k_parts_pay():
    """Narrow weights at 65 and more rows: K parts of the 32-row tiles (us at 100 rows 10.7 on 512 x 4096, 12.5 on 1024 x 6144) against the tiles' eight
    (11.4, 12.9), which are ahead from about 7000 of K on (512 x 8192 14.1 / 13.3)."""
    for M, N, K, tiled in ((100, 512, 4096, False), (256, 512, 4096, False), (80, 1536, 4096, False), (100, 1024, 6144, False), (100, 512, 8192, True),
                           (128, 1024, 14336, True)):
        assert (_tiled_bytes("int4wo", M, N, K, 128) >= 0) == tiled, (M, N, K)


@pytest.mark.parametrize("M,N,K,group,tiled", [
    (33, 2048, 16384, 64, True), (40, 3080, 8320, 128, True), (64, 5120, 13824, 32, True), (47, 1030, 14336, 64, True), (33, 2048, 4096, 64, False),
    (64, 4096, 4096, 64, False), (33, 1024, 8192, 128, False),
])
def test_int4_tiles_at_one_tile_row(M, N, K, group, tiled):
    """33 to 64 rows of narrow weights: tiles in K parts where K is long (2048 x 16384 at 40 rows 32.0 -> 16.2 us), the streaming kernel or its parts where it
    is short.  The tolerance is that of two bf16 roundings of one fp32 sum in another order."""
    from ao_amd import ops

    assert (_tiled_bytes("int4wo", M, N, K, group) >= 0) == tiled
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    packed, qp = ops.int4wo_quantize_pack((torch.randn(N, K, device="cuda", generator=g) * 0.02).bfloat16(), group)
    x = torch.randn(M, K, device="cuda", generator=g).bfloat16()
    y, want = ops.int4wo_linear(x, packed, qp, group, N), (x.float() @ ops.int4wo_dequantize(packed, qp, N, K, group).float().t()).bfloat16()
    rel = ((y.float() - want.float()).norm() / want.float().norm()).item()
    assert rel <= 1e-3 and (y != want).float().mean() <= 0.01, rel


@pytest.mark.parametrize("fmt,M,N,K,group,name", [
    ("int4", 1700, 7000, 512, 64, "int4wo_gemm_lds_kernel<64,2>"), ("int4", 1000, 6400, 512, 128, "int4wo_gemm_lds_kernel<128,1>"),
    ("int4", 300, 4100, 1024, 32, "int4wo_gemm_kwave_kernel"), ("int4", 2750, 1024, 4096, 64, ""), ("int4", 5000, 64, 256, 64, ""),
    ("int8", 2100, 1100, 256, 0, ""), ("int8", 450, 14336, 256, 0, ""), ("fp6", 900, 2048, 256, 0, ""), ("fp6", 3000, 320, 512, 0, ""),
])
def test_every_tile_once(fmt, M, N, K, group, name):
    """Tiles are taken in panels of tile rows, the last of them lower: single weights bit for bit in every tile, panels of one to
    many rows, one or few columns."""
    from ao_amd import _lib, ops

    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    w = torch.randn(N, K, device="cuda", generator=g) * 0.02
    at = torch.randint(0, K, (M,), device="cuda", generator=g)
    x = torch.zeros(M, K, device="cuda", dtype=torch.float16 if fmt == "fp6" else torch.bfloat16)
    x[torch.arange(M, device="cuda"), at] = 1.0
    if fmt == "int4":
        assert _lib.int4wo_linear_plan(M, K, N, group).startswith(name)
        packed, qp = ops.int4wo_quantize_pack(w.bfloat16(), group)
        dq, y = ops.int4wo_dequantize(packed, qp, N, K, group), ops.int4wo_linear(x, packed, qp, group, N)
    elif fmt == "int8":
        q, scale = (w * 3000).round().clamp(-127, 127).to(torch.int8), torch.rand(N, device="cuda", generator=g).bfloat16()
        dq, y = (q.float() * scale.float()[:, None]).bfloat16(), ops.int8wo_linear(x, q, scale)
    else:
        tc, scale = ops.fp6_quantize_pack(w.half(), 3, 2)
        native = ops.fp6_repack(tc, 6)
        dq, y = ops.fp6_dequantize(tc, scale, 3, 2).half(), ops.fp6_linear_native(3, 2, x, native, scale)
    assert torch.equal(y, dq[:, at].t())


# K parts that are no power of two: equal ones and a shorter last one, of pairs of steps (64 x 128 int8 tiles) too, rows and columns that end within a tile
@pytest.mark.parametrize("fmt,M,N,K,plan", [
    ("int8", 40, 5120, 13824, "tile 64x128 parts=6"), ("int8", 61, 10200, 8320, "tile 64x128 parts=3"), ("int8", 77, 10240, 8256, "tile 96x128 parts=3"),
    ("int8", 100, 2300, 4160, "tile 64x64 parts=3"), ("int4wo", 40, 5120, 5120, "tile 64x64 parts=3"), ("int4wo", 90, 5110, 13888, "tile 96x128 parts=6"),
    ("int4wo", 200, 5120, 13824, "tile 128x128 parts=3"), ("fp6", 113, 5120, 13824, "tile 64x128 parts=3"), ("fp6", 77, 5120, 13888, "tile 96x128 parts=6"),
    # tiles times parts that the XCDs cannot share evenly: 41 x 6, 33 x 7
    ("int8", 40, 5128, 13824, "tile 64x128 parts=6"), ("int8", 24, 4104, 14336, "tile 64x128 parts=7"), ("int4wo", 130, 4110, 13888, "tile 192x128 parts=7")])
def test_parts_that_are_no_power_of_two(fmt, M, N, K, plan):
    assert (_plan(M, N, K) if fmt == "int8" else _tiled_plan(fmt, M, N, K)) == plan
    # (the bounds of the helpers: up to 13888 products a sum)
    if fmt == "int8":
        _run(M, N, K)
    elif fmt == "int4wo":
        _int4_tiles(M, N, K, 64)
    else:
        _fp6_tiles(M, N, K, 3, 2)


# Sums of K parts whose rows are 16-byte aligned (a multiple of four columns: four a thread add them) or not (one a thread), stored to rows of any stride:
# streamed row blocks of int8 (up to 16 rows) and of int4 (up to 32), tiles of both.  Activations and int8 weights are views of wider rows with NaN or 127 behind
# their ends; what lies between the rows of the output stays.
@pytest.mark.parametrize("fmt,M,N,K,pad_y", [
    ("int8", 11, 2301, 14336, 0), ("int8", 16, 2302, 14336, 3), ("int8", 9, 2303, 14336, 1), ("int8", 13, 2304, 14336, 1), ("int8", 12, 2304, 14336, 4),
    ("int8", 40, 1021, 14336, 2), ("int8", 70, 1022, 8192, 0), ("int8", 24, 4100, 14336, 5), ("int8", 65, 513, 8192, 0),
    ("int4", 40, 1021, 16384, 2), ("int4", 64, 2050, 14336, 1), ("int4", 47, 1028, 14336, 3), ("int4", 12, 5120, 13824, 5), ("int4", 30, 5124, 13824, 4),
    ("int4", 13, 5000, 8000, 1)])
def test_sums_of_parts_in_rows_of_any_stride(fmt, M, N, K, pad_y):
    from ao_amd import _lib, ops

    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    L, need, st = _lib.lib(), ctypes.c_int64(-1), torch.cuda.current_stream().cuda_stream
    rows = torch.full((M, K + 24), float("nan"), device="cuda").bfloat16()
    x = rows[:, :K]
    x.copy_(torch.randn(M, K, device="cuda", generator=g))
    x[0, 5], x[M // 2, K - 7] = float("inf"), float("-inf")   # in the first and in the last part of K
    if M > 3:
        x[M - 1, K // 2] = float("nan")
    b = torch.randn(N, device="cuda", generator=g).bfloat16()
    y = torch.full((M, N + pad_y), 7.0, device="cuda").bfloat16()
    if fmt == "int8":
        w = torch.full((N, K + 32), 127, device="cuda", dtype=torch.int8)[:, :K]
        w.copy_(torch.randint(-128, 128, (N, K), device="cuda", dtype=torch.int8, generator=g))
        s = (torch.rand(N, device="cuda", generator=g) * 0.01 + 0.001).bfloat16()
        _lib.check(L.ao_amd_int8wo_linear_ws_bytes(M, K, N, ctypes.byref(need)))
        ws = torch.full((need.value // 4,), float("nan"), device="cuda")
        _lib.check(L.ao_amd_int8wo_linear_ws(x.data_ptr(), M, K, K + 24, w.data_ptr(), K + 32, s.data_ptr(), N, b.data_ptr(), y.data_ptr(), _lib.BF16, N + pad_y,
                                             ws.data_ptr(), need.value, st))
        scaled = ((x.float() @ w.float().t()).bfloat16().float() * s.float()).bfloat16()
        want = (scaled.float() + b.float()).bfloat16()
    else:
        packed, qp = ops.int4wo_quantize_pack((torch.randn(N, K, device="cuda", generator=g) * 0.02).bfloat16(), 64)
        _lib.check(L.ao_amd_int4wo_linear_auto_bytes(x.data_ptr(), M, K, K + 24, N, 64, _lib.BF16, ctypes.byref(need)))
        ws = torch.full((need.value // 4,), float("nan"), device="cuda")
        _lib.check(L.ao_amd_int4wo_linear_auto(x.data_ptr(), M, K, K + 24, packed.data_ptr(), qp.data_ptr(), N, 64, b.data_ptr(), y.data_ptr(), _lib.BF16, N + pad_y,
                                               ws.data_ptr(), need.value, st))
        want = (x.float() @ ops.int4wo_dequantize(packed, qp, N, K, 64).float().t() + b.float()).bfloat16()
    assert need.value >= 2 * 4 * M * N   # (in parts)
    assert bool((y[:, N:] == 7.0).all())
    y = y[:, :N]
    assert torch.equal(y.isnan(), want.isnan()) and torch.equal(y.isinf(), want.isinf()) and torch.equal(y[y.isinf()], want[want.isinf()])
    ok = want.isfinite()
    # the bounds of _run, for the rows without a special value (up to 16384 products a sum)
    rel = ((y[ok].float() - want[ok].float()).norm() / want[ok].float().norm()).item()
    assert rel <= 1e-3 and (y[ok] != want[ok]).float().mean() <= 0.01, rel
