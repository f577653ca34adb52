"""ao_amd_int4wo_linear_ws: the int4 linear with a caller-owned workspace, which splits K over workgroups where the tiles
of 17-256 rows leave most CUs idle (same product as ao_amd_int4wo_linear, `aten::_weight_int4pack_mm` as called from
torchao/dtypes/affine_quantized_tensor.py:600-640, summed in another order).  Checked through the C ABI: against the
fp32-accumulated product with the dequantized weight (<= 1e-3 relative L2 after the bf16 rounding, 2e-5 for fp32 output),
one-hot rows bit for bit against ao_amd_int4wo_dequantize, and against the plain entry point."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def _setup(N, K, g, seed):
    from ao_amd import ops
    dev = torch.device("cuda:0")
    w = (torch.randn(N, K, generator=torch.Generator().manual_seed(seed)) * 0.02).bfloat16().to(dev)
    packed, qp = ops.int4wo_quantize_pack(w, g)
    dq = ops.int4wo_dequantize(packed, qp, N, K, g)
    return packed, qp, dq


def _ws_call(x, packed, qp, N, g, bias, fp32, ws_bytes_override=None):
    from ao_amd import _lib
    L = _lib.lib()
    M, K = x.shape
    need = ctypes.c_int64(-1)
    _lib.check(L.ao_amd_int4wo_linear_ws_bytes(M, K, N, g, ctypes.byref(need)))
    nbytes = need.value if ws_bytes_override is None else ws_bytes_override
    ws = torch.empty(max(nbytes // 4, 1), dtype=torch.float32, device=x.device)
    y = torch.empty(M, N, dtype=torch.float32 if fp32 else torch.bfloat16, device=x.device)
    rc = L.ao_amd_int4wo_linear_ws(x.data_ptr(), M, K, x.stride(0), packed.data_ptr(), qp.data_ptr(), N, g,
                                   None if bias is None else bias.data_ptr(), y.data_ptr(), _lib.F32 if fp32 else _lib.BF16, N,
                                   ws.data_ptr() if nbytes else None, nbytes, torch.cuda.current_stream().cuda_stream)
    return rc, y, need.value


# (N, K, g, M, parts the rule gives)
CASES = [
    (4096, 14336, 64, 16, 4), (4096, 14336, 64, 24, 4), (4096, 14336, 64, 32, 4), (4096, 14336, 64, 64, 4),
    (4096, 14336, 64, 100, 2), (4096, 14336, 64, 128, 2), (4096, 14336, 64, 8, 1), (4096, 14336, 64, 256, 1),
    (4096, 4096, 128, 32, 4), (4096, 4096, 128, 64, 4), (4096, 4096, 128, 128, 1), (4096, 4096, 128, 16, 1),
    (6144, 4096, 32, 32, 2), (6144, 4096, 32, 16, 1), (6144, 4096, 32, 64, 1),
    (1024, 4096, 256, 128, 4), (1024, 4096, 256, 256, 4), (1024, 4096, 256, 64, 1),
    (14336, 4096, 64, 32, 1), (4100, 8192, 64, 40, 2), (4099, 8192, 64, 40, 2),
]


@pytest.mark.parametrize("N,K,g,M,parts", CASES)
def test_workspace_linear_matches_the_plain_one_and_the_fp32_product(N, K, g, M, parts):
    from ao_amd import _lib
    print(f"case int4wo_linear_ws N={N} K={K} g={g} M={M} parts={parts}", flush=True)
    L = _lib.lib()
    dev = torch.device("cuda:0")
    assert L.ao_amd_int4wo_linear_ws_parts(M, K, N, g) == parts
    packed, qp, dq = _setup(N, K, g, seed=N + K + g)
    gen = torch.Generator().manual_seed(M)
    x = torch.randn(M, K, generator=gen).bfloat16().to(dev)
    bias = torch.randn(N, generator=gen).bfloat16().to(dev)
    for b in (None, bias):
        for fp32 in (False, True):
            rc, y, need = _ws_call(x, packed, qp, N, g, b, fp32)
            assert rc == 0, L.ao_amd_last_error()
            assert need == (parts * M * N * 4 if parts > 1 else 0)
            ref = x.float() @ dq.float().t() + (0 if b is None else b.float())
            if not fp32:
                ref = ref.bfloat16().float()
            err = float((y.float() - ref).norm() / ref.norm())
            assert err <= (2e-5 if fp32 else 1e-3), (err, fp32)
            y0 = torch.empty_like(y)
            _lib.check(L.ao_amd_int4wo_linear(x.data_ptr(), M, K, K, packed.data_ptr(), qp.data_ptr(), N, g,
                                              None if b is None else b.data_ptr(), y0.data_ptr(),
                                              _lib.F32 if fp32 else _lib.BF16, N, torch.cuda.current_stream().cuda_stream))
            if parts == 1 or N % 4:
                same = bool(torch.equal(y, y0))   # no split (N = 4099: partial rows need a multiple of 4): the same launch
                assert same
            else:
                d = float((y.float() - y0.float()).norm() / y0.float().norm())
                assert d <= (2e-5 if fp32 else 1e-3), d
    # one-hot rows read single columns of the dequantized weight back, bit for bit (the other parts add exact zeros)
    ks = torch.randint(0, K, (M,), generator=gen)
    ks[0], ks[-1] = 0, K - 1
    xh = torch.zeros(M, K, dtype=torch.bfloat16)
    xh[torch.arange(M), ks] = 1.0
    rc, yh, _ = _ws_call(xh.to(dev), packed, qp, N, g, None, False)
    assert rc == 0
    exact = bool(torch.equal(yh, dq[:, ks.to(dev)].t().contiguous()))
    assert exact


def test_workspace_linear_refusals_and_fallbacks():
    from ao_amd import _lib, ops
    L = _lib.lib()
    dev = torch.device("cuda:0")
    N, K, g, M = 4096, 8192, 64, 32
    packed, qp, dq = _setup(N, K, g, seed=5)
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(6)).bfloat16().to(dev)
    rc, _, need = _ws_call(x, packed, qp, N, g, None, False, ws_bytes_override=1024)
    assert rc != 0 and need == 4 * M * N * 4 and b"workspace" in L.ao_amd_last_error()
    # rows that are not 16-byte aligned: the plain kernels take the call, the workspace is left alone
    xp = torch.zeros(M, K + 3, dtype=torch.bfloat16, device=dev)
    xp[:, :K] = x
    rc, y, _ = _ws_call(xp[:, :K], packed, qp, N, g, None, False)
    assert rc == 0
    ref = (x.float() @ dq.float().t()).bfloat16().float()
    assert float((y.float() - ref).norm() / ref.norm()) <= 1e-3
    # the operator takes the same route: same bits as the C call with a workspace
    rc, y_ws, _ = _ws_call(x, packed, qp, N, g, None, False)
    assert rc == 0 and bool(torch.equal(ops.int4wo_linear(x, packed, qp, g, N), y_ws))


# (N, K, group, M, K parts): an even split and a last part that is shorter; row blocks that are no multiple of four, the last one with 4 rows;
# more workgroups than CUs; rows that end before the packed width, read as they are (up to 15) and copied; g = 256 with a packed tile that no row
# reaches (and which makes 50 tiles, eight parts, of 49, which have no eight of one length); 4, 16, 17 and 32 rows; and neighbours of those calls that are not split
@pytest.mark.parametrize("N,K,g,M,parts", [
    (8192, 8192, 64, 16, 2), (5120, 13824, 64, 4, 1), (5120, 13824, 64, 6, 3), (5120, 13824, 32, 13, 3), (5120, 13824, 128, 17, 3),
    (5120, 13824, 64, 32, 3), (5120, 13824, 64, 33, 0), (10240, 8192, 64, 16, 3), (1000, 14336, 128, 16, 8), (2052, 16384, 256, 16, 7),
    (5000, 8000, 256, 13, 3), (5000, 8000, 256, 20, 3), (2048, 6272, 256, 15, 7), (5120, 13768, 128, 15, 3), (5120, 13768, 128, 18, 3), (4096, 4096, 64, 16, 1)])
def test_few_rows_of_narrow_weights_in_parts(N, K, g, M, parts):
    from ao_amd import _lib, ops

    print(f"case int4 rows in parts N={N} K={K} g={g} M={M} parts={parts}", flush=True)
    L, need = _lib.lib(), ctypes.c_int64(-1)
    packed, qp, dq = _setup(N, K, g, seed=N + K + g)
    gen = torch.Generator().manual_seed(M)
    x, bias = torch.randn(M, K, generator=gen).bfloat16().cuda(), torch.randn(N, generator=gen).bfloat16().cuda()
    q = max(128, g)
    copy = 2 * M * (-(-K // q) * q) if K % q else 0
    if parts:   # (0: another route's)
        _lib.check(L.ao_amd_int4wo_linear_auto_bytes(x.data_ptr(), M, K, K, N, g, _lib.BF16, ctypes.byref(need)))
        assert need.value == copy + (4 * parts * M * N if parts > 1 else 0)
    for b in (None, bias):
        ref = x.float() @ dq.float().t() + (0 if b is None else b.float())
        y, y32 = ops.int4wo_linear(x, packed, qp, g, N, b), ops.int4wo_linear(x, packed, qp, g, N, b, True)
        # one rounding to bf16 (2^-9 / sqrt 3 relative, 1.1e-3 against the unrounded, almost nothing against the rounded sum); fp32 sums of K terms
        assert float((y.float() - ref.bfloat16().float()).norm() / ref.norm()) <= 1e-3
        assert float((y32 - ref).norm() / ref.norm()) <= 2e-5
    # one-hot rows read single columns of the dequantized weight back, bit for bit, at both ends of K and of every part
    ks = torch.randint(0, K, (M,), generator=gen)
    ks[0], ks[-1] = 0, K - 1
    if parts > 1:
        per = -(-(-(-K // 128)) // parts) * 128
        for z in range(1, parts):
            if 2 * z < M - 1:
                ks[2 * z - 1], ks[2 * z] = z * per - 1, z * per
    xh = torch.zeros(M, K, dtype=torch.bfloat16)
    xh[torch.arange(M), ks] = 1.0
    assert torch.equal(ops.int4wo_linear(xh.cuda(), packed, qp, g, N), dq[:, ks.cuda()].t().contiguous())


# (N, K, M, parts the rule gives) for ao_amd_fp6_linear_ws
FP6_CASES = [
    (4096, 14336, 16, 4), (4096, 14336, 32, 4), (4096, 14336, 64, 4), (4096, 14336, 100, 2), (4096, 14336, 256, 1),
    (4096, 4096, 32, 4), (4096, 4096, 64, 4), (4096, 4096, 128, 1), (4096, 4096, 16, 1),
    (6144, 4096, 32, 2), (6144, 4096, 64, 1), (1024, 4096, 40, 4), (1024, 4096, 256, 4), (14336, 4096, 32, 1),
    (4096, 8192 + 64, 32, 1),
]


@pytest.mark.parametrize("ebits,mbits", [(3, 2), (2, 3)])
@pytest.mark.parametrize("N,K,M,parts", FP6_CASES)
def test_fp6_workspace_linear(N, K, M, parts, ebits, mbits):
    """ao_amd_fp6_linear_ws (where torchao::quant_llm_linear takes splitK and a [splitK, M, N] workspace,
    torchao/csrc/cuda/fp6_llm/fp6_linear.cu:104-111, 167-168): <= 1e-3 relative L2 of the fp32 product with the dequantized
    weight rounded to fp16, one-hot rows bit for bit, and against the plain entry point.  K = 8256 is not a multiple of
    128: no split."""
    from ao_amd import _lib, ops
    print(f"case fp6_linear_ws N={N} K={K} M={M} parts={parts} e{ebits}m{mbits}", flush=True)
    L = _lib.lib()
    dev = torch.device("cuda:0")
    assert L.ao_amd_fp6_linear_ws_parts(M, K, N) == parts
    gen = torch.Generator().manual_seed(N + K + M)
    w = (torch.randn(N, K, generator=gen) * 0.05).half().to(dev)
    tc, scale = ops.fp6_quantize_pack(w, ebits, mbits)
    native = ops.fp6_repack(tc, 1 + ebits + mbits)
    wd = ops.fp6_dequantize(tc, scale, ebits, mbits).half()      # the kernels multiply fp16(value * scale)
    x = torch.randn(M, K, generator=gen).half().to(dev)
    st = torch.cuda.current_stream().cuda_stream

    def run(xin):
        need = ctypes.c_int64(-1)
        _lib.check(L.ao_amd_fp6_linear_ws_bytes(M, K, N, ctypes.byref(need)))
        assert need.value == (parts * M * N * 4 if parts > 1 else 0)
        ws = torch.empty(max(need.value // 4, 1), dtype=torch.float32, device=dev)
        y = torch.empty(M, N, dtype=torch.float16, device=dev)
        _lib.check(L.ao_amd_fp6_linear_ws(xin.data_ptr(), M, K, native.data_ptr(), scale.data_ptr(), N, ebits, mbits, y.data_ptr(),
                                          ws.data_ptr() if need.value else None, need.value, st))
        return y

    y = run(x)
    ref = (x.float() @ wd.float().t()).half().float()
    err = float((y.float() - ref).norm() / ref.norm())
    assert err <= 1e-3, err
    y0 = torch.empty_like(y)
    _lib.check(L.ao_amd_fp6_linear(x.data_ptr(), M, K, native.data_ptr(), scale.data_ptr(), N, ebits, mbits, y0.data_ptr(), st))
    if parts == 1:
        same = bool(torch.equal(y, y0))
        assert same
    else:
        d = float((y.float() - y0.float()).norm() / y0.float().norm())
        assert d <= 1e-3, d
        # the operator takes the same route
        same = bool(torch.equal(ops.fp6_linear_native(ebits, mbits, x, native, scale), y))
        assert same
    ks = torch.randint(0, K, (M,), generator=gen)
    ks[0], ks[-1] = 0, K - 1
    xh = torch.zeros(M, K, dtype=torch.float16)
    xh[torch.arange(M), ks] = 1.0
    yh = run(xh.to(dev))
    exact = bool(torch.equal(yh, wd[:, ks.to(dev)].t().contiguous()))
    assert exact


# (N, K, M, K parts): every kind of split (four row blocks a workgroup up to 32 rows, tiles of 64 and of 128 columns from 17 and 33 rows on) at the first and
# last row counts of its kernels, a shorter last part, more workgroups than CUs, row blocks that fill neither four nor eight
@pytest.mark.parametrize("ebits,mbits", [(3, 2), (2, 3)])
@pytest.mark.parametrize("N,K,M,parts", [
    (5120, 13824, 4, 3), (5120, 13824, 16, 3), (5120, 13824, 17, 3), (5120, 13824, 32, 3), (5120, 13824, 33, 6), (5120, 13824, 48, 6), (5120, 13824, 49, 6),
    (5120, 13824, 64, 6), (10240, 8192, 16, 3), (4096, 14336, 48, 8), (4096, 4096, 40, 4), (1024, 14336, 30, 8), (1024, 14336, 48, 8), (1024, 14336, 64, 8),
    (2064, 16384, 16, 7), (2064, 16384, 30, 7), (2064, 16384, 64, 7), (5008, 13824, 24, 3), (5008, 13824, 60, 6)])
def test_fp6_rows_in_parts(N, K, M, parts, ebits, mbits):
    from ao_amd import _lib, ops

    print(f"case fp6 rows in parts N={N} K={K} M={M} parts={parts} e{ebits}m{mbits}", flush=True)
    L, need = _lib.lib(), ctypes.c_int64(-1)
    _lib.check(L.ao_amd_fp6_linear_auto_bytes(M, K, N, ctypes.byref(need)))
    assert need.value == 4 * parts * M * N
    n = -(-N // 64) * 64   # the interchange format's rows; the kernels take a multiple of 16 of them
    data, scale = ops.fp6_quantize_pack((torch.randn(n, K, generator=torch.Generator().manual_seed(N)) * 0.02).half().cuda(), ebits, mbits)
    native, w = ops.fp6_repack(data, 6).flatten()[: N // 16 * (K // 128) * 384], ops.fp6_dequantize(data, scale, ebits, mbits)[:N].half()
    scale = scale[:N].contiguous()
    gen = torch.Generator().manual_seed(M)
    x = torch.randn(M, K, generator=gen).half().cuda()
    y = ops.fp6_linear_native(ebits, mbits, x, native, scale)
    ref = (x.float() @ w.float().t()).half().float()
    # one rounding to fp16 (2^-12 / sqrt 3 relative) and fp32 sums in another order: 1e-3 is what the other routes are held to
    assert float((y.float() - ref).norm() / ref.norm()) <= 1e-3
    # one-hot rows read single columns of the weight back, at both ends of K and of every part
    per = -(-(K // 128) // parts) * 128
    ends = [0, K - 1] + [k for z in range(1, parts) for k in (z * per - 1, z * per)]
    ks = torch.tensor([ends[i % len(ends)] for i in range(M)])
    xh = torch.zeros(M, K, dtype=torch.float16)
    xh[torch.arange(M), ks] = 1.0
    assert torch.equal(ops.fp6_linear_native(ebits, mbits, xh.cuda(), native, scale), w[:, ks.cuda()].t().contiguous())


# outputs that begin at any fp16 element: every way of splitting K, and one row count of each that is not split, in the middle of a larger buffer
@pytest.mark.parametrize("N,K,M", [(5120, 13824, 4), (5120, 13824, 12), (5120, 13824, 24), (5120, 13824, 48), (1024, 14336, 64), (4096, 4096, 8)])
@pytest.mark.parametrize("at", [1, 2, 3])
def test_fp6_output_at_any_element(N, K, M, at):
    from ao_amd import _lib, ops

    print(f"case fp6 output at {at} N={N} K={K} M={M}", flush=True)
    L, need = _lib.lib(), ctypes.c_int64(-1)
    data, scale = ops.fp6_quantize_pack((torch.randn(N, K, generator=torch.Generator().manual_seed(N)) * 0.02).half().cuda(), 3, 2)
    native = ops.fp6_repack(data, 6)
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(M)).half().cuda()
    _lib.check(L.ao_amd_fp6_linear_ws_bytes(M, K, N, ctypes.byref(need)))
    ws = _empty_ws(need.value)

    def run(out):
        _lib.check(L.ao_amd_fp6_linear_ws(x.data_ptr(), M, K, native.data_ptr(), scale.data_ptr(), N, 3, 2, out.data_ptr(), ws.data_ptr(), need.value,
                                          torch.cuda.current_stream().cuda_stream))

    want, buf = torch.empty(M * N, dtype=torch.float16, device="cuda"), torch.full((M * N + 8,), 7.0, dtype=torch.float16, device="cuda")
    run(want)
    run(buf[at:])
    assert torch.equal(buf[at:at + M * N], want)   # the same sums, stored in other pieces
    assert bool((buf[:at] == 7.0).all()) and bool((buf[at + M * N:] == 7.0).all())


# Calls with less workspace than the query says, down to what the way needs that they then take (none below 16 rows): int4 in streamed parts, in streamed parts
# of rows that are copied first, and on tiles; FP6 on four row blocks and on tiles.  With less than that a call is refused.
@pytest.mark.parametrize("fmt,N,K,M,less", [
    ("int4", 5120, 13824, 10, 0), ("int4", 5120, 13768, 14, 0), ("int4", 2048, 16384, 40, 0), ("int4", 5120, 13824, 24, 2), ("int4", 5120, 13824, 48, 2),
    ("fp6", 5120, 13824, 10, 0), ("fp6", 1024, 14336, 6, 0), ("fp6", 5120, 13824, 24, 2), ("fp6", 2064, 16384, 60, 4)])
def test_few_rows_with_less_workspace(fmt, N, K, M, less):
    from ao_amd import _lib, ops

    print(f"case less workspace {fmt} N={N} K={K} M={M} less={less}", flush=True)
    L, need, g = _lib.lib(), ctypes.c_int64(-1), 128
    st = torch.cuda.current_stream().cuda_stream
    gen = torch.Generator().manual_seed(M + N)
    if fmt == "int4":
        packed, qp, w = _setup(N, K, g, seed=N + K)
        x, w = torch.randn(M, K, generator=gen).bfloat16().cuda(), w.float()
        query = lambda: L.ao_amd_int4wo_linear_auto_bytes(x.data_ptr(), M, K, K, N, g, _lib.BF16, ctypes.byref(need))
        call = lambda y, ws, n: L.ao_amd_int4wo_linear_auto(x.data_ptr(), M, K, K, packed.data_ptr(), qp.data_ptr(), N, g, None, y.data_ptr(), _lib.BF16, N, ws, n, st)
    else:
        data, scale = ops.fp6_quantize_pack((torch.randn((N + 63) // 64 * 64, K, generator=gen) * 0.02).half().cuda(), 3, 2)
        native, w = ops.fp6_repack(data, 6), ops.fp6_dequantize(data, scale, 3, 2)[:N].half().float()
        x = torch.randn(M, K, generator=gen).half().cuda()
        query = lambda: L.ao_amd_fp6_linear_ws_bytes(M, K, N, ctypes.byref(need))
        call = lambda y, ws, n: L.ao_amd_fp6_linear_ws(x.data_ptr(), M, K, native.data_ptr(), scale.data_ptr(), N, 3, 2, y.data_ptr(), ws, n, st)
    _lib.check(query())
    copy = 2 * M * (-(-K // g) * g) if fmt == "int4" and K % g else 0
    room = copy + 4 * less * M * N
    assert need.value > room
    ref = x.float() @ w.t()
    ws = _empty_ws(need.value)
    for ptr, n in ((ws.data_ptr(), need.value), (ws.data_ptr(), need.value - 16), (ws.data_ptr() if room else None, room)):
        y = torch.full((M, N), float("nan"), device="cuda").to(x.dtype)
        _lib.check(call(y, ptr, n))
        assert float((y.float() - ref.to(x.dtype).float()).norm() / ref.norm()) <= 1e-3   # one rounding of fp32 sums in another order, as in the tests above
    if room:
        assert call(y, ws.data_ptr(), room - 16) != 0 and b"workspace" in L.ao_amd_last_error()


def _empty_ws(nbytes):
    return torch.empty(max(nbytes, 16), dtype=torch.uint8, device="cuda")


# (N, K, group, M, offset of the rows in elements, route)
@pytest.mark.parametrize("N,K,g,M,shift,route", [
    (4096, 4096, 64, 1, 0, "ws"), (4096, 14336, 64, 32, 0, "ws"), (256, 200, 64, 3, 4, "ws"), (1024, 704, 128, 33, 0, "ws"),
    (4096, 4096, 64, 160, 0, "tiled"), (4096, 14336, 64, 160, 0, "tiled"), (4096, 4160, 64, 6, 0, "copied"),
    (4096, 4096, 64, 6, 1, "copied"), (4096, 14208, 256, 32, 0, "copied")])
@pytest.mark.parametrize("fp32", [False, True])
def test_the_one_entry_picks_these_routes(N, K, g, M, shift, route, fp32):
    """ao_amd_int4wo_linear_auto is bit for bit the entry that its rule names, with a workspace of exactly the bytes it asks for."""
    from ao_amd import _lib

    L, code, st = _lib.lib(), _lib.F32 if fp32 else _lib.BF16, torch.cuda.current_stream().cuda_stream
    packed, qp, _ = _setup(N, K, g, 3)
    x = torch.randn(M * K + shift, device="cuda").bfloat16()[shift:].view(M, K)
    bias = torch.randn(N, device="cuda").bfloat16()
    need = ctypes.c_int64(-1)

    def call(name, x, nbytes, ws, *y_dtype):
        y = torch.zeros(M, N, device="cuda", dtype=torch.float32 if fp32 else torch.bfloat16)
        return getattr(L, name)(x.data_ptr(), M, x.shape[1], x.shape[1], packed.data_ptr(), qp.data_ptr(), N, g, bias.data_ptr(), y.data_ptr(),
                                *y_dtype, N, ws, nbytes, st), y

    _lib.check(L.ao_amd_int4wo_linear_auto_bytes(x.data_ptr(), M, K, K, N, g, code, ctypes.byref(need)))
    total, ws = need.value, _empty_ws(need.value)
    rc, got = call("ao_amd_int4wo_linear_auto", x, total, ws.data_ptr() if total else None, code)
    _lib.check(rc)
    if total:
        assert call("ao_amd_int4wo_linear_auto", x, total, None, code)[0] and call("ao_amd_int4wo_linear_auto", x, total - 1, ws.data_ptr(), code)[0]
    if route == "tiled" and not fp32:   # its output is bf16
        _lib.check(L.ao_amd_int4wo_linear_tiled_bytes(M, K, N, g, ctypes.byref(need)))
        assert need.value == total
        rc, want = call("ao_amd_int4wo_linear_tiled", x, total, ws.data_ptr())
    else:
        if route == "copied":
            q = max(128, g)
            x = torch.nn.functional.pad(x, (0, -K % q)).clone()
            assert x.data_ptr() % 16 == 0
        _lib.check(L.ao_amd_int4wo_linear_ws_bytes(M, x.shape[1], N, g, ctypes.byref(need)))
        assert total == need.value + (2 * x.numel() if route == "copied" else 0)
        ws = _empty_ws(need.value)
        rc, want = call("ao_amd_int4wo_linear_ws", x, need.value, ws.data_ptr(), code)
    _lib.check(rc)
    assert torch.equal(got, want)


@pytest.mark.parametrize("N,K,M,route", [(4096, 4096, 2, "ws"), (4096, 14336, 32, "ws"), (4096, 14336, 160, "tiled"), (14336, 4032, 33, "tiled")])
def test_the_one_fp6_entry_picks_these_routes(N, K, M, route):
    from ao_amd import _lib, ops

    L, st = _lib.lib(), torch.cuda.current_stream().cuda_stream
    data, scale = ops.fp6_quantize_pack((torch.randn(N, K, device="cuda") * 0.02).half(), 3, 2)
    native = ops.fp6_repack(data, 6)
    x = torch.randn(M, K, device="cuda").half()
    got, want = torch.zeros(M, N, device="cuda").half(), torch.ones(M, N, device="cuda").half()
    need, part = ctypes.c_int64(-1), ctypes.c_int64(-1)
    _lib.check(L.ao_amd_fp6_linear_auto_bytes(M, K, N, ctypes.byref(need)))
    _lib.check(getattr(L, f"ao_amd_fp6_linear_{route}_bytes")(M, K, N, ctypes.byref(part)))
    assert need.value == part.value >= 0
    ws = _empty_ws(need.value)
    for name, y in (("auto", got), (route, want)):
        _lib.check(getattr(L, f"ao_amd_fp6_linear_{name}")(x.data_ptr(), M, K, native.data_ptr(), scale.data_ptr(), N, 3, 2, y.data_ptr(),
                                                           ws.data_ptr(), need.value, st))
    assert torch.equal(got, want)
