"""Prompt-sized Llama kernels (llama_prefill.hip) against fp32 references of the module chain, and the native pass against the
module-by-module model."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _call(name, *args):
    from ao_amd import _lib

    args = [a.data_ptr() if torch.is_tensor(a) else a for a in args]
    _lib.check(getattr(_lib.lib(), name)(*args, _lib.current_stream(torch.device("cuda"))))


def _rel(a, b):
    return ((a.float() - b.float()).norm() / b.float().norm()).item()


def _qkv(T, n_head, n_kv, dtype, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(T, (n_head + 2 * n_kv) * 128, device="cuda", generator=g).to(dtype)


# tile edges: 32 query rows a wave (64 a workgroup when the waves share a head), 32 positions a tile, every fourth one a group's
@pytest.mark.parametrize("T", [2, 31, 32, 33, 64, 65, 127, 129, 200])
@pytest.mark.parametrize("heads", [(8, 2), (8, 1), (3, 3), (4, 2)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_attention_matches_fp32(T, heads, dtype):
    """rotary embedding + cache write (bit-exact) and attention over an already filled part of the cache.  fp32 reference
    on the same 16-bit inputs; the kernel rounds the probabilities and the output to the type: 2^-9 (bf16) and 2^-12 each,
    relative L2 within 2^-8 / 2^-11."""
    from ao_amd._models.llama.model import apply_rotary_emb, precompute_freqs_cis

    n_head, n_kv = heads
    start, S = 37, T + 37 + 3
    qkv = _qkv(T, n_head, n_kv, dtype)
    freqs = precompute_freqs_cis(S, 128, dtype=dtype, device="cuda")
    pos = torch.arange(start, start + T, device="cuda")
    g = torch.Generator(device="cuda").manual_seed(1)
    kc = torch.randn(n_kv, S, 128, device="cuda", generator=g).to(dtype)
    vc = torch.randn(n_kv, S, 128, device="cuda", generator=g).to(dtype)
    q, k, v = qkv.view(T, n_head + 2 * n_kv, 128).split([n_head, n_kv, n_kv], 1)
    q = apply_rotary_emb(q[None], freqs[pos])[0]
    k_want, v_want = kc.clone(), vc.clone()
    k_want[:, pos] = apply_rotary_emb(k[None], freqs[pos])[0].transpose(0, 1)
    v_want[:, pos] = v.transpose(0, 1)
    out = torch.full((T, n_head * 128), 7.0, device="cuda", dtype=dtype)
    for p in (pos, pos.int()):
        _call("ao_amd_llama_prefill_attention", qkv, int(dtype is torch.float16), freqs, p, int(p.dtype is torch.int64), T, kc, vc,
              n_head, n_kv, 128, S, out)
        assert torch.equal(kc, k_want) and torch.equal(vc, v_want)
        rep = n_head // n_kv
        s = torch.einsum("thd,hsd->hts", q.float(), k_want.float().repeat_interleave(rep, 0)) / math.sqrt(128)
        s.masked_fill_(torch.arange(S, device="cuda")[None, None, :] > pos[None, :, None], float("-inf"))
        want = torch.einsum("hts,hsd->thd", s.softmax(-1), v_want.float().repeat_interleave(rep, 0)).reshape(T, -1)
        assert _rel(out, want) <= (2 ** -8 if dtype is torch.bfloat16 else 2 ** -11)


def test_attention_scattered_and_foreign_positions():
    """Positions need not be consecutive; one outside the cache writes no cache row and leaves a NaN output row."""
    from ao_amd._models.llama.model import precompute_freqs_cis

    T, S, n_head, n_kv = 5, 96, 4, 1
    qkv = _qkv(T, n_head, n_kv, torch.bfloat16)
    freqs = precompute_freqs_cis(S, 128, device="cuda")
    kc, vc = torch.zeros(n_kv, S, 128, device="cuda").bfloat16(), torch.zeros(n_kv, S, 128, device="cuda").bfloat16()
    out = torch.zeros(T, n_head * 128, device="cuda").bfloat16()
    pos = torch.tensor([70, 3, -1, S, 0], device="cuda")
    _call("ao_amd_llama_prefill_attention", qkv, 0, freqs, pos, 1, T, kc, vc, n_head, n_kv, 128, S, out)
    assert out[2:4].isnan().all() and not out[[0, 1, 4]].isnan().any()
    written = kc[0].abs().sum(-1) > 0
    assert written.nonzero().view(-1).tolist() == [0, 3, 70]
    assert torch.equal(out[4].view(n_head, 128), vc[0, :1].expand(n_head, 128))  # sees position 0 only


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,dim", [(1, 8), (3, 2048), (5, 2056), (2, 8192)])
def test_add_rmsnorm_and_silu_mul(rows, dim, dtype):
    """Same roundings as the modules: the sum bit for bit.  A statistic or exponential that differs in the last fp32 bit moves
    the first rounding of a value by at most one step (relative 2^-7 / 2^-10), which the second rounding can widen by one
    more, and by one step of the subnormals (2^-24): few values, and at most two steps each."""
    import torch.nn.functional as F

    from ao_amd._models.llama.model import RMSNorm

    g = torch.Generator(device="cuda").manual_seed(dim)
    x, y = (torch.randn(rows, dim, device="cuda", generator=g).to(dtype) for _ in range(2))
    norm = RMSNorm(dim).to("cuda", dtype)
    with torch.no_grad():
        norm.weight.normal_(1.0, 0.1, generator=g)
        h, n = torch.empty_like(x), torch.empty_like(x)
        _call("ao_amd_add_rmsnorm", x, y, norm.weight, int(dtype is torch.float16), rows, dim, 1e-5, h, n)
        assert torch.equal(h, x + y)
        want = norm(x + y)
        step = 2 ** (-7 if dtype is torch.bfloat16 else -10)
        assert ((n.float() - want.float()).abs() <= 2 * step * want.float().abs() + 2 ** -24).all() and (n != want).float().mean() <= 0.02
        want = F.silu(x) * y
        _call("ao_amd_silu_mul", x, y, int(dtype is torch.float16), rows * dim, x)  # in place over the gate
        assert ((x.float() - want.float()).abs() <= 2 * step * want.float().abs() + 2 ** -24).all() and (x != want).float().mean() <= 0.02


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_silu_mul_over_all_values(dtype):
    """Every finite 16-bit gate and the special ones, times one.  fp32 within a few steps of 2^-24, rounded once: one step of the type at most,
    few values off; below 2^-100 an absolute bound (F.silu's own e^-x overflows there)."""
    x = torch.arange(65536, device="cuda", dtype=torch.int32).to(torch.int16).view(dtype)
    want = (x.double() / (1 + torch.exp(-x.double()))).to(dtype)
    out = torch.empty_like(x)
    _call("ao_amd_silu_mul", x, torch.ones_like(x), int(dtype is torch.float16), x.numel(), out)
    assert torch.equal(out.isnan(), want.isnan())
    ok = ~want.isnan()
    a, b = out[ok].double(), want[ok].double()
    infinite = b.isinf()
    assert torch.equal(a[infinite], b[infinite])
    a, b = a[~infinite], b[~infinite]
    step = 2.0 ** (-7 if dtype is torch.bfloat16 else -10)
    assert ((a - b).abs() <= step * b.abs() + (2.0 ** -100 if dtype is torch.bfloat16 else 2.0 ** -24)).all() and (a != b).double().mean() <= 0.02


@pytest.mark.parametrize("special", [0.0, 69.0, -100.0, float("inf"), float("nan")])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_silu_mul_beside_special_values(dtype, special):
    """Waves of ordinary values (0 < |gate| < 69) leave out what zeros, infinities and large values need; one such value among them changes
    no other's bits.  Every ordinary value, the nearest 16 bits of the fp32 function but for ties that fp32 rounds onto."""
    x = torch.arange(65536, device="cuda", dtype=torch.int32).to(torch.int16).view(dtype)
    x = x[(x != 0) & (x.abs() < 69)]
    x = x[: len(x) // 512 * 512]
    y = x.clone()
    y[5::512] = special
    out = []
    for gate in (x, y):
        out.append(torch.empty_like(gate))
        _call("ao_amd_silu_mul", gate, torch.ones_like(gate), int(dtype is torch.float16), gate.numel(), out[-1])
    same = torch.ones_like(x, dtype=torch.bool)
    same[5::512] = False
    assert torch.equal(out[0][same], out[1][same])
    want = (x.double() / (1 + torch.exp(-x.double()))).to(dtype)
    normal = want.abs() >= torch.finfo(dtype).tiny
    assert (out[0] != want)[normal].sum() <= 2


@pytest.mark.parametrize("rise", [0.4, 6.0, 60.0])
@pytest.mark.parametrize("heads,dtype", [((4, 2), torch.bfloat16), ((3, 3), torch.float16)])
def test_attention_with_rising_scores(rise, heads, dtype):
    """Scores that grow by `rise` every 32 positions, so that every tile raises a row's maximum, by little or by far; and the same ones
    falling, where no tile after a group's first does.  Bound as in test_attention_matches_fp32, doubled for the sums of few large terms."""
    n_head, n_kv = heads
    T = S = 321
    qkv = _qkv(T, n_head, n_kv, dtype) * 0.25
    qkv.view(T, -1, 128)[:, :n_head, 0] = 8.0   # the queries' share of the ramp
    freqs = torch.zeros(S, 64, 2, device="cuda", dtype=dtype)
    freqs[..., 0] = 1.0                         # no rotation
    pos = torch.arange(T, device="cuda")
    for sign in (1, -1):
        qkv.view(T, -1, 128)[:, n_head:n_head + n_kv, 0] = (sign * rise * math.sqrt(128) / 8.0 / 32 * pos)[:, None].to(dtype)
        kc, vc = (torch.zeros(n_kv, S, 128, device="cuda", dtype=dtype) for _ in range(2))
        out = torch.empty(T, n_head * 128, device="cuda", dtype=dtype)
        _call("ao_amd_llama_prefill_attention", qkv, int(dtype is torch.float16), freqs, pos, 1, T, kc, vc, n_head, n_kv, 128, S, out)
        later = torch.ones(T, T, device="cuda", dtype=torch.bool).triu(1)
        for h in range(n_head):
            kv = h * n_kv // n_head
            s = (qkv.view(T, -1, 128)[:, h].float() @ kc[kv].float().t().contiguous() / math.sqrt(128)).masked_fill_(later, float("-inf"))
            want = s.softmax(-1) @ vc[kv].float()
            assert _rel(out.view(T, n_head, 128)[:, h], want) <= 2 * (2 ** -8 if dtype is torch.bfloat16 else 2 ** -11)


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("T", [1, 63, 64])
def test_embed(T, dtype):
    table = torch.randn(100, 264, device="cuda").bfloat16()
    tok = torch.randint(0, 100, (T,), device="cuda", dtype=dtype)
    tok[T // 2] = 100
    out = torch.zeros(T, 264, device="cuda").bfloat16()
    _call("ao_amd_llama_embed", tok, int(dtype is torch.int64), T, table, 100, 264, out)
    keep = [i for i in range(T) if i != T // 2]
    assert torch.equal(out[keep], table[tok[keep].long()]) and out[T // 2].isnan().all()


@pytest.mark.parametrize("quantization", ["int4wo-64", "int8wo", "fp6"])
@pytest.mark.parametrize("T", [2, 17, 130])
def test_native_pass_is_the_module_chain(quantization, T):
    """A prompt and a decode step through the native pass against the modules: same roundings, other summation orders (the
    bound of the decode tests: 3e-2), and the same caches; hooks on a module put the prompt back on the module chain."""
    from ao_amd._models.llama.generate import build_random_model

    model = build_random_model("tiny128", torch.device("cuda"), quantization)
    model.setup_caches(1, 160)
    g = torch.Generator(device="cuda").manual_seed(T)
    tok = torch.randint(0, model.config.vocab_size, (1, T + 1), device="cuda", generator=g)
    pos = torch.arange(T, device="cuda")
    nxt = torch.tensor([T], device="cuda", dtype=torch.int32)
    caches = [c for b in model.layers for c in (b.attention.kv_cache.k_cache, b.attention.kv_cache.v_cache)]

    def both():
        for c in caches:
            c.zero_()
        with torch.no_grad():
            return [model(tok[:, :T], pos), model(tok[:, T:].int(), nxt)] + [c.clone() for c in caches]

    got = both()
    seen = []
    hook = model.layers[1].feed_forward.w2.register_forward_hook(lambda *a: seen.append(1))
    both()
    assert len(seen) == 1  # the prompt; the single token never calls modules
    hook.remove()
    model.use_fused_decode = False
    for a, b in zip(got, both()):
        assert a.shape == b.shape and a.dtype is b.dtype and _rel(a, b) <= 3e-2


@pytest.mark.parametrize("T", [1, 33, 130])
@pytest.mark.parametrize("heads", [(4, 1), (3, 3)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("long", [False, True])
def test_attention_with_negative_positions(T, heads, dtype, long):
    """Counted from the end: bit for bit the other entry at the rows they mean, whose rotary rows stand at those rows in a table of
    its own; a position beyond either end writes no cache row and leaves a NaN row."""
    from ao_amd._models.llama.model import precompute_freqs_cis

    n_head, n_kv = heads
    S, F = 160, 200
    qkv = _qkv(T, n_head, n_kv, dtype)
    freqs = precompute_freqs_cis(F, 128, dtype=dtype, device="cuda")
    rows = torch.randperm(S, device="cuda", generator=torch.Generator(device="cuda").manual_seed(T))[:T]
    negative = torch.arange(T, device="cuda") % 3 == 0
    pos = torch.where(negative, rows - S, rows)
    if T > 1:
        pos[-1], rows[-1], pos[-2], rows[-2] = -S - 1, S, S, S
    own = torch.zeros(S + 1, 64, 2, device="cuda", dtype=dtype)
    own[rows] = freqs[pos.clamp(-F, F - 1)]
    results = []
    for wrap in (True, False):
        kc, vc = (torch.ones(n_kv, S, 128, device="cuda", dtype=dtype) for _ in range(2))
        out = torch.full((T, n_head * 128), 7.0, device="cuda", dtype=dtype)
        p = pos if wrap else rows
        p = p if long else p.int()
        _call("ao_amd_llama_prefill_attention" + ("_wrap" if wrap else ""), qkv, int(dtype is torch.float16), freqs if wrap else own,
              *([F] if wrap else []), p, int(long), T, kc, vc, n_head, n_kv, 128, S, out)
        results.append((out, kc, vc))
    bad = 2 if T > 1 else 0
    for a, b in zip(*results):
        assert torch.equal(a.nan_to_num(9.0), b.nan_to_num(9.0))
    assert results[0][0].isnan().all(1).sum() == bad == results[0][0].isnan().any(1).sum()


@pytest.mark.parametrize("T,heads", [(1025, (8, 2)), (4096, (4, 1)), (2049, (3, 3))])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_long_attention_matches_fp32(T, heads, dtype):
    """As test_attention_matches_fp32, over 33 to 128 tiles of positions; one query head at a time in fp32."""
    from ao_amd._models.llama.model import apply_rotary_emb, precompute_freqs_cis

    n_head, n_kv = heads
    qkv = _qkv(T, n_head, n_kv, dtype)
    freqs = precompute_freqs_cis(T, 128, dtype=dtype, device="cuda")
    pos = torch.arange(T, device="cuda")
    kc, vc = (torch.zeros(n_kv, T, 128, device="cuda", dtype=dtype) for _ in range(2))
    out = torch.empty(T, n_head * 128, device="cuda", dtype=dtype)
    _call("ao_amd_llama_prefill_attention", qkv, int(dtype is torch.float16), freqs, pos, 1, T, kc, vc, n_head, n_kv, 128, T, out)
    q = apply_rotary_emb(qkv.view(1, T, -1, 128)[:, :, :n_head], freqs)[0].float()
    later = torch.ones(T, T, device="cuda", dtype=torch.bool).triu(1)
    for h in range(n_head):
        kv = h * n_kv // n_head
        s = (q[:, h] @ kc[kv].float().t().contiguous() / math.sqrt(128)).masked_fill_(later, float("-inf"))
        want = s.softmax(-1) @ vc[kv].float()
        assert _rel(out.view(T, n_head, 128)[:, h], want) <= (2 ** -8 if dtype is torch.bfloat16 else 2 ** -11)


@pytest.mark.parametrize("T,heads", [(257, (64, 16)), (288, (64, 8)), (1030, (32, 8)), (257, (128, 128)), (352, (132, 22)), (386, (90, 90))])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_attention_of_many_workgroups(T, heads, dtype):
    """The kernel whose tiles serve 128 rows (four heads of 32, or 128 of one): rows and a cache that end within its blocks and tiles, positions in
    any order, two of them outside.  Bound as in test_attention_matches_fp32."""
    from ao_amd._models.llama.model import apply_rotary_emb, precompute_freqs_cis

    n_head, n_kv = heads
    S = T + 9
    qkv = _qkv(T, n_head, n_kv, dtype)
    freqs = precompute_freqs_cis(S, 128, dtype=dtype, device="cuda")
    g = torch.Generator(device="cuda").manual_seed(T)
    pos = torch.randperm(S, device="cuda", generator=g)[:T]
    rows = torch.arange(T, device="cuda") % 100 != 40
    pos[~rows] = S
    kc, vc = (torch.randn(n_kv, S, 128, device="cuda", generator=g).to(dtype) for _ in range(2))
    k_want, v_want = kc.clone(), vc.clone()
    q, k, v = qkv.view(T, n_head + 2 * n_kv, 128)[rows].split([n_head, n_kv, n_kv], 1)
    q = apply_rotary_emb(q[None], freqs[pos[rows]])[0].float()
    k_want[:, pos[rows]] = apply_rotary_emb(k[None], freqs[pos[rows]])[0].transpose(0, 1)
    v_want[:, pos[rows]] = v.transpose(0, 1)
    out = torch.full((T, n_head * 128), 7.0, device="cuda", dtype=dtype)
    _call("ao_amd_llama_prefill_attention", qkv, int(dtype is torch.float16), freqs, pos, 1, T, kc, vc, n_head, n_kv, 128, S, out)
    assert torch.equal(kc, k_want) and torch.equal(vc, v_want) and out[~rows].isnan().all()
    later = torch.arange(S, device="cuda")[None, :] > pos[rows, None]
    for h in range(n_head):
        kv = h * n_kv // n_head
        s = (q[:, h] @ kc[kv].float().t().contiguous() / math.sqrt(128)).masked_fill_(later, float("-inf"))
        want = s.softmax(-1) @ vc[kv].float()
        assert _rel(out.view(T, n_head, 128)[rows, h], want) <= (2 ** -8 if dtype is torch.bfloat16 else 2 ** -11)
