// Mixed matmul over HQQ two-per-byte codes on 32 x 32 x 16 matrix instructions: y[M, N] = a[M, K] @ W[K, N] and, transposed,
// y[M, K] = a[M, N] @ W^T with W = (q - zero) * scale (torchao/prototype/hqq/kernels.py:162-388), for batches beyond the streaming
// kernels of hqq.hip.
//
// A workgroup computes 32 MT rows x 128 columns; its four waves take the 64-wide steps of the reduction round-robin, each over the
// whole tile (MT x 4 blocks of 32 x 32), and add up through LDS at the end: a weight is converted once per row tile, nothing is
// shared inside the loop and there is no barrier.  Both operands of a step come into the wave's own LDS by direct loads, 2 to 4
// steps ahead.  The byte layout [K/2, N] needs no transposition: the weight is the row operand of the matrix instruction, of which a
// lane holds 8 reduction indices of one output column for a slice of 16.
//   forward     lane (r, half) reads the dword of columns 4 r .. 4 r + 3 from the four byte rows of its 8 k; block c takes column c of
//               every dword, so that a lane ends with runs of 4 adjacent outputs;
//   transposed  lane (r, half) reads 32 bytes along n of byte row r of two groups of 32 byte rows; the low nibbles are the outputs
//               2 r of one block, the high ones 2 r + 1 of another.  A reduction that ends inside a step reads zeros beyond.
// What bounds it: the conversion, 4.1 (bf16) or 2.5 (fp16) VALU instructions a weight forward, 5.1 and 2.9 transposed, and the requests,
// 4 MT + 6 of 1 KB a step, each of which holds its wave's issue for some 120 cycles: 1.3 - 2.8 us a step.  96-row tiles convert
// each weight the least often.  11008 x 4096 at 96 rows 68 -> 28 us, 4096 x 4096 at 128 rows 44 -> 20, 12416 x 1600 at 425 rows 71 -> 41
// (dequantization and library product before).
#include <algorithm>
#include <type_traits>

#include "hqq_format.h"
#include "lds_dma.h"

namespace ao {

typedef float ht_f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 ht_bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 ht_f16x8 __attribute__((ext_vector_type(8)));

struct HqqTileArgs {
    const uint8_t* packed;
    const uint16_t *scales, *zeros, *a;
    int64_t lda, M, K, N, group;
    int tiles_m, tiles, per_xcd;
    uint32_t per_group;   // forward: 2^32 / (group / 64) rounded up, exact for the steps that hqq_tile_plan admits, or 0 where a step is a group
    float* part;      // [gridDim.y][M][columns], or null: y is written
    uint16_t* y;
};

// what the lanes past the end of the reduction read: 0 x (q - 0) * 0 adds nothing
__device__ const uint4 hqq_zeros = {0u, 0u, 0u, 0u};

template <int B, int E, class F>
__device__ __forceinline__ void ht_for(F&& f) {
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        ht_for<B + 1, E>(f);
    }
}

template <bool BF16, bool SIGNED, bool TR, int MT>
__global__ __launch_bounds__(256) void hqq_tile_kernel(const HqqTileArgs g) {
    constexpr int W = 4, BM = 32 * MT, BN = 128, SLOTS = 4 * MT;
    constexpr int NA = MT == 1 ? 4 : MT == 2 ? 3 : 2, NC = MT == 1 ? 4 : 3;   // steps in LDS: activations, codes
    constexpr int ASTEP = BM * 128, CSTEP = 4096 + 512;
    constexpr int AREQ = 4 * MT, CREQ = 6, REQ = AREQ + CREQ;
    constexpr int WAVE_LDS = NA * ASTEP + NC * CSTEP, SUM_LDS = 12 * MT * 4096;
    static_assert(WAVE_LDS * W <= 160 * 1024 && SUM_LDS <= 160 * 1024, "LDS of a CU");
    __shared__ __align__(1024) uint8_t lds[WAVE_LDS * W > SUM_LDS ? WAVE_LDS * W : SUM_LDS];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tile = (int)(blockIdx.x & 7) * g.per_xcd + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= g.per_xcd || tile >= g.tiles) return;
    // the row tiles of a weight tile are neighbours on one XCD, whose L2 then holds its codes
    const int tile_n = tile / g.tiles_m, tile_m = tile - tile_n * g.tiles_m;
    const int64_t m0 = (int64_t)tile_m * BM, c0 = (int64_t)tile_n * BN;   // first row, first output column
    const int64_t R = TR ? g.N : g.K, K2 = g.K / 2;
    const int all = (int)((R + 63) / 64), per = (all + (int)gridDim.y - 1) / (int)gridDim.y, first = per * (int)blockIdx.y;
    const int KS = min(per, all - first), nst = (KS - wave + W - 1) / W;   // this wave's steps: first + wave + 4 t
    const int r32 = lane & 31, half = lane >> 5;

    // activation request j: 8 rows x 128 bytes, slot (row, p) holds the 16-byte chunk p ^ (row / 2 % 8)
    uint32_t aoff[AREQ];
#pragma unroll
    for (int j = 0; j < AREQ; ++j) {
        const int row = 8 * j + (lane >> 3);
        const int64_t rel = (m0 + row < g.M ? m0 + row : g.M - 1) - m0;   // rows past M repeat the last one and are not stored
        aoff[j] = (uint32_t)(rel * g.lda * 2) + (((lane & 7) ^ ((row >> 1) & 7)) << 4);
    }
    const uint16_t* const abase = g.a + m0 * g.lda;
    // codes.  Forward: 8 byte rows x 128 columns a request.  Transposed: 16 byte rows x 64 columns a request, slot (row, p) holds
    // chunk p ^ (row / 4 % 4); two blocks of 32 byte rows.  Columns (byte rows) past the end repeat the last ones.
    uint32_t coff[4], soff;
    const uint8_t* cbase;
    const uint16_t *sbase, *zbase;
    if (TR) {
        const int64_t row0 = c0 / 2, g0 = c0 / g.group, groups = g.K / g.group;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int row = 16 * j + (lane >> 2);
            const int64_t rel = (row0 + row < K2 ? row0 + row : K2 - 1) - row0;
            coff[j] = (uint32_t)(rel * g.N) + (((lane & 3) ^ ((row >> 2) & 3)) << 4);
        }
        cbase = g.packed + row0 * g.N;
        int64_t gr = (c0 + 64 * half) / g.group;   // lanes 0 - 31 the first 64 outputs, lanes 32 - 63 the others
        if (gr >= groups) gr = groups - 1;
        soff = (uint32_t)((gr - g0) * g.N * 2) + r32 * 4;
        sbase = g.scales + g0 * g.N;
        zbase = g.zeros + g0 * g.N;
    } else {
        const int64_t n = c0 + (lane & 7) * 16;
#pragma unroll
        for (int j = 0; j < 4; ++j) coff[j] = (uint32_t)((8 * j + (lane >> 3)) * g.N + (n < g.N ? n : g.N - 16) - c0);
        cbase = g.packed + c0;
        soff = (uint32_t)((c0 + 2 * lane < g.N ? 2 * lane : g.N - 2 - c0) * 2);
        sbase = g.scales + c0;
        zbase = g.zeros + c0;
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds + wave * WAVE_LDS;
    const uint8_t* const mine = lds + wave * WAVE_LDS;
    const int tail = TR && g.N % 64 ? all - 1 : -1;   // the step that ends before its 64 columns
    auto step_of = [&](int t) __attribute__((always_inline)) { return first + wave + W * (t < nst ? t : nst - 1); };
    auto request_a = [&](int j, int t, int slot) __attribute__((always_inline)) {
        const int s = step_of(t);
        const uint32_t to = lds0 + slot * ASTEP;
        const int at = j * 1024;
        if (TR && s == tail) {
            const int chunk = (lane & 7) ^ (((8 * j + (lane >> 3)) >> 1) & 7);
            const uint8_t* const p = (const uint8_t*)(abase + (int64_t)s * 64) + aoff[j];
            lds_dma16(to, at, (int64_t)s * 64 + 8 * chunk < g.N ? p : (const uint8_t*)&hqq_zeros);
        } else {
            lds_dma16(to, at, abase + (int64_t)s * 64, aoff[j]);
        }
    };
    auto request_c = [&](int j, int t, int slot) __attribute__((always_inline)) {
        const int s = step_of(t);
        const uint32_t to = lds0 + NA * ASTEP + slot * CSTEP;
        const int at = j < 4 ? j * 1024 : 4096 + (j - 4) * 256;
        if (TR) {
            if (j < 4) {
                const uint8_t* const base = cbase + (int64_t)s * 64;
                const int chunk = (lane & 3) ^ (((16 * j + (lane >> 2)) >> 2) & 3);
                // (codes past the end: the row's first ones of the step, with zero scales)
                lds_dma16(to, at, base, s == tail && (int64_t)s * 64 + 16 * chunk >= g.N ? coff[j] - 16 * chunk : coff[j]);
            } else {
                const uint16_t* const base = (j == 4 ? sbase : zbase) + (int64_t)s * 64;
                if (s == tail)
                    lds_dma4(to, at, (int64_t)s * 64 + 2 * r32 < g.N ? (const uint8_t*)base + soff : (const uint8_t*)&hqq_zeros);
                else
                    lds_dma4(to, at, base, soff);
            }
        } else if (j < 4) {
            lds_dma16(to, at, cbase + (int64_t)s * 32 * g.N, coff[j]);
        } else {
            lds_dma4(to, at, (j == 4 ? sbase : zbase) + (int64_t)(g.per_group ? __umulhi((uint32_t)s, g.per_group) : (uint32_t)s) * g.N, soff);
        }
    };
    auto a_at = [&](int slot) __attribute__((always_inline)) { return mine + slot * ASTEP; };
    auto c_at = [&](int slot) __attribute__((always_inline)) { return mine + NA * ASTEP + slot * CSTEP; };
    auto read_a = [&](const uint8_t* A, int i, int s) __attribute__((always_inline)) {
        return *(const uint4*)(A + (i * 32 + r32) * 128 + (((4 * half + s) ^ ((r32 >> 1) & 7)) << 4));
    };

    union Frag { uint32_t u[4]; uint4 q; };
    Frag fa[2][MT], fb[2][4];
    ht_f32x16 acc[MT][4];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][c][e] = 0.f;

    // Codes of the slices: forward the four dwords (byte rows) of a slice, read two slices ahead; transposed all 32 bytes of the
    // lane's two byte rows, read once a step, and the scales and zeros of a slice's 8 columns, two slices ahead.
    struct Codes { uint32_t d[4]; };
    Codes raw[2];
    uint4 rows[2][2], rows_next[2][2], sl[2][2], zl[2][2];
    uint2 s_next = {0u, 0u}, z_next = {0u, 0u};
    float sf[4], zf[4];
    uint32_t sv[4], zv[4];
    auto read_codes = [&](const uint8_t* C, auto s_c, Codes& out) __attribute__((always_inline)) {
        constexpr int s = decltype(s_c)::value;
#pragma unroll
        for (int i = 0; i < 4; ++i) out.d[i] = *(const uint32_t*)(C + (16 * half + 4 * s + i) * 128 + r32 * 4);
    };
    auto read_rows = [&](const uint8_t* C, uint4 (&out)[2][2]) __attribute__((always_inline)) {
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
#pragma unroll
            for (int h = 0; h < 2; ++h) out[rb][h] = *(const uint4*)(C + rb * 2048 + r32 * 64 + (((2 * half + h) ^ ((r32 >> 2) & 3)) << 4));
    };
    auto read_sz = [&](const uint8_t* C, int s, uint4 (&so)[2], uint4 (&zo)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
            so[rb] = *(const uint4*)(C + 4096 + rb * 128 + half * 64 + s * 16);
            zo[rb] = *(const uint4*)(C + 4352 + rb * 128 + half * 64 + s * 16);
        }
    };
    auto columns = [&](uint2 s2, uint2 z2) __attribute__((always_inline)) {
        const uint32_t ss[2] = {s2.x, s2.y}, zz[2] = {z2.x, z2.y};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if (BF16) {
                sf[c] = __uint_as_float(c & 1 ? ss[c >> 1] & 0xffff0000u : ss[c >> 1] << 16);
                zf[c] = __uint_as_float(c & 1 ? zz[c >> 1] & 0xffff0000u : zz[c >> 1] << 16);
            } else {
                const uint32_t sh = c & 1 ? ss[c >> 1] >> 16 : ss[c >> 1] & 0xffffu, zh = c & 1 ? zz[c >> 1] >> 16 : zz[c >> 1] & 0xffffu;
                sv[c] = sh | (sh << 16);
                zv[c] = zh | (zh << 16);
            }
        }
    };
    // An eighth of a slice's conversion.  Forward: columns o and o + 2 of byte row i (p = 2 i + o).  Transposed: dword i of block rb,
    // nibble o (p = 4 rb + 2 i + o).
    auto convert = [&](auto p_c, auto s_c, const Codes& from, const uint4 (&rw)[2][2], const uint4 (&sx)[2], const uint4 (&zx)[2], Frag (&out)[4])
                       __attribute__((always_inline)) {
        constexpr int p = decltype(p_c)::value, s = decltype(s_c)::value, o = p & 1;
        if constexpr (!TR) {
            constexpr int i = p >> 1;
            if constexpr (BF16) {
                hqq_columns2<SIGNED, o>(from.d[i], zf, sf, out[o].u[i], out[o + 2].u[i]);
            } else {
                uint32_t lo, hi;
                hqq_nibbles<SIGNED>(from.d[i], lo, hi);
                out[o].u[i] = hqq_pair<SIGNED, o, o>(lo, hi, sv[o], zv[o]);
                out[o + 2].u[i] = hqq_pair<SIGNED, o + 2, o + 2>(lo, hi, sv[o + 2], zv[o + 2]);
            }
        } else {
            constexpr int rb = p >> 2, i = (p >> 1) & 1;
            const uint4 v = rw[rb][s >> 1];
            const uint32_t d = s & 1 ? (i ? v.w : v.z) : (i ? v.y : v.x);
            const uint32_t s0 = i ? sx[rb].z : sx[rb].x, s1 = i ? sx[rb].w : sx[rb].y, z0 = i ? zx[rb].z : zx[rb].x, z1 = i ? zx[rb].w : zx[rb].y;
            if constexpr (BF16) {
                if constexpr (o == 0) {   // kept for the high nibbles
                    sf[0] = __uint_as_float(s0 << 16); sf[1] = __uint_as_float(s0 & 0xffff0000u);
                    sf[2] = __uint_as_float(s1 << 16); sf[3] = __uint_as_float(s1 & 0xffff0000u);
                    zf[0] = __uint_as_float(z0 << 16); zf[1] = __uint_as_float(z0 & 0xffff0000u);
                    zf[2] = __uint_as_float(z1 << 16); zf[3] = __uint_as_float(z1 & 0xffff0000u);
                }
                hqq_row<SIGNED, o == 1>(d, zf, sf, out[2 * rb + o].u[2 * i], out[2 * rb + o].u[2 * i + 1]);
            } else {
                uint32_t lo, hi;
                hqq_nibbles<SIGNED>(d, lo, hi);
                const uint32_t n = o ? hi : lo;
                out[2 * rb + o].u[2 * i] = hqq_pair<SIGNED, 0, 1>(n, n, s0, z0);
                out[2 * rb + o].u[2 * i + 1] = hqq_pair<SIGNED, 2, 3>(n, n, s1, z1);
            }
        }
    };

    if (nst > 0) {
#pragma unroll
        for (int t = 0; t < NC - 1; ++t) {
            if (t < NA - 1)
#pragma unroll
                for (int j = 0; j < AREQ; ++j) request_a(j, t, t);
#pragma unroll
            for (int j = 0; j < CREQ; ++j) request_c(j, t, t);
        }
        // step 0 has landed; NA < NC: its activations came in front of both steps' codes
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NA == NC ? (NC - 2) * REQ : CREQ) : "memory");
        if constexpr (TR) {
            read_rows(c_at(0), rows);
            read_sz(c_at(0), 0, sl[0], zl[0]);
            read_sz(c_at(0), 1, sl[1], zl[1]);
        } else {
            columns(*(const uint2*)(c_at(0) + 4096 + r32 * 8), *(const uint2*)(c_at(0) + 4352 + r32 * 8));
            read_codes(c_at(0), std::integral_constant<int, 0>{}, raw[0]);
            read_codes(c_at(0), std::integral_constant<int, 1>{}, raw[1]);
        }
#pragma unroll
        for (int i = 0; i < MT; ++i) fa[0][i].q = read_a(a_at(0), i, 0);
        ht_for<0, 8>([&](auto p) __attribute__((always_inline)) { convert(p, std::integral_constant<int, 0>{}, raw[0], rows, sl[0], zl[0], fb[0]); });

        int ab = 0, cb = 0;   // slots of step t
        for (int t = 0; t < nst; ++t) {
            const int an = ab + 1 == NA ? 0 : ab + 1, cn = cb + 1 == NC ? 0 : cb + 1;
            const int aa = ab == 0 ? NA - 1 : ab - 1, ca = cb == 0 ? NC - 1 : cb - 1;   // left by step t - 1
            ht_for<0, 4>([&](auto s_c) __attribute__((always_inline)) {
                constexpr int s = decltype(s_c)::value, cur = s & 1, nxt = cur ^ 1;
                // codes (and activations) of step t + 1 have landed in front of slice 2, which reads them first
                if constexpr (s == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NA == NC ? (NC - 2) * REQ : REQ) : "memory");
                if constexpr (s == 3 && NA < NC) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(CREQ) : "memory");
                const uint8_t* const C2 = s < 2 ? c_at(cb) : c_at(cn);   // of the slice after the next
                constexpr int s2 = (s + 2) & 3;
                if constexpr (!TR) {
                    if constexpr (s == 3) columns(s_next, z_next);
                    if constexpr (s == 2) {
                        s_next = *(const uint2*)(C2 + 4096 + r32 * 8);
                        z_next = *(const uint2*)(C2 + 4352 + r32 * 8);
                    }
                    read_codes(C2, std::integral_constant<int, s2>{}, raw[cur]);
                } else {
                    if constexpr (s == 2) read_rows(C2, rows_next);
                    if constexpr (s == 3)
#pragma unroll
                        for (int rb = 0; rb < 2; ++rb) {
                            rows[rb][0] = rows_next[rb][0];
                            rows[rb][1] = rows_next[rb][1];
                        }
                    read_sz(C2, s2, sl[cur], zl[cur]);
                }
                ht_for<0, SLOTS>([&](auto q_c) __attribute__((always_inline)) {
                    constexpr int q = decltype(q_c)::value, i = q % MT, c = q / MT;
                    if constexpr (BF16)
                        acc[i][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(ht_bf16x8, fb[cur][c].q),
                                                                            __builtin_bit_cast(ht_bf16x8, fa[cur][i].q), acc[i][c], 0, 0, 0);
                    else
                        acc[i][c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(ht_f16x8, fb[cur][c].q),
                                                                           __builtin_bit_cast(ht_f16x8, fa[cur][i].q), acc[i][c], 0, 0, 0);
                    if constexpr (q < MT) fa[nxt][q].q = s < 3 ? read_a(a_at(ab), q, s + 1) : read_a(a_at(an), q, 0);
                    ht_for<q * 8 / SLOTS, (q + 1) * 8 / SLOTS>([&](auto p) __attribute__((always_inline)) {
                        convert(p, std::integral_constant<int, (s + 1) & 3>{}, raw[nxt], rows, sl[nxt], zl[nxt], fb[nxt]);
                    });
                    if constexpr (s < 2)
                        ht_for<(s * SLOTS + q) * REQ / (2 * SLOTS), (s * SLOTS + q + 1) * REQ / (2 * SLOTS)>([&](auto r_c) __attribute__((always_inline)) {
                            constexpr int r = decltype(r_c)::value;
                            if constexpr (r < AREQ) request_a(r, t + NA - 1, aa);
                            else request_c(r - AREQ, t + NC - 1, ca);
                        });
                    __builtin_amdgcn_sched_barrier(0);
                });
            });
            ab = an;
            cb = cn;
        }
        // the requests past the end have landed before LDS is used again
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    }

    // The four waves add up: wave w finishes the weight rows of accumulator elements 4 w .. 4 w + 3
    __syncthreads();
    float4* const sums = (float4*)lds;
    auto at = [&](int dst, int src, int i, int c) { return sums + (((dst * 3 + (src < dst ? src : src - 1)) * MT + i) * 4 + c) * 64 + lane; };
#pragma unroll
    for (int w = 0; w < W; ++w)
        if (wave != w)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int c = 0; c < 4; ++c) *at(w, wave, i, c) = make_float4(acc[i][c][4 * w], acc[i][c][4 * w + 1], acc[i][c][4 * w + 2], acc[i][c][4 * w + 3]);
    __syncthreads();
    const int64_t cols = TR ? g.K : g.N;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        if (wave != w) continue;
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            float v[4][4];   // [weight row][accumulator]
#pragma unroll
            for (int c = 0; c < 4; ++c) {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e][c] = acc[i][c][4 * w + e];
#pragma unroll
                for (int src = 0; src < W; ++src) {
                    if (src == w) continue;
                    const float4 o = *at(w, src, i, c);
                    v[0][c] += o.x; v[1][c] += o.y; v[2][c] += o.z; v[3][c] += o.w;
                }
            }
            const int64_t m = m0 + 32 * i + r32;
            if (m >= g.M) continue;
            // forward: 16 adjacent columns; transposed: 8 in either block
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int rho = 8 * w + 4 * half + e;
                float4 quad[1] = {make_float4(v[e][0], v[e][1], v[e][2], v[e][3])};
                int64_t col = c0 + 4 * rho;
                if (TR) {
                    // rows e and e + 1 of block 0, then of block 1
                    if (e < 2) {
                        quad[0] = make_float4(v[2 * e][0], v[2 * e][1], v[2 * e + 1][0], v[2 * e + 1][1]);
                        col = c0 + 2 * (8 * w + 4 * half + 2 * e);
                    } else {
                        quad[0] = make_float4(v[2 * e - 4][2], v[2 * e - 4][3], v[2 * e - 3][2], v[2 * e - 3][3]);
                        col = c0 + 64 + 2 * (8 * w + 4 * half + 2 * e - 4);
                    }
                }
                if (col >= cols) continue;
                if (g.part) {
                    *(float4*)(g.part + ((int64_t)blockIdx.y * g.M + m) * cols + col) = quad[0];
                } else {
                    uint16_t o[4];
                    const float f[4] = {quad[0].x, quad[0].y, quad[0].z, quad[0].w};
#pragma unroll
                    for (int k = 0; k < 4; ++k) o[k] = BF16 ? hw_bf16_bits(f[k]) : f32_to_f16_bits(f[k]);
                    *(uint2*)(g.y + m * cols + col) = make_uint2(o[0] | ((uint32_t)o[1] << 16), o[2] | ((uint32_t)o[3] << 16));
                }
            }
        }
    }
}

// Rows of a tile and K parts: the cheapest by a measured model (4096 reduction x 4096 - 128256 columns, 4096 columns x 4096 - 44032, 32 to
// 512 rows, g = 64 and 128).  A workgroup takes 5 us and the table's time for a step of its four waves; rounds over the 256 CUs add up,
// the last one at 0.45 of a full one and up; K parts add a launch and the sums' traffic.
HqqTilePlan hqq_tile_plan(int64_t M, int64_t K, int64_t N, int64_t group, bool transposed, bool bf16, int max_parts) {
    static const double step_us[2][2][3] = {{{1.27, 1.51, 1.89}, {1.33, 1.62, 2.18}}, {{1.54, 1.67, 2.06}, {1.94, 2.20, 2.78}}};
    HqqTilePlan best{0, 0, 0, 1, 1e30};
    const int64_t R = transposed ? N : K, C = transposed ? K : N;
    if (group <= 0 || group % 64 || K % group || N % 16 || M < 1 || M >= (1 << 24) || R >= (1 << 24) || C >= (1 << 24)) return best;
    const int64_t steps = (R + 63) / 64, tiles_n = (C + 127) / 128;
    // the kernel divides a step by d = group / 64 as the high word of step * ceil(2^32 / d), exact while step * (d - 1) < 2^32
    if (!transposed && (steps - 1) * (group / 64 - 1) >= ((int64_t)1 << 32)) return best;
    for (int mt = 1; mt <= 3; ++mt) {
        const int64_t tiles_m = (M + 32 * mt - 1) / (32 * mt);
        if (tiles_m * tiles_n >= (1 << 24)) continue;
        for (int z = 1; z <= max_parts; z *= 2) {
            const int64_t per = (steps + z - 1) / z;
            if (z > 1 && (per < 8 || (z - 1) * per >= steps)) break;
            const double rounds = (double)(tiles_m * tiles_n * z) / 256.0, full = (double)(int64_t)rounds, rest = rounds - full;
            const double one = 5.0 + (double)((per + 3) / 4) * step_us[bf16][transposed][mt - 1];
            double us = full * one + (rest == 0.0 ? 0.0 : full == 0.0 ? one * (0.8 + 0.2 * rest) : one * (0.45 + 0.45 * rest));
            if (z > 1) us += 3.0 + 1.5e-6 * (double)(M * C * z);
            if (us < best.us) best = HqqTilePlan{32 * mt, (int)tiles_m, (int)tiles_n, z, us};
        }
    }
    return best;
}

// The tiles' plan where they are the faster route.  Beyond 64 rows the other one writes the weight in 16 bits and calls the library product: 11008 x
// 4096 at 96 / 235 rows 68 / 76 us against 28 / 56; 128256 x 4096 at 79 / 253 rows 749 / 899 against 170 / 427; 1024 x 4096 at 228 rows
// 16.4 against 14.5; 14336 x 4096 at 433 rows 94 against 99.  Its time is estimated with a lead for products of 45 GFLOP on, where the
// library catches up (and twice the rate beyond the rows that were measured).  Transposed products whose reduction is at most one and
// a half times as long as their output is wide have an estimate of their own, from weights of up to 71 M at 65 to 512 rows: the library holds up there (K x
// N, bf16, 16-bit weight and library / tiles at 192 and 384 rows: 11008 x 4096 60 / 45, 70 / 86; 14336 x 4096 70 / 45, 86 / 86; 4096 x 6144 52 / 27, 44 / 40, 51 / 58 at 512;
// 5120 x 5120 49 / 30, 44 / 47; 8192 x 8192 92 / 50, 96 / 84, 106 / 135 at 448), and a little on wide weights forward (4096 x 14336 at 448 rows 95 / 98,
// 4096 x 32000 of fp16 at 512 193 / 198).
// Up to 64 rows the other one is the streaming kernel of hqq.hip, timed against the tiles on 31 weights from 4096 x 4096 to 14336 x 14336 and 4096 x
// 128256, groups of 64.  Its time is estimated from its plan's costs, the weight and the rows times the weight (the activations are read again for every 64
// columns), with the factors that lose least by choosing wrong: 0.3 % of the best of both over all of them (3.2 % of bf16 and 1.4 % of fp16 forward by the
// weight's size and a lead), and no tiles where they were never ahead.  us streamed / tiled, forward, bf16 (K x N): one row 8192 x 8192 15.7 / 18.8, 5120 x 13824 18.0 / 20.3,
// 4096 x 32000 27.4 / 26.9; 17 rows 14336 x 4096 16.3 / 18.8, 13824 x 5120 19.4 / 25.7, 24 rows 8192 x 28672 52.3 / 47.5; 33 rows 4096 x 4096 10.6 / 13.7, 13824 x 5120 23.3 / 29.1,
// 5120 x 13824 23.7 / 23.2; 64 rows 13824 x 5120 28.5 / 29.6, 4096 x 11008 24.7 / 21.8.  fp16: 32 rows 13824 x 5120 20.2 / 22.6, 5120 x 13824 20.0 / 18.8.  Transposed,
// fp16: 17 rows 8192 x 28672 36.6 / 42.3, 32 rows 44.9 / 42.2, 40 rows 4096 x 11008 18.6 / 19.0, 11008 x 4096 21.8 / 20.0; bf16, whose rule is an older one (0.3 % lost): 33 / 64 rows
// 8192 x 28672 54.6 / 64.3, 71.2 / 64.1, 14336 x 4096 21.7 / 24.5, 26.4 / 25.5.  Chosen wrong by most: transposed bf16 18944 x 3584 at 48 rows 38.5 / 33.0, fp16 8192 x 4096 at
// 56 rows 16.6 / 14.5; forward bf16 8192 x 28672 at 16 rows 43.7 / 47.6.
HqqTilePlan hqq_tile_route(int64_t M, int64_t K, int64_t N, int64_t group, bool transposed, bool bf16) {
    const HqqTilePlan none{0, 0, 0, 1, 1e30};
    const double weights = (double)K * (double)N, rows = (double)M, flops = 2.0 * rows * weights;
    // the size of the weight first: a plan takes a tenth of a microsecond of host time, which bounds calls on small weights
    if (weights < (M > 64 ? 0.0 : !transposed ? (M > 32 ? 2e7 : 3e7) : M > 32 ? (bf16 ? 4e7 : 2e7) : M > 16 && !bf16 ? 2e7 : 1e30)) return none;
    const HqqTilePlan p = hqq_tile_plan(M, K, N, group, transposed, bf16);
    if (!p.rows) return none;
    double other = 1e30, lead = 1.0;
    if (M > 512) {
        other = 10.0 + weights * 0.55e-6 + flops / 1.2e9;
    } else if (M > 64) {
        other = 14.0 + weights * 0.8e-6 + flops / 0.9e9;
        if (flops >= 4.5e10) other *= transposed || N <= 2 * K ? 0.82 : 0.8;
        if (transposed && 2 * N <= 3 * K && weights < 1e8) other = std::min(other, 20.0 + 0.61e-6 * weights + rows * (0.0016e-6 * weights - 0.009));
    } else if (transposed && bf16) {
        other = 0.88 * (5.6 + (0.18 + 0.0022 * rows) * weights * 1e-6 + 0.065 * rows + 4.5e-6 * rows * (double)K);
        lead = 0.92;
    } else {
        // constant, factor of the plan's costs, us a million weights, a row more; up to 32 rows and beyond
        static const double by[3][2][4] = {{{3.4, 0.23, 0.13, 0.0022}, {3.1, 0.70, -0.002, 0.0030}},       // forward, fp16
                                           {{4.9, 0.56, 0.053, 0.0009}, {1.8, 1.12, -0.064, 0.0018}},      // forward, bf16
                                           {{4.6, 0.65, -0.002, 0.0026}, {4.4, 1.11, -0.021, 0.0017}}};    // transposed, fp16
        const double* c = by[transposed ? 2 : bf16][M > 32];
        other = c[0] + c[1] * hqq_stream_us(M, K, N, group, transposed) + (c[2] + c[3] * rows) * weights * 1e-6;
    }
    return lead * p.us < other ? p : none;
}

template <bool BF16, bool SIGNED, bool TR>
static void launch_rows(int rows, dim3 grid, const HqqTileArgs& g, hipStream_t st) {
    switch (rows) {
        case 32: hipLaunchKernelGGL((hqq_tile_kernel<BF16, SIGNED, TR, 1>), grid, dim3(256), 0, st, g); break;
        case 64: hipLaunchKernelGGL((hqq_tile_kernel<BF16, SIGNED, TR, 2>), grid, dim3(256), 0, st, g); break;
        default: hipLaunchKernelGGL((hqq_tile_kernel<BF16, SIGNED, TR, 3>), grid, dim3(256), 0, st, g); break;
    }
}
template <bool BF16, bool SIGNED>
static void launch_direction(bool transposed, int rows, dim3 grid, const HqqTileArgs& g, hipStream_t st) {
    if (transposed) launch_rows<BF16, SIGNED, true>(rows, grid, g, st);
    else launch_rows<BF16, SIGNED, false>(rows, grid, g, st);
}

void launch_hqq_tile(const HqqTilePlan& p, const uint8_t* packed, const uint16_t* scales, const uint16_t* zeros, const uint16_t* a, int64_t lda,
                     int64_t M, int64_t K, int64_t N, int64_t group, bool is_signed, bool bf16, bool transposed, float* part, uint16_t* y,
                     hipStream_t st) {
    const int tiles = p.tiles_m * p.tiles_n, per_xcd = (tiles + 7) / 8;
    const HqqTileArgs g{packed, scales, zeros, a, lda, M, K, N, group, p.tiles_m, tiles, per_xcd,
                        group == 64 ? 0u : (uint32_t)((((uint64_t)1 << 32) + group / 64 - 1) / (uint64_t)(group / 64)), p.parts > 1 ? part : nullptr, y};
    const dim3 grid((unsigned)(per_xcd * 8), (unsigned)p.parts);
    if (bf16) is_signed ? launch_direction<true, true>(transposed, p.rows, grid, g, st) : launch_direction<true, false>(transposed, p.rows, grid, g, st);
    else is_signed ? launch_direction<false, true>(transposed, p.rows, grid, g, st) : launch_direction<false, false>(transposed, p.rows, grid, g, st);
    if (p.parts > 1) launch_hqq_finish(part, p.parts, M * (transposed ? K : N), bf16, y, st);
}

}  // namespace ao

using namespace ao;

extern "C" int ao_amd_hqq_mixed_mm_tiled_bytes(int64_t M, int64_t K, int64_t N, int64_t group_size, int dtype, int transposed, int64_t* bytes) {
    AO_REQUIRE(bytes, "null pointer argument");
    AO_REQUIRE(M >= 1 && K > 0 && N > 0 && group_size > 0, "need positive M, K, N and group size");
    const HqqTilePlan p = hqq_tile_route(M, K, N, group_size, transposed != 0, dtype == AO_BF16);
    *bytes = !p.rows ? -1 : p.parts > 1 ? (int64_t)p.parts * M * (transposed ? K : N) * (int64_t)sizeof(float) : 0;
    return 0;
}

extern "C" int ao_amd_hqq_mixed_mm_tiled(const void* a, int64_t M, int64_t lda, const void* packed_2xint4, int is_signed, int64_t K, int64_t N,
                                         const void* scales, const void* zeros, int64_t group_size, int dtype, int transposed, void* workspace,
                                         int64_t workspace_bytes, void* y, void* stream) {
    AO_REQUIRE(a && packed_2xint4 && scales && zeros && y, "null pointer argument");
    AO_REQUIRE(dtype == AO_BF16 || dtype == AO_F16, "activations, scales, zeros and output must be bf16 or f16, got code %d", dtype);
    AO_REQUIRE(M >= 1 && K > 0 && N > 0, "need positive M, K and N");
    HqqTilePlan p = hqq_tile_plan(M, K, N, group_size, transposed != 0, dtype == AO_BF16);
    AO_REQUIRE(p.rows, "the tiled product needs the group size a multiple of 64 that divides K, N a multiple of 16 and sizes below 2^24, got K=%lld N=%lld group=%lld",
               (long long)K, (long long)N, (long long)group_size);
    AO_REQUIRE(lda >= (transposed ? N : K) && lda % 8 == 0 && lda < (1ll << 24), "activation rows must be 16-byte aligned and as long as the reduction");
    AO_REQUIRE(((((uintptr_t)a) | ((uintptr_t)packed_2xint4) | ((uintptr_t)scales) | ((uintptr_t)zeros) | ((uintptr_t)y) | ((uintptr_t)workspace)) & 15) == 0,
               "buffers must be 16-byte aligned");
    if (p.parts > 1 && (!workspace || workspace_bytes < p.parts * M * (transposed ? K : N) * (int64_t)sizeof(float)))
        p = hqq_tile_plan(M, K, N, group_size, transposed != 0, dtype == AO_BF16, 1);
    launch_hqq_tile(p, (const uint8_t*)packed_2xint4, (const uint16_t*)scales,
                    (const uint16_t*)zeros, (const uint16_t*)a, lda, M, K, N, group_size, is_signed != 0, dtype == AO_BF16, transposed != 0,
                    (float*)workspace, (uint16_t*)y, (hipStream_t)stream);
    AO_LAUNCH_CHECK();
    return 0;
}
