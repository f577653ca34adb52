// Tiled product y[M,N] = x[M,K] @ dequant(W[N,K])^T for batches beyond the streaming kernels, generic over the weight format.
//
// A workgroup of WM x WN x KW waves computes a tile of 32 MT WM activation rows x 32 NT WN weight rows; a wave owns MT x NT blocks of
// 32x32x16 matrix instructions.  With WM = 1 it has all rows of the tile, so every weight is dequantized once per tile.  192 x 128
// tiles of int8 and FP6, whose dequantization is short, have WM = 2: twice the conversions, but two waves on a SIMD (int8
// 192 rows, 14336 x 4096 46.0 -> 42.7 us, 333 rows 11008 x 4096 44.5 -> 42.1, by this alone; with the rest below 45.9 -> 40.3; FP6 40.6 -> 38.9, 41.7 -> 40.8; int4
// 45.9 -> 57.8, so not there.
// 256 x 128, 192 x 256 and 256 x 256 tiles of that kind were no faster than what they would replace).  With KW > 1 the
// groups of WN waves take the 64-wide K steps round-robin and add their accumulators through LDS at the end.  Both
// operands of a step come into LDS by direct loads (no registers, no LDS store instructions) through a ring of STAGES
// buffers with one barrier per step.  Weights are stored in LDS as they are in memory and dequantized by the wave that
// multiplies them, in registers, on the way into the matrix instruction.
//
// The weight is the row operand of the matrix instruction: a lane of the result holds 4 consecutive outputs of one
// activation row (8-byte stores), and the order of the 64 reduction indices within a step is free as long as both
// operands agree, so a lane half takes 32 consecutive k of its rows: a format's natural contiguous run.
//
// What bounds it (ablations on 14336 x 4096 int8, 64 - 256 rows): with one wave per SIMD nothing overlaps inside the wave, so
// LDS reads, conversion and requests add to the matrix time; and a step's data takes 0.7 us from the last-level cache, so
// the bytes in flight per CU set the pace of small tiles.  Requests three steps ahead instead of two took 128 x 128 tiles
// at 256 rows from 51 to 38 us; two groups along K (two waves per SIMD) took 64 x 128 tiles from 29 to 24 us.  A CU takes 125
// bytes a nanosecond from its XCD's L2, but only 55 to 70 while the weights come from memory: requests return in order, so
// those behind a weight wait with it.  More buffers than four change nothing then (six measured), and neither do wider
// tiles for a wave (64 columns, half the LDS reads).  Every instruction of the loop counts, also the scalar ones and the
// wait states: buffers named by their byte offset, 32-bit step offsets, the LDS address added into m0 by one instruction and
// conversions that the compiler knows (in place of asm statements, behind which it places a wait state each) took the int4
// loop of 96 x 128 tiles from 273 to 224 instructions and 5120 x 13824 at 427 rows from 96.3 to 89.6 us, 4096 x 14336 at 1254 rows
// from 179 to 164; int8 and FP6 loops are 5 to 10 % shorter and 0 to 2 % faster.
#pragma once
#include "lds_dma.h"
#include "tile_order.h"
#include <type_traits>

namespace ao {

typedef float tg_f32x16 __attribute__((ext_vector_type(16)));

struct TileGemmArgs {
    const uint16_t* x; int64_t M, K, ldx;
    const uint8_t* w; int64_t ldw;      // weight and its row (or 16-row block) stride in bytes
    const void* scale;                  // bf16 / fp16 row scales, or the int4 (scale, zero) words
    const uint16_t* bias;               // or null
    int64_t N;
    uint16_t* y; int64_t ldy;
    TileOrder order;
    const uint16_t* residual; int64_t ldres;   // y += residual, or null
    const uint16_t* gate; int64_t ldgate;      // y = silu(gate) * y, or null
    int group_shift;                    // int4: log2 of the group size
    float* parts;                       // K in parts: fp32 partial products [order.parts][M][N], or null
};

template <int N>
__device__ __forceinline__ void tg_wait_barrier() {
    // lgkmcnt: this wave's reads of the buffer that the next requests overwrite have returned
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// A weight format F describes a block of 32 weight rows of one 64-wide K step:
//   REQ, BLOCK_BYTES      requests that bring it into LDS, and its bytes there
//   PAIR                  whether two steps' worth is brought in at once (a row's 64 k are half a 128-byte line)
//   lane_offset(a, n0, n, r, lane)   this lane's offset of request r from the tile's base, rows n ..
//   request(a, n0, s, r, lds, at, off)   issues request r of step s, which lands at `lds` + the constant `at`
//   Raw read(block, lane, odd)       a lane's share: row lane % 32, the 32 k of half lane / 32 (PAIR: of the first or second step)
//   Ready prepare(raw, row)          whatever is computed once per step
//   Piece piece(ready, s, d)         two dequantized weights: dword d of the 8 k of slice s, up to
//   uint32_t pack(piece)             the work left for the end of the slice
//   mul, columns, finish, combine    the matrix instruction and the epilogue
template <class F, int WN, int KW, int MT, int NT, int WM>
__global__ __launch_bounds__(64 * WM * WN * KW) void tile_gemm_kernel(const TileGemmArgs a) {
    constexpr int G = WM * WN, BM = 32 * MT * WM, BN = 32 * NT * WN;
    constexpr bool PAIR = F::PAIR;
    constexpr int ABYTES = BM * 128, BBYTES = WN * NT * F::BLOCK_BYTES, STAGE = ABYTES + BBYTES;
    constexpr int STAGES = KW * 4 * STAGE <= 160 * 1024 ? 4 : 3;
    // with PAIR the weights have a ring of their own, of three pairs of steps
    constexpr int RING = PAIR ? STAGES * ABYTES + 6 * BBYTES : STAGES * STAGE;
    static_assert(!PAIR || KW * RING <= 160 * 1024, "LDS of a CU");
    // With three buffers an odd step would wait for its own requests and those of the pair, and not for the step that it reads next
    static_assert(!PAIR || STAGES == 4, "PAIR's waits count four activation buffers");
    constexpr int AREQ = ABYTES / 1024 / G, WREQ = F::REQ * (PAIR ? 2 : 1), BREQ = NT * WREQ / WM, REQ = AREQ + BREQ;
    static_assert(AREQ * G * 1024 == ABYTES && BREQ * WM == NT * WREQ && (NT % WM == 0 || NT == 1), "every wave issues the same number of requests");
    constexpr int ACC = MT * NT * 4096;   // bytes of one wave's accumulators
    constexpr int LDS = KW * RING > (KW - 1) * G * ACC ? KW * RING : (KW - 1) * G * ACC;
    __shared__ __align__(1024) uint8_t lds[LDS];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int group = wave / G, gw = wave % G, wn = gw % WN, wm = WM == 1 ? 0 : gw / WN;
    int tile_m, tile_n, part;
    tile_at(a.order, (int)blockIdx.x, tile_m, tile_n, part);
    const int64_t m0 = (int64_t)tile_m * BM, n0 = (int64_t)tile_n * BN;
    // this workgroup's run of 64-wide K steps: all of them, or the part-th of order.parts equal parts
    // (PAIR: whole pairs, and the groups take pairs; a last part may be left without any and stores zeros)
    constexpr int UNIT = PAIR ? 2 : 1;
    const int all = (int)(a.K / 64), per = (all / UNIT + a.order.parts - 1) / a.order.parts * UNIT, first = per * part;
    const int KS = PAIR ? max(min(per, all - first), 0) : min(per, all - first);
    const int nst = PAIR ? KS / (2 * KW) * 2 + min(KS % (2 * KW), 2) : (KS + KW - 1) / KW;

    // Activation request j of a wave: 8 rows x 128 bytes, slot (row, p) holds k chunk p ^ (row / 2 % 8), so that the fragment
    // reads below (16 rows, one chunk) cover all banks.  Rows past M repeat the last one; their outputs are not stored.
    uint32_t aoff[AREQ], boff[BREQ];
#pragma unroll
    for (int j = 0; j < AREQ; ++j) {
        const int row = (gw * AREQ + j) * 8 + (lane >> 3);
        const int64_t rel = (m0 + row < a.M ? m0 + row : a.M - 1) - m0;
        aoff[j] = (uint32_t)(rel * a.ldx * 2) + (((lane & 7) ^ ((row >> 1) & 7)) << 4);
    }
#pragma unroll
    for (int j = 0; j < BREQ; ++j) {
        const int r = wm * BREQ + j;   // of the NT x WREQ requests of its columns, which WM waves share
        boff[j] = F::lane_offset(a, n0, n0 + (wn * NT + r / WREQ) * 32, r % WREQ, lane);
    }
    const uint16_t* const abase = a.x + m0 * a.ldx;
    // Buffers are named by their byte offset within the ring: activations A_STEP apart, weights behind them
    constexpr int A_STEP = PAIR ? ABYTES : STAGE, A_END = STAGES * A_STEP, B_STEP = 2 * BBYTES, B_END = 3 * B_STEP;   // (B_: PAIR)
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds + group * RING;
    const uint32_t lds_a = lds0 + gw * AREQ * 1024, lds_b = lds0 + (PAIR ? A_END : ABYTES) + wn * NT * UNIT * F::BLOCK_BYTES +
                   wm * (NT % WM == 0 ? NT / WM * UNIT * F::BLOCK_BYTES : BREQ * 1024);
    // request r of step t: the activations' into `buf`, then the weights'; with PAIR first the weights of steps t .. t + 1, into pair
    // buffer `buf`, then the activations
    auto request = [&](int r, int t, int buf) __attribute__((always_inline)) {
        const bool weights = PAIR ? r < BREQ : r >= AREQ;
        const int i = PAIR == weights ? r : weights ? r - AREQ : r - BREQ;
        // (a request past the end repeats the last step's and is not used)
        int s;
        if constexpr (PAIR) {
            s = min(first + (t >> 1) * 2 * KW + 2 * group + (t & 1), max(min(first + KS, all) - (weights ? 2 : 1), 0));
        } else {
            s = t * KW + group;
            s = first + (s < KS ? s : KS - 1);
        }
        if (weights)
            F::request(a, n0, s, NT % WM == 0 ? i % WREQ : wm * BREQ + i, lds_b + buf, i / WREQ * UNIT * F::BLOCK_BYTES + i % WREQ * 1024, boff[i]);
        else
            lds_dma16(lds_a + buf, i * 1024, (const uint8_t*)abase + (uint32_t)s * 128u, aoff[i]);
    };

    tg_f32x16 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
    const int r32 = lane & 31, half = lane >> 5;
    typename F::Row row_const[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) row_const[j] = F::row(a, n0 + (wn * NT + j) * 32 + r32);

    // Steps 0 .. STAGES - 2 are requested; from then on step t multiplies buffer t and requests step t + STAGES - 1 into the buffer
    // that step t - 1 has left.  The step's barrier stands in front of its last slice, where every wave has read what it needs of
    // buffer t and step t + 1 has to have landed: the last slice reads the first fragments of the next step, so no wave starts
    // a step by waiting for LDS, and a request has STAGES - 2 steps and three quarters to arrive.  (With the barrier at the end of a
    // step, which then had to see step t + 2 arrive, the three-buffer shapes had less than one: 64 x 64 tiles of int8 at 106
    // rows, 4888 x 3456, 18.4 -> 14.4 us.)  A slice is MT x NT slots of one matrix instruction each; its share of the
    // conversion, the LDS reads and the requests are dealt out over the slots.
    //
    // PAIR: an even step t requests the weights of steps t + 4 and t + 5 into the pair buffer that steps t - 2 and t - 1 have left.
    // An int8 row's 64 k of one step are half a line of the L1, which has passed on by the time the other half is asked for:
    // 13824 x 5120 at 113 rows 37.5 -> 34.0 us, 14336 x 4096 at 128 / 1149 / 2000 rows 29.5 / 133.8 / 242 -> 27.3 / 129.8 / 234.  (With
    // two pairs in the ring, requested two steps ahead, 96 x 128 tiles lost 8 %; with three they do not gain, nor do 192 x 128.)
    constexpr int SLOTS = MT * NT, PIECES = NT * 4;
#pragma unroll
    for (int t = 0; t < STAGES - 1; ++t)
#pragma unroll
        for (int r = 0; r < REQ; ++r) {
            if (!PAIR || r >= BREQ) request(r, t, t * A_STEP);
            else if (t < 2) request(r, 2 * t, t * B_STEP);
        }
    // this lane's weights of a step (with PAIR of a pair) in buffer `buf`, its activation fragment of slice s
    auto b_at = [&](int buf, int j) { return lds + group * RING + (PAIR ? A_END : ABYTES) + buf + (wn * NT + j) * UNIT * F::BLOCK_BYTES; };
    int a_lane[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) a_lane[s] = group * RING + wm * MT * 4096 + r32 * 128 + (((4 * half + s) ^ ((r32 >> 1) & 7)) << 4);
    auto read_a = [&](int buf, int i, int s) __attribute__((always_inline)) { return *(const uint4*)(lds + (a_lane[s] + buf) + i * 4096); };
    union Frag { uint32_t u[4]; uint4 q; };
    Frag fa[2][MT], fb[2][NT];
    typename F::Raw raw[NT];
    typename F::Ready ready[NT];
    tg_wait_barrier<PAIR ? (STAGES - 2) * AREQ + BREQ : (STAGES - 2) * REQ>();
#pragma unroll
    for (int j = 0; j < NT; ++j) ready[j] = F::prepare(F::read(b_at(0, j), lane, false), row_const[j]);
#pragma unroll
    for (int i = 0; i < MT; ++i) fa[0][i].q = read_a(0, i, 0);
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int d = 0; d < 4; ++d) fb[0][j].u[d] = F::pack(F::piece(ready[j], 0, d));
    int prev = A_END - A_STEP, buf = 0, pair = 0;   // the buffer of the step before, this step's, its pair's
    // (a group that has one step less runs one less; a test around every matrix instruction of that step cost 2 to 5 %)
    const int own = PAIR ? KS / (2 * KW) * 2 + min(max(KS % (2 * KW) - 2 * group, 0), 2) : (KS - group + KW - 1) / KW;
    auto step = [&](int t, auto odd) __attribute__((always_inline)) {
        constexpr bool ODD = decltype(odd)::value;   // of PAIR's two steps
        constexpr int NREQ = PAIR && ODD ? AREQ : REQ;
        const int next = buf + A_STEP == A_END ? 0 : buf + A_STEP;
        const int pair_prev = pair == 0 ? B_END - B_STEP : pair - B_STEP;
        if (PAIR && ODD) pair = pair + B_STEP == B_END ? 0 : pair + B_STEP;   // (from here on the next step's)
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int cur = s & 1, nxt = cur ^ 1;
            typename F::Piece piece[PIECES];
            if (s == 3) {
                tg_wait_barrier<PAIR ? (STAGES - 2) * AREQ + BREQ : (STAGES - 2) * REQ>();
#pragma unroll
                for (int j = 0; j < NT; ++j) raw[j] = F::read(b_at(PAIR ? pair : next, j), lane, !ODD);
            }
#pragma unroll
            for (int q = 0; q < SLOTS; ++q) {
                const int i = q % MT, j = q / MT;
                acc[i][j] = F::mul(fb[cur][j].q, fa[cur][i].q, acc[i][j]);
                if (q < MT) fa[nxt][q].q = s < 3 ? read_a(buf, q, s + 1) : read_a(next, q, 0);
                if (s == 3 && q == 1)
#pragma unroll
                    for (int j2 = 0; j2 < NT; ++j2) ready[j2] = F::prepare(raw[j2], row_const[j2]);
                // (the last slice's pieces are the next step's first, whose codes arrive in its first slot)
                const int p0 = s < 3 ? q * PIECES / SLOTS : q == 0 ? 0 : (q - 1) * PIECES / (SLOTS - 1);
                const int p1 = s < 3 ? (q + 1) * PIECES / SLOTS : q * PIECES / (SLOTS - 1);
#pragma unroll
                for (int p = p0; p < p1; ++p) piece[p] = F::piece(ready[p / 4], (s + 1) & 3, p % 4);
                if (q == SLOTS - 1)
#pragma unroll
                    for (int p = 0; p < PIECES; ++p) fb[nxt][p / 4].u[p % 4] = F::pack(piece[p]);
                if (s < 2)
#pragma unroll
                    for (int r = (s * SLOTS + q) * NREQ / (2 * SLOTS); r < (s * SLOTS + q + 1) * NREQ / (2 * SLOTS); ++r) {
                        if (PAIR && !ODD && r < BREQ) request(r, t + 4, pair_prev);
                        else request(PAIR && ODD ? r + BREQ : r, t + STAGES - 1, prev);
                    }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        prev = buf;
        buf = next;
    };
    if constexpr (PAIR) {
        for (int t = 0; t < own; t += 2) {   // (a group's steps are whole pairs)
            step(t, std::false_type());
            step(t + 1, std::true_type());
        }
    } else {
        for (int t = 0; t < own; ++t) step(t, std::false_type());
    }
    if (KW > 1)
        for (int t = own; t < nst; ++t) tg_wait_barrier<0>();   // the barriers of the steps that this group does not have
    // requests past the end have landed before LDS is used again or the workgroup ends
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    if (KW > 1) {
        __syncthreads();
        float* mine = (float*)(lds + ((group > 0 ? group - 1 : 0) * G + gw) * ACC) + lane * 4;
        if (group > 0)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j)
#pragma unroll
                    for (int e = 0; e < 16; e += 4)
                        *(float4*)(mine + ((i * NT + j) * 4 + e / 4) * 256) =
                            make_float4(acc[i][j][e], acc[i][j][e + 1], acc[i][j][e + 2], acc[i][j][e + 3]);
        __syncthreads();
        if (group > 0) return;
#pragma unroll
        for (int g = 0; g < KW - 1; ++g)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j)
#pragma unroll
                    for (int e = 0; e < 16; e += 4) {
                        const float4 v = *(const float4*)((const float*)(lds + (g * G + gw) * ACC) + lane * 4 + ((i * NT + j) * 4 + e / 4) * 256);
                        acc[i][j][e] += v.x; acc[i][j][e + 1] += v.y; acc[i][j][e + 2] += v.z; acc[i][j][e + 3] += v.w;
                    }
    }
    // acc[i][j][e]: output row m = 32 i + lane % 32, column n = 32 j + 8 (e / 4) + 4 (lane / 32) + e % 4
    const bool wide = (a.ldy & 3) == 0 && ((uintptr_t)a.y & 7) == 0;
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int e = 0; e < 16; e += 4) {
            const int64_t n = n0 + (wn * NT + j) * 32 + 8 * (e >> 2) + 4 * half;
            const typename F::Cols cols = F::columns(a, n);
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                const int64_t m = m0 + (wm * MT + i) * 32 + r32;
                if (m >= a.M) continue;
                if (a.parts) {
                    float* dst = a.parts + ((int64_t)part * a.M + m) * a.N + n;
                    if ((a.N & 3) == 0 && n + 3 < a.N)
                        *(float4*)dst = make_float4(acc[i][j][e], acc[i][j][e + 1], acc[i][j][e + 2], acc[i][j][e + 3]);
                    else
#pragma unroll
                        for (int v = 0; v < 4; ++v)
                            if (n + v < a.N) dst[v] = acc[i][j][e + v];
                    continue;
                }
                uint16_t o[4];
#pragma unroll
                for (int v = 0; v < 4; ++v) o[v] = F::finish(acc[i][j][e + v], cols, v);
                F::combine(a, m, n, o);
                uint16_t* dst = a.y + m * a.ldy + n;
                if (wide && n + 3 < a.N) {
                    *(uint2*)dst = make_uint2(o[0] | ((uint32_t)o[1] << 16), o[2] | ((uint32_t)o[3] << 16));
                } else {
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        if (n + v < a.N) dst[v] = o[v];
                }
            }
        }
}

// Adds the K parts of a tile_gemm_kernel and finishes as that kernel does: W columns a thread, 4 or, where rows of sums are not 16-byte aligned, 1.
// (Latency bounds it.  Four columns a thread of such rows, one load after the other under a condition, cost 2 to 4 us more, which the estimates of K parts do not
// have: int8 1093 x 6144 at 10 rows in eight parts 12.5 -> 9.9 us, 4098 x 14336 at 16 rows 24.3 -> 20.9; int4 695 x 4416 at 52 rows 14.2 -> 11.5.)
template <class F, int W>
__global__ __launch_bounds__(256) void tile_finish_kernel(const TileGemmArgs a, int nparts) {
    const int64_t per_row = a.N / W, i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t m = i / per_row, n = (i - m * per_row) * W;
    if (m >= a.M) return;
    float sum[W];
#pragma unroll
    for (int v = 0; v < W; ++v) sum[v] = 0.f;
    for (int p = 0; p < nparts; ++p) {
        const float* src = a.parts + ((int64_t)p * a.M + m) * a.N + n;
        if constexpr (W == 4) {
            const float4 v = *(const float4*)src;
            sum[0] += v.x; sum[1] += v.y; sum[2] += v.z; sum[3] += v.w;
        } else {
            sum[0] += src[0];
        }
    }
    const typename F::Cols cols = F::columns(a, n);
    uint16_t o[W];
#pragma unroll
    for (int v = 0; v < W; ++v) o[v] = F::finish(sum[v], cols, v);
    uint16_t* dst = a.y + m * a.ldy + n;
    if constexpr (W == 4) {
        if ((a.ldy & 3) == 0 && ((uintptr_t)a.y & 7) == 0) {
            *(uint2*)dst = make_uint2(o[0] | ((uint32_t)o[1] << 16), o[2] | ((uint32_t)o[3] << 16));
            return;
        }
    }
#pragma unroll
    for (int v = 0; v < W; ++v) dst[v] = o[v];
}

// Tile shape and K parts for M x N x K: the cheapest by a measured model.  A shape costs `one` us for a wave of workgroups
// over 4096 of K with one workgroup on a CU and `two` with two (0: only one fits), 6 us of it whatever K is; K parts add a
// second launch, something with each doubling and the traffic of their fp32 sums (TilePartCost: us, us, us for four million sums).
struct TileShape {
    int bm, bn;
    double one, two;
    int max_parts = 8;
};
struct TilePlan {
    int shape, parts;
    double us;
};
struct TilePartCost {
    double launch = 1.5, doubling = 1.0, sums = 8.0;
    double lead = 1.0;   // K parts have to take less than this share of the whole K's estimate
    bool uneven = true;  // part counts that are no power of two
};
// us of one shape whose M x N has `tiles` tiles, with K in `z` parts of `per` steps
inline double tile_us(const TileShape& s, int64_t tiles, int64_t per, int z, int64_t M, int64_t N, int64_t K, const TilePartCost& c) {
    const int shift = s.two > 0 ? 9 : 8;   // two workgroups fit a CU, or one
    const int64_t wgs = tiles * z, full = wgs >> shift, rest = wgs & (((int64_t)1 << shift) - 1);
    auto us = [&](double t) { return 6.0 + (t - 6.0) * (double)per / 64.0; };
    const double one = us(s.one), wave = s.two > 0 ? us(s.two) : one;
    // (CUs that read a large weight at once share the memory: 120 workgroups take 0.7 to 0.97 of the time of 224)
    const double alone = full == 0 && rest < 256 && N * K >= ((int64_t)1 << 25) ? 0.85 + 0.15 * (double)rest / 256.0 : 1.0;
    // (the first CU with two workgroups sets the time, and the more there are the more they slow each other down)
    const double t = (double)full * wave + (rest == 0 ? 0.0 : rest <= 256 ? one * alone : one + (wave - one) * (0.4 + 0.6 * (double)(rest - 256) / 256.0));
    constexpr double LOG2[9] = {0.0, 0.0, 1.0, 1.585, 2.0, 2.322, 2.585, 2.807, 3.0};
    return z == 1 ? t : t + c.launch + LOG2[z] * c.doubling + c.sums * 1e-6 * (double)(M * N * z) / 4.0;
}
// Part counts that are no power of two fill the chip where a weight has 48, 80 or 160 tiles, but the estimates do not rank them finely: of 154
// calls (33 to 1000 rows, 21 weights) those with an estimate below 0.945 of the best power of two took 0.90 of its time on average and 1.03 at most, the others 1.02 (and
// up to 1.19), and weights below 2^23 gained nothing (1024 x 4096 0.96 to 1.04).  us in powers of two / other parts: int8 10240 x 8192 at 77 / 128 rows 39.7 /
// 31.0, 41.2 / 38.2, 9000 x 6144 at 48 rows 25.0 / 22.0, 5120 x 13824 at 200 rows 52.5 / 45.0; int4 5120 x 13824 at 256 rows 66.2 / 49.4, 5120 x 5120 at 40 rows
// 15.3 / 14.2.  Not for shapes with few parts, whose sums are large (int4 5120 x 5120 at 420 rows in three of 256 x 128, 36.8 / 46.4).
inline TilePlan tile_plan(const TileShape* shapes, int nshapes, int64_t M, int64_t N, int64_t K, int max_parts,
                          const TilePartCost& c = TilePartCost()) {
    TilePlan best{-1, 1, 1e30}, whole = best, uneven = best;
    constexpr int MOST = 16;
    int64_t tiles[MOST];   // (a call plans twice: the divisions stand outside the loop over the parts)
    for (int i = 0; i < nshapes && i < MOST; ++i) tiles[i] = (M + shapes[i].bm - 1) / shapes[i].bm * ((N + shapes[i].bn - 1) / shapes[i].bn);
    const int64_t steps = K / 64;
    const bool all = c.uneven && N * K >= ((int64_t)1 << 23);
    for (int z = 1; z <= (max_parts < 8 ? max_parts : 8); ++z) {
        const bool power = (z & (z - 1)) == 0;
        if (!power && !all) continue;
        const int64_t per = (steps + z - 1) / z;
        if (z > 1 && per < 8) break;
        if ((z - 1) * per >= steps) continue;   // the last part would be empty
        for (int i = 0; i < nshapes && i < MOST; ++i) {
            if (z > shapes[i].max_parts || (!power && shapes[i].max_parts < 8)) continue;
            const double t = tile_us(shapes[i], tiles[i], per, z, M, N, K, c);
            TilePlan& to = power ? best : uneven;
            if (t < to.us) to = TilePlan{i, z, t};
            if (z == 1 && t < whole.us) whole = TilePlan{i, z, t};
        }
    }
    if (uneven.us < 0.945 * best.us) best = uneven;
    return best.us < c.lead * whole.us ? best : whole;
}

// The launches of a plan: tile_grid once, tile_launch with the shape's constants, tile_finish.
// row_bytes: a weight row's bytes in a 64-wide step.
inline void tile_grid(TileGemmArgs& a, const TileShape& s, int row_bytes, int parts) {
    a.order = tile_order((a.M + s.bm - 1) / s.bm, (a.N + s.bn - 1) / s.bn, s.bm * 128, s.bn * row_bytes);
    a.order.parts = parts;
    if (parts == 1) a.parts = nullptr;
}
template <class F, int WN, int KW, int MT, int NT, int WM = 1>
void tile_launch(const TileGemmArgs& a, hipStream_t st) {
    hipEvent_t ev0 = g_prof_start, ev1 = g_prof_stop;
    g_prof_start = g_prof_stop = nullptr;
    hipExtLaunchKernelGGL((tile_gemm_kernel<F, WN, KW, MT, NT, WM>), dim3(a.order.workgroups()), dim3(64 * WM * WN * KW), 0, st,
                          ev0, ev1, 0, a);
}
template <class F>
void tile_finish(const TileGemmArgs& a, int parts, hipStream_t st) {
    if (parts == 1) return;
    const bool quads = a.N % 4 == 0;
    const dim3 grid((unsigned)((a.M * (quads ? a.N / 4 : a.N) + 255) / 256)), block(256);
    if (quads) hipLaunchKernelGGL((tile_finish_kernel<F, 4>), grid, block, 0, st, a, parts);
    else hipLaunchKernelGGL((tile_finish_kernel<F, 1>), grid, block, 0, st, a, parts);
}

}  // namespace ao
