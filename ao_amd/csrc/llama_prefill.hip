// Prompt-sized work of the Llama harness between the quantized linears (batch 1, head_dim 128):
//
//   rope + cache write   torchao/_models/llama/model.py:196-203  (keys rotated and stored at input_pos, values stored)
//   attention            torchao/_models/llama/model.py:205-210  (query row i over the cache positions 0 .. input_pos[i])
//   residual + RMSNorm   torchao/_models/llama/model.py:162-165, 232-244
//   SiLU(gate) * up      torchao/_models/llama/model.py:229
//
// Module by module these were some 30 launches a layer over fp32 temporaries and an attention that walked the whole cache
// under a boolean mask: 4 layers of Llama-3-8B widths at 1000 positions spent 2.1 of 4.8 ms in them.
#include "llama_elem.h"

namespace ao {

typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4p_t __attribute__((ext_vector_type(4)));   // loads that wait in registers: a uint4 struct is kept in scratch

// 32x32x16 product, 8 elements of a 16-bit type per lane and operand
template <class E> struct Mfma32;
template <> struct Mfma32<ElemBf16> {
    typedef __bf16 x8 __attribute__((ext_vector_type(8)));
    static __device__ __forceinline__ f32x16_t mul(uint4 a, uint4 b, f32x16_t c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(x8, a), __builtin_bit_cast(x8, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t pack(float lo, float hi) { return hw_bf16_pack(lo, hi); }
};
template <> struct Mfma32<ElemF16> {
    typedef _Float16 x8 __attribute__((ext_vector_type(8)));
    static __device__ __forceinline__ f32x16_t mul(uint4 a, uint4 b, f32x16_t c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(x8, a), __builtin_bit_cast(x8, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t pack(float lo, float hi) {
        return (uint32_t)f32_to_f16_bits(lo) | ((uint32_t)f32_to_f16_bits(hi) << 16);
    }
};

__device__ __forceinline__ int64_t position(const void* pos, int pos_is_i64, int64_t i) {
    return pos_is_i64 ? ((const int64_t*)pos)[i] : (int64_t)((const int32_t*)pos)[i];
}

// The cache row of a position and its row of the rotary table.  With wrap, the rows of that table (at least S), a negative position
// counts from the end of either.  row -1: outside the cache.
struct Position {
    int64_t row, freq;
};
__device__ __forceinline__ Position locate(const void* pos, int pos_is_i64, int64_t i, int64_t S, int64_t wrap) {
    const int64_t p = position(pos, pos_is_i64, i);
    const bool behind = wrap > 0 && p < 0;
    const int64_t row = behind ? p + S : p;
    return row >= 0 && row < S ? Position{row, behind ? p + wrap : p} : Position{-1, 0};
}

// Rotates the consecutive pairs (2i, 2i+1) of 8 elements d .. d+7 of a head: fp32 products rounded one by one, the result
// rounded to the element type, as the module does.  `cs` holds the four (cos, sin) pairs.
template <class E>
__device__ __forceinline__ uint4 rotate8(uint4 x, uint4 cs) {
    const uint32_t u[4] = {x.x, x.y, x.z, x.w}, f[4] = {cs.x, cs.y, cs.z, cs.w};
    uint32_t o[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float x0 = E::lo(u[j]), x1 = E::hi(u[j]), c = E::lo(f[j]), s = E::hi(f[j]);
        o[j] = (uint32_t)E::to_bits(x0 * c - x1 * s) | ((uint32_t)E::to_bits(x1 * c + x0 * s) << 16);
    }
    return make_uint4(o[0], o[1], o[2], o[3]);
}

// Keys rotated and values as they are, into row input_pos[t] of the caches.  One thread per 8 elements; a row outside the
// cache is not written.
template <class E>
__global__ __launch_bounds__(256) void prefill_cache_kernel(const uint16_t* __restrict__ qkv, const uint16_t* __restrict__ freqs,
                                                            int64_t wrap, const void* __restrict__ pos, int pos_is_i64, int T,
                                                            int n_head, int n_kv, int64_t S, uint16_t* __restrict__ k_cache,
                                                            uint16_t* __restrict__ v_cache) {
    const int per_row = 2 * n_kv * 16;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int t = (int)(i / per_row), c = (int)(i % per_row);
    if (t >= T) return;
    const Position p = locate(pos, pos_is_i64, t, S, wrap);
    if (p.row < 0) return;
    const int head = c >> 4, d = (c & 15) * 8;
    const uint4 x = *(const uint4*)(qkv + ((int64_t)t * (n_head + 2 * n_kv) + n_head + head) * 128 + d);
    if (head < n_kv)
        *(uint4*)(k_cache + ((int64_t)head * S + p.row) * 128 + d) = rotate8<E>(x, *(const uint4*)(freqs + p.freq * 128 + d));
    else
        *(uint4*)(v_cache + ((int64_t)(head - n_kv) * S + p.row) * 128 + d) = x;
}

// Causal attention of T query rows over the cache, flash style.
//
// GROUPS = 8 / WAVES groups of WAVES waves walk the cache in tiles of 32 positions, every GROUPS-th one each; a wave owns 32 query rows of one
// head, the same ones in all groups, whose maxima, sums and accumulators meet at the end: each group finishes its share of the columns.  HEADS of a
// group's waves are query heads of one KV head (grouped-query models: one K / V tile serves them all), the others are consecutive 32-row blocks.
//
// Both products are 32x32x16 matrix instructions with the query on the column side: S^T = K Q^T leaves a lane with 16 scores
// of ONE query row per 32 positions, so the softmax statistics are lane-local up to one exchange between the wave's
// halves, the rescaling of O^T = V^T P^T is one multiply per accumulator, and the 8 probabilities a lane already holds are
// its operand of the second product: that product may take positions in any order as long as both operands agree, so V^T is
// stored in LDS in the order the first product leaves them in (lane half h of step s: positions 16 s + 4 h + 0..3 and
// 16 s + 8 + 4 h + 0..3).  V is turned on its way into LDS: a lane loads 2 columns of 8 positions and writes two 16-byte runs.
// LDS rows are XOR-swizzled in 16-byte chunks (fragment reads of 16 lanes cover all banks).  Tiles are double-buffered
// through registers, one barrier per tile; the first one is requested before the positions are known (any tile lies within the cache).
//
// The accumulators are rescaled in tiles that raise a maximum.  (Only where a score passes the kept maximum by 2^8 saves most of these 64
// multiplications, but then the largest probability of a row is no longer 1, which 16 bits hold exactly: 400 rows over 40 heads were 0.00188
// from the result in 64 bits instead of 0.00174, for 1 us of 28 at 1000 positions.)
//
// Bound by the chain of a tile (scores, maximum, exponentials, second product) and by what brings tiles into LDS (requests, V's turn, writes).  Groups
// of two: a short prompt pays the start, where a group rotates its share of the eight query fragments and reads the others from LDS (some 450
// instructions for all), and one whose workgroups are resident at once its longest rows, which four groups share.  Llama-3-8B widths, 61 / 130 / 1000
// positions 8.1 / 7.9 / 27.8 us; with two groups of four waves, 64 positions a tile and all fragments rotated by each wave 11.4 / 13.4 / 34.8.  Groups of
// four: a tile serves 128 rows instead of 64, for half the staging a wave.  Both at 2048 / 4096 / 8192 positions: 32 heads over 8 77 / 241 / 842 -> 63 / 197 /
// 690 us, 64 over 8 143 / 466 / 1714 -> 114 / 372 / 1355, 40 over 40 105 / 324 / 1131 -> 93 / 274 / 918; each group's largest probability of a row is
// exact in 16 bits, so fewer groups are a little further from 64 bits (bf16, 1300 positions 0.00196 -> 0.00198, as far as two groups always were).
template <class E, int WAVES, int HEADS>
__global__ __launch_bounds__(512) void prefill_attention_kernel(const uint16_t* __restrict__ qkv, const uint16_t* __restrict__ freqs,
                                                                int64_t wrap, const void* __restrict__ pos, int pos_is_i64,
                                                                int T, int n_head, int n_kv, int64_t S, const uint16_t* __restrict__ k_cache,
                                                                const uint16_t* __restrict__ v_cache, uint16_t* __restrict__ out) {
    typedef Mfma32<E> MM;
    constexpr int GROUPS = 8 / WAVES, KEYS = 32;
    __shared__ uint4 lds[GROUPS][2][2][KEYS * 16];   // [group][K / V][buffer]
    __shared__ uint4 q_lds[WAVES][8][64];            // [wave][fragment][lane]
    __shared__ int wave_last[WAVES];
    const int group = __builtin_amdgcn_readfirstlane(threadIdx.x / (64 * WAVES));
    uint4 (*const ks)[KEYS * 16] = lds[group][0];   // [key][chunk of 8 d], chunk ^ (key & 15)
    uint4 (*const vs)[KEYS * 16] = lds[group][1];   // [d / 2][(d & 1) * 4 + (chunk of 8 keys ^ (d / 4 & 3))]
    const int tid = threadIdx.x % (64 * WAVES), lane = tid & 63, col = lane & 31, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tile = gridDim.y - 1 - blockIdx.y;   // the rows that see most positions start first
    const int head = blockIdx.x * HEADS + wave % HEADS, row0 = (tile * (WAVES / HEADS) + wave / HEADS) * 32;
    const int kv = head / (n_head / n_kv);
    const uint16_t* kc = k_cache + (int64_t)kv * S * 128;
    const uint16_t* vc = v_cache + (int64_t)kv * S * 128;

    constexpr int KROWS = 4 * WAVES, KLOADS = KEYS / KROWS, RUNS = KEYS / 8 / WAVES;   // rows of K a pass of the threads, passes; runs of 8 positions of V
    u32x4p_t kr[KLOADS];
    uint32_t vr[8 * RUNS];
    const int smax = (int)S - 1;
    // this lane's shares of a tile: 16 bytes of rows tid / 16 + KROWS i, two columns of the 8 positions of run (step, half) = wave * RUNS + g
    auto vrow = [&](int g, int j) { return 16 * ((wave * RUNS + g) >> 1) + 4 * ((wave * RUNS + g) & 1) + (j & 3) + 8 * (j >> 2); };
    const uint32_t koff = (tid >> 4) * 256 + (tid & 15) * 16, voff = vrow(0, 0) * 256 + lane * 4;
    auto fetch = [&](int t) {
        const int base = t * KEYS;
        if (base + KEYS - 1 <= smax) {
            const char* const kb = (const char*)(kc + (int64_t)base * 128);
            const char* const vb = (const char*)(vc + (int64_t)base * 128);
#pragma unroll
            for (int i = 0; i < KLOADS; ++i) kr[i] = *(const u32x4p_t*)(kb + koff + i * (KROWS * 256));
#pragma unroll
            for (int g = 0; g < RUNS; ++g)
#pragma unroll
                for (int j = 0; j < 8; ++j) vr[g * 8 + j] = *(const uint32_t*)(vb + voff + (4 * g + (j & 3) + 8 * (j >> 2)) * 256);
        } else {   // the cache ends within the tile: its last row instead
#pragma unroll
            for (int i = 0; i < KLOADS; ++i) {
                const int key = min(base + i * KROWS + (tid >> 4), smax);
                kr[i] = *(const u32x4p_t*)(kc + (int64_t)key * 128 + (tid & 15) * 8);
            }
#pragma unroll
            for (int g = 0; g < RUNS; ++g)
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int key = min(base + vrow(g, j), smax);
                    vr[g * 8 + j] = *(const uint32_t*)(vc + (int64_t)key * 128 + 2 * lane);
                }
            asm volatile("");   // (keeps the compiler from making one set of loads, with computed addresses, of both)
        }
    };
    auto stash = [&](int b) {
#pragma unroll
        for (int i = 0; i < KLOADS; ++i) {
            const int key = i * KROWS + (tid >> 4);
            *(u32x4p_t*)&ks[b][key * 16 + ((tid & 15) ^ (key & 15))] = kr[i];
        }
#pragma unroll
        for (int g = 0; g < RUNS; ++g) {
            const int c = (wave * RUNS + g) ^ ((lane >> 1) & 3);
            uint32_t even[4], odd[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                even[j] = __builtin_amdgcn_perm(vr[g * 8 + 2 * j + 1], vr[g * 8 + 2 * j], 0x05040100u);
                odd[j] = __builtin_amdgcn_perm(vr[g * 8 + 2 * j + 1], vr[g * 8 + 2 * j], 0x07060302u);
            }
            vs[b][lane * 8 + c] = make_uint4(even[0], even[1], even[2], even[3]);
            vs[b][lane * 8 + 4 + c] = make_uint4(odd[0], odd[1], odd[2], odd[3]);
        }
    };
    fetch(group);

    // this lane's query row: position, rotated fragments
    const int row = row0 + col;
    const int srow = row < T ? row : T - 1;
    const Position p = locate(pos, pos_is_i64, srow, S, wrap);
    const int last = row < T ? (int)p.row : -1;     // last position the row sees; -1: none
#pragma unroll
    for (int s = 0; s < WAVES; ++s) {   // each group rotates its share of the eight
        const int d = 16 * (WAVES * group + s) + 8 * half;
        q_lds[wave][WAVES * group + s][lane] = rotate8<E>(*(const uint4*)(qkv + ((int64_t)srow * (n_head + 2 * n_kv) + head) * 128 + d),
                                                      *(const uint4*)(freqs + p.freq * 128 + d));
    }
    int hi = last, lo = last;
#pragma unroll
    for (int o = 16; o >= 1; o >>= 1) {
        hi = max(hi, __shfl_xor(hi, o, 64));
        lo = min(lo, __shfl_xor(lo, o, 64));
    }
    hi = __builtin_amdgcn_readfirstlane(hi);
    lo = __builtin_amdgcn_readfirstlane(lo);
    if (lane == 0) wave_last[wave] = hi;   // (the same in every group)
    stash(0);
    __syncthreads();
    uint4 q[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) q[s] = q_lds[wave][s][lane];
    int seen = wave_last[0];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) seen = max(seen, wave_last[w]);
    const int ntile = __builtin_amdgcn_readfirstlane((seen + KEYS) / KEYS);

    f32x16_t o[4];
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[b][r] = 0.f;
    float m = -INFINITY, sum = 0.f;                 // running maximum and (this lane's share of the) sum, base 2
    const float scale = 0.08838834764831845f * 1.4426950408889634f;  // 1 / sqrt(128), log2(e)

    int b = 0;
    for (int t = group; t < ntile + group; t += GROUPS, b ^= 1) {   // as many passes in every group: they share the barrier
        if (t + GROUPS < ntile) fetch(t + GROUPS);
        __syncthreads();                            // tile t is in LDS; everybody is done with the other buffer
        if (t < ntile && t * KEYS <= hi) {
            f32x16_t s2;
#pragma unroll
            for (int r = 0; r < 16; ++r) s2[r] = 0.f;
            // (all fragments of K, and then of V, are requested at once: a read in front of each product waited for each)
            u32x4p_t f[8];
#pragma unroll
            for (int s = 0; s < 8; ++s) f[s] = *(const u32x4p_t*)&ks[b][col * 16 + ((2 * s + half) ^ (col & 15))];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < 8; ++s) s2 = MM::mul(__builtin_bit_cast(uint4, f[s]), q[s], s2);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int db = 0; db < 4; ++db) {
                    const int d = db * 32 + col;
                    f[s * 4 + db] = *(const u32x4p_t*)&vs[b][(d >> 1) * 8 + (d & 1) * 4 + ((2 * s + half) ^ ((d >> 2) & 3))];
                }
            __builtin_amdgcn_sched_barrier(0);
            if (t * KEYS + KEYS - 1 > lo)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (t * KEYS + 8 * (r >> 2) + 4 * half + (r & 3) > last) s2[r] = -INFINITY;
            float tmax = -INFINITY;
#pragma unroll
            for (int r = 0; r < 16; ++r) tmax = fmaxf(tmax, s2[r]);
            tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64)) * scale;
            if (__any(tmax > m)) {
                const float m2 = fmaxf(m, tmax), alpha = __builtin_amdgcn_exp2f(m - (m2 == -INFINITY ? 0.f : m2));
                m = m2;
                sum *= alpha;
#pragma unroll
                for (int bb = 0; bb < 4; ++bb)
#pragma unroll
                    for (int r = 0; r < 16; ++r) o[bb][r] *= alpha;
            }
            const float base = m == -INFINITY ? 0.f : m;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                s2[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s2[r], scale, -base));
                sum += s2[r];
            }
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const int r = 8 * s;
                const uint4 pb = make_uint4(MM::pack(s2[r], s2[r + 1]), MM::pack(s2[r + 2], s2[r + 3]), MM::pack(s2[r + 4], s2[r + 5]),
                                            MM::pack(s2[r + 6], s2[r + 7]));
#pragma unroll
                for (int db = 0; db < 4; ++db) o[db] = MM::mul(__builtin_bit_cast(uint4, f[s * 4 + db]), pb, o[db]);
            }
        }
        if (t + GROUPS < ntile) stash(b ^ 1);
    }
    // The groups' maxima, sums and accumulators meet: a group finishes its share of the four blocks of 32 columns
    __syncthreads();
    constexpr int BLOCKS = 4 / GROUPS;
    float4* const parts = (float4*)lds;        // [block][from][wave][4][lane]
    float2* const stats = (float2*)q_lds;      // [group][wave][lane]
    static_assert(4 * (GROUPS - 1) * WAVES * 4 * 64 * 16 <= sizeof(lds) && 8 * 64 * 8 <= sizeof(q_lds), "partial sums");
    auto part_at = [&](int block, int from) {
        return parts + ((block * (GROUPS - 1) + (from < block / BLOCKS ? from : from - 1)) * WAVES + wave) * 256 + lane;
    };
#pragma unroll
    for (int b = 0; b < 4; ++b)
        if (b / BLOCKS != group)
#pragma unroll
            for (int r = 0; r < 16; r += 4) part_at(b, group)[r * 16] = make_float4(o[b][r], o[b][r + 1], o[b][r + 2], o[b][r + 3]);
    stats[(group * WAVES + wave) * 64 + lane] = make_float2(m, sum);
    __syncthreads();
    float2 ms[GROUPS];
    float top = -INFINITY;
#pragma unroll
    for (int g = 0; g < GROUPS; ++g) {
        ms[g] = stats[(g * WAVES + wave) * 64 + lane];
        top = fmaxf(top, ms[g].x);
    }
    const float base = top == -INFINITY ? 0.f : top;
    sum = 0.f;
#pragma unroll
    for (int g = 0; g < GROUPS; ++g) {
        ms[g].x = __builtin_amdgcn_exp2f(ms[g].x - base);
        sum += ms[g].y * ms[g].x;
    }
    sum += __shfl_xor(sum, 32, 64);
    const float inv = 1.0f / sum;                   // a row that sees nothing (a position outside the cache) becomes NaN
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        if (b / BLOCKS != group) continue;
#pragma unroll
        for (int r = 0; r < 16; ++r) o[b][r] *= ms[b / BLOCKS].x;
#pragma unroll
        for (int from = 0; from < GROUPS; ++from) {
            if (from == b / BLOCKS) continue;
#pragma unroll
            for (int r = 0; r < 16; r += 4) {
                const float4 v = part_at(b, from)[r * 16];
                o[b][r] += v.x * ms[from].x;
                o[b][r + 1] += v.y * ms[from].x;
                o[b][r + 2] += v.z * ms[from].x;
                o[b][r + 3] += v.w * ms[from].x;
            }
        }
        if (row < T) {
            uint16_t* const dst = out + ((int64_t)row * n_head + head) * 128 + b * 32 + 4 * half;
#pragma unroll
            for (int r = 0; r < 16; r += 4)
                *(uint2*)(dst + 8 * (r >> 2)) = make_uint2(MM::pack(o[b][r] * inv, o[b][r + 1] * inv), MM::pack(o[b][r + 2] * inv, o[b][r + 3] * inv));
        }
    }
}

// h = x + y, n = rmsnorm(h) * w: one workgroup per row, the row in registers (dim a multiple of 8, at most 8192).
template <class E>
__global__ __launch_bounds__(256) void add_rmsnorm_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ y,
                                                          const uint16_t* __restrict__ w, int dim, float eps,
                                                          uint16_t* __restrict__ h, uint16_t* __restrict__ n) {
    constexpr int MAXC = 4;
    __shared__ float part[4];
    const int64_t row = blockIdx.x;
    const int nchunk = dim / 8;
    uint32_t v[MAXC][4];
    uint4 g[MAXC];
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < MAXC; ++c) {
        const int i = threadIdx.x + c * 256;
        if (i < nchunk) {
            const uint4 a4 = ((const uint4*)(x + row * dim))[i], b4 = ((const uint4*)(y + row * dim))[i];
            g[c] = ((const uint4*)w)[i];
            const uint32_t a[4] = {a4.x, a4.y, a4.z, a4.w}, b[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                v[c][j] = (uint32_t)E::to_bits(E::lo(a[j]) + E::lo(b[j])) | ((uint32_t)E::to_bits(E::hi(a[j]) + E::hi(b[j])) << 16);
                const float lo = E::lo(v[c][j]), hi = E::hi(v[c][j]);
                ss += lo * lo + hi * hi;
            }
        }
    }
    ss = wave_sum(ss);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = ss;
    __syncthreads();
    const float r = rsqrtf((part[0] + part[1] + part[2] + part[3]) / (float)dim + eps);
#pragma unroll
    for (int c = 0; c < MAXC; ++c) {
        const int i = threadIdx.x + c * 256;
        if (i < nchunk) {
            const uint32_t gg[4] = {g[c].x, g[c].y, g[c].z, g[c].w};
            uint32_t o[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                o[j] = (uint32_t)E::to_bits(E::rne(E::lo(v[c][j]) * r) * E::lo(gg[j])) |
                       ((uint32_t)E::to_bits(E::rne(E::hi(v[c][j]) * r) * E::hi(gg[j])) << 16);
            ((uint4*)(h + row * dim))[i] = make_uint4(v[c][0], v[c][1], v[c][2], v[c][3]);
            ((uint4*)(n + row * dim))[i] = make_uint4(o[0], o[1], o[2], o[3]);
        }
    }
}

// x / (1 + e^-x) from t = e^-|x|: x / (1 + t), or x t / (1 + t) below zero, so that the divisor lies in 1 .. 2 and takes the hardware's
// reciprocal; the quotient is corrected once by its remainder, with what the divisor and the product were rounded by.  The exponent of e^-|x| = 2^hi e^lo is
// split in two.  Over all 16-bit values at most 1.40e-7 off, 2.1e-8 in the mean (expf and an IEEE division: 1.43e-7, 3.0e-8, and 45 instructions a value).
// ANY: also zeros (whose sign the correction would lose), infinities (which have no remainder) and values whose t is a subnormal, which the exponential
// flushes (it is scaled by 2^64 on the way; 1 + t is 1 either way); the others are 0 < |x| < 69.
template <bool ANY>
__device__ __forceinline__ float silu(float x) {
    const float a = -fabsf(x), hi = a * 1.44269504088896340736f;
    const float lo = __builtin_fmaf(hi, 1.904654299957768e-09f, __builtin_fmaf(hi, -0.693147182464599609375f, a));
    const int up = ANY && hi < -100.f ? 64 : 0;
    const float e = __builtin_amdgcn_exp2f(hi + (float)up);
    const float t = ANY && e == 0.f ? 0.f : __builtin_fmaf(e, lo, e);   // (an infinite x: lo is no number)
    const float d = 1.0f + t, d_lo = t - (d - 1.0f), r = __builtin_amdgcn_rcpf(d), s = x < 0.f ? t : 1.0f;
    const float n = x * s, n_lo = __builtin_fmaf(x, s, -n);
    const float q = n * r, rest = __builtin_fmaf(-d_lo, q, __builtin_fmaf(-d, q, n)) + n_lo;
    float y = ANY && __builtin_amdgcn_classf(n, 0x264) ? q : __builtin_fmaf(rest, r, q);
    asm("" : "+v"(y));   // (without it the compiler rounds to fp16 in the fma itself where ANY is false, so that bits hung on the wave's other values)
    return ANY && x < 0.f ? __builtin_ldexpf(y, -up) : y;
}

// out = silu(gate) * up, 8 elements per thread; silu is rounded to the element type before the product, as F.silu leaves it.
// 1000 x 14336, six sets of buffers in turn, 17.6 us, 4.9 TB/s, close to the rate of a copy; with expf and a division 18.5, with one Newton step on the
// reciprocal 17.4 (one set of buffers 16.5 / 18.9 / 17.3).
template <class E>
__global__ __launch_bounds__(256) void silu_mul_kernel(const uint16_t* gate, const uint16_t* __restrict__ up, int64_t n8,
                                                       uint16_t* out) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n8) return;
    const uint4 a4 = ((const uint4*)gate)[i], b4 = ((const uint4*)up)[i];
    const uint32_t a[4] = {a4.x, a4.y, a4.z, a4.w}, b[4] = {b4.x, b4.y, b4.z, b4.w};
    float least = INFINITY, most = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        least = fminf(least, fminf(fabsf(E::lo(a[j])), fabsf(E::hi(a[j]))));
        most = fmaxf(most, fmaxf(fabsf(E::lo(a[j])), fabsf(E::hi(a[j]))));
    }
    uint32_t o[4];
    auto rows = [&](auto any) __attribute__((always_inline)) {
        constexpr bool ANY = decltype(any)::value;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float s0 = E::rne(silu<ANY>(E::lo(a[j]))), s1 = E::rne(silu<ANY>(E::hi(a[j])));
            o[j] = (uint32_t)E::to_bits(s0 * E::lo(b[j])) | ((uint32_t)E::to_bits(s1 * E::hi(b[j])) << 16);
        }
    };
    if (__any(!(least > 0.f && most < 69.f))) rows(std::true_type());
    else rows(std::false_type());
    ((uint4*)out)[i] = make_uint4(o[0], o[1], o[2], o[3]);
}

// Rows of the embedding table.  A token outside the table leaves a row of NaN (both 16-bit types: all bits set).
__global__ __launch_bounds__(256) void embed_kernel(const void* __restrict__ tokens, int is_i64, const uint4* __restrict__ table,
                                                    int64_t vocab, int row16, uint4* __restrict__ out) {
    const int64_t t = blockIdx.x, tok = position(tokens, is_i64, t);
    const bool ok = tok >= 0 && tok < vocab;
    for (int i = blockIdx.y * 256 + threadIdx.x; i < row16; i += gridDim.y * 256)
        out[t * row16 + i] = ok ? table[tok * row16 + i] : make_uint4(~0u, ~0u, ~0u, ~0u);
}

static bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

struct PrefillAttention {
    const uint16_t *qkv, *freqs;
    int64_t wrap;   // rows of freqs from whose end negative positions count, 0: they are outside
    const void* pos;
    int pos_is_i64;
    int64_t T;
    uint16_t *k_cache, *v_cache;
    int n_head, n_kv;
    int64_t S;
    uint16_t* out;
};

template <class E>
static void prefill_attention(const PrefillAttention& a, hipStream_t st) {
    const int T = (int)a.T;
    const int64_t chunks = a.T * 2 * a.n_kv * 16;
    hipLaunchKernelGGL(prefill_cache_kernel<E>, dim3((unsigned)((chunks + 255) / 256)), dim3(256), 0, st, a.qkv, a.freqs, a.wrap,
                       a.pos, a.pos_is_i64, T, a.n_head, a.n_kv, a.S, a.k_cache, a.v_cache);
    const int rep = a.n_head / a.n_kv;
    auto go = [&](auto kernel, int waves, int heads) {
        const int rows = 32 * waves / heads;
        hipLaunchKernelGGL(kernel, dim3(a.n_head / heads, (T + rows - 1) / rows), dim3(512), 0, st, a.qkv, a.freqs, a.wrap, a.pos, a.pos_is_i64, T,
                           a.n_head, a.n_kv, a.S, a.k_cache, a.v_cache, a.out);
    };
    // Groups of two until their workgroups take a third round (us of groups of two / four: 32 heads over 8 at 1000 / 1200 positions 29.2 / 31.0, 40.7 /
    // 36.6; 40 over 40 at 700 / 800 28.3 / 29.0, 35.6 / 31.4; 8 over 4 at 4096 / 8192 72 / 92, 232 / 205), or, where a short prompt's tiles serve four heads
    // and starting is most of the time, a second (64 over 8 at 200 / 300 / 500 11.3 / 13.4, 17.0 / 15.8, 22.6 / 21.3; 32 over 8 at 600 / 900 18.8 / 23.1, 27.0 / 28.3).
    const int64_t workgroups = rep % 2 == 0 ? (int64_t)a.n_head / 2 * ((T + 31) / 32) : (int64_t)a.n_head * ((T + 63) / 64);
    if (workgroups > (rep % 4 == 0 && T <= 512 ? 256 : 512)) {
        if (rep % 4 == 0) go(prefill_attention_kernel<E, 4, 4>, 4, 4);
        else go(prefill_attention_kernel<E, 4, 1>, 4, 1);
    } else if (rep % 2 == 0) {
        go(prefill_attention_kernel<E, 2, 2>, 2, 2);
    } else {
        go(prefill_attention_kernel<E, 2, 1>, 2, 1);
    }
}

static int prefill_attention_entry(const PrefillAttention& a, int is_f16, int head_dim, void* stream) {
    AO_REQUIRE(a.qkv && a.freqs && a.pos && a.k_cache && a.v_cache && a.out, "null pointer argument");
    AO_REQUIRE(head_dim == 128, "prefill attention is built for head_dim 128, got %d", head_dim);
    AO_REQUIRE(a.n_kv > 0 && a.n_head > 0 && a.n_head % a.n_kv == 0, "n_head=%d must be a multiple of n_kv=%d", a.n_head, a.n_kv);
    AO_REQUIRE(a.n_head <= 65535 && a.T >= 0 && a.T <= 1 << 20 && a.S > 0 && a.S <= 1 << 20, "T=%lld, max_seq=%lld out of range",
               (long long)a.T, (long long)a.S);
    AO_REQUIRE(a.wrap == 0 || a.wrap >= a.S, "freqs_cis has %lld rows for a cache of %lld positions", (long long)a.wrap, (long long)a.S);
    AO_REQUIRE(aligned16(a.qkv) && aligned16(a.freqs) && aligned16(a.k_cache) && aligned16(a.v_cache) && aligned16(a.out),
               "16-byte aligned tensors needed");
    if (a.T == 0) return 0;
    if (is_f16)
        prefill_attention<ElemF16>(a, (hipStream_t)stream);
    else
        prefill_attention<ElemBf16>(a, (hipStream_t)stream);
    AO_LAUNCH_CHECK();
    return 0;
}

}  // namespace ao

using namespace ao;

extern "C" int ao_amd_llama_prefill_attention(const void* qkv, int is_f16, const void* freqs_cis, const void* positions, int pos_is_i64,
                                              int64_t T, void* k_cache, void* v_cache, int n_head, int n_kv, int head_dim,
                                              int64_t max_seq, void* out, void* stream) {
    return prefill_attention_entry({(const uint16_t*)qkv, (const uint16_t*)freqs_cis, 0, positions, pos_is_i64, T, (uint16_t*)k_cache,
                                    (uint16_t*)v_cache, n_head, n_kv, max_seq, (uint16_t*)out}, is_f16, head_dim, stream);
}

extern "C" int ao_amd_llama_prefill_attention_wrap(const void* qkv, int is_f16, const void* freqs_cis, int64_t freqs_len,
                                                   const void* positions, int pos_is_i64, int64_t T, void* k_cache, void* v_cache,
                                                   int n_head, int n_kv, int head_dim, int64_t max_seq, void* out, void* stream) {
    AO_REQUIRE(freqs_len > 0, "freqs_len=%lld must be positive", (long long)freqs_len);
    return prefill_attention_entry({(const uint16_t*)qkv, (const uint16_t*)freqs_cis, freqs_len, positions, pos_is_i64, T, (uint16_t*)k_cache,
                                    (uint16_t*)v_cache, n_head, n_kv, max_seq, (uint16_t*)out}, is_f16, head_dim, stream);
}

extern "C" int ao_amd_add_rmsnorm(const void* x, const void* y, const void* weight, int is_f16, int64_t rows, int64_t dim, float eps,
                                  void* sum, void* normed, void* stream) {
    AO_REQUIRE(x && y && weight && sum && normed, "null pointer argument");
    AO_REQUIRE(rows >= 0 && rows <= INT32_MAX && dim > 0 && dim <= 8192 && dim % 8 == 0, "rows=%lld, dim=%lld: dim must be a multiple of 8, at most 8192",
               (long long)rows, (long long)dim);
    AO_REQUIRE(aligned16(x) && aligned16(y) && aligned16(weight) && aligned16(sum) && aligned16(normed), "16-byte aligned tensors needed");
    if (rows == 0) return 0;
    if (is_f16)
        hipLaunchKernelGGL(add_rmsnorm_kernel<ElemF16>, dim3((unsigned)rows), dim3(256), 0, (hipStream_t)stream, (const uint16_t*)x,
                           (const uint16_t*)y, (const uint16_t*)weight, (int)dim, eps, (uint16_t*)sum, (uint16_t*)normed);
    else
        hipLaunchKernelGGL(add_rmsnorm_kernel<ElemBf16>, dim3((unsigned)rows), dim3(256), 0, (hipStream_t)stream, (const uint16_t*)x,
                           (const uint16_t*)y, (const uint16_t*)weight, (int)dim, eps, (uint16_t*)sum, (uint16_t*)normed);
    AO_LAUNCH_CHECK();
    return 0;
}

extern "C" int ao_amd_silu_mul(const void* gate, const void* up, int is_f16, int64_t n, void* out, void* stream) {
    AO_REQUIRE(gate && up && out, "null pointer argument");
    AO_REQUIRE(n >= 0 && n % 8 == 0 && n / 8 / 256 < INT32_MAX, "n=%lld must be a multiple of 8", (long long)n);
    AO_REQUIRE(aligned16(gate) && aligned16(up) && aligned16(out), "16-byte aligned tensors needed");
    if (n == 0) return 0;
    const dim3 grid((unsigned)((n / 8 + 255) / 256));
    if (is_f16)
        hipLaunchKernelGGL(silu_mul_kernel<ElemF16>, grid, dim3(256), 0, (hipStream_t)stream, (const uint16_t*)gate, (const uint16_t*)up,
                           n / 8, (uint16_t*)out);
    else
        hipLaunchKernelGGL(silu_mul_kernel<ElemBf16>, grid, dim3(256), 0, (hipStream_t)stream, (const uint16_t*)gate, (const uint16_t*)up,
                           n / 8, (uint16_t*)out);
    AO_LAUNCH_CHECK();
    return 0;
}

extern "C" int ao_amd_llama_embed(const void* tokens, int is_i64, int64_t T, const void* table, int64_t vocab, int64_t dim, void* out,
                                  void* stream) {
    AO_REQUIRE(tokens && table && out, "null pointer argument");
    AO_REQUIRE(T >= 0 && T <= INT32_MAX && vocab > 0 && dim > 0 && dim % 8 == 0, "T=%lld, dim=%lld: dim must be a multiple of 8",
               (long long)T, (long long)dim);
    AO_REQUIRE(aligned16(table) && aligned16(out), "16-byte aligned tensors needed");
    if (T == 0) return 0;
    // one row: spread over a few workgroups, many rows: one each
    const dim3 grid((unsigned)T, T >= 64 ? 1u : (unsigned)((dim / 8 + 255) / 256));
    hipLaunchKernelGGL(embed_kernel, grid, dim3(256), 0, (hipStream_t)stream, tokens, is_i64, (const uint4*)table, vocab, (int)(dim / 8),
                       (uint4*)out);
    AO_LAUNCH_CHECK();
    return 0;
}
