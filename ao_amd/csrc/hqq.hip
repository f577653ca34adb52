// HQQ-format int4 weights (torchao/prototype/hqq): dequantization for the mixed matmul.
//
// The reference's Triton kernel (torchao/prototype/hqq/kernels.py:200-380) multiplies activations with a weight kept
// as `pack_2xint4(W_q.T)`: uint8 [K/2, N], byte (k2, n) = W_q[n][2*k2] | W_q[n][2*k2 + 1] << 4
// (torchao/prototype/hqq/mixed_mm.py:13-35), with scales and zeros of shape [K/group, N] in the activation dtype, and
// dequantizes in that dtype, op by op: w = (q - zero) * scale (kernels.py:358).  The products (x @ W over K, and x @ W^T over N,
// which the backward pass of a fine-tuning run needs) are fused below and in hqq_tile.hip.  For what those do not take the
// dequantization is a pass of its own into a [K, N] matrix of the activation dtype, followed by a plain library GEMM: the packed layout is N-major, so a thread that takes 16 consecutive bytes of one k2 row produces two 32-byte
// runs of the output rows 2*k2 and 2*k2 + 1, and neighbouring threads continue those rows.
#include <type_traits>

#include "hqq_format.h"

namespace ao {

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

template <bool BF16, bool SIGNED>
__global__ __launch_bounds__(256) void hqq_dequantize_kernel(const uint8_t* __restrict__ packed, const uint16_t* __restrict__ scales,
                                                             const uint16_t* __restrict__ zeros, int64_t K, int64_t N,
                                                             int64_t group, uint16_t* __restrict__ out) {
    const int64_t chunks = N / 16;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (K / 2) * chunks) return;
    const int64_t k2 = i / chunks, n0 = (i % chunks) * 16;
    const int64_t g = (2 * k2) / group;
    union { u32x4_t v; uint8_t b[16]; } q;
    q.v = *reinterpret_cast<const u32x4_t*>(packed + k2 * N + n0);
    union { u32x4_t v[2]; uint16_t h[16]; } s, z, lo, hi;
    const u32x4_t* sp = reinterpret_cast<const u32x4_t*>(scales + g * N + n0);
    const u32x4_t* zp = reinterpret_cast<const u32x4_t*>(zeros + g * N + n0);
    s.v[0] = sp[0]; s.v[1] = sp[1];
    z.v[0] = zp[0]; z.v[1] = zp[1];
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        // the reference unpacks with (qb << 4) >> 4 and qb >> 4 in the storage dtype: logical shifts for uint8,
        // arithmetic (sign-extending) shifts for int8 (kernels.py:324-326)
        const int ql = SIGNED ? ((int)(int8_t)(q.b[e] << 4)) >> 4 : (q.b[e] & 15);
        const int qh = SIGNED ? ((int)(int8_t)q.b[e]) >> 4 : (q.b[e] >> 4);
        if (BF16) {
            const float sf = bf16_bits_to_f32(s.h[e]), zf = bf16_bits_to_f32(z.h[e]);
            lo.h[e] = hw_bf16_bits(hw_rne_bf16((float)ql - zf) * sf);
            hi.h[e] = hw_bf16_bits(hw_rne_bf16((float)qh - zf) * sf);
        } else {
            _Float16 sf, zf;
            __builtin_memcpy(&sf, &s.h[e], 2);
            __builtin_memcpy(&zf, &z.h[e], 2);
            const _Float16 wl = ((_Float16)ql - zf) * sf, wh = ((_Float16)qh - zf) * sf;  // each op rounds to fp16
            __builtin_memcpy(&lo.h[e], &wl, 2);
            __builtin_memcpy(&hi.h[e], &wh, 2);
        }
    }
    u32x4_t* o0 = reinterpret_cast<u32x4_t*>(out + (2 * k2) * N + n0);
    u32x4_t* o1 = reinterpret_cast<u32x4_t*>(out + (2 * k2 + 1) * N + n0);
    o0[0] = lo.v[0]; o0[1] = lo.v[1];
    o1[0] = hi.v[0]; o1[1] = hi.v[1];
}

// ---------------------------------------------------------------- fused mixed matmul for few activation rows
// y[M, N] = a[M, K] @ W[K, N] with W dequantized on the fly (the forward product of the reference's Triton kernel,
// torchao/prototype/hqq/kernels.py:162-388, for the decode-sized batches where a dequantize pass + library GEMM moves
// five times the bytes).  The packed layout is N-major, so lanes go along N: a lane owns 4 adjacent columns (one dword
// of a byte row = 8 codes: 4 columns x 2 consecutive k), a wave 256 columns, and walks a run of byte rows; the
// activations a[m][2 k2], a[m][2 k2 + 1] are the same for every lane and come through scalar loads.  K is cut into
// gridDim.y slices x 4 waves; the waves of a workgroup add up in LDS and each slice leaves fp32 partial sums
// part[slice][m][n], which hqq_mm_finish_kernel adds and rounds.  Every weight is rounded exactly as the dequantize
// kernel above rounds it.
template <bool BF16, bool SIGNED, int MB>
__global__ __launch_bounds__(256) void hqq_mm_small_kernel(const uint8_t* __restrict__ packed, const uint16_t* __restrict__ scales,
                                                           const uint16_t* __restrict__ zeros, const uint16_t* __restrict__ a,
                                                           int64_t lda, int M, int64_t K, int64_t N, int64_t group,
                                                           int rows_per_wave, float* __restrict__ part) {
    __shared__ float red[4][MB][256];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t n0 = ((int64_t)blockIdx.x * 64 + lane) * 4;
    const bool live = n0 < N;   // N is a multiple of 4
    const int64_t K2 = K / 2;
    const int64_t r0 = ((int64_t)blockIdx.y * 4 + wave) * rows_per_wave;
    const int64_t r1 = r0 + rows_per_wave < K2 ? r0 + rows_per_wave : K2;
    float acc[MB][4];
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[m][c] = 0.f;
    const uint32_t* arow[MB];
#pragma unroll
    for (int m = 0; m < MB; ++m) arow[m] = reinterpret_cast<const uint32_t*>(a + (int64_t)(m < M ? m : M - 1) * lda);
    auto widen = [](uint16_t h) -> float {
        if (BF16) return bf16_bits_to_f32(h);
        _Float16 f;
        __builtin_memcpy(&f, &h, 2);
        return (float)f;
    };
    // (q - zero) * scale, each op rounded to the storage dtype, as a float
    auto weight = [&](int q, float zf, float sf) -> float {
        if (BF16) return hw_rne_bf16(hw_rne_bf16((float)q - zf) * sf);
        const _Float16 w = ((_Float16)q - (_Float16)zf) * (_Float16)sf;
        return (float)w;
    };
    int64_t g_cur = -1;
    float sf[4] = {0.f, 0.f, 0.f, 0.f}, zf[4] = {0.f, 0.f, 0.f, 0.f};
    auto load_group = [&](int64_t k2) {
        const int64_t g = (2 * k2) / group;
        if (g != g_cur && live) {
            g_cur = g;
            const uint2 sv = *reinterpret_cast<const uint2*>(scales + g * N + n0);
            const uint2 zv = *reinterpret_cast<const uint2*>(zeros + g * N + n0);
            sf[0] = widen((uint16_t)sv.x); sf[1] = widen((uint16_t)(sv.x >> 16)); sf[2] = widen((uint16_t)sv.y); sf[3] = widen((uint16_t)(sv.y >> 16));
            zf[0] = widen((uint16_t)zv.x); zf[1] = widen((uint16_t)(zv.x >> 16)); zf[2] = widen((uint16_t)zv.y); zf[3] = widen((uint16_t)(zv.y >> 16));
        }
    };
    // one byte row: 8 codes of the lane's 4 columns, times the row's two activations of every row m
    auto row = [&](uint32_t d, const uint32_t (&av)[MB]) {
        float wl[4], wh[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const uint32_t b = (d >> (8 * c)) & 0xffu;
            // the reference unpacks with (qb << 4) >> 4 and qb >> 4 in the storage dtype (kernels.py:324-326)
            const int ql = SIGNED ? ((int)(int8_t)(uint8_t)(b << 4)) >> 4 : (int)(b & 15u);
            const int qh = SIGNED ? ((int)(int8_t)(uint8_t)b) >> 4 : (int)(b >> 4);
            wl[c] = weight(ql, zf[c], sf[c]);
            wh[c] = weight(qh, zf[c], sf[c]);
        }
#pragma unroll
        for (int m = 0; m < MB; ++m) {
            const float a0 = widen((uint16_t)av[m]), a1 = widen((uint16_t)(av[m] >> 16));
#pragma unroll
            for (int c = 0; c < 4; ++c) acc[m][c] += a0 * wl[c] + a1 * wh[c];
        }
    };
    int64_t k2 = r0;
    // four byte rows per trip: their code dwords and the 8 activations of every row m (one 16-byte scalar load each,
    // the address is the same in every lane) are requested together
    for (; k2 + 4 <= r1; k2 += 4) {
        uint32_t d[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) d[r] = live ? *reinterpret_cast<const uint32_t*>(packed + (k2 + r) * N + n0) : 0u;
        uint32_t av[4][MB];
#pragma unroll
        for (int m = 0; m < MB; ++m) {
            const uint32_t* p = arow[m] + k2;
            av[0][m] = p[0]; av[1][m] = p[1]; av[2][m] = p[2]; av[3][m] = p[3];
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            load_group(k2 + r);
            row(d[r], av[r]);
        }
    }
    for (; k2 < r1; ++k2) {
        load_group(k2);
        const uint32_t d = live ? *reinterpret_cast<const uint32_t*>(packed + k2 * N + n0) : 0u;
        uint32_t av[MB];
#pragma unroll
        for (int m = 0; m < MB; ++m) av[m] = arow[m][k2];
        row(d, av);
    }
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int c = 0; c < 4; ++c) red[wave][m][lane * 4 + c] = acc[m][c];
    __syncthreads();
    // 256 threads: column threadIdx.x of the block, all rows
    const int64_t n = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (n < N) {
#pragma unroll
        for (int m = 0; m < MB; ++m)
            if (m < M)
                part[((int64_t)blockIdx.y * M + m) * N + n] = red[0][m][threadIdx.x] + red[1][m][threadIdx.x] +
                                                              red[2][m][threadIdx.x] + red[3][m][threadIdx.x];
    }
}

// V sums a thread: four where all of them are whole aligned runs, one elsewhere (an odd number of rows over K = 2 mod 4 outputs of the
// transposed product, a workspace that is only 4-byte aligned)
template <bool BF16, int V>
__global__ __launch_bounds__(256) void hqq_mm_finish_kernel(const float* __restrict__ part, int slices, int64_t count,
                                                            uint16_t* __restrict__ y) {
    const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * V;
    if (i >= count) return;   // (V divides count)
    float s[V];
#pragma unroll
    for (int e = 0; e < V; ++e) s[e] = 0.f;
    for (int z = 0; z < slices; ++z) {
        const float* const src = part + (int64_t)z * count + i;
        if constexpr (V == 4) {
            const float4 v = *reinterpret_cast<const float4*>(src);
            s[0] += v.x; s[1] += v.y; s[2] += v.z; s[3] += v.w;
        } else {
            s[0] += src[0];
        }
    }
    uint16_t o[V];
#pragma unroll
    for (int e = 0; e < V; ++e) o[e] = BF16 ? hw_bf16_bits(s[e]) : f32_to_f16_bits(s[e]);
    if (V == 4 && ((uintptr_t)y & 7) == 0)
        *reinterpret_cast<uint2*>(y + i) = make_uint2(o[0] | ((uint32_t)o[1 % V] << 16), o[2 % V] | ((uint32_t)o[3 % V] << 16));
    else
#pragma unroll
        for (int e = 0; e < V; ++e) y[i + e] = o[e];
}
void launch_hqq_finish(const float* part, int slices, int64_t count, bool bf16, uint16_t* y, hipStream_t st) {
    auto go = [&](auto kernel, int v) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)((count / v + 255) / 256)), dim3(256), 0, st, part, slices, count, y);
    };
    // (part is 16-byte aligned and so is every slice behind it)
    if (count % 4 == 0 && ((uintptr_t)part & 15) == 0) bf16 ? go(hqq_mm_finish_kernel<true, 4>, 4) : go(hqq_mm_finish_kernel<false, 4>, 4);
    else bf16 ? go(hqq_mm_finish_kernel<true, 1>, 1) : go(hqq_mm_finish_kernel<false, 1>, 1);
}

// K slices of the small-M product: enough waves to occupy the chip, at least 8 byte rows per wave
static int hqq_mm_slices(int64_t K, int64_t N) {
    const int64_t colblocks = (N + 255) / 256, K2 = K / 2;
    int64_t s = (4096 + colblocks * 4 - 1) / (colblocks * 4);
    const int64_t most = (K2 + 31) / 32;   // 4 waves x 8 rows
    if (s > most) s = most;
    if (s < 1) s = 1;
    if (s > 64) s = 64;
    return (int)s;
}

// ---------------------------------------------------------------- fused mixed matmul on the matrix cores, up to 64 rows
// Both products of the reference's Triton kernel (torchao/prototype/hqq/kernels.py:162-388) with the weight dequantized
// in registers: forward y[M, N] = a[M, K] @ W (reduction over K) and transposed y[M, K] = a[M, N] @ W^T (reduction over
// N, the product a backward pass needs).  v_mfma_f32_16x16x32 contracts 32 reduction indices; a lane of its weight
// operand holds 8 of them for ONE output column, and any order of the 32 is fine as long as the activation operand uses
// the same one.  The byte layout [K/2, N] (two consecutive k per byte, N fastest) fits both products without a
// transposition:
//   forward     lane (j = lane % 16, kb = lane / 16) loads one dword from each of the 4 byte rows k2 = 16 s + 4 kb + r
//               at columns n = 64 tile + 4 j + c: 8 consecutive k for each of 4 columns.  MFMA c (of 4) takes the 8
//               weights of column c, so its output column j is n = 64 tile + 4 j + c and a lane ends with 4 adjacent
//               outputs of a row.
//   transposed  lane (j, nb) loads 16 bytes of byte row k2 = 16 tile + j at n = 64 s + 16 nb + e: 16 reduction indices
//               for the two output columns k = 2 k2 (low nibbles) and 2 k2 + 1 (high nibbles): 4 MFMAs (low / high x
//               two halves of 8) into two accumulators, and a lane ends with the adjacent outputs k, k + 1 of a row.
// A wave step covers 2048 weights either way.  The reduction is cut over gridDim.y x 4 waves; the waves of a workgroup
// add up in LDS and every slice leaves fp32 partial sums part[slice][m][col] for hqq_mm_finish_kernel.  Every weight
// is rounded twice to the storage dtype, exactly as hqq_dequantize_kernel rounds it.
typedef __bf16 hqq_bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 hqq_f16x8_t __attribute__((ext_vector_type(8)));
typedef float hqq_f32x4_t __attribute__((ext_vector_type(4)));

template <bool BF16>
__device__ __forceinline__ hqq_f32x4_t hqq_mfma(const u32x4_t a, const uint32_t (&b)[4], hqq_f32x4_t c) {
    if (BF16) {
        union { u32x4_t q; hqq_bf16x8_t v; } xa, xb;
        xa.q = a;
        xb.q = u32x4_t{b[0], b[1], b[2], b[3]};
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa.v, xb.v, c, 0, 0, 0);
    } else {
        union { u32x4_t q; hqq_f16x8_t v; } xa, xb;
        xa.q = a;
        xb.q = u32x4_t{b[0], b[1], b[2], b[3]};
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(xa.v, xb.v, c, 0, 0, 0);
    }
}

// Waves of a workgroup: each takes a run of the reduction, and they add up in LDS.  A step's loads take a microsecond and a
// wave keeps one step ahead in flight (tiles_ahead), so the runs are kept short and the waves many; eight of them to a
// workgroup keep the number of fp32 partial sums in memory where four waves with runs of eight steps had it.  Two steps ahead up to 16 rows, in three
// sets of fragments used in turn, took 14.8 / 15.8 us for one and 16 rows of fp16 14336 x 4096 where one takes 13.6 / 14.3, one ahead in two such sets 32 rows
// transposed of 4096 x 11008 16.2 where the copy from set to set takes 15.4: the step's code stands once then.

// RB (transposed product): blocks of 16 byte rows per wave.  With two of them in one quantization group the activation
// fragments and the scales and zeros, 128 bytes a lane and step, serve 32 bytes of codes instead of 16.
template <bool BF16, bool SIGNED, bool TRANSPOSED, int MB, int RB, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void hqq_mm_mfma_kernel(const uint8_t* __restrict__ packed, const uint16_t* __restrict__ scales,
                                                          const uint16_t* __restrict__ zeros, const uint16_t* __restrict__ a,
                                                          int64_t lda, int M, int64_t K, int64_t N, int64_t group,
                                                          int steps, int steps_per_wave, float* __restrict__ part) {
    static_assert(TRANSPOSED || RB == 1, "the forward product takes one block of columns per wave");
    constexpr int NACC = TRANSPOSED ? 2 * RB : 4;   // accumulators per block of 16 activation rows
    __shared__ float red[WAVES][NACC * 4][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane & 15, q4 = lane >> 4;
    const int64_t K2 = K / 2;
    const int s0 = ((int)blockIdx.y * WAVES + wave) * steps_per_wave;
    const int s1 = s0 + steps_per_wave < steps ? s0 + steps_per_wave : steps;
    hqq_f32x4_t acc[MB][NACC];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int c = 0; c < NACC; ++c) acc[mb][c] = hqq_f32x4_t{0.f, 0.f, 0.f, 0.f};
    // activation rows of this lane (operand row j of every block of 16); rows past M read row M - 1 and are not written
    const uint16_t* arow[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        const int m = mb * 16 + j;
        arow[mb] = a + (int64_t)(m < M ? m : M - 1) * lda;
    }
    const u32x4_t zero4 = {0u, 0u, 0u, 0u};

    if (!TRANSPOSED) {
        // columns past N (a multiple of 4) repeat the last ones and are not stored
        const int64_t n_at = (int64_t)blockIdx.x * 64 + 4 * j, n0 = n_at < N ? n_at : N - 4;
        struct Frag { uint32_t d[4]; uint2 s, z; u32x4_t x[MB]; };
        const uint32_t eighths = (uint32_t)(group / 8);
        const int shift = (eighths & (eighths - 1)) == 0 ? __builtin_ctz(eighths) : -1;
        const int tail = K2 % 16 ? steps - 1 : -1;   // the step that ends before its 16 byte rows
        auto load = [&](Frag& f, int s) __attribute__((always_inline)) {
            const int64_t at = (int64_t)s * 16 + 4 * q4, k2 = at < K2 ? at : K2 - 4;   // K is a multiple of 8: the lane's 4 byte rows exist together
            // group is a multiple of 8: one group for the lane's 8 k
            const uint32_t eighth = (uint32_t)k2 >> 2;
            const int64_t g = shift >= 0 ? eighth >> shift : eighth / eighths;
#pragma unroll
            for (int r = 0; r < 4; ++r) f.d[r] = *reinterpret_cast<const uint32_t*>(packed + (k2 + r) * N + n0);
            f.s = *reinterpret_cast<const uint2*>(scales + g * N + n0);
            f.z = *reinterpret_cast<const uint2*>(zeros + g * N + n0);
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) f.x[mb] = *reinterpret_cast<const u32x4_t*>(arow[mb] + 2 * k2);
        };
        auto compute = [&](Frag& f, int s) __attribute__((always_inline)) {
            if (s == tail && (int64_t)s * 16 + 4 * q4 >= K2) {   // 0 x (0 - 0) * 0
#pragma unroll
                for (int r = 0; r < 4; ++r) f.d[r] = 0u;
                f.s = f.z = uint2{0u, 0u};
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) f.x[mb] = zero4;
            }
            uint32_t sv[4], zv[4];   // a column's value twice
            float sf[4], zf[4];
            const uint32_t ss[2] = {f.s.x, f.s.y}, zz[2] = {f.z.x, f.z.y};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                if constexpr (BF16) {
                    sf[c] = __uint_as_float(c & 1 ? ss[c >> 1] & 0xffff0000u : ss[c >> 1] << 16);
                    zf[c] = __uint_as_float(c & 1 ? zz[c >> 1] & 0xffff0000u : zz[c >> 1] << 16);
                } else {
                    const uint32_t sh = (c & 1) ? ss[c >> 1] >> 16 : ss[c >> 1] & 0xffffu, zh = (c & 1) ? zz[c >> 1] >> 16 : zz[c >> 1] & 0xffffu;
                    sv[c] = sh | (sh << 16);
                    zv[c] = zh | (zh << 16);
                }
            }
            uint32_t lo[4], hi[4], w[4][4];   // w: [column][byte row]
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if constexpr (BF16) hqq_columns<SIGNED>(f.d[r], zf, sf, w[0][r], w[1][r], w[2][r], w[3][r]);
                else hqq_nibbles<SIGNED>(f.d[r], lo[r], hi[r]);
            }
            // both nibbles of byte c belong to column c
            auto column = [&](auto c_c) {
                constexpr int c = decltype(c_c)::value;
                if constexpr (!BF16)
#pragma unroll
                    for (int r = 0; r < 4; ++r) w[c][r] = hqq_pair<SIGNED, c, c>(lo[r], hi[r], sv[c], zv[c]);
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) acc[mb][c] = hqq_mfma<BF16>(f.x[mb], w[c], acc[mb][c]);
            };
            column(std::integral_constant<int, 0>());
            column(std::integral_constant<int, 1>());
            column(std::integral_constant<int, 2>());
            column(std::integral_constant<int, 3>());
        };
        tiles_ahead<Frag>(s0, s1, 1, load, compute);
    } else {
        int64_t k2[RB];
        bool live[RB];
        const uint8_t* prow[RB];
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            k2[rb] = (int64_t)blockIdx.x * 16 * RB + 16 * rb + j;
            live[rb] = k2[rb] < K2;
            prow[rb] = packed + (live[rb] ? k2[rb] : 0) * N;
        }
        const int64_t g = live[0] ? (2 * k2[0]) / group : 0;   // RB == 2: the host has checked that both blocks share it
        const int64_t g_block = (int64_t)blockIdx.x * 32 * RB / group;   // of the block's first row, which exists
        const uint16_t* srow = scales + g * N;
        const uint16_t* zrow = zeros + g * N;
        struct Frag { u32x4_t d[RB], x[MB][2]; };
        const int tail = N % 64 ? steps - 1 : -1;   // the step that ends before its 64 columns
        auto column = [&](int s) {
            const int64_t at = (int64_t)s * 64 + 16 * q4;
            return at < N ? at : N - 16;   // N is a multiple of 16
        };
        auto load = [&](Frag& f, int s) __attribute__((always_inline)) {
            const int64_t n = column(s);
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) f.d[rb] = *reinterpret_cast<const u32x4_t*>(prow[rb] + n);
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                for (int h = 0; h < 2; ++h) f.x[mb][h] = *reinterpret_cast<const u32x4_t*>(arow[mb] + n + 8 * h);
        };
        const HqqRowMatrices rows(lane);
        auto compute = [&](Frag& f, int s, u32x4_t (&sc)[2], u32x4_t (&ze)[2], auto element_wise) __attribute__((always_inline)) {
            if (s == tail && (int64_t)s * 64 + 16 * q4 >= N) {   // 0 x (0 - 0) * 0
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) f.d[rb] = zero4;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    sc[h] = ze[h] = zero4;
#pragma unroll
                    for (int mb = 0; mb < MB; ++mb) f.x[mb][h] = zero4;
                }
            }
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if constexpr (BF16 && !decltype(element_wise)::value) {
                    HqqRowScales sz[2];   // of indices 8 h .. + 3, + 4 .. + 7
                    sz[0] = rows.scales(sc[h].x, sc[h].y, ze[h].x, ze[h].y);
                    sz[1] = rows.scales(sc[h].z, sc[h].w, ze[h].z, ze[h].w);
#pragma unroll
                    for (int rb = 0; rb < RB; ++rb) {
                        const uint32_t dd[4] = {f.d[rb].x, f.d[rb].y, f.d[rb].z, f.d[rb].w};
                        uint32_t lo[4], hi[4];
#pragma unroll
                        for (int i = 0; i < 2; ++i) rows.template weights<SIGNED>(dd[2 * h + i], sz[i], lo[2 * i], lo[2 * i + 1], hi[2 * i], hi[2 * i + 1]);
#pragma unroll
                        for (int mb = 0; mb < MB; ++mb) {
                            acc[mb][2 * rb] = hqq_mfma<BF16>(f.x[mb][h], lo, acc[mb][2 * rb]);
                            acc[mb][2 * rb + 1] = hqq_mfma<BF16>(f.x[mb][h], hi, acc[mb][2 * rb + 1]);
                        }
                    }
                    continue;
                }
                const uint32_t ss[4] = {sc[h].x, sc[h].y, sc[h].z, sc[h].w};
                const uint32_t zz[4] = {ze[h].x, ze[h].y, ze[h].z, ze[h].w};
                float sf[8], zf[8];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    sf[2 * i] = __uint_as_float(ss[i] << 16);
                    sf[2 * i + 1] = __uint_as_float(ss[i] & 0xffff0000u);
                    zf[2 * i] = __uint_as_float(zz[i] << 16);
                    zf[2 * i + 1] = __uint_as_float(zz[i] & 0xffff0000u);
                }
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) {
                    const uint32_t dd[4] = {f.d[rb].x, f.d[rb].y, f.d[rb].z, f.d[rb].w};
                    uint32_t lo[4], hi[4];
#pragma unroll
                    for (int i = 0; i < 4; i += 2) {
                        // reduction indices 8 h + 2 i .. + 3: the four bytes of dword 2 h + i / 2
                        const uint32_t d = dd[2 * h + (i >> 1)];
                        if constexpr (BF16) {
                            hqq_row<SIGNED, false>(d, zf + 2 * i, sf + 2 * i, lo[i], lo[i + 1]);
                            hqq_row<SIGNED, true>(d, zf + 2 * i, sf + 2 * i, hi[i], hi[i + 1]);
                        } else {
                            uint32_t nl, nh;
                            hqq_nibbles<SIGNED>(d, nl, nh);
                            lo[i] = hqq_pair<SIGNED, 0, 1>(nl, nl, ss[i], zz[i]);
                            hi[i] = hqq_pair<SIGNED, 0, 1>(nh, nh, ss[i], zz[i]);
                            lo[i + 1] = hqq_pair<SIGNED, 2, 3>(nl, nl, ss[i + 1], zz[i + 1]);
                            hi[i + 1] = hqq_pair<SIGNED, 2, 3>(nh, nh, ss[i + 1], zz[i + 1]);
                        }
                    }
#pragma unroll
                    for (int mb = 0; mb < MB; ++mb) {
                        acc[mb][2 * rb] = hqq_mfma<BF16>(f.x[mb][h], lo, acc[mb][2 * rb]);
                        acc[mb][2 * rb + 1] = hqq_mfma<BF16>(f.x[mb][h], hi, acc[mb][2 * rb + 1]);
                    }
                }
            }
        };
        // Where all 16 byte rows of a block share their group, a wave brings the scales and zeros of its columns into LDS, CHUNK steps at a
        // time: read by each lane they were 4 of the 8 (16 rows) to 14 (64 rows) requests of a step, for a sixteenth of their bytes, and a CU takes
        // some 45 bytes a cycle of them (32 rows x 4096 x 11008 of bf16 / fp16 with the unconditional requests alone 18.5 / 18.9 us, with this 16.2 / 16.9).
        constexpr int CHUNK = NACC * 4;   // 256 bytes a step, in the wave's own part of what the waves add up in later
        uint16_t* const s_lds = reinterpret_cast<uint16_t*>(&red[wave][0][0]);
        uint16_t* const z_lds = s_lds + CHUNK * 64;
        bool direct = group % 32 != 0;
        // bf16: whether scales and zeros allow the matrix instructions is looked at as they pass, and once more where one may be 0.  Two block rows: in front
        // of a chunk's products; one: at the end, as the chunks are short (16 rows of 13824 x 5120 in groups of 32 22.6 -> 24.1 us in front, 23.0 at the end; 32
        // rows x 4096 x 11008 in groups of 64 16.0 -> 16.2 in front, 16.5 at the end).
        HqqOrdinary ordinary;
        if (!direct) {
            for (int c0 = s0; c0 < s1; c0 += CHUNK) {
                const int c1 = c0 + CHUNK < s1 ? c0 + CHUNK : s1;
                const int64_t n_end = (int64_t)c1 * 64 < N ? (int64_t)c1 * 64 : N;
                u32x4_t in[2][CHUNK / 8];
#pragma unroll
                for (int i = 0; i < CHUNK / 8; ++i) {
                    const int64_t at = (int64_t)c0 * 64 + i * 512 + lane * 8, n = at < n_end ? at : n_end - 8;
                    in[0][i] = *reinterpret_cast<const u32x4_t*>(scales + g_block * N + n);
                    in[1][i] = *reinterpret_cast<const u32x4_t*>(zeros + g_block * N + n);
                }
                if (BF16) {   // (a lane's columns past the end of the run are the last ones again)
                    HqqOrdinary here;
#pragma unroll
                    for (int i = 0; i < 2 * (CHUNK / 8); ++i)
#pragma unroll
                        for (int e = 0; e < 4; ++e) here.see(in[i & 1][i >> 1][e]);
                    if (RB == 1) {
                        ordinary.most = __builtin_elementwise_max(ordinary.most, here.most);
                    } else {
                        bool all = here.all();
                        if (!all) {
                            all = true;
#pragma unroll
                            for (int i = 0; i < 2 * (CHUNK / 8); ++i)
#pragma unroll
                                for (int e = 0; e < 4; ++e) all &= HqqOrdinary::with_zeros(in[i & 1][i >> 1][e]);
                        }
                        direct = __any(!all);
                        if (direct) break;
                    }
                }
#pragma unroll
                for (int i = 0; i < CHUNK / 8; ++i) {
                    *reinterpret_cast<u32x4_t*>(s_lds + i * 512 + lane * 8) = in[0][i];
                    *reinterpret_cast<u32x4_t*>(z_lds + i * 512 + lane * 8) = in[1][i];
                }
                asm volatile("" ::: "memory");   // (one wave: its LDS operations are done in order)
                tiles_ahead<Frag>(c0, c1, 1, load, [&](Frag& f, int s) __attribute__((always_inline)) {
                    const uint16_t* const at = s_lds + (s - c0) * 64 + 16 * q4;
                    u32x4_t sc[2], ze[2];
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        sc[h] = *reinterpret_cast<const u32x4_t*>(at + 8 * h);
                        ze[h] = *reinterpret_cast<const u32x4_t*>(at + CHUNK * 64 + 8 * h);
                    }
                    compute(f, s, sc, ze, std::integral_constant<bool, !BF16>());
                });
                asm volatile("" ::: "memory");
            }
        }
        if (BF16 && group % 32 == 0) {   // 2^-9 of the sums; of no use where a scale or zero was beyond the range
            if (RB == 1 && __any(!ordinary.all())) {
                const int64_t n_end = (int64_t)s1 * 64 < N ? (int64_t)s1 * 64 : N;
                bool all = true;
                for (int64_t n = (int64_t)s0 * 64 + lane * 8; n < n_end; n += 512) {
                    const u32x4_t sc = *reinterpret_cast<const u32x4_t*>(scales + g_block * N + n), ze = *reinterpret_cast<const u32x4_t*>(zeros + g_block * N + n);
#pragma unroll
                    for (int e = 0; e < 4; ++e) all &= HqqOrdinary::with_zeros(sc[e]) & HqqOrdinary::with_zeros(ze[e]);
                }
                direct = __any(!all);
            }
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                for (int c = 0; c < NACC; ++c)
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[mb][c][r] = direct ? 0.f : acc[mb][c][r] * HqqRowMatrices::DOWN;
        }
        if (direct)   // other group sizes, and scales or zeros beyond the range
            for (int s = s0; s < s1; ++s) {
                Frag f;
                u32x4_t sc[2], ze[2];
                load(f, s);
                const int64_t n = column(s);
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    sc[h] = *reinterpret_cast<const u32x4_t*>(srow + n + 8 * h);
                    ze[h] = *reinterpret_cast<const u32x4_t*>(zrow + n + 8 * h);
                }
                compute(f, s, sc, ze, std::true_type());
            }
    }

    // the waves of the workgroup add up, one block of 16 rows at a time: thread (wave w < 4, lane) sums element r = w of
    // every accumulator, which is output row 4 (lane / 16) + w of the block and NACC adjacent columns
    const int64_t cols = TRANSPOSED ? K : N;
    const int64_t col0 = TRANSPOSED ? 2 * ((int64_t)blockIdx.x * 16 * RB + j) : (int64_t)blockIdx.x * 64 + 4 * j;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        if (mb) __syncthreads();
#pragma unroll
        for (int c = 0; c < NACC; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) red[wave][c * 4 + r][lane] = acc[mb][c][r];
        __syncthreads();
        if (wave >= 4) continue;
        const int m = mb * 16 + 4 * q4 + wave;
        float v[NACC];
#pragma unroll
        for (int c = 0; c < NACC; ++c) {
            v[c] = red[0][c * 4 + wave][lane];
#pragma unroll
            for (int w = 1; w < WAVES; ++w) v[c] += red[w][c * 4 + wave][lane];
        }
        float* o = part + ((int64_t)blockIdx.y * M + m) * cols + col0;
        if (TRANSPOSED) {
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
                if (m < M && col0 + 32 * rb < cols) *reinterpret_cast<float2*>(o + 32 * rb) = float2{v[2 * rb], v[2 * rb + 1]};
        } else if (m < M && col0 < cols) {
            *reinterpret_cast<float4*>(o) = float4{v[0], v[1], v[NACC - 2], v[NACC - 1]};
        }
    }
}

// reduction steps (32 k forward, 64 n transposed), output tiles and the slices of the reduction over workgroups
struct HqqMfmaPlan { int waves, rb, tiles, steps, slices, steps_per_wave; double us; };
static HqqMfmaPlan hqq_mfma_plan(int64_t M, int64_t K, int64_t N, bool transposed, int64_t group) {
    HqqMfmaPlan p{};
    p.steps = (int)(transposed ? (N + 63) / 64 : (K + 31) / 32);
    // Cheapest by a measured model (in us, 1 to 64 rows, 4096 and 11008 wide): a CU takes 0.12 us for a kilobyte of codes with
    // all its waves together, eight at least, plus the start of each run, and its workgroups come in whole rounds; a slice costs its fp32 partial
    // sums, written and read.  (With 0.15 us and half the start, from when every step waited for the next one's requests, 32 rows
    // transposed of 11008 x 4096 took 22.6 us, with these 19.8, and one row 16.0, 13.8; by the present loop 17.6 and 12.6.)
    // Two blocks of 16 byte rows (64 values of k) per wave in the transposed product where they share their group.
    // Transposed products whose groups leave one block row to a wave keep those costs: short chunks of scales, or (groups that are no multiple of 32)
    // scales that each lane requests itself, with no step ahead: 13824 x 5120 at one row in groups of 8 21.3 us at the lower costs, 19.3 at
    // these, 64 rows of fp16 4608 x 11008 39.4, 36.6.  (A step ahead for groups of 8 gives one row 1 us and takes 0.7 to 1.7 us from 16 to 32 rows: eight waves
    // a CU hide the requests, and the second set of scales costs registers.)
    const bool single = transposed && group % 64 != 0;
    const int most_slices = M <= 16 ? 16 : 8;
    double best = 1e30;
    for (int rb = 1; rb <= (transposed && group % 64 == 0 ? 2 : 1); ++rb) {
        const int tiles = (int)(transposed ? (K / 2 + 16 * rb - 1) / (16 * rb) : (N + 63) / 64);
        for (int waves = 8; waves >= 4 * rb; waves -= 4)   // (four waves of block pairs do not fit the registers twice)
            for (int slices = 1; slices <= most_slices; ++slices) {
                if (slices > 1 && p.steps < 2 * waves * slices) break;   // runs of at least two steps
                const int per = (p.steps + slices * waves - 1) / (slices * waves), z = (p.steps + per * waves - 1) / (per * waves);
                if (z != slices) continue;
                // (a block pair reads scales, zeros and activations once for both)
                const int64_t on_cu = ((int64_t)tiles * z + 255) / 256 * waves;
                const double us = (single ? 0.15 : 0.12) * (rb == 2 ? 1.4 : 1.0) * (double)(on_cu > 8 ? on_cu : 8) * (per + (single ? 0.7 : 1.5)) +
                                  2e-6 * (double)(M * (transposed ? K : N)) * z;
                if (us < best) {
                    best = us;
                    p = HqqMfmaPlan{waves, rb, tiles, p.steps, z, per, us};
                }
            }
    }
    return p;
}

double hqq_stream_us(int64_t M, int64_t K, int64_t N, int64_t group, bool transposed) { return hqq_mfma_plan(M, K, N, transposed, group).us; }

}  // namespace ao

using namespace ao;

extern "C" int ao_amd_hqq_mixed_mm_workspace(int64_t M, int64_t K, int64_t N, int64_t* bytes) {
    AO_REQUIRE(bytes, "null pointer argument");
    AO_REQUIRE(M >= 1 && M <= 16 && K > 0 && N > 0 && K % 2 == 0, "need 1 <= M <= 16, K even, got M=%lld K=%lld N=%lld",
               (long long)M, (long long)K, (long long)N);
    *bytes = (int64_t)hqq_mm_slices(K, N) * M * N * (int64_t)sizeof(float);
    return 0;
}

extern "C" int ao_amd_hqq_mixed_mm(const void* a, int64_t M, int64_t K, int64_t lda, const void* packed_2xint4, int is_signed,
                                   int64_t N, const void* scales, const void* zeros, int64_t group_size, int dtype,
                                   void* workspace, int64_t workspace_bytes, void* y, void* stream) {
    AO_REQUIRE(a && packed_2xint4 && scales && zeros && workspace && y, "null pointer argument");
    AO_REQUIRE(dtype == AO_BF16 || dtype == AO_F16, "activations, scales, zeros and output must be bf16 or f16, got code %d", dtype);
    AO_REQUIRE(M >= 1 && M <= 16, "the fused product takes 1 to 16 activation rows, got M=%lld (dequantize and use a GEMM beyond)", (long long)M);
    AO_REQUIRE(K > 0 && N > 0 && K % 2 == 0 && N % 4 == 0, "need K even and N a multiple of 4, got K=%lld N=%lld", (long long)K, (long long)N);
    AO_REQUIRE(group_size > 0 && group_size % 2 == 0 && K % group_size == 0, "group_size %lld must be even and divide K=%lld",
               (long long)group_size, (long long)K);
    AO_REQUIRE(lda >= K && lda % 2 == 0 && (((uintptr_t)a) & 3) == 0, "activation rows must be 4-byte aligned with stride >= K");
    AO_REQUIRE(((((uintptr_t)packed_2xint4) & 3) | (((uintptr_t)scales) & 7) | (((uintptr_t)zeros) & 7)) == 0 && (N % 4) == 0,
               "packed codes must be 4-byte, scales and zeros 8-byte aligned");
    int64_t need = 0;
    if (int rc = ao_amd_hqq_mixed_mm_workspace(M, K, N, &need)) return rc;
    AO_REQUIRE(workspace_bytes >= need && (((uintptr_t)workspace) & 3) == 0, "workspace of %lld bytes needed, got %lld",
               (long long)need, (long long)workspace_bytes);
    const int slices = hqq_mm_slices(K, N);
    const int64_t K2 = K / 2;
    const int rows_per_wave = (int)((K2 + (int64_t)slices * 4 - 1) / ((int64_t)slices * 4));
    const dim3 grid((unsigned)((N + 255) / 256), (unsigned)slices);
    hipStream_t st = (hipStream_t)stream;
    const uint8_t* p = (const uint8_t*)packed_2xint4;
    const uint16_t *s = (const uint16_t*)scales, *z = (const uint16_t*)zeros, *av = (const uint16_t*)a;
    float* part = (float*)workspace;
#define AO_HQQ_MM(BF, SG, MBV) \
    hipLaunchKernelGGL((hqq_mm_small_kernel<BF, SG, MBV>), grid, dim3(256), 0, st, p, s, z, av, lda, (int)M, K, N, group_size, rows_per_wave, part)
#define AO_HQQ_MM_M(BF, SG)                  \
    do {                                     \
        if (M <= 4) AO_HQQ_MM(BF, SG, 4);    \
        else if (M <= 8) AO_HQQ_MM(BF, SG, 8); \
        else AO_HQQ_MM(BF, SG, 16);          \
    } while (0)
    if (dtype == AO_BF16) {
        if (is_signed) AO_HQQ_MM_M(true, true); else AO_HQQ_MM_M(true, false);
    } else {
        if (is_signed) AO_HQQ_MM_M(false, true); else AO_HQQ_MM_M(false, false);
    }
#undef AO_HQQ_MM_M
#undef AO_HQQ_MM
    AO_LAUNCH_CHECK();
    launch_hqq_finish(part, slices, M * N, dtype == AO_BF16, (uint16_t*)y, st);
    AO_LAUNCH_CHECK();
    return 0;
}


extern "C" int ao_amd_hqq_dequantize(const void* packed_2xint4, int is_signed, int64_t K, int64_t N, const void* scales,
                                     const void* zeros, int64_t group_size, int dtype, void* out, void* stream) {
    AO_REQUIRE(packed_2xint4 && scales && zeros && out, "null pointer argument");
    AO_REQUIRE(dtype == AO_BF16 || dtype == AO_F16, "scales, zeros and output must be bf16 or f16, got code %d", dtype);
    AO_REQUIRE(K > 0 && N > 0 && K % 2 == 0 && N % 16 == 0, "need K even and N a multiple of 16, got K=%lld N=%lld",
               (long long)K, (long long)N);
    AO_REQUIRE(group_size > 0 && group_size % 2 == 0 && K % group_size == 0,
               "group_size %lld must be even and divide K=%lld", (long long)group_size, (long long)K);
    AO_REQUIRE(((((uintptr_t)packed_2xint4) | ((uintptr_t)scales) | ((uintptr_t)zeros) | ((uintptr_t)out)) & 15) == 0,
               "buffers must be 16-byte aligned");
    const int64_t n = (K / 2) * (N / 16);
    AO_REQUIRE((n + 255) / 256 <= 0x7fffffff, "weight too large for one launch");
    dim3 grid((unsigned)((n + 255) / 256));
    hipStream_t st = (hipStream_t)stream;
    const uint8_t* p = (const uint8_t*)packed_2xint4;
    const uint16_t *s = (const uint16_t*)scales, *z = (const uint16_t*)zeros;
    uint16_t* o = (uint16_t*)out;
    if (dtype == AO_BF16) {
        if (is_signed) hipLaunchKernelGGL((hqq_dequantize_kernel<true, true>), grid, dim3(256), 0, st, p, s, z, K, N, group_size, o);
        else hipLaunchKernelGGL((hqq_dequantize_kernel<true, false>), grid, dim3(256), 0, st, p, s, z, K, N, group_size, o);
    } else {
        if (is_signed) hipLaunchKernelGGL((hqq_dequantize_kernel<false, true>), grid, dim3(256), 0, st, p, s, z, K, N, group_size, o);
        else hipLaunchKernelGGL((hqq_dequantize_kernel<false, false>), grid, dim3(256), 0, st, p, s, z, K, N, group_size, o);
    }
    AO_LAUNCH_CHECK();
    return 0;
}

extern "C" int ao_amd_hqq_mixed_mm_mfma_workspace(int64_t M, int64_t K, int64_t N, int transposed, int64_t* bytes) {
    AO_REQUIRE(bytes, "null pointer argument");
    AO_REQUIRE(M >= 1 && M <= 64 && K > 0 && N > 0 && K % 2 == 0, "need 1 <= M <= 64, K even, got M=%lld K=%lld N=%lld",
               (long long)M, (long long)K, (long long)N);
    // whatever the group size and the type: the plans depend on whether it is a multiple of 64, and on the type
    const int a = hqq_mfma_plan(M, K, N, transposed != 0, 64).slices, b = hqq_mfma_plan(M, K, N, transposed != 0, 2).slices;
    int most = a > b ? a : b;
    for (int bf16 = 0; bf16 < 2; ++bf16) {
        const HqqTilePlan t = hqq_tile_route(M, K, N, 64, transposed != 0, bf16 != 0);
        if (t.rows && t.parts > most) most = t.parts;
    }
    *bytes = (int64_t)most * M * (transposed ? K : N) * (int64_t)sizeof(float);
    return 0;
}

extern "C" int ao_amd_hqq_mixed_mm_mfma(const void* a, int64_t M, int64_t lda, const void* packed_2xint4, int is_signed, int64_t K,
                                        int64_t N, const void* scales, const void* zeros, int64_t group_size, int dtype,
                                        int transposed, void* workspace, int64_t workspace_bytes, void* y, void* stream) {
    AO_REQUIRE(a && packed_2xint4 && scales && zeros && workspace && y, "null pointer argument");
    AO_REQUIRE(dtype == AO_BF16 || dtype == AO_F16, "activations, scales, zeros and output must be bf16 or f16, got code %d", dtype);
    AO_REQUIRE(M >= 1 && M <= 64, "the fused product takes 1 to 64 activation rows, got M=%lld (dequantize and use a GEMM beyond)", (long long)M);
    AO_REQUIRE(K > 0 && N > 0 && K < (1ll << 31) && N < (1ll << 31), "K and N must be positive and below 2^31, got K=%lld N=%lld",
               (long long)K, (long long)N);
    AO_REQUIRE(group_size > 0 && K % group_size == 0, "group_size %lld must divide K=%lld", (long long)group_size, (long long)K);
    if (transposed) {
        AO_REQUIRE(K % 2 == 0 && N % 16 == 0 && group_size % 2 == 0,
                   "the transposed product needs K even, N a multiple of 16 and an even group size, got K=%lld N=%lld group=%lld",
                   (long long)K, (long long)N, (long long)group_size);
        AO_REQUIRE(lda >= N, "activation row stride %lld below N=%lld", (long long)lda, (long long)N);
    } else {
        AO_REQUIRE(K % 8 == 0 && N % 4 == 0 && group_size % 8 == 0,
                   "the forward product needs K and the group size multiples of 8 and N a multiple of 4, got K=%lld N=%lld group=%lld",
                   (long long)K, (long long)N, (long long)group_size);
        AO_REQUIRE(lda >= K, "activation row stride %lld below K=%lld", (long long)lda, (long long)K);
    }
    AO_REQUIRE(lda % 8 == 0 && (((uintptr_t)a) & 15) == 0, "activation rows must be 16-byte aligned (stride a multiple of 8 elements)");
    AO_REQUIRE(((((uintptr_t)packed_2xint4) | ((uintptr_t)scales) | ((uintptr_t)zeros)) & 15) == 0,
               "packed codes, scales and zeros must be 16-byte aligned");
    int64_t need = 0;
    if (int rc = ao_amd_hqq_mixed_mm_mfma_workspace(M, K, N, transposed, &need)) return rc;
    AO_REQUIRE(workspace_bytes >= need && (((uintptr_t)workspace) & 15) == 0, "16-byte aligned workspace of %lld bytes needed, got %lld",
               (long long)need, (long long)workspace_bytes);
    const HqqTilePlan t = hqq_tile_route(M, K, N, group_size, transposed != 0, dtype == AO_BF16);
    if (t.rows && (((uintptr_t)y) & 15) == 0 && lda < (1 << 24)) {
        launch_hqq_tile(t, (const uint8_t*)packed_2xint4, (const uint16_t*)scales, (const uint16_t*)zeros, (const uint16_t*)a, lda, M, K, N, group_size,
                        is_signed != 0, dtype == AO_BF16, transposed != 0, (float*)workspace, (uint16_t*)y, (hipStream_t)stream);
        AO_LAUNCH_CHECK();
        return 0;
    }
    const HqqMfmaPlan p = hqq_mfma_plan(M, K, N, transposed != 0, group_size);
    const dim3 grid((unsigned)p.tiles, (unsigned)p.slices);
    hipStream_t st = (hipStream_t)stream;
    const uint8_t* pk = (const uint8_t*)packed_2xint4;
    const uint16_t *s = (const uint16_t*)scales, *z = (const uint16_t*)zeros, *av = (const uint16_t*)a;
    float* part = (float*)workspace;
#define AO_HQQ_MFMA(BF, SG, TR, MBV, RBV)                                                                                       \
    if (p.waves == 8 || RBV == 2) hipLaunchKernelGGL((hqq_mm_mfma_kernel<BF, SG, TR, MBV, RBV, 8>), grid, dim3(512), 0, st, pk, s, z, av, lda, (int)M, K, N, \
                       group_size, p.steps, p.steps_per_wave, part); \
    else hipLaunchKernelGGL((hqq_mm_mfma_kernel<BF, SG, TR, MBV, 1, 4>), grid, dim3(256), 0, st, pk, s, z, av, lda, (int)M, K, N, \
                       group_size, p.steps, p.steps_per_wave, part)
#define AO_HQQ_MFMA_M(BF, SG, TR, RBV)                     \
    do {                                                   \
        if (M <= 16) { AO_HQQ_MFMA(BF, SG, TR, 1, RBV); }      \
        else if (M <= 32) { AO_HQQ_MFMA(BF, SG, TR, 2, RBV); } \
        else { AO_HQQ_MFMA(BF, SG, TR, 4, RBV); }              \
    } while (0)
#define AO_HQQ_MFMA_T(BF, SG)                                            \
    do {                                                                 \
        if (transposed && p.rb == 2) AO_HQQ_MFMA_M(BF, SG, true, 2);     \
        else if (transposed) AO_HQQ_MFMA_M(BF, SG, true, 1);             \
        else AO_HQQ_MFMA_M(BF, SG, false, 1);                            \
    } while (0)
    if (dtype == AO_BF16) {
        if (is_signed) AO_HQQ_MFMA_T(true, true); else AO_HQQ_MFMA_T(true, false);
    } else {
        if (is_signed) AO_HQQ_MFMA_T(false, true); else AO_HQQ_MFMA_T(false, false);
    }
#undef AO_HQQ_MFMA_T
#undef AO_HQQ_MFMA_M
#undef AO_HQQ_MFMA
    AO_LAUNCH_CHECK();
    launch_hqq_finish(part, p.slices, M * (transposed ? K : N), dtype == AO_BF16, (uint16_t*)y, st);
    AO_LAUNCH_CHECK();
    return 0;
}
