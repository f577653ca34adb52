// FP6 weight-only linear on the tiled product of tile_gemm.h: native tiles (fp6.hip: 16 rows x 128 k in 1536 bytes) come into
// LDS as they are, one conversion instruction per lane and 64-wide K step makes 32 fp16 values, and a packed fp16 multiply per
// pair applies the row's scale with the one rounding of the reference kernel, fp16(fp6 * scale): 17 VALU instructions for 32
// weights, so the tiles are bounded by what tile_gemm.h names, the bytes in flight and the LDS reads of the activations.  The
// kernels of fp6.hip at these row counts move the activations through registers and convert the weight in every wave.
#include "tile_gemm.h"

namespace ao {

int fp6_ws_parts(int64_t M, int64_t K, int64_t N);   // fp6.hip: the power of two that the 32- and 64-row tiles are split in

typedef _Float16 ft_f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 ft_f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 ft_f16x32 __attribute__((ext_vector_type(32)));
typedef uint32_t ft_u32x6 __attribute__((ext_vector_type(6)));

template <bool E3M2>
struct Fp6Tile {
    static constexpr bool PAIR = false;
    typedef uint32_t Piece;
    static __device__ __forceinline__ uint32_t pack(Piece p) { return p; }
    static constexpr int REQ = 2, BLOCK_BYTES = 2048;   // 1 KB of first dwords, 512 bytes of last dwords and their repetition
    struct Row { ft_f16x2 scale; };
    struct Raw { uint4 lo; uint2 hi; };     // 32 codes of 6 bits
    struct Ready { ft_f16x32 v; ft_f16x2 scale; };
    struct Cols {};

    static __device__ __forceinline__ uint32_t lane_offset(const TileGemmArgs& a, int64_t n0, int64_t n, int r, int lane) {
        const int64_t nblocks = a.N / 16;
        // first dwords: 32 lanes of 16 bytes a row block; last dwords: 16 lanes (8 bytes a weight row and k half)
        int64_t nb = n / 16 + (r == 0 ? lane >> 5 : (lane >> 4) & 1);
        if (nb >= nblocks) nb = nblocks - 1;   // a row block past N repeats the last one; its columns are not stored
        return (uint32_t)((nb - n0 / 16) * a.ldw) + (r == 0 ? lane & 31 : lane & 15) * 16;
    }
    static __device__ __forceinline__ void request(const TileGemmArgs& a, int64_t n0, int s, int r, uint32_t lds, int at, uint32_t off) {
        const uint8_t* const tile = a.w + (n0 / 16) * a.ldw + (uint32_t)((s >> 1) * 1536 + (s & 1) * (r == 0 ? 512 : 256));
        lds_dma16(lds, at, tile, off + (r == 0 ? 0 : 1024));
    }
    static __device__ __forceinline__ Row row(const TileGemmArgs& a, int64_t n) {
        const _Float16 s = __builtin_bit_cast(_Float16, ((const uint16_t*)a.scale)[n < a.N ? n : a.N - 1]);
        return Row{{s, s}};
    }
    static __device__ __forceinline__ Raw read(const uint8_t* block, int lane, bool) {
        const int slot = ((lane & 16) << 1) + (lane >> 5) * 16 + (lane & 15);   // row lane % 32, half lane / 32
        return Raw{*(const uint4*)(block + slot * 16), *(const uint2*)(block + 1024 + slot * 8)};
    }
    static __device__ __forceinline__ Ready prepare(const Raw& r, const Row& row) {
        const ft_u32x6 p = {r.lo.x, r.lo.y, r.lo.z, r.lo.w, r.hi.x, r.hi.y};
        Ready out;
        out.v = E3M2 ? __builtin_amdgcn_cvt_scalef32_pk32_f16_bf6(p, 1.0f) : __builtin_amdgcn_cvt_scalef32_pk32_f16_fp6(p, 1.0f);
        out.scale = row.scale;
        return out;
    }
    static __device__ __forceinline__ uint32_t piece(const Ready& r, int s, int d) {
        const ft_f16x2 v = {r.v[8 * s + 2 * d], r.v[8 * s + 2 * d + 1]};
        return __builtin_bit_cast(uint32_t, v * r.scale);
    }
    static __device__ __forceinline__ tg_f32x16 mul(uint4 w, uint4 x, tg_f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(ft_f16x8, w), __builtin_bit_cast(ft_f16x8, x), c, 0, 0, 0);
    }
    static __device__ __forceinline__ Cols columns(const TileGemmArgs&, int64_t) { return Cols(); }
    static __device__ __forceinline__ uint16_t finish(float acc, const Cols&, int) { return f32_to_f16_bits(acc); }
    static __device__ __forceinline__ void combine(const TileGemmArgs&, int64_t, int64_t, uint16_t (&)[4]) {}
};

// us at K = 4096, 192 to 256 workgroups (14336, 6144 and 4096 columns)
static const TileShape kFp6Shapes[] = {
    {64, 64, 17.4, 0.0},     // four groups along K
    {64, 128, 24.6, 0.0},    // two groups
    {96, 128, 30.5, 0.0},    // two groups
    {128, 128, 35.9, 0.0},   // two groups
    {192, 128, 47.7, 0.0},   // eight waves of 96 x 32
    {128, 256, 62.0, 0.0},   // 128 x 64 a wave
    {192, 256, 87.0, 0.0},   // eight waves
};

template <bool E3M2>
static void launch_shape(TileGemmArgs a, const TilePlan& p, hipStream_t st) {
    typedef Fp6Tile<E3M2> F;
    tile_grid(a, kFp6Shapes[p.shape], 48, p.parts);
    switch (p.shape) {
        case 0: tile_launch<F, 2, 4, 2, 1>(a, st); break;
        case 1: tile_launch<F, 4, 2, 2, 1>(a, st); break;
        case 2: tile_launch<F, 4, 2, 3, 1>(a, st); break;
        case 3: tile_launch<F, 4, 2, 4, 1>(a, st); break;
        case 4: tile_launch<F, 4, 1, 3, 1, 2>(a, st); break;
        case 5: tile_launch<F, 4, 1, 4, 2>(a, st); break;
        default: tile_launch<F, 8, 1, 6, 1>(a, st); break;
    }
    tile_finish<F>(a, p.parts, st);
}

static TilePlan fp6_tile_plan(int64_t M, int64_t N, int64_t K, int max_parts) {
    // (a short lead of K parts over the whole K is none; us in the parts that the estimates prefer / whole: 8192 x 8192 at 65 / 96 rows, four of 96 x 128, 29.8 /
    // 25.1, 32.4 / 26.5, 8192 x 7168 at 80 rows 27.4 / 22.7; two of 96 x 128: 6144 x 4096 at 140 rows 20.2 / 16.2, 5120 x 5120 at 256 rows 25.2 / 20.8; but
    // 4096 x 14336 at 256 rows, four of 128 x 128, 43.0 / 44.2, 5120 x 13824 at 129 rows, two of 64 x 128, 36.9 / 39.2)
    TilePartCost parts;
    parts.lead = 0.89;
    // (in powers of two / three or six parts: 5120 x 13824 at 96 / 128 / 256 rows 33.8 / 30.9, 40.7 / 33.0, 49.1 / 46.4; 10240 x 8192 at 40 / 77 / 113 rows 26.0 / 27.6, 30.3 /
    // 33.1, 34.3 / 36.1; 9000 x 6144 and 5120 x 5120 level.  The line is drawn between these weights: a part has to be long enough to pay for its sums, and where
    // between 8192 and 13824 that begins was not measured)
    parts.uneven = K >= 10240;
    return tile_plan(kFp6Shapes, (int)(sizeof(kFp6Shapes) / sizeof(kFp6Shapes[0])), M, N, K, max_parts, parts);
}

// Whether the tiled product is the faster one.  The kernels of fp6.hip cost, by measurement at 33 to 1000 rows on 16 weights from
// 768 x 1024 to 28672 x 8192: 32 x 64 tiles 4 us and 8 us per round over the CUs and 4096 of K, 64 x 64 tiles 4 and 14, and
// 128 x 128 tiles 50 for one round and 37 for each of several.  us, those /
// tiled: 14336 x 4096 at 65 / 160 / 256 / 384 / 768 rows 30 / 24, 44 / 30, 56 / 40, 68 / 49, 114 / 88; 4096 x 14336 at 160 / 512 / 1000 rows
// 57 / 35, 97 / 74, 169 / 120; 4096 x 4096 at 128 / 384 / 1000 rows 12.3 / 15.0, 27 / 21, 50 / 39; 5120 x 5120 at 96 / 384 rows 14.4 /
// 18.0, 34 / 32; 1024 x 4096 at 512 / 640 rows 12.6 / 15.4, 17.8 / 16.8.  At 33 to 64 rows the others are 32 x 64 tiles, whose one round over
// the CUs ends at 8192 columns: beyond, the tiles are ahead by 0 to 32 % (those / tiled at 33 and 64 rows: 8448 x 4096 16.9 / 11.8, 17.7 /
// 12.1; 14336 x 4096 18.0 / 16.3, 19.0 / 17.6; 14336 x 2048 10.5 / 8.7, 11.0 / 9.4; 16384 x 2048 10.6 / 9.9, 11.4 / 11.2; 28672 x 8192 54 / 43, 60 /
// 46); below it only where that round is long and its workgroups leave room for two K parts (5120 x 5120 14.0 / 12.4, 14.1 / 13.7; 6400 x
// 7168 19.2 / 16.7, 19.6 / 18.9; but 8192 x 4096 12.2 / 13.1 at 33 and 12.5 / 13.6 at 56 rows, 7168 x 6144 16.8 / 15.7, 16.9 / 17.7, 8192 x 7168 20.0 / 20.4,
// 20.6 / 22.3).  Weights below 26 M were not measured there.
// Those lines for 33 to 64 rows were drawn against unsplit 32 x 64 tiles.  The parts that ao_amd_fp6_linear_ws has since (fp6.hip: fp6_rows_plan) are ahead of the tiles on
// most of these weights, but ao_amd_fp6_linear_auto asks here first and does not compare the two.  us tiled / in parts at 40 and 64 rows: 10240 x 8192 24.0 / 19.7, 26.6 / 24.0; 9216 x
// 8192 23.7 / 19.3, 26.4 / 23.7; 6400 x 7168 17.1 / 15.1, 18.7 / 19.5; 5376 x 7168 16.8 / 14.1, 18.3 / 16.2; 12032 x 8192 24.6 / 23.6, 27.2 / 29.8; level: 5120 x 5120 12.5 / 12.8, 13.0 /
// 14.1; 8448 x 4096 14.0 / 14.1, 15.5 / 16.7.
// Where the others split K over workgroups (fp6.hip: fp6_ws_parts) they are kept but for 65 to 96 rows of weights from 50 M on (4096 x
// 14336 at 64 / 66 / 96 rows 20.9 / 20.9, 31.0 / 22.2, 32.3 / 24.1; 4096 x 4096 at 66 rows 11.9 / 13.4).
static bool fp6_tiled(int64_t M, int64_t N, int64_t K) {
    if (K % 64 != 0 || N % 16 != 0 || M <= 32 || M * N >= ((int64_t)1 << 40) || 192 * K * 2 >= ((int64_t)1 << 32)) return false;
    if (fp6_ws_parts(M, K, N) != 1 && (M <= 64 || M > 96 || N * K < 50000000)) return false;
    const double tile_us = fp6_tile_plan(M, N, K, 8).us;
    // streamed once per 16 rows there (14336 x 4032 at 33 / 128 / 1000 rows 22 / 50 / 305 us, tiled 20 / 24 / 119; 4096 x 4160 at 65 / 128 /
    // 1000 rows 14 / 17 / 96, tiled 16 / 16 / 41)
    if (K % 128 != 0) return tile_us < 5.0 + 8.5e-8 * (double)(N * K) * (double)((M + 15) / 16);
    if (M <= 64) return N * K >= 26000000 && (N > 8192 || (N <= 6400 && K >= 5120));
    // (the 128 x 128 tiles of fp6.hip were never ahead there: 14336 x 4096 at 1200 / 1500 rows 169 / 178 tiled)
    if (M >= 1024 && N >= 2048) return true;
    const int64_t big = (N + 127) / 128 * ((M + 127) / 128), mid = (N + 63) / 64 * ((M + 63) / 64), small = (N + 63) / 64 * ((M + 31) / 32);
    const double k = (double)K / 4096.0;
    const double us = big >= 256 ? k * (big > 256 ? 37.0 * (double)((big + 255) / 256) : 50.0)
                      : mid >= 192 ? 4.0 + 14.0 * k * (double)((mid + 255) / 256)
                                   : 4.0 + 8.0 * k * (double)((small + 255) / 256);
    return tile_us < (big >= 256 ? 0.9 : 1.0) * us;
}

}  // namespace ao

using namespace ao;

extern "C" int ao_amd_fp6_linear_tiled_bytes(int64_t M, int64_t K, int64_t N, int64_t* bytes) {
    AO_REQUIRE(bytes, "null pointer argument");
    AO_REQUIRE(M >= 0 && K > 0 && N > 0, "need M >= 0 and positive K, N");
    *bytes = -1;
    if (!fp6_tiled(M, N, K)) return 0;
    const TilePlan p = fp6_tile_plan(M, N, K, 8);
    *bytes = p.parts > 1 ? p.parts * M * N * (int64_t)sizeof(float) : 0;
    return 0;
}

extern "C" int ao_amd_fp6_linear_tiled_plan(int64_t M, int64_t K, int64_t N, char* out, int64_t out_cap) {
    AO_REQUIRE(out && out_cap > 0 && M > 0 && N > 0 && K > 0 && K % 64 == 0, "need positive M and N, K a multiple of 64, and a buffer");
    const TilePlan p = fp6_tile_plan(M, N, K, 8);
    snprintf(out, (size_t)out_cap, "tile %dx%d parts=%d", kFp6Shapes[p.shape].bm, kFp6Shapes[p.shape].bn, p.parts);
    return 0;
}

extern "C" int ao_amd_fp6_linear_tiled(const void* x_f16, int64_t M, int64_t K, const void* weights_native, const void* scale_f16, int64_t N,
                                       int ebits, int mbits, void* out_f16, void* workspace, int64_t workspace_bytes, void* stream) {
    AO_REQUIRE(x_f16 && weights_native && scale_f16 && out_f16, "null pointer argument");
    AO_REQUIRE((ebits == 3 && (mbits == 1 || mbits == 2)) || (ebits == 2 && (mbits == 2 || mbits == 3)),
               "native tiles hold e3m2, e2m3, e2m2 and e3m1, got e%dm%d", ebits, mbits);   // 5-bit codes in their 6-bit form
    AO_REQUIRE(K > 0 && K % 64 == 0, "Expected in_features to be a multiple of 64, but received %lld", (long long)K);
    AO_REQUIRE(N > 0 && N % 16 == 0, "out_features must be a positive multiple of 16, got %lld", (long long)N);
    AO_REQUIRE(M >= 0, "negative batch");
    AO_REQUIRE((((uintptr_t)x_f16) & 15) == 0 && (((uintptr_t)weights_native) & 15) == 0 && (((uintptr_t)workspace) & 15) == 0,
               "buffers must be 16-byte aligned");
    // per-lane offsets within a tile are 32 bits wide
    AO_REQUIRE(192 * K * 2 < ((int64_t)1 << 32) && M * N < ((int64_t)1 << 40), "operands too large");
    if (M == 0) return 0;
    TilePlan p = fp6_tile_plan(M, N, K, 8);
    if (p.parts > 1 && (!workspace || workspace_bytes < p.parts * M * N * (int64_t)sizeof(float))) p = fp6_tile_plan(M, N, K, 1);
    const TileGemmArgs a{(const uint16_t*)x_f16, M, K, K, (const uint8_t*)weights_native, round_up(K, 128) / 128 * 1536, scale_f16, nullptr, N,
                         (uint16_t*)out_f16, N, TileOrder(), nullptr, 0, nullptr, 0, 0, (float*)workspace};
    if (ebits == 3) launch_shape<true>(a, p, (hipStream_t)stream);
    else launch_shape<false>(a, p, (hipStream_t)stream);
    AO_LAUNCH_CHECK();
    return 0;
}

extern "C" int ao_amd_fp6_linear_auto_bytes(int64_t M, int64_t K, int64_t N, int64_t* bytes) {
    if (int rc = ao_amd_fp6_linear_tiled_bytes(M, K, N, bytes)) return rc;
    return *bytes >= 0 ? 0 : ao_amd_fp6_linear_ws_bytes(M, K, N, bytes);
}

extern "C" int ao_amd_fp6_linear_auto(const void* x_f16, int64_t M, int64_t K, const void* weights_native, const void* scale_f16, int64_t N,
                                      int ebits, int mbits, void* out_f16, void* workspace, int64_t workspace_bytes, void* stream) {
    AO_REQUIRE(M >= 0 && K > 0 && N > 0, "need M >= 0 and positive K, N");
    if (fp6_tiled(M, N, K))
        return ao_amd_fp6_linear_tiled(x_f16, M, K, weights_native, scale_f16, N, ebits, mbits, out_f16, workspace, workspace_bytes, stream);
    return ao_amd_fp6_linear_ws(x_f16, M, K, weights_native, scale_f16, N, ebits, mbits, out_f16, workspace, workspace_bytes, stream);
}
