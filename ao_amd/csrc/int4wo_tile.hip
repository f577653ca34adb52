// int4 weight-only linear between the streaming kernels and the prefill kernels, on the tiled product of tile_gemm.h:
// y[M, N] = x[M, K] . dequant(W)[N, K]^T, torchao/dtypes/affine_quantized_tensor.py:600-640.  The packed codes of 32 weight
// rows and one 64-wide K step are one request of 1 KB (two runs of 512 bytes), their (scale, zero) words a second one.
//
// What bounds it: the exact two-rounding dequantization, 33 VALU instructions per 8 weights, against MT matrix instructions
// (MT = rows of the tile / 32).  Two waves per SIMD (two groups along K) overlap one wave's dequantization with the other's
// matrix instructions: 96 x 128 tiles of 14336 x 4096 at 160 rows take 36 us, where the 128 x 64 tiles of int4wo_gemm.hip, one
// wave per SIMD and a second round, take 45.
#include "int4wo_linear.h"
#include "tile_gemm.h"

namespace ao {

struct Int4Tile {
    static constexpr bool PAIR = false;
    typedef uint32_t Piece;
    static __device__ __forceinline__ uint32_t pack(Piece p) { return p; }
    static constexpr int REQ = 2, BLOCK_BYTES = 1024 + 256;
    struct Row { uint32_t even, odd, one; };   // masks of the even and odd pairs, the fp16 pair (1024, 1024)
    struct Raw { uint4 codes; uint32_t qp; };   // 32 consecutive k of one row, the scale and zero of their group
    struct Ready { uint32_t w[4]; float s, c, s16, c16, z; Row k; };   // c = -1032 s, s16 = s / 16, c16 = -72 s
    struct Cols { float bias[4]; };

    // in_features as packed, a multiple of max(128, group); the K steps end at in_features, a multiple of 64
    static __device__ __forceinline__ int64_t padded_k(const TileGemmArgs& a) { return a.ldw >> 3; }
    // this lane's row within the block, its k half within the step: (lane % 16 + 16 * block half, lane / 16 % 2)
    static __device__ __forceinline__ uint32_t lane_offset(const TileGemmArgs& a, int64_t n0, int64_t n, int r, int lane) {
        const int64_t nblocks = (a.N + 15) / 16;
        int64_t nb = n / 16 + (lane >> 5);
        if (nb >= nblocks) nb = nblocks - 1;   // a row block past N repeats the last one; its columns are not stored
        const int64_t rel = nb - n0 / 16;
        const int half = (lane >> 4) & 1, row = lane & 15;
        if (r == 0) return (uint32_t)(rel * a.ldw) + (half * 16 + row) * 16;
        // one word per row and group: a 64-wide step has two groups of 32 or lies within one
        return (uint32_t)(rel * (padded_k(a) >> a.group_shift) * 64) + (a.group_shift == 5 ? half * 64 : 0) + row * 4;
    }
    static __device__ __forceinline__ void request(const TileGemmArgs& a, int64_t n0, int s, int r, uint32_t lds, int at, uint32_t off) {
        if (r == 0)
            lds_dma16(lds, at, a.w + (n0 / 16) * a.ldw + (uint32_t)s * 512u, off);
        else
            lds_dma4(lds, at, (const uint8_t*)a.scale + (n0 / 16) * (padded_k(a) >> a.group_shift) * 64 + (((uint32_t)s * 64u) >> a.group_shift) * 64u, off);
    }
    static __device__ __forceinline__ Row row(const TileGemmArgs&, int64_t) {
        Row k;   // in registers, so that one instruction masks and inserts
        asm("s_mov_b32 %0, 0x000F000F" : "=s"(k.even));
        asm("s_mov_b32 %0, 0x00F000F0" : "=s"(k.odd));
        asm("v_mov_b32 %0, 0x64006400" : "=v"(k.one));
        return k;
    }
    static __device__ __forceinline__ Raw read(const uint8_t* block, int lane, bool) {
        const int slot = ((lane & 16) << 1) + (lane >> 5) * 16 + (lane & 15);   // row lane % 32, half lane / 32
        return Raw{*(const uint4*)(block + slot * 16), *(const uint32_t*)(block + 1024 + slot * 4)};
    }
    static __device__ __forceinline__ Ready prepare(const Raw& r, const Row& k) {
        const float s = __uint_as_float(r.qp << 16);
        return Ready{{r.codes.x, r.codes.y, r.codes.z, r.codes.w}, s, -1032.0f * s, 0.0625f * s, -72.0f * s, __uint_as_float(r.qp & 0xffff0000u), k};
    }
    // (vector conversions: element by element, the compiler adds a permutation to each packed one)
    static __device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
        typedef float f32x2 __attribute__((ext_vector_type(2)));
        typedef __bf16 b16x2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{lo, hi}), b16x2));
    }
    // a zero low operand: the rounded value lands in the high half, where it is an fp32 again
    static __device__ __forceinline__ float high_bf16(float f) { return __uint_as_float(pack_bf16(0.f, f)); }
    // Codes 2 d and 2 d + 1 of dword s as dequantize_affine rounds them: t = bf16((q - 8) * scale), w = bf16(t + zero).  The
    // pairs sit at bits (0, 16), (4, 20), (8, 24), (12, 28): masked and or'ed into the fp16 pair 1024 + q (1024 + 16 q for odd
    // pairs, whose factor goes into the scale), widened and scaled by one mixed fma each, exact in fp32.
    static __device__ __forceinline__ uint32_t piece(const Ready& r, int s, int d) {
        const uint32_t w = d < 2 ? r.w[s] : r.w[s] >> 8;
        typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
        const f16x2 p = __builtin_bit_cast(f16x2, (w & (d & 1 ? r.k.odd : r.k.even)) | r.k.one);
        const float sc = d & 1 ? r.s16 : r.s, c = d & 1 ? r.c16 : r.c;
        const float t0 = high_bf16(__builtin_fmaf((float)p.x, sc, c)), t1 = high_bf16(__builtin_fmaf((float)p.y, sc, c));
        return pack_bf16(t0 + r.z, t1 + r.z);
    }
    static __device__ __forceinline__ tg_f32x16 mul(uint4 w, uint4 x, tg_f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, w), __builtin_bit_cast(bf16x8_t, x), c, 0, 0, 0);
    }
    static __device__ __forceinline__ Cols columns(const TileGemmArgs& a, int64_t n) {
        Cols c;
#pragma unroll
        for (int v = 0; v < 4; ++v) c.bias[v] = a.bias ? bf16_bits_to_f32(a.bias[n + v < a.N ? n + v : a.N - 1]) : 0.f;
        return c;
    }
    static __device__ __forceinline__ uint16_t finish(float acc, const Cols& c, int v) { return f32_to_bf16_bits(acc + c.bias[v]); }
    static __device__ __forceinline__ void combine(const TileGemmArgs&, int64_t, int64_t, uint16_t (&)[4]) {}
};

// us at K = 4096, fitted to 128 calls (36 to 2000 rows of eight weights from 1024 x 4096 to 28672 x 8192), every shape and number of parts
// timed: the choice is within 0.7 % of the fastest on average (1.2 % with the costs from before the loops were shortened: 100 rows of
// 14336 x 4096 28.1 -> 25.9 us, 128 of 13824 x 5120 34.0 -> 30.8, 333 of 5120 x 5120 39.7 -> 31.3, 1400 of 6144 x 4096 99 -> 90).  Sums of parts
// cost more than a call alone shows: 1000 rows of 4096 x 14336 take 127 us on 256 x 256 tiles in four parts, 126 on 128 x 128 tiles and 141 on
// 256 x 128 in two, but within a prompt the four parts are 2 to 3 % of the pass slower than either.
static const TileShape kInt4Shapes[] = {
    {64, 64, 17.9, 0.0},     // four groups along K
    {64, 128, 31.2, 0.0},    // two groups
    {96, 128, 34.5, 0.0},    // two groups
    {128, 128, 36.9, 0.0},   // two groups
    {192, 128, 55.2, 0.0},
    {256, 128, 68.0, 0.0},
    // the kernels of int4wo_gemm.hip, which have no K parts of their own: in_features of the packed width only
    {256, 128, 59.0, 120.0, 4},
    {256, 256, 96.2, 0.0, 4},
};
static constexpr TilePartCost kInt4Parts{0.5, 0.5, 7.2};
static constexpr int kInt4Own = 6, kInt4All = 8;

static TilePlan int4wo_tile_plan(int64_t M, int64_t N, int64_t K, int max_parts) {
    return tile_plan(kInt4Shapes, K % 256 == 0 && M >= 128 ? kInt4All : kInt4Own, M, N, K, max_parts, kInt4Parts);
}

// us of the kernel that ao_amd_int4wo_linear(_ws) runs, by measurement at 33 to 1000 rows on 16 weights from 768 x 1024 to 28672 x
// 8192; 0 where it is not one of the tile kernels (few rows: the weight is streamed).  K as packed.
static double int4wo_other_us(int64_t M, int64_t N, int64_t K, int64_t g) {
    Int4Kernel kernel;
    if (!int4wo_plain_kernel(M, K, N, g, &kernel)) return 0.0;
    const int parts = ao_amd_int4wo_linear_ws_parts(M, K, N, g);
    const int64_t per = (K / 128 + parts - 1) / parts;
    // (33 to 64 rows, one tile row: the ws kernel's parts are powers of two and its 64 x 64 tiles without the tiled product's pipeline.  us there / tiled at 33, 64
    // rows: 5120 x 13824 31.7 / 23.5, 32.8 / 24.3; 8192 x 8192 24.1 / 22.3, 24.8 / 23.0; 4096 x 14336 23.2 / 22.2, 22.6 / 22.1; up to 16 tiles a part it is level or ahead:
    // 4096 x 4096 11.9 / 12.4, 13.0 / 13.2; 4096 x 6144 13.2 / 13.9, 14.5 / 14.5)
    if (parts > 1 && M <= 64) return per >= 20 ? 8.0 + 0.46 * (double)per : 0.0;
    if (kernel == Int4Kernel::streaming) {
        // Four blocks of streamed rows (weights of 768 row blocks and up) are behind the tiles, except where the weight has very many rows and the batch
        // few.  us at 33 / 48 rows, streamed / tiled: 12288 x 1024 8.6 / 8.4, 9.1 / 8.3; 14336 x 4096 18.9 / 17.2, 19.3 / 17.3; 13824 x 5120 22.1 / 19.9, 23.8 / 20.2; 16384
        // x 8192 31.8 / 29.8, 32.9 / 30.8; 28672 x 8192 53.4 / 50.6, 57.0 / 51.4; 65536 x 1024 23.6 / 21.3, 25.5 / 22.0; 65600 x 4096 (whose last tiles begin a third
        // round) 69.8 / 80.7, 77.4 / 83.8, 88.9 / 84.0 at 56; 128256 x 4096 111 / 121, 124 / 126, 142 / 128 at 56; but 128256 x 1024 42.3 / 40.3, 46.0 / 41.4.  Rows that
        // end early, 18837 x 1088 14.9 / 12.0, 16.1 / 12.8.  Up to 32 rows (two blocks) the streaming kernel is ahead: 14336 x 1024 at 32 rows 7.7 / 8.3,
        // 65536 x 4096 49.0 / 58.1.
        const int64_t blocks = (N + 15) / 16;
        // Narrower ones are streamed 16 rows and one block a workgroup, or four blocks where K is long; an estimate of each.  us streamed / tiled at 33, 40 rows: 2048
        // x 16384 25.1 / 16.1, 32.0 / 16.2; 3072 x 8192 22.0 / 14.7, 23.8 / 14.8; 1024 x 14336 17.8 / 14.3; 3584 x 18944 44.4 / 23.4; 256 x 28672 30.7 / 19.1 (40); ahead where K
        // is short: 2048 x 4096 8.6 / 11.7 (33), 1024 x 8192 11.6 / 12.4 (33).
        const double tiles = (double)(K / 128), full = (double)(blocks * ((M + 15) / 16)) / 256.0;
        if (blocks < 768) return fmin(2.6 + 0.12 * tiles * fmax(1.0, full), 6.2 + 0.05 * (double)M + 0.35 * tiles);
        return blocks <= 4096 || M > 48 ? 1e9 : 0.0;
    }
    const double k = (double)K / 4096.0;
    auto rounds = [&](int bm, int bn) { return (double)((M + bm - 1) / bm * ((N + bn - 1) / bn)) / 256.0; };
    auto up = [](double r) { return (double)(int64_t)(r + 255.0 / 256.0); };
    if (kernel == Int4Kernel::lds_256x256 || kernel == Int4Kernel::lds_256x128) {
        const double rw = rounds(256, 256);
        if (kernel == Int4Kernel::lds_256x256) return 6.0 + 100.0 * k * (rw < 1.0 ? 0.4 + 0.6 * rw : up(rw));   // CUs that run at once slow each other down
        // (1400 / 2000 rows of 4096 x 14336 230 / 247 us, tiled 186 / 217)
        const double r = rounds(256, 128), full = (double)(int64_t)r, rest = r - full, round = K > 8192 ? 62.0 : 52.5;
        return 14.0 + k * (round * full + (rest == 0.0 ? 0.0 : full > 0.0 && rest <= 0.5 ? 28.0 : round));
    }
    if (kernel == Int4Kernel::kwave) {
        const double r = up(rounds(128, 64));
        const bool three = (M + 95) / 96 == (M + 127) / 128;   // its 96-row tiles
        // (one round over 14336 of K: 427 / 512 rows of 4096 x 14336 80 / 78 us, tiled 70 / 73)
        return 6.0 + (three ? (r > 1.0 ? 17.5 : 16.5) : r > 1.0 || K >= 8192 ? 20.5 : 18.5) * k * r;
    }
    // (short K: the sums of eight parts cost the tiles more than they save.  us in K parts there / tiled at 100 rows: 512 x 4096 10.7 / 11.4, 1024 x 4096
    // 11.1 / 12.6, 1536 x 4096 11.5 / 12.0, 1024 x 2048 10.3 / 10.4, 1024 x 6144 12.5 / 12.9; 512 x 8192 14.1 / 13.3, 1024 x 14336 20.0 / 16.5)
    if (parts > 1) return K < 7168 ? 0.0 : 4.0 + 8.0 * k;
    if (kernel == Int4Kernel::tiles_128x128) return 90.0 * k * rounds(128, 128) / 2.0;
    if (rounds(64, 64) >= 0.75) return 5.0 + (K >= 8192 ? 14.0 : 18.0) * k * up(rounds(64, 64));
    return 4.0 + 10.4 * k * up(rounds(32, 64));
}

// Whether the tiled product is the faster one.  us, the others / tiled: 14336 x 4096 at 64 / 128 / 160 / 256 / 384 / 512 rows 23.8 / 21.3,
// 24.4 / 31.3, 44.8 / 37.4, 46.9 / 42.5, 62.9 / 57.3, 63.8 / 67.2; 4096 x 14336 at 96 / 160 / 640 / 1000 rows 32.7 / 26.8, 53.9 / 39.5, 124 /
// 108, 137 / 123; 8192 x 28672 at 448 rows 275 / 207; 4096 x 4096 at 128 / 256 / 512 / 768 rows 14.7 / 15.9, 23.5 / 19.6, 24.6 / 31.6, 44.1 / 37.6; 11008 x 4096 at 48 / 96 / 384
// rows 26.2 / 18.5, 35.1 / 25.2, 66.1 / 56.5; 8192 x 28672 at 96 rows 114 / 74.  The estimates hold to some 10 %: a lead of 5 % is asked for.
static bool int4wo_tiled(int64_t M, int64_t N, int64_t K, int64_t g) {
    if (!valid_group(g) || K % 64 != 0 || M <= 32 || M * N >= ((int64_t)1 << 40)) return false;
    // in_features that were padded to whole tiles of the packed layout: the others take activations copied to that width first
    const int64_t Kp = round_up(K, g > 128 ? g : 128);
    const double other = int4wo_other_us(M, N, Kp, g);
    if (other <= 0.0) return false;
    const TilePlan plan = int4wo_tile_plan(M, N, K, 8);
    Int4Kernel kernel;
    // (the plan may be the very launch that the dispatch makes)
    if (plan.shape >= kInt4Own && plan.parts == 1 && int4wo_plain_kernel(M, Kp, N, g, &kernel) &&
        kernel == (plan.shape == kInt4Own ? Int4Kernel::lds_256x128 : Int4Kernel::lds_256x256))
        return false;
    // (sums whose rows are not 16-byte aligned are stored one by one, which the estimates of K parts do not have.  Up to 64 rows, us in the other kernels / tiled:
    // 4481 x 3584 at 56 rows 12.7 / 14.1, 667 x 4416 at 39 rows 10.4 / 11.3, 4277 x 3584 at 59 rows 13.2 / 14.2)
    const double single = M <= 64 && plan.parts > 1 && N % 4 != 0 ? 0.8 : 0.0;
    // (rows that end early are copied for the others: 4 us, up to 64 rows 2.5.  3400 x 1472 at 38 rows 9.2 copied and streamed / 10.1 tiled, 912 x 4672 at 57 rows 11.4 / 12.2)
    return plan.us + single < (Kp == K ? 0.95 * other : other + (M <= 64 ? 2.5 : 4.0));
}

// x [M, K] with row stride ldx -> y [M, Kp], zeros beyond K, 8 elements a thread: activations whose rows are not 16-byte aligned
// or end before the packed width.  The kernel that reads such rows as they are does it element by element, for every 16 weight
// rows again; a copy is 2 to 3 us and the launch's gap.
__global__ __launch_bounds__(256) void pad_rows_kernel(const uint16_t* __restrict__ x, int64_t M, int64_t K, int64_t ldx, int64_t Kp,
                                                       bool vec, uint16_t* __restrict__ y) {
    const int64_t per_row = Kp / 8, i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t m = i / per_row, k = (i - m * per_row) * 8;
    if (m >= M) return;
    const uint16_t* src = x + m * ldx + k;
    uint4 out;
    if (vec && k + 8 <= K) {
        out = *(const uint4*)src;
    } else {
        uint32_t v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = k + e < K ? src[e] : 0u;
        out = make_uint4(v[0] | (v[1] << 16), v[2] | (v[3] << 16), v[4] | (v[5] << 16), v[6] | (v[7] << 16));
    }
    *(uint4*)(y + m * Kp + k) = out;
}

// Which route a plain linear takes and what its workspace holds: the copied rows first, then the K parts.
struct Int4Auto {
    bool tiled;
    bool as_is;           // the plain kernel reads the rows itself: nothing is copied (the workspace keeps the size that callers know)
    int64_t Kp;           // the width of the copied rows, 0: read as they are
    int stream_parts;     // K parts of the streaming kernel with four row blocks, 1: not split
    int64_t copy, parts;  // bytes
};
// room: the workspace that the call has.  Up to 64 rows a call without room for the K parts takes the way of one that needs less or none.
static int int4wo_auto(const void* x, int64_t M, int64_t K, int64_t ldx, int64_t N, int64_t g, int y_dtype, int64_t room, Int4Auto* r) {
    *r = Int4Auto{false, false, 0, 1, 0, 0};
    const bool aligned = (ldx & 7) == 0 && (((uintptr_t)x) & 15) == 0;
    if (M > 32 && y_dtype == AO_BF16 && aligned && 256 * ldx * 2 < ((int64_t)1 << 32)) {
        int64_t need = -1;
        if (int rc = ao_amd_int4wo_linear_tiled_bytes(M, K, N, g, &need)) return rc;
        if (need >= 0 && (M > 64 || need <= room)) {
            r->tiled = true;
            r->parts = need;
            return 0;
        }
    }
    // Rows that the kernel cannot read (int4wo_takes_short_rows) are copied to the packed width where the copy (2 to 3 us with its launch) costs less than the
    // element-wise kernel loses, whose time follows the length of the rows, or the whole product where the weight is large.  us a call
    // as they are / copied: 4096 x 4160 at 1 / 6 / 16 / 64 rows 15.5 / 18 / 35 / 121, 10.5 / 10.0 / 10.5 / 16.4; 14336 x 4032 at 1 / 16
    // rows 30 / 114, 13.5 / 15.5; 1024 x 2112 at 1 / 2 / 8 / 16 rows 13.9 / 8.9 / 12.9 / 19.8, about 9.5; 1024 x 704 up to 64 rows 7
    // to 9, about 9.
    AO_REQUIRE(valid_group(g), "group size must be 32, 64, 128 or 256, got %lld", (long long)g);
    const int64_t Kp = round_up(K, g > 128 ? g : 128), rows = M < 16 ? M : 16;
    if (M > 0 && (K != Kp || !aligned) && (N * K * (M + 4) >= 50000000 || K * (M == 1 ? 13 : rows + 4) >= 18000)) {
        r->Kp = Kp;
        r->copy = M * Kp * 2;
        r->as_is = aligned && K % 8 == 0 && int4wo_takes_short_rows(M, N, g);
    }
    r->stream_parts = (K == Kp && aligned) || r->Kp ? int4wo_stream_parts(M, r->as_is ? K : Kp, N, g) : 1;
    if (r->stream_parts > 1) {
        r->parts = r->stream_parts * M * N * (int64_t)sizeof(float);
        if (r->copy + r->parts <= room) return 0;
        r->stream_parts = 1;
    }
    return ao_amd_int4wo_linear_ws_bytes(M, r->Kp ? Kp : K, N, g, &r->parts);
}

}  // namespace ao

using namespace ao;

extern "C" int ao_amd_int4wo_linear_tiled_bytes(int64_t M, int64_t K, int64_t N, int64_t g, int64_t* bytes) {
    AO_REQUIRE(bytes, "null pointer argument");
    AO_REQUIRE(M >= 0 && K > 0 && N > 0, "need M >= 0 and positive K, N");
    *bytes = -1;
    if (!int4wo_tiled(M, N, K, g)) return 0;
    const TilePlan p = int4wo_tile_plan(M, N, K, 8);
    *bytes = p.parts > 1 ? p.parts * M * N * (int64_t)sizeof(float) : 0;
    return 0;
}

extern "C" int ao_amd_int4wo_linear_tiled_plan(int64_t M, int64_t K, int64_t N, char* out, int64_t out_cap) {
    AO_REQUIRE(out && out_cap > 0 && M > 0 && N > 0 && K > 0 && K % 64 == 0, "need positive M and N, K a multiple of 64, and a buffer");
    const TilePlan p = int4wo_tile_plan(M, N, K, 8);
    snprintf(out, (size_t)out_cap, "tile %dx%d parts=%d", kInt4Shapes[p.shape].bm, kInt4Shapes[p.shape].bn, p.parts);
    return 0;
}

extern "C" int ao_amd_int4wo_linear_tiled(const void* x_bf16, int64_t M, int64_t K, int64_t ldx, const void* packed, const void* qparams,
                                          int64_t N, int64_t g, const void* bias_bf16, void* y_bf16, int64_t ldy, void* workspace,
                                          int64_t workspace_bytes, void* stream) {
    AO_REQUIRE(x_bf16 && packed && qparams && y_bf16, "null pointer argument");
    AO_REQUIRE(valid_group(g), "group size must be 32, 64, 128 or 256, got %lld", (long long)g);
    AO_REQUIRE(M >= 0 && N > 0 && K > 0 && K % 64 == 0, "the tiled int4 product needs in_features to be a multiple of 64, got %lld", (long long)K);
    if (M == 0) return 0;
    AO_REQUIRE(ldx >= K && ldy >= N, "row strides (ldx=%lld, ldy=%lld) smaller than the rows", (long long)ldx, (long long)ldy);
    AO_REQUIRE((((uintptr_t)x_bf16) & 15) == 0 && (ldx & 7) == 0 && (((uintptr_t)packed) & 15) == 0 && (((uintptr_t)workspace) & 15) == 0,
               "activation rows, packed codes and workspace must be 16-byte aligned");
    // per-lane offsets within a tile are 32 bits wide
    AO_REQUIRE(256 * ldx * 2 < ((int64_t)1 << 32) && M * N < ((int64_t)1 << 40), "operands too large");
    TilePlan p = int4wo_tile_plan(M, N, K, 8);
    if (p.parts > 1 && (!workspace || workspace_bytes < p.parts * M * N * (int64_t)sizeof(float))) p = int4wo_tile_plan(M, N, K, 1);
    TileGemmArgs a{(const uint16_t*)x_bf16, M, K, ldx, (const uint8_t*)packed, round_up(K, g > 128 ? g : 128) * 8, qparams, (const uint16_t*)bias_bf16, N,
                   (uint16_t*)y_bf16, ldy, TileOrder(), nullptr, 0, nullptr, 0, g == 32 ? 5 : g == 64 ? 6 : g == 128 ? 7 : 8, (float*)workspace};
    hipStream_t st = (hipStream_t)stream;
    tile_grid(a, kInt4Shapes[p.shape], 32, p.parts);
    switch (p.shape) {
        case 0: tile_launch<Int4Tile, 2, 4, 2, 1>(a, st); break;
        case 1: tile_launch<Int4Tile, 4, 2, 2, 1>(a, st); break;
        case 2: tile_launch<Int4Tile, 4, 2, 3, 1>(a, st); break;
        case 3: tile_launch<Int4Tile, 4, 2, 4, 1>(a, st); break;
        case 4: tile_launch<Int4Tile, 4, 1, 6, 1>(a, st); break;
        case 5: tile_launch<Int4Tile, 4, 1, 8, 1>(a, st); break;
        default: {
            LinearArgs l{};
            l.x = a.x; l.M = M; l.K = l.Kp = K; l.ldx = ldx;
            l.packed = (const uint4*)packed; l.qparams = (const uint32_t*)qparams; l.N = N;
            l.ksplit = p.parts;
            if (p.parts == 1) {
                l.bias = a.bias; l.y = a.y; l.ldy = ldy;
            } else {
                l.y = a.parts; l.y_is_f32 = 1; l.ldy = N;
            }
            launch_int4wo_gemm_lds_parts(l, g, p.shape - kInt4Own + 1, st);
        }
    }
    tile_finish<Int4Tile>(a, p.parts, st);
    AO_LAUNCH_CHECK();
    return 0;
}

extern "C" int ao_amd_pad_rows(const void* x, int64_t M, int64_t K, int64_t ldx, int64_t Kp, void* y, void* stream) {
    AO_REQUIRE(x && y, "null pointer argument");
    AO_REQUIRE(M >= 0 && K > 0 && ldx >= K && Kp >= K && Kp % 8 == 0, "need M >= 0, ldx >= K > 0 and Kp >= K a multiple of 8");
    AO_REQUIRE((((uintptr_t)y) & 15) == 0, "output must be 16-byte aligned");
    const int64_t blocks = (M * (Kp / 8) + 255) / 256;
    AO_REQUIRE(blocks < ((int64_t)1 << 31), "operand too large");
    if (M == 0) return 0;
    const bool vec = (((uintptr_t)x) & 15) == 0 && (ldx & 7) == 0;
    hipLaunchKernelGGL(pad_rows_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, (const uint16_t*)x, M, K, ldx, Kp, vec, (uint16_t*)y);
    AO_LAUNCH_CHECK();
    return 0;
}

extern "C" int ao_amd_int4wo_linear_auto_bytes(const void* x_bf16, int64_t M, int64_t K, int64_t ldx, int64_t N, int64_t g, int y_dtype,
                                               int64_t* bytes) {
    AO_REQUIRE(bytes, "null pointer argument");
    AO_REQUIRE(M >= 0 && K > 0 && N > 0, "need M >= 0 and positive K, N");
    Int4Auto r;
    if (int rc = int4wo_auto(x_bf16, M, K, ldx, N, g, y_dtype, INT64_MAX, &r)) return rc;
    *bytes = r.copy + r.parts;
    return 0;
}

extern "C" int ao_amd_int4wo_linear_auto(const void* x_bf16, int64_t M, int64_t K, int64_t ldx, const void* packed, const void* qparams,
                                         int64_t N, int64_t g, const void* bias_bf16, void* y, int y_dtype, int64_t ldy, void* workspace,
                                         int64_t workspace_bytes, void* stream) {
    AO_REQUIRE(M >= 0 && K > 0 && N > 0, "need M >= 0 and positive K, N");
    AO_REQUIRE(ldx >= K && ldy >= N, "row strides (ldx=%lld, ldy=%lld) smaller than the rows (K=%lld, N=%lld)", (long long)ldx, (long long)ldy,
               (long long)K, (long long)N);
    Int4Auto r;
    const int64_t room = workspace && (((uintptr_t)workspace) & 15) == 0 ? workspace_bytes : 0;
    if (int rc = int4wo_auto(x_bf16, M, K, ldx, N, g, y_dtype, room, &r)) return rc;
    AO_REQUIRE(r.copy + r.parts <= (room > 0 ? room : 0),
               "16-byte aligned workspace of %lld bytes needed (ao_amd_int4wo_linear_auto_bytes), got %lld", (long long)(r.copy + r.parts),
               (long long)workspace_bytes);
    if (r.tiled)
        return ao_amd_int4wo_linear_tiled(x_bf16, M, K, ldx, packed, qparams, N, g, bias_bf16, y, ldy, workspace, r.parts, stream);
    if (r.as_is && r.stream_parts == 1) return ao_amd_int4wo_linear(x_bf16, M, K, ldx, packed, qparams, N, g, bias_bf16, y, y_dtype, ldy, stream);
    if (r.Kp && !r.as_is) {
        if (int rc = ao_amd_pad_rows(x_bf16, M, K, ldx, r.Kp, workspace, stream)) return rc;
        x_bf16 = workspace;
        K = ldx = r.Kp;
        if (!r.parts) return int4wo_linear_copied_rows(x_bf16, M, K, packed, qparams, N, g, bias_bf16, y, y_dtype, ldy, stream);
    }
    if (r.stream_parts > 1)
        return int4wo_linear_stream_parts(x_bf16, M, K, ldx, packed, qparams, N, g, bias_bf16, y, y_dtype, ldy, r.stream_parts,
                                          (uint8_t*)workspace + r.copy, stream);
    if (!r.parts) return ao_amd_int4wo_linear(x_bf16, M, K, ldx, packed, qparams, N, g, bias_bf16, y, y_dtype, ldy, stream);
    return ao_amd_int4wo_linear_ws(x_bf16, M, K, ldx, packed, qparams, N, g, bias_bf16, y, y_dtype, ldy, (uint8_t*)workspace + r.copy,
                                   r.parts, stream);
}
