// int8 weight-only linear for batches beyond the streaming kernels (int8wo_linear.hip): y = bf16(bf16(x @ W^T) * scale) (+ bias),
// torchao/dtypes/affine_quantized_tensor.py:641-665, on the tiled product of tile_gemm.h.  The plain [N, K] int8 rows are
// copied into LDS as they are and converted by the multiplying wave (an int8 is exact in bf16: two byte conversions and a
// pack per pair), where the earlier route wrote the whole weight as bf16, called the library GEMM and scaled the
// result in a third pass.  11008 x 4096 at 333 rows: 22 + 43 + 6 us -> 44.
#include "int8wo_gemm.h"
#include "int4wo_linear.h"

namespace ao {

typedef __bf16 i8_bf16x8 __attribute__((ext_vector_type(8)));

template <bool PAIR_>
struct Int8Tile {
    static constexpr bool PAIR = PAIR_;
    static constexpr int REQ = 2, BLOCK_BYTES = 2048;   // 32 rows x 64 bytes
    struct Row {};
    struct Raw { uint4 v[2]; };             // 32 consecutive k of one row
    typedef Raw Ready;
    struct Cols { float scale[4], bias[4]; bool has_bias; };

    // request r: 8 rows x 128 bytes, two steps; slot (row, p) holds 16-byte chunk p ^ (row / 2 % 8): conflict-free reads.  Where K is no
    // multiple of 128, 16 rows x 64 bytes with chunk p ^ (row / 4 % 4).
    static __device__ __forceinline__ uint32_t lane_offset(const TileGemmArgs& a, int64_t n0, int64_t n, int r, int lane) {
        const int row = PAIR ? r * 8 + (lane >> 3) : r * 16 + (lane >> 2);
        const int64_t rel = (n + row < a.N ? n + row : a.N - 1) - n0;   // rows past N repeat the last one
        return (uint32_t)(rel * a.ldw) + ((PAIR ? (lane & 7) ^ ((row >> 1) & 7) : (lane & 3) ^ ((row >> 2) & 3)) << 4);
    }
    static __device__ __forceinline__ void request(const TileGemmArgs& a, int64_t n0, int s, int r, uint32_t lds, int at, uint32_t off) {
        lds_dma16(lds, at, a.w + n0 * a.ldw + (uint32_t)s * 64u, off);
    }
    static __device__ __forceinline__ Row row(const TileGemmArgs&, int64_t) { return Row(); }
    static __device__ __forceinline__ Raw read(const uint8_t* block, int lane, bool odd) {
        const int n = lane & 31, half = lane >> 5;
        Raw r;
#pragma unroll
        for (int c = 0; c < 2; ++c)
            r.v[c] = *(const uint4*)(block + (PAIR ? n * 128 + (((4 * odd + 2 * half + c) ^ ((n >> 1) & 7)) << 4)
                                                   : n * 64 + (((2 * half + c) ^ ((n >> 2) & 3)) << 4)));
        return r;
    }
    static __device__ __forceinline__ Ready prepare(const Raw& r, const Row&) { return r; }
    // dword d (k = 8 s + 2 d, + 1) of slice s; a pack right behind its byte conversions would wait for them
    struct Piece { float f0, f1; };
    static __device__ __forceinline__ uint32_t pack(const Piece& p) { return hw_bf16_pack(p.f0, p.f1); }
    static __device__ __forceinline__ Piece piece(const Ready& r, int s, int d) {
        const uint4 v = r.v[s >> 1];
        const uint32_t w = s & 1 ? (d < 2 ? v.z : v.w) : (d < 2 ? v.x : v.y);
        float f0, f1;
        if (d & 1)
            asm("v_cvt_f32_i32_sdwa %0, sext(%2) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_2\n\t"
                "v_cvt_f32_i32_sdwa %1, sext(%2) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_3" : "=&v"(f0), "=&v"(f1) : "v"(w));
        else
            asm("v_cvt_f32_i32_sdwa %0, sext(%2) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_0\n\t"
                "v_cvt_f32_i32_sdwa %1, sext(%2) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_1" : "=&v"(f0), "=&v"(f1) : "v"(w));
        return Piece{f0, f1};
    }
    static __device__ __forceinline__ tg_f32x16 mul(uint4 w, uint4 x, tg_f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(i8_bf16x8, w), __builtin_bit_cast(i8_bf16x8, x), c, 0, 0, 0);
    }
    static __device__ __forceinline__ Cols columns(const TileGemmArgs& a, int64_t n) {
        Cols c;
        c.has_bias = a.bias != nullptr;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int64_t i = n + v < a.N ? n + v : a.N - 1;
            c.scale[v] = bf16_bits_to_f32(((const uint16_t*)a.scale)[i]);
            c.bias[v] = a.bias ? bf16_bits_to_f32(a.bias[i]) : 0.f;
        }
        return c;
    }
    static __device__ __forceinline__ uint16_t finish(float acc, const Cols& c, int v) {
        const float y = rne_bf16(acc) * c.scale[v];
        return f32_to_bf16_bits(c.has_bias ? rne_bf16(y) + c.bias[v] : y);
    }
    // the residual and gated epilogues of the streaming kernels, on the rounded result
    static __device__ __forceinline__ void combine(const TileGemmArgs& a, int64_t m, int64_t n, uint16_t (&o)[4]) {
        if (!a.residual && !a.gate) return;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            if (n + v >= a.N) break;
            const float y = bf16_bits_to_f32(o[v]);
            o[v] = f32_to_bf16_bits(a.residual ? y + bf16_bits_to_f32(a.residual[m * a.ldres + n + v])
                                               : silu_bf16(bf16_bits_to_f32(a.gate[m * a.ldgate + n + v])) * y);
        }
    }
};

// us at K = 4096 with one and two workgroups on a CU (14336 columns, 224 workgroups, 448 for the second figure)
static const TileShape kInt8Shapes[] = {
    {64, 128, 26.4, 0.0},    // two groups of 4 waves along K
    {96, 128, 32.0, 52.7},
    {128, 128, 35.2, 0.0},   // two groups; 14336 of K 115 us, one group of four waves 122
    {192, 128, 44.4, 0.0},   // eight waves of 96 x 32
    {128, 256, 57.0, 0.0},   // eight waves; four of 128 x 64 each are 7 % slower
    {64, 64, 20.0, 0.0},     // four groups along K
    {192, 256, 77.8, 0.0},   // eight waves
};

TilePlan int8wo_gemm_plan(int64_t M, int64_t N, int64_t K, int max_parts) {
    TileShape shapes[7];
    for (int i = 0; i < 7; ++i) shapes[i] = kInt8Shapes[i];
    // (128 x 128 tiles take 8 % more for every K step of long rows: 5120 x 13824 at 640 rows 114 us, 128 x 256 in two K parts 106; 4096 x 14336 at 780 rows
    // 120 / 113, at 400 rows in two parts 71.5, 128 x 256 in four 70.4; 8192 x 8192 at 512 rows 71)
    if (K >= 8192) shapes[2].one = 37.5;
    // (the figures above are those of a weight from memory; 96 x 128 tiles of a smaller one with long rows take less: 1024 x 8192 at 1280 / 1400 rows in two K parts 36.3 /
    // 37.5 us, 192 x 128 in four 38.9 / 42.0; 2048 x 8192 at 700 rows 40.3 / 41.6, 2048 x 14336 at 290 rows 35.4 / 36.6)
    if (K >= 8192 && N * K < ((int64_t)1 << 25)) shapes[1].one = 30.0;
    return tile_plan(shapes, 7, M, N, K, max_parts);
}

void int8wo_gemm_describe(const TilePlan& p, char* out, size_t cap) {
    snprintf(out, cap, "tile %dx%d parts=%d", kInt8Shapes[p.shape].bm, kInt8Shapes[p.shape].bn, p.parts);
}

template <bool PAIR>
static bool launch_paired(const TileGemmArgs& a, const TilePlan& p, hipStream_t st) {
    typedef Int8Tile<PAIR> F;
    switch (p.shape) {
        case 0: tile_launch<F, 4, 2, 2, 1>(a, st); return true;
        case 4: tile_launch<F, 8, 1, 4, 1>(a, st); return true;
        default: return false;
    }
}

void launch_int8wo_gemm(TileGemmArgs a, const TilePlan& p, hipStream_t st) {
    tile_grid(a, kInt8Shapes[p.shape], 64, p.parts);
    if (!(a.K % 128 == 0 ? launch_paired<true>(a, p, st) : launch_paired<false>(a, p, st))) {
        switch (p.shape) {
            case 1: tile_launch<Int8Tile<false>, 4, 1, 3, 1>(a, st); break;
            case 2: tile_launch<Int8Tile<false>, 4, 2, 4, 1>(a, st); break;
            case 3: tile_launch<Int8Tile<false>, 4, 1, 3, 1, 2>(a, st); break;
            case 5: tile_launch<Int8Tile<false>, 2, 4, 2, 1>(a, st); break;
            default: tile_launch<Int8Tile<false>, 8, 1, 6, 1>(a, st); break;
        }
    }
    tile_finish<Int8Tile<false>>(a, p.parts, st);
}

void int8wo_finish_parts(const TileGemmArgs& a, int parts, hipStream_t st) { tile_finish<Int8Tile<false>>(a, parts, st); }

}  // namespace ao
