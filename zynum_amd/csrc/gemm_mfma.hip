// Plain FP64 / FP32 GEMM on gfx950 matrix cores (v_mfma_f64_16x16x4_f64,
// v_mfma_f32_16x16x4_f32).
//
// Replaces Zynum's packed-B CPU micro-kernel (packed_simd.zig:140-199), its
// B-panel / A-transpose packing (packing.zig:45-80,131-139) and the alpha/beta
// epilogue (epilogue.zig:10-39).  Design:
//   * one workgroup of 256 threads (4 wave64s in a 2x2 grid) owns a BM x BN
//     tile of C; every wave owns (BM/2) x (BN/2) accumulated in 16x16 MFMA
//     blocks held in registers for the whole K loop;
//   * op(A) and op(B) K-slices (BK deep) are staged in LDS as k-major
//     [BK][BM] / [BK][BN] panels, double buffered: global loads for slice t+1
//     are issued into registers before the MFMAs of slice t and written to the
//     other LDS buffer afterwards, one barrier per slice;
//   * column-major operands are read with 16-byte coalesced loads along the
//     contiguous dimension whatever the transpose (M/N-contiguous for A / B^T,
//     K-contiguous for A^T / B); transposition happens on the LDS write;
//   * edge tiles (M, N, K not multiples of the tile) use guarded scalar loads
//     with zero fill; interior tiles run unguarded;
//   * tile ids are remapped so each of the 8 XCDs gets a contiguous block of
//     tiles in grouped (super-row) order, keeping shared A/B panels in its L2;
//   * products of aligned operands skip the register staging: direct-to-LDS
//     loads fill a 4-stage ring (gemm_dma.hpp), on the tile that dma_plan or
//     f32_plan picks for the shape, the leftover output tiles split over K.
#include <algorithm>

#include "common.hpp"
#include "gemm.hpp"
#include "gemm_dma.hpp"
#include "gemm_f32_split.hpp"
#include "gemm_pieces.hpp"
#include "gemm_tile.hpp"

// Tile rows per super-row of the grouped tile order; a build knob for tuning.
#ifndef ZG_GROUP_M
#define ZG_GROUP_M 8
#endif

namespace zg {

template <typename T, class CF, bool TA, bool TB, int VEC>
__global__ __launch_bounds__(CF::NT) __attribute__((amdgpu_waves_per_eu(CF::OCC > 0 ? CF::OCC : 1)))
void gemm_mfma_kernel(GemmArgs<T> p) {
    __shared__ __attribute__((aligned(16))) T lds_a[tile_lds_a<T, CF>()];
    __shared__ __attribute__((aligned(16))) T lds_b[tile_lds_b<T, CF>()];
    const int total = p.tiles_m * p.tiles_n;
    int tm, tn;
    grouped_tile(xcd_remap(blockIdx.x, total), p.tiles_m, p.tiles_n, p.group_m, tm, tn);
    gemm_tile<T, CF, TA, TB, VEC>(p, tm * CF::BM, tn * CF::BN, lds_a, lds_b);
}

// Direct-load form (gemm_dma.hpp).
template <bool TA, bool TB, class CF>
__global__ __launch_bounds__(CF::NT) __attribute__((amdgpu_waves_per_eu(CF::OCC))) void gemm_dma_kernel(
    PieceArgs<typename CF::T> p) {
    using T = typename CF::T;
    __shared__ __attribute__((aligned(32))) T lds[CF::LDS];
    int tm, tn;
    grouped_tile(piece_tile(p, blockIdx.x), p.g.tiles_m, p.g.tiles_n, p.g.group_m, tm, tn);
    const int m0 = tm * CF::BM, n0 = tn * CF::BN;
    gemm_tile_dma<TA, TB, CF>(piece_of<T, TA, TB, CF::BM, CF::BN>(p, blockIdx.x, m0, n0), m0, n0, lds);
}

// Split-K form for shapes with few output tiles and a long K: blockIdx.y
// selects a K range [k0, k0 + kchunk) of the product, written unscaled
// (alpha 1, beta 0: the accumulator itself) to its own slice of the partial
// buffer; splitk_reduce_kernel sums the slices in increasing order and applies
// the alpha/beta epilogue.
template <typename T, class CF, bool TA, bool TB, int VEC>
__global__ __launch_bounds__(CF::NT) __attribute__((amdgpu_waves_per_eu(CF::OCC > 0 ? CF::OCC : 1)))
void gemm_splitk_kernel(GemmArgs<T> p, int kchunk, int64_t part_stride) {
    __shared__ __attribute__((aligned(16))) T lds_a[tile_lds_a<T, CF>()];
    __shared__ __attribute__((aligned(16))) T lds_b[tile_lds_b<T, CF>()];
    const int k0 = (int)blockIdx.y * kchunk;
    GemmArgs<T> q = p;
    q.k = min(kchunk, p.k - k0);
    q.a = TA ? p.a + k0 : p.a + (int64_t)k0 * p.lda;
    q.b = TB ? p.b + (int64_t)k0 * p.ldb : p.b + k0;
    q.c = p.c + (int64_t)blockIdx.y * part_stride;
    const int total = p.tiles_m * p.tiles_n;
    int tm, tn;
    grouped_tile(xcd_remap(blockIdx.x, total), p.tiles_m, p.tiles_n, p.group_m, tm, tn);
    gemm_tile<T, CF, TA, TB, VEC>(q, tm * CF::BM, tn * CF::BN, lds_a, lds_b);
}

template <typename T>
__global__ void splitk_reduce_kernel(int m, int n, int parts, const T* __restrict__ part, int64_t part_stride,
                                     T alpha, T beta, T* __restrict__ c, int64_t ldc) {
    const int64_t total = (int64_t)m * n;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
        T acc = part[e];
        for (int s = 1; s < parts; ++s) acc += part[s * part_stride + e];
        T* cp = c + (e / m) * ldc + e % m;
        *cp = epilogue(alpha, beta, acc, cp);
    }
}

template <typename T>
__global__ void scale_kernel(int m, int n, T beta, T* __restrict__ c, int64_t ldc) {
    const int64_t total = (int64_t)m * n;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t j = e / m, i = e % m;
        T* cp = c + j * ldc + i;
        *cp = (beta == T(0)) ? T(0) : beta * *cp;
    }
}

template <typename T>
hipError_t scale_launch(int m, int n, T beta, T* c, int64_t ldc, hipStream_t stream) {
    if (m <= 0 || n <= 0) return hipSuccess;
    const int64_t total = (int64_t)m * n;
    int blocks = (int)((total + 255) / 256);
    if (blocks > 65536) blocks = 65536;
    scale_kernel<T><<<blocks, 256, 0, stream>>>(m, n, beta, c, ldc);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// dispatch
// ---------------------------------------------------------------------------
template <typename T, class CF, int VEC>
static hipError_t launch_cfg(const GemmDesc<T>& d, hipStream_t stream) {
    GemmArgs<T> p;
    p.m = d.m; p.n = d.n; p.k = d.k;
    p.lda = d.lda; p.ldb = d.ldb; p.ldc = d.ldc;
    p.alpha = d.alpha; p.beta = d.beta;
    p.a = d.a; p.b = d.b; p.c = d.c;
    p.tiles_m = (d.m + CF::BM - 1) / CF::BM;
    p.tiles_n = (d.n + CF::BN - 1) / CF::BN;
    p.group_m = ZG_GROUP_M;
    const int grid = p.tiles_m * p.tiles_n;
    if (!d.ta && !d.tb) gemm_mfma_kernel<T, CF, false, false, VEC><<<grid, CF::NT, 0, stream>>>(p);
    else if (!d.ta && d.tb) gemm_mfma_kernel<T, CF, false, true, VEC><<<grid, CF::NT, 0, stream>>>(p);
    else if (d.ta && !d.tb) gemm_mfma_kernel<T, CF, true, false, VEC><<<grid, CF::NT, 0, stream>>>(p);
    else gemm_mfma_kernel<T, CF, true, true, VEC><<<grid, CF::NT, 0, stream>>>(p);
    return hipGetLastError();
}

template <typename T, class CF>
static hipError_t launch_vec(const GemmDesc<T>& d, hipStream_t stream) {
    constexpr int V = 16 / sizeof(T);
    const uintptr_t mask = 15;
    const bool aligned = ((reinterpret_cast<uintptr_t>(d.a) & mask) == 0) &&
                         ((reinterpret_cast<uintptr_t>(d.b) & mask) == 0) && (d.lda % V == 0) &&
                         (d.ldb % V == 0);
    if (aligned) return launch_cfg<T, CF, V>(d, stream);
    return launch_cfg<T, CF, 1>(d, stream);
}

// BK is given for FP64; FP32 uses twice the depth (same bytes per slice).
template <typename T, int BM, int BN, int BK64, int WM, int WN, int OCC>
static hipError_t launch_shape(const GemmDesc<T>& d, hipStream_t stream) {
    constexpr int BK = (sizeof(T) == 8) ? BK64 : 2 * BK64;
    return launch_vec<T, TileCfg<BM, BN, BK, WM, WN, OCC>>(d, stream);
}

// ---------------------------------------------------------------------------
// direct-load plan (FP64)
// ---------------------------------------------------------------------------
enum DmaTile : int { kDma128x128, kDma128x64, kDma64x128, kDma64x64 };

// Shares of a CU's 0.307 TFLOP/s from 4096^3 and 2048^3 (several tiles on a
// CU) and 2048^3, 1024^3 (one); a tile costs 96 k more than its depth.  The
// estimates are within 10 % of 1024^3 .. 8192^3 and of 256 .. 1024-row
// updates.  Splitting the leftover tiles: 3072 x 1536 x 3072, 576 tiles of
// 128x64, 558 us whole and 435 us with the last 64 split in 4; 2500^3 608 and
// 493 us; 512^3 (64 tiles in 4 ranges) 35.5 and 29.5 us a synchronous call,
// 128 x 128 x 4096 158 and 35 us.
static PiecePlan dma_plan(int m, int n, int k, bool may_split) {
    static const PieceTile kSizes[] = {{128, 128, 0.94, 0.80}, {128, 64, 0.92, 0.75}, {64, 128, 0.915, 0.75}, {64, 64, 0.87, 0.71}};
    return piece_plan(kSizes, m, n, k, 0.307e6, 96.0, 64, sizeof(double), may_split ? kGemmScratchMax : 0);
}

template <class CF>
static hipError_t launch_dma(const GemmDesc<typename CF::T>& d, hipStream_t stream, const PiecePlan& plan,
                             typename CF::T* part) {
    using T = typename CF::T;
    PieceArgs<T> p;
    int grid;
    if (!piece_args<T, CF::BM, CF::BN>(p, d, plan, part, ZG_GROUP_M, &grid)) return hipErrorInvalidValue;
    if (!d.ta && !d.tb) gemm_dma_kernel<false, false, CF><<<grid, CF::NT, 0, stream>>>(p);
    else if (!d.ta && d.tb) gemm_dma_kernel<false, true, CF><<<grid, CF::NT, 0, stream>>>(p);
    else if (d.ta && !d.tb) gemm_dma_kernel<true, false, CF><<<grid, CF::NT, 0, stream>>>(p);
    else gemm_dma_kernel<true, true, CF><<<grid, CF::NT, 0, stream>>>(p);
    const hipError_t e = hipGetLastError();
    return e != hipSuccess ? e : piece_sum_launch<T, CF::BM, CF::BN>(p, stream);
}

static hipError_t launch_dma_plan(const GemmDesc<double>& d, hipStream_t stream, const PiecePlan& plan, double* part) {
    switch (plan.tile) {
        case kDma128x128: return launch_dma<Dma128x128>(d, stream, plan, part);
        case kDma128x64: return launch_dma<Dma128x64>(d, stream, plan, part);
        case kDma64x128: return launch_dma<Dma64x128>(d, stream, plan, part);
        default: return launch_dma<Dma64x64<double>>(d, stream, plan, part);
    }
}

// FP32: the direct-load tiles or, for deep products, the bf16 matrix cores
// (gemm_f32_split.hip), whichever is estimated faster.  Shares of a CU in
// TFLOP/s (0.614 peak) from 4096^3, 1024 x 8192 x 256 and 2048 x 2048 x 256,
// and 1024^3, 512^3 for one tile on a CU.  Measured against the register-staged
// tiles: 1024^3 24.6 us (37.8), 512^3 13.7 (20.3), 256^3 8.7 (12.0), 64 x 2048 x
// 512 13.4 (20.3), TN 2048 x 2048 x 256 23.1 (29.8).
struct F32Plan {
    bool split;  // on the bf16 cores
    PiecePlan plan;
};

static F32Plan f32_plan(int m, int n, int k, bool may_split) {
    static const PieceTile kSizes[] = {{128, 64, 0.53, 0.43}, {64, 128, 0.535, 0.43}, {64, 64, 0.47, 0.37}};
    F32Plan f;
    f.plan = piece_plan(kSizes, m, n, k, 1.0e6, 96.0, 64, sizeof(float), may_split ? kGemmScratchMax : 0);
    PiecePlan deep;
    f.split = f32_split_plan(m, n, k, may_split, &deep) && deep.us < 0.9 * f.plan.us;
    if (f.split) f.plan = deep;
    return f;
}

static hipError_t launch_f32_plan(const GemmDesc<float>& d, hipStream_t stream, const F32Plan& f, float* part) {
    if (f.split) return gemm_f32_split_launch(d, stream, f.plan, part);
    switch (f.plan.tile) {
        case 0: return launch_dma<DmaCfg<float, 128, 64, 4, 1, 1, 3>>(d, stream, f.plan, part);
        case 1: return launch_dma<DmaCfg<float, 64, 128, 2, 2, 1, 3>>(d, stream, f.plan, part);
        default: return launch_dma<Dma64x64<float>>(d, stream, f.plan, part);
    }
}

// The direct-load tiles that walk K in one chain: the 64x64 tile with one
// k-group in the place of the one with two (its shares: 1024^3 52 us against
// 42), nothing split over K, FP32 on the FP32 instruction.  FP32 products of
// many 128x128 tiles take the table's register-staged tile: 4096^3 1.03 ms
// against 1.06 (2048^3 156 us against 140).
template <typename T>
static PiecePlan chain_plan(int m, int n, int k) {
    static const PieceTile kSizes64[] = {{128, 128, 0.94, 0.80}, {128, 64, 0.92, 0.75}, {64, 128, 0.915, 0.75}, {64, 64, 0.85, 0.57}};
    static const PieceTile kSizes32[] = {{128, 64, 0.53, 0.43}, {64, 128, 0.535, 0.43}, {64, 64, 0.47, 0.30}};
    if constexpr (sizeof(T) == 8) return piece_plan(kSizes64, m, n, k, 0.307e6, 96.0, 64, sizeof(T), 0);
    else return piece_plan(kSizes32, m, n, k, 1.0e6, 96.0, 64, sizeof(T), 0);
}

template <typename T>
hipError_t gemm_launch_chain(const GemmDesc<T>& d, hipStream_t stream) {
    const bool product = d.m > 0 && d.n > 0 && d.k > 0 && d.alpha != T(0);
    const bool staged = sizeof(T) == 4 && (int64_t)(d.m / 128) * (d.n / 128) >= 4 * kCus;
    if (!product || staged || !dma_shape_ok<T>(d.ta, d.tb, d.m, d.n, d.a, d.b))
        return gemm_launch<T>(d, stream, product ? pick_tile(d.m, d.n, d.k, (int)sizeof(T), d.ta, d.tb) : kTileAuto);
    const PiecePlan plan = chain_plan<T>(d.m, d.n, d.k);
    if constexpr (sizeof(T) == 8) {
        if (plan.tile == kDma64x64) return launch_dma<Dma64x64k1<T>>(d, stream, plan, nullptr);
        return launch_dma_plan(d, stream, plan, nullptr);
    } else {
        if (plan.tile == 2) return launch_dma<Dma64x64k1<T>>(d, stream, plan, nullptr);
        return launch_f32_plan(d, stream, F32Plan{false, plan}, nullptr);
    }
}

template <typename T>
hipError_t gemm_launch(const GemmDesc<T>& d, hipStream_t stream, int tile) {
    if (d.m <= 0 || d.n <= 0) return hipSuccess;
    if (d.k <= 0 || d.alpha == T(0)) return scale_launch<T>(d.m, d.n, d.beta, d.c, d.ldc, stream);
    return gemm_launch_product<T>(d, stream, tile);
}

template <typename T>
hipError_t gemm_launch_product(const GemmDesc<T>& d, hipStream_t stream, int tile) {
    if (d.m <= 0 || d.n <= 0) return hipSuccess;
    if (d.k <= 0) return scale_launch<T>(d.m, d.n, d.beta, d.c, d.ldc, stream);
    if (tile == kTileAuto) {
        if (dma_shape_ok<T>(d.ta, d.tb, d.m, d.n, d.a, d.b)) {
            if constexpr (sizeof(T) == 8) return launch_dma_plan(d, stream, dma_plan(d.m, d.n, d.k, false), nullptr);
            else return launch_f32_plan(d, stream, f32_plan(d.m, d.n, d.k, false), nullptr);
        }
        tile = pick_tile(d.m, d.n, d.k, (int)sizeof(T), d.ta, d.tb);
    }
    switch (tile) {
        case kTile64x64: return launch_shape<T, 64, 64, 16, 2, 2, 0>(d, stream);
        case kTile128x128: return launch_shape<T, 128, 128, 16, 2, 2, 1>(d, stream);
        case kTile128x128o2: return launch_shape<T, 128, 128, 16, 2, 2, 2>(d, stream);
        case kTile128x64: return launch_shape<T, 128, 64, 16, 2, 2, 2>(d, stream);
        case kTile64x128: return launch_shape<T, 64, 128, 16, 2, 2, 2>(d, stream);
        case kTile128x128k32: return launch_shape<T, 128, 128, 32, 2, 2, 1>(d, stream);
        case kTile128x128w8: return launch_shape<T, 128, 128, 16, 4, 2, 2>(d, stream);
        case kTile64x64k32:
            return launch_shape<T, 64, 64, 32, 2, 2, 0>(d, stream);
        case kTile256x128w8: return launch_shape<T, 256, 128, 16, 4, 2, 1>(d, stream);
        case kTile128x256w8: return launch_shape<T, 128, 256, 16, 2, 4, 1>(d, stream);
        case kTile128x128w8k8: return launch_shape<T, 128, 128, 8, 4, 2, 2>(d, stream);
        case kTile128x128w16:
            if constexpr (sizeof(T) == 8) {
                if (dma_shape_ok<T>(d.ta, d.tb, d.m, d.n, d.a, d.b)) {
                    PiecePlan plan;
                    plan.tile = kDma128x128;
                    plan.full = ((d.m + 127) / 128) * ((d.n + 127) / 128);
                    return launch_dma_plan(d, stream, plan, nullptr);
                }
            }
            return launch_shape<T, 128, 128, 16, 4, 4, 4>(d, stream);
        default: return hipErrorInvalidValue;
    }
}

// Split-K plan on the 64x64 tile: split when fewer than 128 tiles would run
// and K >= 1024, into enough K ranges (each a multiple of 32 and at least
// 256 deep, at most 64 of them) to give about 512 workgroups.
static int gemm_splitk_plan(int m, int n, int k, int* kchunk) {
    const int64_t tiles = (int64_t)((m + 63) / 64) * ((n + 63) / 64);
    if (tiles >= 128 || k < 1024) return 1;
    int64_t parts = std::min<int64_t>({(512 + tiles - 1) / tiles, (int64_t)k / 256, 64});
    if (parts < 2) return 1;
    int64_t kc = ((k + parts - 1) / parts + 31) / 32 * 32;
    parts = (k + kc - 1) / kc;
    if (parts < 2) return 1;
    *kchunk = (int)kc;
    return (int)parts;
}

template <typename T>
static hipError_t gemm_splitk_launch(const GemmDesc<T>& d, hipStream_t stream, T* part, int parts, int kchunk) {
    using CF = TileCfg<64, 64, (sizeof(T) == 8) ? 16 : 32, 2, 2, 0>;
    GemmArgs<T> p;
    p.m = d.m; p.n = d.n; p.k = d.k;
    p.lda = d.lda; p.ldb = d.ldb; p.ldc = d.m;
    p.alpha = T(1); p.beta = T(0);
    p.a = d.a; p.b = d.b; p.c = part;
    p.tiles_m = (d.m + CF::BM - 1) / CF::BM;
    p.tiles_n = (d.n + CF::BN - 1) / CF::BN;
    p.group_m = ZG_GROUP_M;
    const int64_t stride = (int64_t)d.m * d.n;
    constexpr int V = 16 / sizeof(T);
    const bool vec = ((reinterpret_cast<uintptr_t>(d.a) & 15) == 0) && ((reinterpret_cast<uintptr_t>(d.b) & 15) == 0) &&
                     (d.lda % V == 0) && (d.ldb % V == 0) && (kchunk % V == 0);
    const dim3 grid(p.tiles_m * p.tiles_n, parts);
#define ZG_SPLITK(TA, TB, VV) gemm_splitk_kernel<T, CF, TA, TB, VV><<<grid, CF::NT, 0, stream>>>(p, kchunk, stride)
    if (vec) {
        if (!d.ta && !d.tb) ZG_SPLITK(false, false, V);
        else if (!d.ta && d.tb) ZG_SPLITK(false, true, V);
        else if (d.ta && !d.tb) ZG_SPLITK(true, false, V);
        else ZG_SPLITK(true, true, V);
    } else {
        if (!d.ta && !d.tb) ZG_SPLITK(false, false, 1);
        else if (!d.ta && d.tb) ZG_SPLITK(false, true, 1);
        else if (d.ta && !d.tb) ZG_SPLITK(true, false, 1);
        else ZG_SPLITK(true, true, 1);
    }
#undef ZG_SPLITK
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    int blocks = (int)std::min<int64_t>(4096, (stride + 255) / 256);
    splitk_reduce_kernel<T><<<blocks, 256, 0, stream>>>(d.m, d.n, parts, part, stride, d.alpha, d.beta, d.c, d.ldc);
    return hipGetLastError();
}

template <typename T>
size_t gemm_scratch_bytes(const GemmDesc<T>& d, bool waits) {
    if (d.m <= 0 || d.n <= 0 || d.k <= 0 || d.alpha == T(0)) return 0;
    int kchunk = 0;
    const int parts = gemm_splitk_plan(d.m, d.n, d.k, &kchunk);
    if (parts <= 1 && !waits) return 0;
    if constexpr (sizeof(T) == 8) {
        if (dma_shape_ok<T>(d.ta, d.tb, d.m, d.n, d.a, d.b)) return dma_plan(d.m, d.n, d.k, true).scratch;
    } else {
        if (dma_shape_ok<T>(d.ta, d.tb, d.m, d.n, d.a, d.b)) return f32_plan(d.m, d.n, d.k, true).plan.scratch;
    }
    return parts > 1 ? (size_t)parts * d.m * d.n * sizeof(T) : 0;
}

template <typename T>
hipError_t gemm_launch_scratch(const GemmDesc<T>& d, hipStream_t stream, T* part) {
    if constexpr (sizeof(T) == 8) {
        if (dma_shape_ok<T>(d.ta, d.tb, d.m, d.n, d.a, d.b)) return launch_dma_plan(d, stream, dma_plan(d.m, d.n, d.k, true), part);
    } else {
        if (dma_shape_ok<T>(d.ta, d.tb, d.m, d.n, d.a, d.b))
            return launch_f32_plan(d, stream, f32_plan(d.m, d.n, d.k, true), part);
    }
    int kchunk = 0;
    const int parts = gemm_splitk_plan(d.m, d.n, d.k, &kchunk);
    return gemm_splitk_launch<T>(d, stream, part, parts, kchunk);
}

template size_t gemm_scratch_bytes<double>(const GemmDesc<double>&, bool);
template size_t gemm_scratch_bytes<float>(const GemmDesc<float>&, bool);
template hipError_t gemm_launch_scratch<double>(const GemmDesc<double>&, hipStream_t, double*);
template hipError_t gemm_launch_scratch<float>(const GemmDesc<float>&, hipStream_t, float*);
template hipError_t gemm_launch_chain<double>(const GemmDesc<double>&, hipStream_t);
template hipError_t gemm_launch_chain<float>(const GemmDesc<float>&, hipStream_t);
template hipError_t gemm_launch<double>(const GemmDesc<double>&, hipStream_t, int);
template hipError_t gemm_launch<float>(const GemmDesc<float>&, hipStream_t, int);
template hipError_t gemm_launch_product<double>(const GemmDesc<double>&, hipStream_t, int);
template hipError_t gemm_launch_product<float>(const GemmDesc<float>&, hipStream_t, int);
template hipError_t scale_launch<double>(int, int, double, double*, int64_t, hipStream_t);
template hipError_t scale_launch<float>(int, int, float, float*, int64_t, hipStream_t);

}  // namespace zg
