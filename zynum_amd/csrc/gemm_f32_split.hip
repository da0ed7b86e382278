// FP32 GEMM on the bf16 matrix cores.
//
// v_mfma_f32_16x16x4_f32 multiplies at 157 TFLOP/s, the bf16 instructions at
// 2.5 PFLOP/s.  A float of 24 significant bits is exactly the sum of three
// bf16 (8 bits each, rounded to nearest, so |x1| <= 2^-8 |x| and |x2| <=
// 2^-17 |x|), and a product of two parts is exact in FP32: Henry, Tang and
// Heinecke, "Leveraging the bfloat16 artificial intelligence datatype for
// higher-precision computations" (ARITH 2019), whose six part products these
// are.  The three left out are at most 2^-24 |a b| together (1.0038986 squared
// loses 2^-24.01), one rounding of an FP32 product; six products take 6/16 of
// the FP32 instruction's time.
//
// Sums of many terms are more exact than the FP32 instruction's, which rounds
// after every k where this rounds six times in 16.  2-norm error against 64
// bits, uniform operands: 320 deep 2.63e-7 (FP32 instruction 3.21e-7), 512
// 3.37e-7 (4.05e-7), 4096 1.00e-6 (1.15e-6), 8192 1.44e-6 (1.62e-6); 40 calls of
// GEMM, SYMM and TRSM drawn over their sizes, FP32 and complex, 0.32 .. 0.96 of
// it.  Sums of few terms are less exact: 4096 deep with one entry in 16 of A
// not zero 0.99 of the FP32 instruction's error, one in 64 1.11, one in 256
// 1.23, a single term 1.31 (1.39 units in the last place at most, not 0.5; with
// all nine products still 1.29: it is the bf16 unit's own sum).  A forced tile
// is the FP32 instruction.
//
// The parts are formed while an operand is staged, so no pass over memory and
// no workspace is added: global loads put 16 k of a row in registers, a share
// of them is split between the MFMAs of each 32-row block and goes to LDS as
// three planes of 32-byte rows (the fragment reads are linear: no bank
// conflicts), two stages deep.  256x256 tiles of 8 waves, each 128x64 as 4x2
// blocks of v_mfma_f32_32x32x16_bf16, two waves per SIMD.  One barrier per
// stage, before the last row block: the next stage's first fragments are read
// as that block's products free their registers (without it the MFMAs wait
// for 9 fragment reads of every wave, 4 %).
//
// What bounds it: the MFMA pipes are 75 % busy at 8192^3 and the clock falls
// to 1.79 GHz under that load (2.36 GHz on a quarter of the chip): 1.40 PFLOP/s
// of bf16 products, 4.70 ms against 8.43 ms with FP32 MFMAs.  4096^3 0.61 ms
// against 1.09, 2048^3 118 us (128x128 tiles) against 163.
//
// Range.  Inputs are multiplied by 2^24 before the split, so that every part of
// any finite float, subnormal ones too, is a normal bf16 (its last bit is
// 2^-125 at least), and the sums by 2^-48 in the epilogue.  What has no such
// sum (an infinity, a NaN, an entry past 2^104, a product past 2^80) is formed
// by the FP32 direct-load tile before anything is written, with the FP32
// instruction's own results (of a tile split over K, that K range).  An entry
// shows when its stage is split, a sum at the end: 4096^3 0.61 ms without such
// entries or with subnormal ones (1.09 on FP32 tiles throughout), 1.30 when
// every tile meets one at once, 1.72 somewhere on its way, 1.87 at its end.
#include "common.hpp"
#include "gemm.hpp"
#include "gemm_dma.hpp"
#include "gemm_f32_split.hpp"
#include "gemm_tile.hpp"

namespace zg {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));
typedef float v4f_u __attribute__((ext_vector_type(4), aligned(4)));

template <int BM_, int BN_, int WM_, int WN_>
struct SplitCfg {
    static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, NT = 64 * WM_ * WN_;
};
using Split256 = SplitCfg<256, 256, 2, 4>;
using Split128 = SplitCfg<128, 128, 2, 4>;

// the FP32 tile for what the split cannot hold, run by the same workgroup
template <class CF>
using SplitWide = DmaCfg<float, 128, 128, 4, CF::NT / 256, 1, 2>;

constexpr int kSplitK = 16;  // k per stage
constexpr float kSplitScale = 0x1p24f, kSplitUnscale = 0x1p-48f;

// a pair of floats as three bf16 pairs; `sum` becomes NaN when a part is not finite
__device__ __forceinline__ void split_pair(float x, float y, uint32_t (&p)[3], float& sum) {
    v2f r = {x * kSplitScale, y * kSplitScale};
#pragma unroll
    for (int s = 0; s < 3; ++s) {
        const v2bf h = __builtin_convertvector(r, v2bf);
        p[s] = __builtin_bit_cast(uint32_t, h);
        if (s < 2) {
            r.x -= __uint_as_float(p[s] << 16);
            r.y -= __uint_as_float(p[s] & 0xffff0000u);
        }
    }
    // (an infinite part leaves a NaN here; the finite rests are below 2^111)
    sum += r.x;
    sum += r.y;
}

// one operand's part of a stage: R rows of 16 k, as three bf16 planes
template <int R, bool KCONTIG, int NT>
struct SplitStage {
    static constexpr int E = R * kSplitK / NT;             // elements per thread
    static constexpr int U = KCONTIG ? 4 : (E < 8 ? E : 8);  // k per unit
    static constexpr int NU = E / U;                        // units per thread
    static constexpr int PER = kSplitK / U;                 // units per row
    float v[E];
    uint32_t p[U / 2][3];
    const float* base[KCONTIG ? NU : 1];
    uint32_t row[NU];
    int64_t ld;

    __device__ __forceinline__ void init(const float* x, int64_t ldx, int r0, int rlim, int tid) {
        ld = ldx;
#pragma unroll
        for (int i = 0; i < NU; ++i) {
            const int u = tid + NT * i;
            if constexpr (KCONTIG) {
                base[i] = x + (int64_t)min(r0 + u / PER, rlim - 1) * ldx + (u % PER) * U;
            } else {
                row[i] = (uint32_t)min(r0 + u % R, rlim - 1);
                base[0] = x;
            }
        }
    }
    template <bool FULL>
    __device__ __forceinline__ void load(int k0, int klim, int tid) {
#pragma unroll
        for (int i = 0; i < NU; ++i) {
            const int u = tid + NT * i;
            if constexpr (KCONTIG) {
                const float* q = base[i] + k0;
                if (FULL) {
                    const v4f_u t = *(const gptr<const v4f_u>)to_global(q);
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[i * 4 + e] = t[e];
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[i * 4 + e] = (k0 + (u % PER) * U + e < klim) ? q[e] : 0.0f;
                }
            } else {
                const int kk = k0 + __builtin_amdgcn_readfirstlane(u / R) * U;
                const float* q = base[0] + (int64_t)kk * ld;
#pragma unroll
                for (int e = 0; e < U; ++e) {
                    if (FULL) v[i * U + e] = to_global(q)[row[i]];
                    else v[i * U + e] = (kk + e < klim) ? to_global(q)[row[i]] : 0.0f;
                    q += ld;
                }
            }
        }
    }
    // half h of this thread's elements (in units' order) to parts; complete units are written
    __device__ __forceinline__ void store(char* lds, int h, int tid, float& sum) {
#pragma unroll
        for (int x = h * (E / 2); x < (h + 1) * (E / 2); x += 2) {
            const int i = x / U, e = x % U;
            split_pair(v[x], v[x + 1], p[e / 2], sum);
            if (e + 2 == U) {
                const int u = tid + NT * i;
                const int r = KCONTIG ? u / PER : u % R, kq = KCONTIG ? u % PER : u / R;
#pragma unroll
                for (int s = 0; s < 3; ++s) {
                    char* d = lds + s * (R * 32) + r * 32 + kq * (U * 2);
                    if constexpr (U == 8) *reinterpret_cast<v4u*>(d) = v4u{p[0][s], p[1][s], p[2][s], p[3][s]};
                    else *reinterpret_cast<v2u*>(d) = v2u{p[0][s], p[1][s]};
                }
            }
        }
    }
};

template <bool TA, bool TB, class CF>
__global__ __launch_bounds__(CF::NT) __attribute__((amdgpu_waves_per_eu(2))) void gemm_f32_split_kernel(PieceArgs<float> args) {
    constexpr int BM = CF::BM, BN = CF::BN, NT = CF::NT;
    constexpr int FM = BM / CF::WM / 32, FN = BN / CF::WN / 32;
    constexpr int PA = BM * 32, PB = BN * 32;  // bytes per plane
    constexpr int STAGE = 3 * (PA + PB);
    static_assert(FM % 2 == 0, "block FM reuses the registers of block 0");
    using CG = SplitWide<CF>;
    __shared__ __attribute__((aligned(32))) char lds[CG::LDS * 4 > 2 * STAGE ? CG::LDS * 4 : 2 * STAGE];
    __shared__ int out_of_range[2][NT / 64];  // by stage % 2: whether this wave has split an entry out of range
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm0 = (wave % CF::WM) * (BM / CF::WM), wn0 = (wave / CF::WM) * (BN / CF::WN);
    int tm, tn;
    grouped_tile(piece_tile(args, blockIdx.x), args.g.tiles_m, args.g.tiles_n, args.g.group_m, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;
    const GemmArgs<float> p = piece_of<float, TA, TB, BM, BN>(args, blockIdx.x, m0, n0);

    SplitStage<BM, TA, NT> sa;
    SplitStage<BN, !TB, NT> sb;
    sa.init(p.a, p.lda, m0, p.m, tid);
    sb.init(p.b, p.ldb, n0, p.n, tid);
    float sum = 0.0f;  // NaN once this thread has split an entry out of range

    v16f acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

    const int lr = lane & 31, lh = lane >> 5;
    auto frag = [&](const char* base, int r) { return *reinterpret_cast<const v8bf*>(base + r * 32 + lh * 16); };
    auto barrier = [&]() {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    v8bf fb[FN][3], fa[2][3];
    // one 32-row block against every column block, part products s0 .. s1 - 1
    // of (0,2) (1,1) (0,1) (2,0) (1,0) (0,0): B's smallest parts are done first
    auto mma = [&](int i, int s0, int s1) {
        constexpr int ia[6] = {0, 1, 0, 2, 1, 0}, ib[6] = {2, 1, 1, 0, 0, 0};
#pragma unroll
        for (int s = s0; s < s1; ++s)
#pragma unroll
            for (int j = 0; j < FN; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[j][ib[s]], fa[i & 1][ia[s]], acc[i][j], 0, 0, 0);
    };
    auto read_a = [&](const char* la, int i) {
#pragma unroll
        for (int s = 0; s < 3; ++s) fa[i & 1][s] = frag(la + s * PA, wm0 + i % FM * 32 + lr);
    };
    auto read_b = [&](const char* lb, int s) {
#pragma unroll
        for (int j = 0; j < FN; ++j) fb[j][s] = frag(lb + s * PB, wn0 + j * 32 + lr);
    };

    const int nk = p.k / kSplitK;  // whole stages
    bool stop = false;  // a wave has split one, by the next stage at the latest (the same for every wave)
    if (nk > 0) {
        sa.template load<true>(0, p.k, tid);
        sb.template load<true>(0, p.k, tid);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            sa.store(lds, h, tid, sum);
            sb.store(lds + 3 * PA, h, tid, sum);
        }
        const int k1 = min(1, nk - 1) * kSplitK;
        sa.template load<true>(k1, p.k, tid);
        sb.template load<true>(k1, p.k, tid);
        barrier();
        read_a(lds, 0);
#pragma unroll
        for (int s = 2; s >= 0; --s) read_b(lds + 3 * PA, s);
    }
    for (int t = 0; t < nk && !stop; ++t) {
        const char* la = lds + (t & 1) * STAGE;
        char* ln = lds + ((t + 1) & 1) * STAGE;
        const int k2 = min(t + 2, nk - 1) * kSplitK;  // the last stages are loaded again past the end, unused
#pragma unroll
        for (int i = 0; i < FM - 1; ++i) {
            read_a(la, i + 1);
            mma(i, 0, 6);
            // a share of the next stage's parts goes to the other buffer
#pragma unroll
            for (int h = 0; h < 4; ++h) {
                if (h * (FM - 1) / 4 != i) continue;
                if (h < 2) sa.store(ln, h, tid, sum);
                else sb.store(ln + 3 * PA, h - 2, tid, sum);
                if (h == 1) sa.template load<true>(k2, p.k, tid);
                if (h == 3) sb.template load<true>(k2, p.k, tid);
            }
            // the conversions between the MFMAs
#pragma unroll
            for (int s = 0; s < 6 * FN; ++s) {
                __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x2, 3, 0);
                if (s < 3) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        // the next stage is written: its first fragments are read as the last
        // block's products free their registers
        out_of_range[t & 1][wave] = __builtin_amdgcn_ballot_w64(sum != sum) != 0;  // (written again two barriers on)
        barrier();
        const int found = out_of_range[t & 1][lane & (NT / 64 - 1)];
        read_a(ln, FM);
        mma(FM - 1, 0, 1);
        __builtin_amdgcn_sched_barrier(0);
        read_b(ln + 3 * PA, 2);
        mma(FM - 1, 1, 3);
        __builtin_amdgcn_sched_barrier(0);
        read_b(ln + 3 * PA, 1);
        mma(FM - 1, 3, 6);
        __builtin_amdgcn_sched_barrier(0);
        read_b(ln + 3 * PA, 0);
        stop = __builtin_amdgcn_ballot_w64(found != 0) != 0;
    }
    if (nk * kSplitK < p.k && !stop) {
        // (nobody reads the buffer of stage nk but for fragments that are not used)
        sa.template load<false>(nk * kSplitK, p.k, tid);
        sb.template load<false>(nk * kSplitK, p.k, tid);
        char* ln = lds + (nk & 1) * STAGE;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            sa.store(ln, h, tid, sum);
            sb.store(ln + 3 * PA, h, tid, sum);
        }
        barrier();
#pragma unroll
        for (int s = 2; s >= 0; --s) read_b(ln + 3 * PA, s);
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            read_a(ln, i);
            mma(i, 0, 6);
        }
    }

    // tiles outside the split's range: the FP32 tile on this tile's 128x128 parts
    bool bad = stop || sum != sum;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) bad |= (__float_as_uint(acc[i][j][e]) & 0x7f800000u) == 0x7f800000u;
    if (__syncthreads_or(bad)) {
#pragma unroll 1
        for (int s = 0; s < (BM / 128) * (BN / 128); ++s) {
            const int mm = m0 + s % (BM / 128) * 128, nn = n0 + s / (BM / 128) * 128;
            if (mm < p.m && nn < p.n) gemm_tile_dma<TA, TB, CG>(p, mm, nn, reinterpret_cast<float*>(lds));
            __syncthreads();
        }
        return;
    }
    // (C^T is formed, as in the other tiles: a result item is 32 consecutive
    // rows of two columns of C)
    const float alpha = p.alpha, beta = p.beta;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const int row = m0 + wm0 + i * 32 + lr;
        if (row >= p.m) continue;
#pragma unroll
        for (int j = 0; j < FN; ++j)
        {
            float v[16];
#pragma unroll
            for (int g = 0; g < 16; ++g) v[g] = acc[i][j][g] * kSplitUnscale;
            auto col = [&](int g) { return n0 + wn0 + j * 32 + (g & 3) + 8 * (g >> 2) + 4 * lh; };
            write_back<float>(alpha, beta, v, [&](int g) { return col(g) < p.n; },
                              [&](int g) { return p.c + (int64_t)col(g) * p.ldc + row; });
        }
    }
}

// Taken from 320 deep, where its error was measured from (above); the caller
// compares the estimate with the FP32 tiles'.  Shares of a CU in TFLOP/s, from 4096^3, 8192^3, 8192 x 8192
// x 512 (256x256) and 4096^3, 2048^3, 1536 x 1536 x 300 (128x128); a tile costs
// 200 k more than its depth.
bool f32_split_plan(int m, int n, int k, bool may_split, PiecePlan* plan) {
    static const PieceTile kSizes[] = {{256, 256, 0.92, 0.92}, {128, 128, 0.76, 0.66}};
    if (k < 320) return false;
    *plan = piece_plan(kSizes, m, n, k, 1.0e6, 200.0, 256, sizeof(float), may_split ? kGemmScratchMax : 0);
    return true;
}

template <class CF>
static hipError_t launch_split(const GemmDesc<float>& d, hipStream_t stream, const PiecePlan& plan, float* part) {
    PieceArgs<float> p;
    int grid;
    if (!piece_args<float, CF::BM, CF::BN>(p, d, plan, part, 8, &grid)) return hipErrorInvalidValue;
    if (!d.ta && !d.tb) gemm_f32_split_kernel<false, false, CF><<<grid, CF::NT, 0, stream>>>(p);
    else if (!d.ta && d.tb) gemm_f32_split_kernel<false, true, CF><<<grid, CF::NT, 0, stream>>>(p);
    else if (d.ta && !d.tb) gemm_f32_split_kernel<true, false, CF><<<grid, CF::NT, 0, stream>>>(p);
    else gemm_f32_split_kernel<true, true, CF><<<grid, CF::NT, 0, stream>>>(p);
    const hipError_t e = hipGetLastError();
    return e != hipSuccess ? e : piece_sum_launch<float, CF::BM, CF::BN>(p, stream);
}

hipError_t gemm_f32_split_launch(const GemmDesc<float>& d, hipStream_t stream, const PiecePlan& plan, float* part) {
    if (plan.tile == 0) return launch_split<Split256>(d, stream, plan, part);
    return launch_split<Split128>(d, stream, plan, part);
}

}  // namespace zg
