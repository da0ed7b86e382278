// FP32 GEMM on the bf16 matrix cores.
//
// v_mfma_f32_16x16x4_f32 multiplies at 157 TFLOP/s, the bf16 instructions at
// 2.5 PFLOP/s.  A float of 24 significant bits is exactly the sum of three
// bf16 (8 bits each, rounded to nearest, so |x1| <= 2^-8 |x| and |x2| <=
// 2^-17 |x|), and a product of two parts is exact in FP32: Henry, Tang and
// Heinecke, "Leveraging the bfloat16 artificial intelligence datatype for
// higher-precision computations" (ARITH 2019).  All part products but a2 b2
// are formed, which is at most 2^-34 |a b|; eight take 8/16 of the FP32
// instruction's time.  (Without a1 b2 and a2 b1, 16 % faster, a product is
// short of up to 2^-24 of itself, one FP32 rounding.)
//
// The products a0 b0 are summed apart from the others.  The bf16 instructions
// round a sum once in 16 k, but not to nearest: with all products in one sum
// the low parts' roundings dominate, 2 times the FP32 instruction's error where
// one entry in 16 of A is not zero, and 64 units in the last place on constant
// operands.  The low sum's roundings are 2^-8 of that, and the two sums are
// added at the end.  Error against 64 bits, 2-norm (FP32 instruction): uniform
// operands 333 deep 9.2e-8 (3.27e-7), 4096 deep 3.75e-7 (1.15e-6), positive ones
// 3.0e-7 (8.4e-7), one entry of A in 4, 16, 64, 256 not zero 2.0e-7, 9.4e-8,
// 5.1e-8, 3.2e-8 (5.7e-7, 2.9e-7, 1.45e-7, 7.6e-8), a single term 2.58e-8
// (2.58e-8; 0.51 units in the last place at most, 0.50), constant operands
// 5.9e-8 (5.9e-8): on nothing tried larger than the FP32 instruction's.
//
// The parts are formed while an operand is staged, so no pass over memory and
// no workspace is added: global loads put 16 k of a row in registers, they are
// split between the MFMAs and go to LDS as three planes of 32-byte rows (the
// fragment reads are linear; the writes conflict, 11 % of the LDS cycles).  Waves of 64x64 as 2x2 blocks of
// v_mfma_f32_32x32x16_bf16, two sums each, two waves per SIMD: 256x128 tiles of
// 8 waves, or 128x128 of 4 and two workgroups on a CU.  Three stages in LDS, one
// barrier per stage, between the two row blocks: the stage after next is written
// and the next one's first fragments are read while products run.  (Every wait
// inside the loop counts what it needs: with LDS or memory waits for everything
// at the loop's top 4096^3 takes 0.90 ms.)
//
// What bounds it is the MFMAs, 77 % busy, and the chip's power: under this load
// the clock falls to 1.5 .. 1.65 GHz (2.4 with few CUs busy), and a CU then
// reaches 0.72 TFLOP/s (4096^3), with half of the CUs idle 0.98.  4096^3 0.77 ms
// (FP32 tiles 1.08), 8192^3 6.1 ms (8.5), 2048^3 135 us (155).
//
// Range.  Inputs are multiplied by 2^24 before the split, so that every part of
// any finite float, subnormal ones too, is a normal bf16 (its last bit is
// 2^-125 at least), and the sums by 2^-48 in the epilogue.  What has no such
// sum (an infinity, a NaN, an entry past 2^103, a product past 2^80) is formed
// by the FP32 direct-load tile before anything is written, with the FP32
// instruction's own results (of a tile split over K, that K range).  An entry
// shows when its stage is split, a sum at the end: 4096^3 0.77 ms without such
// entries or with subnormal ones (1.08 on FP32 tiles throughout), 1.26 when
// every tile meets one at once, 1.79 somewhere on its way, 1.97 at its end.
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
using SplitTall = SplitCfg<256, 128, 4, 2>;
using SplitSquare = SplitCfg<128, 128, 2, 2>;

// the FP32 tile for what the split cannot hold, run by the same workgroup
template <class CF>
using SplitWide = DmaCfg<float, 128, 128, 4, CF::NT / 256, 1, 2>;

constexpr int kSplitK = 16;  // k per stage
constexpr float kSplitScale = 0x1p24f, kSplitUnscale = 0x1p-48f;
constexpr float kSplitMax = 0x1p103f;  // smaller entries have finite parts

// a pair of floats as three bf16 pairs
__device__ __forceinline__ void split_pair(float x, float y, uint32_t (&p)[3]) {
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
}

// one operand's part of a stage: R rows of 16 k, as three bf16 planes of
// 32-byte rows.  The 16-byte halves of every other eight rows are exchanged:
// 8-byte writes of one k along the rows then fall on distinct banks.
template <int R, bool KCONTIG, int NT>
struct SplitStage {
    static constexpr int E = R * kSplitK / NT;             // elements per thread
    static constexpr int U = KCONTIG ? 4 : E;              // k per unit
    static constexpr int NU = E / U;                        // units per thread
    static constexpr int PER = kSplitK / U;                 // units per row
    static_assert(U == 4 || U == 8, "a unit is one write per plane");
    float v[E];
    uint32_t p[U / 2][3];
    const float* src[NU];  // what the next load reads: the unit's row (KCONTIG), else its first k-row
    uint32_t row;          // byte offset of this thread's element in a k-row
    int64_t ld, step;

    __device__ __forceinline__ void init(const float* x, int64_t ldx, int r0, int rlim, int tid) {
        ld = ldx;
        if constexpr (KCONTIG) {
#pragma unroll
            for (int i = 0; i < NU; ++i) {
                const int u = tid + NT * i;
                src[i] = x + (int64_t)min(r0 + u / PER, rlim - 1) * ldx + (u % PER) * U;
            }
            step = kSplitK;
        } else {
            // (320 k-rows and more: a row of 2^32 bytes would be a matrix of a terabyte)
            src[0] = x + (int64_t)(__builtin_amdgcn_readfirstlane(tid / R) * U) * ldx;
            row = (uint32_t)min(r0 + tid % R, rlim - 1) * 4u;
            step = kSplitK * ldx;
        }
    }
    __device__ __forceinline__ void advance() {
#pragma unroll
        for (int i = 0; i < NU; ++i) src[i] += step;
    }
    // FULL: a whole stage; else its first `left` k, zeros behind them
    template <bool FULL>
    __device__ __forceinline__ void load(int tid, int left = kSplitK) {
#pragma unroll
        for (int i = 0; i < NU; ++i) {
            const int kk = KCONTIG ? (tid + NT * i) % PER * U : __builtin_amdgcn_readfirstlane(tid / R) * U;
            const float* q = src[i];
            uint32_t off = KCONTIG ? 0u : row;
            asm volatile("" : "+v"(off));  // (a 32-bit offset beside the scalar address)
            if constexpr (KCONTIG && FULL) {
                const v4f_u t = *(const gptr<const v4f_u>)to_global(q);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[i * 4 + e] = t[e];
            } else {
#pragma unroll
                for (int e = 0; e < U; ++e) {
                    const gptr<const char> at = (gptr<const char>)to_global(q) + off;
                    v[i * U + e] = FULL || kk + e < left ? *(gptr<const float>)at : 0.0f;
                    q += KCONTIG ? 1 : ld;
                }
            }
        }
    }
    // half h of this thread's elements (in units' order) to parts; complete
    // units are written.  `big` is the largest magnitude, NaN behind a NaN.
    __device__ __forceinline__ void store(char* lds, int h, int tid, float& big) {
#pragma unroll
        for (int x = h * (E / 2); x < (h + 1) * (E / 2); x += 2) {
            const int i = x / U, e = x % U;
            split_pair(v[x], v[x + 1], p[e / 2]);
            big = __builtin_elementwise_maximum(__builtin_elementwise_maximum(big, __builtin_fabsf(v[x])), __builtin_fabsf(v[x + 1]));
            if (e + 2 == U) {
                const int u = tid + NT * i;
                const int r = KCONTIG ? u / PER : u % R, kq = KCONTIG ? u % PER : u / R;
#pragma unroll
                for (int s = 0; s < 3; ++s) {
                    char* d = lds + s * (R * 32) + r * 32 + (kq * (U * 2) ^ ((r >> 3 & 1) << 4));
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
    constexpr int STAGE = 3 * (PA + PB), NS = 3;
    static_assert(FM == 2 && FN == 2, "a wave owns 64 x 64");
    using CG = SplitWide<CF>;
    static_assert(CG::LDS * 4 <= NS * STAGE, "the FP32 tile fits");
    __shared__ __attribute__((aligned(32))) char lds[NS * STAGE];
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
    float big = 0.0f;  // largest entry this thread has split

    v16f hi[FM][FN], lo[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) hi[i][j][e] = lo[i][j][e] = 0.0f;

    const int lr = lane & 31, lh = lane >> 5, half = (lh ^ (lr >> 3 & 1)) * 16;
    auto frag = [&](const char* base, int r) { return *reinterpret_cast<const v8bf*>(base + r * 32 + half); };
    auto barrier = [&]() {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    v8bf fb[FN][3], fa[FM][3];
    // One 32-row block against both column blocks, part products s0 .. s1 - 1, B's
    // smallest parts first: the first kB2 use b2, up to kB1 b1, the rest b0.
    constexpr int kB2 = 2, kB1 = 5, kAll = 8;
    auto mma = [&](int i, int s0, int s1) {
        constexpr int ia[kAll] = {1, 0, 2, 1, 0, 2, 1, 0}, ib[kAll] = {2, 2, 1, 1, 1, 0, 0, 0};
#pragma unroll
        for (int s = s0; s < s1; ++s)
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                v16f& acc = s + 1 == kAll ? hi[i][j] : lo[i][j];
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[j][ib[s]], fa[i][ia[s]], acc, 0, 0, 0);
            }
    };
    auto read_a = [&](const char* la, int i) {
#pragma unroll
        for (int s = 0; s < 3; ++s) fa[i][s] = frag(la + s * PA, wm0 + i * 32 + lr);
    };
    auto read_b = [&](const char* lb, int s) {
#pragma unroll
        for (int j = 0; j < FN; ++j) fb[j][s] = frag(lb + s * PB, wn0 + j * 32 + lr);
    };

    const int nk = p.k / kSplitK;  // whole stages
    bool stop = false;  // a wave has split one, by the next stage at the latest (the same for every wave)
    // the MFMAs of n part products, five vector instructions beside each
    auto schedule = [&](auto n) {
#pragma unroll
        for (int g = 0; g < decltype(n)::value * FN; ++g) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x2, 5, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    int at = 0;  // the stage's buffer
    if (nk > 0) {
        // stages 0 and 1 in LDS, stage 2 on its way (past the end: the last one
        // again, unused).  The order of the loads is the loop's own, so that its
        // waits count the same ones on the way in.
#pragma unroll
        for (int u = 0; u < 3; ++u) {
            sa.template load<true>(tid);
            __builtin_amdgcn_sched_barrier(0);
            sb.template load<true>(tid);
            __builtin_amdgcn_sched_barrier(0);
            if (u + 1 < nk) {
                sa.advance();
                sb.advance();
            }
            if (u == 2) break;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                sa.store(lds + u * STAGE, h, tid, big);
                sb.store(lds + u * STAGE + 3 * PA, h, tid, big);
            }
        }
        barrier();
        read_a(lds, 0);
#pragma unroll
        for (int s = 2; s >= 0; --s) {
            __builtin_amdgcn_sched_barrier(0);
            read_b(lds + 3 * PA, s);
        }
        __builtin_amdgcn_sched_barrier(0);
        for (int t = 0; t < nk && !stop; ++t) {
            const int next = at == (NS - 1) * STAGE ? 0 : at + STAGE, over = next == (NS - 1) * STAGE ? 0 : next + STAGE;
            const char *la = lds + at, *l1 = lds + next;
            char* l2 = lds + over;
            const bool more = t + 4 < nk;  // (past the end the last stage is loaded again, unused)
            // rows 0 .. 31 of the wave's block; A's parts of the stage after next
            read_a(la, 1);
            mma(0, 0, kAll);
            sa.store(l2, 0, tid, big);
            sa.store(l2, 1, tid, big);
            sa.template load<true>(tid);
            if (more) sa.advance();
            schedule(std::integral_constant<int, kAll>{});
            // every wave is done with the stage before this one, and has written all of the next
            out_of_range[t & 1][wave] = __builtin_amdgcn_ballot_w64(!(big < kSplitMax)) != 0;  // (written again two barriers on)
            barrier();
            const int found = out_of_range[t & 1][lane & (NT / 64 - 1)];
            // rows 32 .. 63; the next stage's first fragments as registers come free
            read_a(l1, 0);
            mma(1, 0, kB2);
            __builtin_amdgcn_sched_barrier(0);
            read_b(l1 + 3 * PA, 2);
            mma(1, kB2, kB1);
            sb.store(l2 + 3 * PA, 0, tid, big);
            schedule(std::integral_constant<int, kB1 - kB2>{});
            read_b(l1 + 3 * PA, 1);
            mma(1, kB1, kAll);
            sb.store(l2 + 3 * PA, 1, tid, big);
            sb.template load<true>(tid);
            if (more) sb.advance();
            schedule(std::integral_constant<int, kAll - kB1>{});
            read_b(l1 + 3 * PA, 0);
            stop = __builtin_amdgcn_ballot_w64(found != 0) != 0;
            at = next;
        }
    }
    if (nk * kSplitK < p.k && !stop) {
        // (nobody reads the buffer of stage nk but for fragments that are not used)
        if (nk > 0) {  // (src is at the last whole stage)
            sa.advance();
            sb.advance();
        }
        sa.template load<false>(tid, p.k - nk * kSplitK);
        sb.template load<false>(tid, p.k - nk * kSplitK);
        char* ln = lds + at;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            sa.store(ln, h, tid, big);
            sb.store(ln + 3 * PA, h, tid, big);
        }
        barrier();
#pragma unroll
        for (int s = 2; s >= 0; --s) read_b(ln + 3 * PA, s);
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            read_a(ln, i);
            mma(i, 0, kAll);
        }
    }

    // tiles outside the split's range: the FP32 tile on this tile's 128x128 parts
    bool bad = stop || !(big < kSplitMax);
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                hi[i][j][e] += lo[i][j][e];
                bad |= (__float_as_uint(hi[i][j][e]) & 0x7f800000u) == 0x7f800000u;
            }
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
            for (int g = 0; g < 16; ++g) v[g] = hi[i][j][g] * kSplitUnscale;
            auto col = [&](int g) { return n0 + wn0 + j * 32 + (g & 3) + 8 * (g >> 2) + 4 * lh; };
            write_back<float>(alpha, beta, v, [&](int g) { return col(g) < p.n; },
                              [&](int g) { return p.c + (int64_t)col(g) * p.ldc + row; });
        }
    }
}

// Taken from 320 deep, where its error was measured from (above); the caller
// compares the estimate with the FP32 tiles'.  Shares of a CU in TFLOP/s: between
// those of a full chip, whose clock falls (256x128 tiles 0.72 at 4096^3, 0.85 at
// 8192 x 8192 x 512; 128x128 0.67 and 0.84), and of a part of one (0.98; 0.60 one
// tile to a CU).  With the full chip's, products of 10 to 200 us that gain (2097 x
// 7837 x 760: 207 us against 238 on FP32 tiles) stay on the FP32 tiles; with
// these, of 56 drawn products none is slower than there.  A tile costs 200 k
// more than its depth.
bool f32_split_plan(int m, int n, int k, bool may_split, PiecePlan* plan) {
    static const PieceTile kSizes[] = {{256, 128, 0.92, 0.92}, {128, 128, 0.85, 0.66}};
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
    if (plan.tile == 0) return launch_split<SplitTall>(d, stream, plan, part);
    return launch_split<SplitSquare>(d, stream, plan, part);
}

}  // namespace zg
