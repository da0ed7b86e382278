// DTRSM and DSYRK on the GEMM core.
//
// TRSM (triangular.zig:155-249 solves one column at a time with trsv and
// streams the whole triangle per right-hand side) is recast recursively, as
// in the reference's blocked template (structured_blocked.zig:315-374):
// split the triangle in two halves, solve the first, update the second with
// one GEMM (B2 -= op(A)21 X1, plain FP64 MFMA or split precision), recurse.
// Triangles of at most 256 unknowns are one launch: 64-row blocks solved in
// FP64 with four lanes per vector (column of B for side L, row for side R)
// and the vector's unknowns in registers, in the reference's per-step order
// x_k /= a_kk; x_i = fma(a_ik, -x_k, x_i) (matrix_vector/triangular.zig:
// 375-385), their coupling subtracted with MFMAs in between.
//
// SYRK (symmetric.zig:180-279, one strided dot per element) runs as one launch
// over the lower (or upper) triangle of output tiles with the GEMM tile routine;
// diagonal tiles write only their stored triangle, so the other triangle is
// never touched (structured_blocked.zig:158-201 commits the same way).
#include <math.h>

#include <algorithm>
#include <utility>

#include "common.hpp"
#include "gemm.hpp"
#include "gemm_dma.hpp"
#include "gemm_pieces.hpp"
#include "gemm_tile.hpp"
#include "ops.hpp"
#include "runtime.hpp"

namespace zg {

// ---------------------------------------------------------------------------
// B <- alpha * B (a plain multiply, as scaleDenseColumns, triangular.zig:52-59)
// ---------------------------------------------------------------------------
template <typename T>
__global__ void mul_kernel(int m, int n, T alpha, T* __restrict__ b, int64_t ldb) {
    const int64_t total = (int64_t)m * n;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t j = e / m, i = e % m;
        b[j * ldb + i] = alpha * b[j * ldb + i];
    }
}

// ---------------------------------------------------------------------------
// leaf solve: nb <= 64 unknowns per vector
// ---------------------------------------------------------------------------
constexpr int kLeaf = 64;

template <typename T>
struct LeafArgs {
    const T* a;
    int64_t lda;
    T* b;
    int64_t ldb;
    int left;      // side L: vectors are columns of B, unknowns are rows i0..i0+nb
    int lower_eff; // op(A) is lower triangular
    int trans, unit;
    int i0, nb;    // unknowns [i0, i0 + nb) along the triangle
    int nvec;      // number of vectors (n for side L, m for side R)
};

template <typename T>
__device__ __forceinline__ T op_a(const LeafArgs<T>& p, int r, int c) {
    return p.trans ? p.a[(int64_t)r * p.lda + c] : p.a[(int64_t)c * p.lda + r];
}

// Leaf kernel: a quad of lanes per vector, 16 vectors per workgroup (one
// wave).  The unknowns are numbered in solve order (u = i forward, u = 63 - i
// backward, so a backward solve is a forward one in u); lane q of a quad holds
// unknowns u = 4j + q in x[j].  Step k takes the owner lane's (q = k % 4)
// final x_k to the whole quad with one DPP broadcast, divides it by the
// diagonal in every lane and eliminates it, one FMA per later unknown of the
// lane, in the reference's per-column order x_k /= a_kk;
// x_i = fma(a_ik, -x_k, x_i) (matrix_vector/triangular.zig:375-385).  The
// coefficients of a step are laid out in LDS per lane position and negated,
// Cs[k][q][j] = -a_{4j+q, k} (so no negation of x_k sits between the
// division and the FMAs), and read two steps ahead of their use; the
// diagonals are read as broadcasts.  A lane does a quarter of the FMAs and
// reads a quarter of the coefficients of the one-lane-per-vector form, and
// the grid has four times the waves: with one wave per SIMD the solve is
// bound by instruction issue, and the per-step division, which every lane
// executes, is then the largest share.  Unknowns past nb are padding:
// diagonal 1 and zero coefficients, so they stay 0 and eliminate nothing.
constexpr int kQuad = 4;                  // lanes per vector
constexpr int kLeafU = kLeaf / kQuad;     // unknowns per lane
constexpr int kLeafThreads = 64;
constexpr int kLeafVecs = kLeafThreads / kQuad;  // vectors per workgroup
constexpr int kLeafAhead = 2;             // steps whose coefficients are read ahead
constexpr int kLdsQ = kLeafU + 2;         // per-lane-position row (odd in 16-byte units: no bank conflict)
constexpr int kLdsK = kQuad * kLdsQ + 2;  // per-step row (odd in 16-byte units: lanes that store one step each)

template <typename T>
__device__ __forceinline__ T quad_bcast(T v, int src);
template <>
__device__ __forceinline__ double quad_bcast<double>(double v, int src) {
    // DPP quad_perm [src, src, src, src] on both halves; src is a constant at every call
    const uint64_t u = __double_as_longlong(v);
    int lo = (int)(uint32_t)u, hi = (int)(uint32_t)(u >> 32);
    switch (src) {
        case 0: lo = __builtin_amdgcn_mov_dpp(lo, 0x00, 0xf, 0xf, false); hi = __builtin_amdgcn_mov_dpp(hi, 0x00, 0xf, 0xf, false); break;
        case 1: lo = __builtin_amdgcn_mov_dpp(lo, 0x55, 0xf, 0xf, false); hi = __builtin_amdgcn_mov_dpp(hi, 0x55, 0xf, 0xf, false); break;
        case 2: lo = __builtin_amdgcn_mov_dpp(lo, 0xaa, 0xf, 0xf, false); hi = __builtin_amdgcn_mov_dpp(hi, 0xaa, 0xf, 0xf, false); break;
        default: lo = __builtin_amdgcn_mov_dpp(lo, 0xff, 0xf, 0xf, false); hi = __builtin_amdgcn_mov_dpp(hi, 0xff, 0xf, 0xf, false); break;
    }
    return __longlong_as_double((long long)(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo));
}
template <>
__device__ __forceinline__ float quad_bcast<float>(float v, int src) {
    int x = __float_as_int(v);
    switch (src) {
        case 0: x = __builtin_amdgcn_mov_dpp(x, 0x00, 0xf, 0xf, false); break;
        case 1: x = __builtin_amdgcn_mov_dpp(x, 0x55, 0xf, 0xf, false); break;
        case 2: x = __builtin_amdgcn_mov_dpp(x, 0xaa, 0xf, 0xf, false); break;
        default: x = __builtin_amdgcn_mov_dpp(x, 0xff, 0xf, 0xf, false); break;
    }
    return __int_as_float(x);
}

// coefficients (and diagonal) of step K into ring slot K % (kLeafAhead + 1);
// cq points at this lane's Cs[0][q][0]
template <typename T, bool UNIT, int K>
__device__ __forceinline__ void leaf_fetch(T (&c)[kLeafAhead + 1][kLeafU], T (&d)[kLeafAhead + 1], const T* cq,
                                           const T* Dg) {
    if constexpr (K < kLeaf) {
        constexpr int slot = K % (kLeafAhead + 1), j0 = K / kQuad;
#pragma unroll
        for (int j = j0; j < kLeafU; ++j) c[slot][j] = cq[K * kLdsK + j];
        if constexpr (!UNIT) d[slot] = Dg[K];
    }
}

template <typename T, bool UNIT, int K>
__device__ __forceinline__ void leaf_step(T (&x)[kLeafU], T (&c)[kLeafAhead + 1][kLeafU], T (&d)[kLeafAhead + 1],
                                          const T* cq, const T* Dg, int q, T& upd) {
    leaf_fetch<T, UNIT, K + kLeafAhead>(c, d, cq, Dg);
    constexpr int slot = K % (kLeafAhead + 1), jo = K / kQuad, o = K % kQuad;
    // x_k from its owner lane: for o > 0 the previous step's update of slot
    // jo, which is what lane o kept there (q > o - 1), taken before the selects
    T xk = quad_bcast<T>(o == 0 ? x[jo] : upd, o);
    if constexpr (!UNIT) xk = xk / d[slot];
    // the coefficients are stored negated: fma(-a_ik, x_k, x_i) is
    // fma(a_ik, -x_k, x_i) bit for bit
#pragma unroll
    for (int j = jo + 1; j < kLeafU; ++j) x[j] = fma_t(c[slot][j], xk, x[j]);
    // slot jo: unknown k in the owner, earlier (solved) unknowns below it,
    // later ones above
    // (unpredictable: selects, not branches around the FMA and the division)
    upd = fma_t(c[slot][jo], xk, x[jo]);
    const T keep = __builtin_unpredictable(q > o) ? upd : x[jo];
    x[jo] = __builtin_unpredictable(q == o) ? xk : keep;
    // one scheduling region per step: the reads stay ahead, register pressure
    // and compile time stay bounded
    __builtin_amdgcn_sched_barrier(0);
}

template <typename T, bool UNIT, int... K>
__device__ __forceinline__ void leaf_solve(T (&x)[kLeafU], const T* cq, const T* Dg, int q,
                                           std::integer_sequence<int, K...>) {
    T c[kLeafAhead + 1][kLeafU];
    T d[kLeafAhead + 1];
#pragma unroll
    for (int s = 0; s < kLeafAhead; ++s) {
#pragma unroll
        for (int j = s / kQuad; j < kLeafU; ++j) c[s][j] = cq[s * kLdsK + j];
        if constexpr (!UNIT) d[s] = Dg[s];
    }
    T upd = T(0);
    (leaf_step<T, UNIT, K>(x, c, d, cq, Dg, q, upd), ...);
}

// Coefficients of the 64-block whose first stored element is ablk, its stored
// columns c0 .. c0 + NC - 1: thread t takes stored row t, av[c] = stored column
// c0 + c (the wave reads one contiguous column per load), and dv = the
// diagonal of equation t.  Every load is issued before the first is used.  A
// full block (nb = 64) needs no clamping; otherwise rows and columns past nb
// repeat the last one.
template <typename T, typename P, int NC>
__device__ __forceinline__ void leaf_coeffs_load(T (&av)[NC], T& dv, P ablk, int64_t lda, int nb, int t, int c0 = 0) {
    const int tc = min(t, nb - 1);
    if (nb == kLeaf) {
        P col = ablk + t + (int64_t)c0 * lda;
#pragma unroll
        for (int c = 0; c < NC; ++c, col += lda) av[c] = *col;
    } else {
#pragma unroll
        for (int c = 0; c < NC; ++c) av[c] = ablk[(int64_t)min(c0 + c, nb - 1) * lda + tc];
    }
    dv = ablk[(int64_t)tc * lda + tc];
}

// The block's coefficients into LDS in solve order, negated,
// Cs[k][q][j] = -M_{4j+q, k} (M the equation matrix of the block), and its
// diagonal into Dg.  Side L
// solves op(A) x = b (M = op(A) block), side R solves x op(A) = b, i.e.
// op(A)^T x^T = b^T (M = op(A)^T block), so the stored element (row r,
// column c) is M[r][c] for side L without transpose and for side R with it,
// and M[c][r] otherwise (swap).  Every (equation, unknown) pair has its own
// slot.  A full block needs no zeroing: every slot a step reads for a later
// unknown holds its coefficient, and the other slots only feed updates that
// the owner selection discards.  A partial block zeroes the slots of padding
// and of the other triangle; padding equations get diagonal 1.
template <typename T, bool FWD, bool UNIT, int NC>
__device__ __forceinline__ void leaf_coeffs_store(T* Cs, T* Dg, const T (&av)[NC], T dv, int nb, int t, bool swap,
                                                  int c0 = 0) {
    if constexpr (!UNIT) Dg[FWD ? t : kLeaf - 1 - t] = (t < nb) ? dv : T(1);
    auto slot = [](int i, int k) {  // slot of M[i][k]
        const int ui = FWD ? i : kLeaf - 1 - i, uk = FWD ? k : kLeaf - 1 - k;
        return uk * kLdsK + (ui % kQuad) * kLdsQ + ui / kQuad;
    };
    auto keep = [&](int i, int k) {  // a coefficient some step reads
        const int ui = FWD ? i : kLeaf - 1 - i, uk = FWD ? k : kLeaf - 1 - k;
        return i < nb && k < nb && ui > uk;
    };
    if (nb == kLeaf) {
        if (swap) {
#pragma unroll
            for (int c = 0; c < NC; ++c) Cs[slot(c0 + c, t)] = -av[c];
        } else {
#pragma unroll
            for (int c = 0; c < NC; ++c) Cs[slot(t, c0 + c)] = -av[c];
        }
    } else {
        if (swap) {
#pragma unroll
            for (int c = 0; c < NC; ++c) Cs[slot(c0 + c, t)] = -(keep(c0 + c, t) ? av[c] : T(0));
        } else {
#pragma unroll
            for (int c = 0; c < NC; ++c) Cs[slot(t, c0 + c)] = -(keep(t, c0 + c) ? av[c] : T(0));
        }
    }
}

template <typename T, bool FWD, bool UNIT>
__global__ __launch_bounds__(kLeafThreads) void trsm_leaf_kernel(LeafArgs<T> p) {
    __shared__ __attribute__((aligned(16))) T Cs[kLeaf * kLdsK];  // Cs[k][q][j] = -a_{4j+q, k} (solve order)
    __shared__ T Dg[kLeaf];                      // diagonal in solve order (1 for padding)
    __shared__ T Xs[kLeafVecs * (kLeaf + 1)];    // side L: vectors staged for the transposition
    const int t = threadIdx.x, q = t & (kQuad - 1), vv = t / kQuad;
    const int v0 = blockIdx.x * kLeafVecs, v = v0 + vv;  // this quad's vector
    const int nb = p.nb;
    const int tc = min(t, nb - 1);
    auto idx = [](int u) { return FWD ? u : kLeaf - 1 - u; };  // solve order -> index in the block
    // Every load of a phase is issued before the first is used (one memory
    // round trip per phase).
    T av[kLeaf], dv;
    leaf_coeffs_load(av, dv, p.a + (int64_t)p.i0 * p.lda + p.i0, p.lda, nb, t);
    T x[kLeafU];
    if (p.left) {
        // vector v is column v of B, unknown i row i0 + i: the wave reads
        // columns (contiguous rows), transposed through LDS below
        T bv[kLeafVecs];
        const T* bblk = p.b + p.i0 + tc;
        if (v0 + kLeafVecs <= p.nvec) {
            const T* col = bblk + (int64_t)v0 * p.ldb;
#pragma unroll
            for (int w = 0; w < kLeafVecs; ++w, col += p.ldb) bv[w] = *col;
        } else {
#pragma unroll
            for (int w = 0; w < kLeafVecs; ++w) bv[w] = bblk[(int64_t)min(v0 + w, p.nvec - 1) * p.ldb];
        }
#pragma unroll
        for (int w = 0; w < kLeafVecs; ++w) Xs[w * (kLeaf + 1) + t] = bv[w];
    }
    // vector v is row v of B for side R, unknown i column i0 + i
    const T* bvec = p.b + (int64_t)p.i0 * p.ldb + min(v, p.nvec - 1);
    auto load_x = [&](T (&xx)[kLeafU]) {
        if (p.left) {
#pragma unroll
            for (int j = 0; j < kLeafU; ++j) xx[j] = Xs[vv * (kLeaf + 1) + idx(kQuad * j + q)];
        } else {
#pragma unroll
            for (int j = 0; j < kLeafU; ++j) xx[j] = bvec[(int64_t)min(idx(kQuad * j + q), nb - 1) * p.ldb];
        }
#pragma unroll
        for (int j = 0; j < kLeafU; ++j)
            if (idx(kQuad * j + q) >= nb) xx[j] = T(0);
    };
    if (!p.left) load_x(x);
    leaf_coeffs_store<T, FWD, UNIT>(Cs, Dg, av, dv, nb, t, (p.left != 0) == (p.trans != 0));
    __syncthreads();
    if (p.left) load_x(x);
    leaf_solve<T, UNIT>(x, Cs + q * kLdsQ, Dg, q, std::make_integer_sequence<int, kLeaf>{});
    if (p.left) {
        __syncthreads();
#pragma unroll
        for (int j = 0; j < kLeafU; ++j) Xs[vv * (kLeaf + 1) + idx(kQuad * j + q)] = x[j];
        __syncthreads();
        T* bblk = p.b + p.i0 + t;
        if (t < nb) {
            if (v0 + kLeafVecs <= p.nvec) {
                T* col = bblk + (int64_t)v0 * p.ldb;
#pragma unroll
                for (int w = 0; w < kLeafVecs; ++w, col += p.ldb) *col = Xs[w * (kLeaf + 1) + t];
            } else {
#pragma unroll
                for (int w = 0; w < kLeafVecs; ++w)
                    if (v0 + w < p.nvec) bblk[(int64_t)(v0 + w) * p.ldb] = Xs[w * (kLeaf + 1) + t];
            }
        }
    } else if (v < p.nvec) {
#pragma unroll
        for (int j = 0; j < kLeafU; ++j)
            if (idx(kQuad * j + q) < nb) p.b[(int64_t)(p.i0 + idx(kQuad * j + q)) * p.ldb + v] = x[j];
    }
}

// ---------------------------------------------------------------------------
// block solve: up to 256 unknowns per vector in one launch
// ---------------------------------------------------------------------------
// Below 256 unknowns the recursion's launches are latency-bound: a 64-row
// leaf over 8192 vectors and the 64- and 128-deep updates between leaves
// each take 10-15 us on MI355X for a few microseconds of work.  The block
// kernel keeps a workgroup's 16 vectors (all 256 unknowns) in LDS and runs
// the same recursion inside: each 64-block is solved by the leaf's quad
// solve, and its coupling to every later 64-block of the 256 is subtracted
// with 16 x 16 x 4 MFMAs, the workgroup's 16 vectors being the MFMA's 16
// columns (B_t -= M_ts X_s, as the recursion's GEMM updates).
//
// One or two waves solve, four update.  Step k (64-blocks in solve order) has
// two phases.  A(k): the coupling of block k to block k - 1 is subtracted (the
// near update, whose coefficients were read during B(k - 1)), and block k's
// coefficients go to LDS.  B(k): block k is solved; the updating waves read the
// coefficients of the near update A(k + 1) and subtract the coupling of blocks
// k + 1 and later to block k - 1 (the far updates), which the solve of block k
// does not need.  Only the solves and the near updates are on the critical path.
//
// Four updating waves, each 16 rows of every update (a near update is then 16
// MFMAs in a row, 0.5 us, not 64 on one wave) and a quarter of the next block's
// coefficients, read during the solve.  G groups of 16 vectors, each with a
// solving wave of its own: one while every workgroup has a CU to itself, else
// two, which share the coefficients and their reads.
// 256 unknowns, FP64, with one updating wave, workgroups of 16 vectors and wave 0
// reading its coefficients -> now (a synchronous call, 11 us of it launch and
// wait): 4096 vectors 47.9 -> 41.3 us, unit diagonal 43.9 -> 33.6; 8192 vectors
// 51.7 -> 46.4, transposed 59.0 -> 47.1; FP32 8192 vectors, right side 52.9 -> 36.6.
// (Five waves for two workgroups of one group on a CU exceed its registers:
// 67.4.)  What is left: 4.5 us of dependent steps per 64-block.
constexpr int kBlock = 256;
constexpr int kBlockUpd = 4;  // updating waves
constexpr int kXsV = kBlock + 4;  // LDS row per vector (4 mod 32 doubles: the MFMA reads spread over the banks)
constexpr int kTileK = kLeaf / 4;  // MFMA k-steps per 64-block

// row of item r of lane l in a 16 x 16 MFMA result (column l % 16)
template <typename T>
__device__ __forceinline__ int mfma_d_row(int r, int l);
template <>
__device__ __forceinline__ int mfma_d_row<double>(int r, int l) { return 4 * r + (l >> 4); }
template <>
__device__ __forceinline__ int mfma_d_row<float>(int r, int l) { return 4 * (l >> 4) + r; }

template <typename T, bool FWD, bool UNIT, int G>
__global__ __launch_bounds__(kLeafThreads * (G + kBlockUpd)) void trsm_block_kernel(LeafArgs<T> p) {
    constexpr int VECS = G * kLeafVecs, NTH = kBlockUpd * kLeafThreads;
    __shared__ __attribute__((aligned(16))) T Cs[kLeaf * kLdsK];  // current 64-block, as in the leaf
    __shared__ T Dg[kLeaf];
    __shared__ T Xs[VECS * kXsV];  // Xs[w][i]: unknown i of vector v0 + w (0 past len)
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int t = tid & (kLeafThreads - 1), q = t & (kQuad - 1), vv = t / kQuad;
    const int lr = t & 15, lk = t >> 4;  // MFMA operand lane coordinates
    const int v0 = blockIdx.x * VECS;
    const int len = p.nb, nsub = (len + kLeaf - 1) / kLeaf;
    const bool swap = (p.left != 0) == (p.trans != 0);
    const gptr<const T> a0 = to_global(p.a) + (int64_t)p.i0 * p.lda + p.i0;
    const gptr<T> b = to_global(p.b);
    auto sub = [&](int k) { return FWD ? k : nsub - 1 - k; };  // k-th 64-block in solve order
    auto idx = [](int u) { return FWD ? u : kLeaf - 1 - u; };

    // updating wave u: 16 stored columns of a 64-block's own coefficients
    constexpr int NC = kLeaf / kBlockUpd;
    const int u = wave - G;
    T av[NC], dv;
    auto load_block = [&](int k) {  // coefficients of the k-th 64-block into av, dv
        const int s0 = sub(k) * kLeaf;
        int64_t ld = p.lda;
        asm volatile("" : "+s"(ld));  // the column offsets are recomputed per block, not kept in registers
        leaf_coeffs_load(av, dv, a0 + (int64_t)s0 * ld + s0, ld, min(kLeaf, len - s0), t, NC * u);
    };
    auto store_block = [&](int k) {
        leaf_coeffs_store<T, FWD, UNIT>(Cs, Dg, av, dv, min(kLeaf, len - sub(k) * kLeaf), t, swap, NC * u);
    };

    // Coupling tiles.  Tile (kt, rt) of source ks: rows sub(kt) * 64 +
    // 16 rt + [0, 16) of M against the source block's 64 unknowns; A operand:
    // lane l holds M[row0 + l % 16][s0 + 4 kk + l / 16].  Indices are clamped
    // into [0, len): a row past len only feeds a padding unknown (solved
    // last, coupled to nothing, never stored); a column past len (a partial
    // first block of a backward solve) is masked to zero before use.
    const int64_t si = swap ? p.lda : 1, sk = swap ? 1 : p.lda;
    auto load_tile = [&](int kt, int rt, int ks, T (&am)[kTileK]) {
        const int s0 = sub(ks) * kLeaf;
        const gptr<const T> ai = a0 + (int64_t)min(sub(kt) * kLeaf + 16 * rt + lr, len - 1) * si;
        int64_t step = sk;
        asm volatile("" : "+s"(step));  // (as above)
#pragma unroll
        for (int kk = 0; kk < kTileK; ++kk) am[kk] = ai[(int64_t)min(s0 + 4 * kk + lk, len - 1) * step];
        __builtin_amdgcn_sched_barrier(0);  // issued here, consumed later
    };
    // B_t -= M_ts X_s as B_t + M_ts (-X_s); xb[g] is -X_s of vector group g as
    // the B operand: lane l holds -X[s0 + 4 kk + l / 16][vector l % 16]
    auto mma_tile = [&](int kt, int rt, int ks, T (&am)[kTileK], const T (&xb)[G][kTileK]) {
        const int s0 = sub(ks) * kLeaf;
        if (len - s0 < kLeaf) {
#pragma unroll
            for (int kk = 0; kk < kTileK; ++kk)
                if (s0 + 4 * kk + lk >= len) am[kk] = T(0);
        }
        const int i0 = sub(kt) * kLeaf + 16 * rt;
        typename Mfma<T>::acc_t acc[G];
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[g][r] = Xs[(16 * g + lr) * kXsV + i0 + mfma_d_row<T>(r, t)];
#pragma unroll
        for (int kk = 0; kk < kTileK; ++kk)
#pragma unroll
            for (int g = 0; g < G; ++g) acc[g] = Mfma<T>::mma(am[kk], xb[g][kk], acc[g]);
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int r = 0; r < 4; ++r) Xs[(16 * g + lr) * kXsV + i0 + mfma_d_row<T>(r, t)] = acc[g][r];
    };
    // The vectors' unknowns of one 64-block, rows [r0, r0 + 64), between B
    // and Xs, by the updating threads: every load (or LDS read) is issued
    // before the first store.  Rows past len are 0 in Xs and not
    // written back; vectors past nvec are not written back.
    constexpr int E = kLeaf * VECS / NTH;
    static_assert(NTH % VECS == 0, "a thread keeps its vector");
    auto rows_in = [&](int r0) {
        int64_t ldb = p.ldb;
        int th = tid - G * kLeafThreads;
        asm volatile("" : "+s"(ldb), "+v"(th));  // (as above)
        T xv[E];
        if (p.left) {
            // consecutive threads read consecutive rows of one column
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int f = th + NTH * e, w = f / kLeaf, i = r0 + f % kLeaf;
                xv[e] = b[(int64_t)min(v0 + w, p.nvec - 1) * ldb + p.i0 + min(i, len - 1)];
            }
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int f = th + NTH * e, w = f / kLeaf, i = r0 + f % kLeaf;
                Xs[w * kXsV + i] = (i < len) ? xv[e] : T(0);
            }
        } else {
            // consecutive threads read consecutive vectors of one row
            const int w = th % VECS;
            const gptr<const T> col = b + (int64_t)p.i0 * ldb + min(v0 + w, p.nvec - 1);
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int i = r0 + (th + NTH * e) / VECS;
                xv[e] = col[(int64_t)min(i, len - 1) * ldb];
            }
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int i = r0 + (th + NTH * e) / VECS;
                Xs[w * kXsV + i] = (i < len) ? xv[e] : T(0);
            }
        }
    };
    auto rows_out = [&](int r0) {
        int64_t ldb = p.ldb;
        int th = tid - G * kLeafThreads;
        asm volatile("" : "+s"(ldb), "+v"(th));  // (as above)
        T xv[E];
        if (p.left) {
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int f = th + NTH * e;
                xv[e] = Xs[(f / kLeaf) * kXsV + r0 + f % kLeaf];
            }
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int f = th + NTH * e, w = f / kLeaf, i = r0 + f % kLeaf;
                if (v0 + w < p.nvec && i < len) b[(int64_t)(v0 + w) * ldb + p.i0 + i] = xv[e];
            }
        } else {
            const int w = th % VECS;
#pragma unroll
            for (int e = 0; e < E; ++e) xv[e] = Xs[w * kXsV + r0 + (th + NTH * e) / VECS];
            if (v0 + w < p.nvec) {
                const gptr<T> col = b + (int64_t)p.i0 * ldb + v0 + w;
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    const int i = r0 + (th + NTH * e) / VECS;
                    if (i < len) col[(int64_t)i * ldb] = xv[e];
                }
            }
        }
    };
    // Each wave runs its own loop (its registers are allocated for its own
    // work, not for both); the loops meet at the same barriers, two per
    // 64-block, which end phases A(k) and B(k).
    if (wave < G) {
        T* xs = Xs + (wave * kLeafVecs + vv) * kXsV;
        for (int k = 0; k < nsub; ++k) {
            __syncthreads();  // end of A(k)
            const int r0 = sub(k) * kLeaf;
            T x[kLeafU];
#pragma unroll
            for (int j = 0; j < kLeafU; ++j) x[j] = xs[r0 + idx(kQuad * j + q)];
            leaf_solve<T, UNIT>(x, Cs + q * kLdsQ, Dg, q, std::make_integer_sequence<int, kLeaf>{});
#pragma unroll
            for (int j = 0; j < kLeafU; ++j) xs[r0 + idx(kQuad * j + q)] = x[j];
            __syncthreads();  // end of B(k)
        }
        return;
    }
    T xb[G][kTileK];  // -X of the last solved block
    T nm[kTileK];     // the near update's coefficients
    load_block(0);
    // the first-solved block's unknowns; the others are read during its solve,
    // and each block is written back during the next one's
    rows_in(sub(0) * kLeaf);
    for (int k = 0; k < nsub; ++k) {
        if (k > 0) {
#pragma unroll
            for (int g = 0; g < G; ++g)
#pragma unroll
                for (int kk = 0; kk < kTileK; ++kk)
                    xb[g][kk] = -Xs[(16 * g + lr) * kXsV + sub(k - 1) * kLeaf + 4 * kk + lk];
            mma_tile(k, u, k - 1, nm, xb);
        }
        store_block(k);
        __syncthreads();  // end of A(k)
        if (k + 1 < nsub) {
            load_tile(k + 1, u, k, nm);
            load_block(k + 1);
        }
        if (k == 0) {
            // before the first update reads them
#pragma unroll 1
            for (int k2 = 1; k2 < nsub; ++k2) rows_in(sub(k2) * kLeaf);
        } else {
            rows_out(sub(k - 1) * kLeaf);  // final since B(k - 1)
            T am[kTileK];
#pragma unroll 1
            for (int kt = k + 1; kt < nsub; ++kt) {
                load_tile(kt, u, k - 1, am);
                mma_tile(kt, u, k - 1, am, xb);
            }
        }
        __syncthreads();  // end of B(k)
    }
    rows_out(sub(nsub - 1) * kLeaf);
}

// ---------------------------------------------------------------------------
// recursion
// ---------------------------------------------------------------------------
namespace {
template <typename T>
struct TrsmCtx {
    bool left, lower_eff, trans, unit;
    int m, n;
    const T* a;
    int64_t lda;
    T* b;
    int64_t ldb;
    hipStream_t s;
    int mode, mode_param;
    // partial sums of updates split over K (null: none split)
    T* part = nullptr;
    size_t part_bytes = 0;
    size_t* want = nullptr;  // set: nothing is launched, the bytes that part should hold are noted
};

// op(A)[r0.., c0..] as a GEMM operand (pointer, transpose flag)
template <typename T>
const T* sub_opa(const TrsmCtx<T>& c, int r0, int c0) {
    return c.trans ? c.a + r0 * c.lda + c0 : c.a + c0 * c.lda + r0;
}

// smallest m, n and k of an off-diagonal update that runs in split precision
#ifndef ZG_SPLIT_UPDATE_MIN
#define ZG_SPLIT_UPDATE_MIN 1024
#endif
constexpr int kSplitUpdateMin = ZG_SPLIT_UPDATE_MIN;

template <typename T>
int gemm_update(const TrsmCtx<T>& c, bool ta, bool tb, int m, int n, int k, const T* a, int64_t lda, const T* b,
                int64_t ldb, T* cc, int64_t ldc) {
    if (m <= 0 || n <= 0 || k <= 0) return ZYNUM_GPU_OK;
    if constexpr (sizeof(T) == 8) {
        // Split precision pays only on large updates: its operand preparation
        // and reconstruction are fixed costs that the small updates at the
        // bottom of the recursion cannot amortise, so those run on FP64 MFMA
        // (same or smaller error).
        if (c.mode != ZYNUM_GPU_MODE_PLAIN && std::min(std::min(m, n), k) >= kSplitUpdateMin)
            return c.want != nullptr ? ZYNUM_GPU_OK
                                     : ozaki_dgemm(ta, tb, m, n, k, -1.0, a, lda, b, ldb, 1.0, cc, ldc, c.s, c.mode,
                                                   c.mode_param);
    }
    GemmDesc<T> d;
    d.ta = ta; d.tb = tb; d.m = m; d.n = n; d.k = k;
    d.lda = lda; d.ldb = ldb; d.ldc = ldc;
    d.alpha = T(-1); d.beta = T(1);
    d.a = a; d.b = b; d.c = cc;
    // With scratch, an update with few output tiles is split over K (256 x 1792 x
    // 1556: one walk of K is 66 us): 256 vectors, 3348 unknowns 803 -> 650 us, 805
    // vectors, 3501 unknowns 979 -> 858.  The updates at the bottom of the recursion
    // run on the direct-load tiles too: 256 x 8192 x 256 28 us, 256 x 256 x 256 14
    // (35 and 20 on register-staged 64x64 tiles; FP32 17 and 9, 22 and 14).
    const size_t want = c.want != nullptr || c.part != nullptr ? gemm_scratch_bytes<T>(d, true) : 0;
    if (c.want != nullptr) {
        *c.want = std::max(*c.want, want);
        return ZYNUM_GPU_OK;
    }
    if (want > 0 && want <= c.part_bytes) return status_from_hip(gemm_launch_scratch<T>(d, c.s, c.part));
    return status_from_hip(gemm_launch<T>(d, c.s, kTileAuto));
}

template <typename T>
int leaf(const TrsmCtx<T>& c, int i0, int nb) {
    LeafArgs<T> p;
    p.a = c.a; p.lda = c.lda; p.b = c.b; p.ldb = c.ldb;
    p.left = c.left; p.lower_eff = c.lower_eff; p.trans = c.trans; p.unit = c.unit;
    p.i0 = i0; p.nb = nb;
    p.nvec = c.left ? c.n : c.m;
    const int grid = (p.nvec + kLeafVecs - 1) / kLeafVecs;
    // forward substitution when the equations are lower triangular
    const bool fwd = c.left ? c.lower_eff : !c.lower_eff;
    if (fwd) {
        if (c.unit) trsm_leaf_kernel<T, true, true><<<grid, kLeafThreads, 0, c.s>>>(p);
        else trsm_leaf_kernel<T, true, false><<<grid, kLeafThreads, 0, c.s>>>(p);
    } else {
        if (c.unit) trsm_leaf_kernel<T, false, true><<<grid, kLeafThreads, 0, c.s>>>(p);
        else trsm_leaf_kernel<T, false, false><<<grid, kLeafThreads, 0, c.s>>>(p);
    }
    return status_from_hip(hipGetLastError());
}

// Solves the unknowns [i0, i0 + len), 64 < len <= kBlock, in one launch.
template <typename T>
int block(const TrsmCtx<T>& c, int i0, int len) {
    LeafArgs<T> p;
    p.a = c.a; p.lda = c.lda; p.b = c.b; p.ldb = c.ldb;
    p.left = c.left; p.lower_eff = c.lower_eff; p.trans = c.trans; p.unit = c.unit;
    p.i0 = i0; p.nb = len;
    p.nvec = c.left ? c.n : c.m;
    const int groups = (p.nvec + kLeafVecs - 1) / kLeafVecs;
    const bool fwd = c.left ? c.lower_eff : !c.lower_eff;
    auto run = [&](auto g) {
        constexpr int G = decltype(g)::value, NT = kLeafThreads * (G + kBlockUpd);
        const int grid = (groups + G - 1) / G;
        if (fwd) {
            if (c.unit) trsm_block_kernel<T, true, true, G><<<grid, NT, 0, c.s>>>(p);
            else trsm_block_kernel<T, true, false, G><<<grid, NT, 0, c.s>>>(p);
        } else {
            if (c.unit) trsm_block_kernel<T, false, true, G><<<grid, NT, 0, c.s>>>(p);
            else trsm_block_kernel<T, false, false, G><<<grid, NT, 0, c.s>>>(p);
        }
    };
    if (groups <= kCus) run(std::integral_constant<int, 1>{});
    else run(std::integral_constant<int, 2>{});
    return status_from_hip(hipGetLastError());
}

// A range of unknowns (rows of X for side L, columns for side R).
struct Range {
    int lo, len;
};

// The two halves of the unknowns [i0, i0 + len) in solve order: f is solved
// first.  Forward when the equations are lower triangular (side L with op(A)
// lower, side R with op(A) upper).
template <typename T>
void halves(const TrsmCtx<T>& c, int i0, int len, Range& f, Range& g) {
    int h = (len / 2 + kLeaf - 1) / kLeaf * kLeaf;
    if (h >= len) h = len - kLeaf;
    const bool forward = c.left ? c.lower_eff : !c.lower_eff;
    if (forward) {
        f = {i0, h};
        g = {i0 + h, len - h};
    } else {
        f = {i0 + h, len - h};
        g = {i0, h};
    }
}

// Unknowns r -= coupling to the solved unknowns s:
// side L, B[r, :] -= op(A)[r, s] X[s, :]; side R, B[:, r] -= X[:, s] op(A)[s, r].
template <typename T>
int update_range(const TrsmCtx<T>& c, Range r, Range s) {
    if (c.left)
        return gemm_update(c, c.trans, false, r.len, c.n, s.len, sub_opa(c, r.lo, s.lo), c.lda, c.b + s.lo, c.ldb,
                           c.b + r.lo, c.ldb);
    return gemm_update(c, false, c.trans, c.m, r.len, s.len, c.b + (int64_t)s.lo * c.ldb, c.ldb,
                       sub_opa(c, s.lo, r.lo), c.lda, c.b + (int64_t)r.lo * c.ldb, c.ldb);
}

// Solves the unknowns [i0, i0 + len): the first half, the update of the
// second half, the second half (structured_blocked.zig:315-374 blocks the
// same way).  One stream: the far half of a large update on a second stream
// beside the near half's solve slows that solve by more than it hides (8192 x
// 8192 9.40 against 9.30 ms, 500 vectors 1.86 against 1.80).
template <typename T>
int solve(const TrsmCtx<T>& c, int i0, int len) {
    if (len <= kBlock && c.want != nullptr) return ZYNUM_GPU_OK;
    if (len <= kLeaf) return leaf(c, i0, len);
    if (len <= kBlock) return block(c, i0, len);
    Range f, g;
    halves(c, i0, len, f, g);
    int st;
    if ((st = solve(c, f.lo, f.len))) return st;
    if ((st = update_range(c, g, f))) return st;
    return solve(c, g.lo, g.len);
}
}  // namespace

template <typename T>
static TrsmCtx<T> trsm_ctx(char side, char uplo, bool trans, char diag, int m, int n, const T* a, int64_t lda, T* b,
                           int64_t ldb, hipStream_t s, int mode, int mode_param) {
    TrsmCtx<T> c;
    c.left = (side == 'L');
    c.lower_eff = (uplo == 'L') != trans;
    c.trans = trans;
    c.unit = (diag == 'U');
    c.m = m; c.n = n; c.a = a; c.lda = lda; c.b = b; c.ldb = ldb; c.s = s;
    c.mode = mode; c.mode_param = mode_param;
    return c;
}

template <typename T>
size_t trsm_scratch_bytes(char side, char uplo, bool trans, int m, int n, const T* a, int64_t lda, T* b, int64_t ldb,
                          int mode) {
    TrsmCtx<T> c = trsm_ctx<T>(side, uplo, trans, 'N', m, n, a, lda, b, ldb, nullptr, mode, 0);
    size_t want = 0;
    c.want = &want;
    const int len = c.left ? m : n;
    if (len > kBlock) (void)solve(c, 0, len);
    return want;
}

template <typename T>
int trsm_device(char side, char uplo, bool trans, char diag, int m, int n, T alpha, const T* a, int64_t lda, T* b,
                int64_t ldb, hipStream_t s, int mode, int mode_param, T* part, size_t part_bytes) {
    if (m <= 0 || n <= 0) return ZYNUM_GPU_OK;
    if (alpha != T(1)) {
        const int64_t total = (int64_t)m * n;
        const int blocks = (int)std::min<int64_t>(65536, (total + 255) / 256);
        mul_kernel<T><<<blocks, 256, 0, s>>>(m, n, alpha, b, ldb);
        const int st = status_from_hip(hipGetLastError());
        if (st) return st;
    }
    TrsmCtx<T> c = trsm_ctx(side, uplo, trans, diag, m, n, a, lda, b, ldb, s, mode, mode_param);
    c.part = part;
    c.part_bytes = part_bytes;
    return solve(c, 0, c.left ? m : n);
}

// ---------------------------------------------------------------------------
// SYRK
// ---------------------------------------------------------------------------
// The large-shape GEMM tile: 16 waves of 32x32, two workgroups per CU; BK 16
// for FP64, 32 for FP32 (the same bytes per slice).
template <typename T>
using SyrkCfg = TileCfg<128, 128, (sizeof(T) == 8) ? 16 : 32, 4, 4, 4>;

// Triangle tiles in a cache-friendly order: the lower triangle of the tn x tn
// tile grid is cut into 8 x 8 super-tiles, walked in triangular order, with
// the tiles of each super-tile in row order; the workgroup index is first
// remapped so each XCD takes a contiguous run of that order.  The workgroups
// running together on one XCD then share a few A and B panels, as the grouped
// order of the plain GEMM does.  TRI 2 (upper) takes the transposed tile.
constexpr int kSyrkGroup = 8;

template <int TRI>
__device__ __forceinline__ void tri_tile(int t, int tn, int& ti, int& tj) {
    const int G = kSyrkGroup, ns = (tn + G - 1) / G;
    int I = 0, J = 0;
    for (I = 0; I < ns; ++I) {
        const int r0 = I * G, r1 = min(tn, r0 + G);
        bool found = false;
        for (J = 0; J <= I; ++J) {
            const int c0 = J * G, c1 = min(tn, c0 + G);
            int cnt = 0;  // tiles (i, j) of the super-tile with j <= i
            if (J < I) cnt = (r1 - r0) * (c1 - c0);
            else for (int i = r0; i < r1; ++i) cnt += min(c1, i + 1) - c0;
            if (t < cnt) { found = true; break; }
            t -= cnt;
        }
        if (found) break;
    }
    const int r0 = I * G, c0 = J * G, c1 = min(tn, c0 + G);
    int i = r0;
    for (;; ++i) {
        const int w = (J < I) ? (c1 - c0) : (min(c1, i + 1) - c0);
        if (t < w) break;
        t -= w;
    }
    const int j = c0 + t;
    ti = (TRI == 1) ? i : j;
    tj = (TRI == 1) ? j : i;
}

template <typename T, bool TA, int TRI, int VEC>
__global__ __launch_bounds__(SyrkCfg<T>::NT) __attribute__((amdgpu_waves_per_eu(SyrkCfg<T>::OCC)))
void syrk_kernel(GemmArgs<T> p, int tiles) {
    using CF = SyrkCfg<T>;
    __shared__ __attribute__((aligned(16))) T lds_a[tile_lds_a<T, CF>()];
    __shared__ __attribute__((aligned(16))) T lds_b[tile_lds_b<T, CF>()];
    int ti, tj;
    tri_tile<TRI>(xcd_remap(blockIdx.x, tiles), p.tiles_m, ti, tj);
    // C = alpha * op(A) op(A)^T + beta * C: the B operand is A with the other transpose
    gemm_tile<T, CF, TA, !TA, VEC, TRI>(p, ti * CF::BM, tj * CF::BN, lds_a, lds_b);
}

// Triangle tiles on the direct-load tiles, the leftover ones split over K.
template <bool TA, int TRI, class CF>
__global__ __launch_bounds__(CF::NT) __attribute__((amdgpu_waves_per_eu(CF::OCC))) void syrk_dma_kernel(
    PieceArgs<typename CF::T> p) {
    using T = typename CF::T;
    __shared__ __attribute__((aligned(32))) T lds[CF::LDS];
    int ti, tj;
    tri_tile<TRI>(piece_tile(p, blockIdx.x), p.g.tiles_m, ti, tj);
    const int m0 = ti * CF::BM, n0 = tj * CF::BN;
    gemm_tile_dma<TA, !TA, CF, TRI>(piece_of<T, TA, !TA, CF::BM, CF::BN>(p, blockIdx.x, m0, n0), m0, n0, lds);
}

// The unsplit form for many 128x128 tiles: the leftover tiles (past `full`) as
// quarters on the 64x64 tile with one k-group, the same order of every sum.
template <typename T>
using SyrkDma = DmaCfg<T, 128, 128, 4, 1, 1, 2>;
template <bool TA, int TRI, typename T>
__global__ __launch_bounds__(SyrkDma<T>::NT) __attribute__((amdgpu_waves_per_eu(2))) void syrk_quarters_kernel(
    GemmArgs<T> p, int full) {
    using CF = SyrkDma<T>;
    using CQ = Dma64x64k1<T>;
    static_assert(CF::NT == CQ::NT && CQ::LDS <= CF::LDS, "one workgroup runs either");
    __shared__ __attribute__((aligned(32))) T lds[CF::LDS];
    const int wg = blockIdx.x, r = wg - full;
    int ti, tj;
    tri_tile<TRI>(r < 0 ? xcd_remap(wg, full) : full + r / 4, p.tiles_m, ti, tj);
    if (r < 0) return gemm_tile_dma<TA, !TA, CF, TRI>(p, ti * 128, tj * 128, lds);
    const int m0 = ti * 128 + 64 * (r & 1), n0 = tj * 128 + 32 * (r & 2);
    // a quarter outside C or in the other triangle
    if (m0 >= p.m || n0 >= p.n || (TRI == 1 && m0 < n0) || (TRI == 2 && m0 > n0)) return;
    gemm_tile_dma<TA, !TA, CQ, TRI>(p, m0, n0, lds);
}

template <typename T>
hipError_t syrk_quarters_launch(GemmArgs<T> p, int tiles, bool lower, bool trans, hipStream_t s) {
    p.tiles_m = p.tiles_n = (p.n + 127) / 128;
    const int full = tiles / kCus * kCus, grid = full + 4 * (tiles - full);
    constexpr int NT = SyrkDma<T>::NT;
    if (lower) {
        if (trans) syrk_quarters_kernel<true, 1, T><<<grid, NT, 0, s>>>(p, full);
        else syrk_quarters_kernel<false, 1, T><<<grid, NT, 0, s>>>(p, full);
    } else {
        if (trans) syrk_quarters_kernel<true, 2, T><<<grid, NT, 0, s>>>(p, full);
        else syrk_quarters_kernel<false, 2, T><<<grid, NT, 0, s>>>(p, full);
    }
    return hipGetLastError();
}

template <int TRI, class CF>
__global__ __launch_bounds__(256) void syrk_sum_kernel(PieceArgs<typename CF::T> p) {
    constexpr int BLOCKS = CF::BM * CF::BN / 1024;
    const int tile = blockIdx.x / BLOCKS;
    int ti, tj;
    tri_tile<TRI>(p.full + tile, p.g.tiles_m, ti, tj);
    piece_sum<typename CF::T, CF::BM, CF::BN, TRI>(p, tile, (blockIdx.x % BLOCKS) * 1024 + threadIdx.x, ti * CF::BM,
                                                   tj * CF::BN);
}

template <class CF>
hipError_t syrk_dma_launch(const GemmArgs<typename CF::T>& g, const PiecePlan& plan, bool lower, bool trans,
                           typename CF::T* part, hipStream_t s) {
    PieceArgs<typename CF::T> p;
    p.g = g;
    p.g.tiles_m = p.g.tiles_n = (g.n + CF::BN - 1) / CF::BN;
    const int tiles = p.g.tiles_m * (p.g.tiles_m + 1) / 2, rest = tiles - plan.full;
    int grid;
    if (!piece_args(p, plan, part, tiles, &grid)) return hipErrorInvalidValue;
    if (lower) {
        if (trans) syrk_dma_kernel<true, 1, CF><<<grid, CF::NT, 0, s>>>(p);
        else syrk_dma_kernel<false, 1, CF><<<grid, CF::NT, 0, s>>>(p);
    } else {
        if (trans) syrk_dma_kernel<true, 2, CF><<<grid, CF::NT, 0, s>>>(p);
        else syrk_dma_kernel<false, 2, CF><<<grid, CF::NT, 0, s>>>(p);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || rest == 0) return e;
    const int blocks = rest * (CF::BM * CF::BN / 1024);
    if (lower) syrk_sum_kernel<1, CF><<<blocks, 256, 0, s>>>(p);
    else syrk_sum_kernel<2, CF><<<blocks, 256, 0, s>>>(p);
    return hipGetLastError();
}

// Tile size and leftover split of a triangle, as the plain GEMM's plans (the
// same shares of a CU).
template <typename T>
PiecePlan syrk_plan(int n, int k, size_t scratch_max) {
    static const PieceTile kSizes64[] = {{128, 128, 0.94, 0.80}, {64, 64, 0.87, 0.71}};
    static const PieceTile kSizes32[] = {{128, 128, 0.54, 0.27}, {64, 64, 0.47, 0.37}};
    return piece_plan(sizeof(T) == 8 ? kSizes64 : kSizes32, n, n, k, sizeof(T) == 8 ? 0.307e6 : 1.0e6, 96.0, 64, sizeof(T),
                      scratch_max, true);
}

// Without scratch, a triangle of two rounds of 128x128 tiles or more leaves its
// last tiles % 256 to quarters: 8192 x 4096 3.94 ms, 4096 x 2048 568 us (whole
// 64x64 tiles 4.47 ms and 620 us; split over K, with scratch, 3.87 and 526).
constexpr int kSyrkQuarters = 2 * kCus;

// Triangle-tile launch: the direct-load tiles, else (operands off their
// alignment) the register-staged one.  part: the split's partial sums, null
// when nothing is to be split.
template <typename T>
hipError_t syrk_launch(const GemmArgs<T>& p, int tiles, bool lower, bool trans, T* part, hipStream_t s) {
    if (dma_shape_ok<T>(trans, !trans, p.m, p.n, p.a, p.b)) {
        const int nt = (p.n + 127) / 128, tiles128 = nt * (nt + 1) / 2;
        if (part == nullptr && tiles128 >= kSyrkQuarters) return syrk_quarters_launch(p, tiles128, lower, trans, s);
        const PiecePlan plan = syrk_plan<T>(p.n, p.k, part != nullptr ? kGemmScratchMax : 0);
        return plan.tile == 0 ? syrk_dma_launch<SyrkDma<T>>(p, plan, lower, trans, part, s)
                              : syrk_dma_launch<Dma64x64<T>>(p, plan, lower, trans, part, s);
    }
    constexpr int V = 16 / sizeof(T);
    const bool vec = ((reinterpret_cast<uintptr_t>(p.a) & 15) == 0) && ((reinterpret_cast<uintptr_t>(p.b) & 15) == 0) &&
                     (p.lda % V == 0) && (p.ldb % V == 0);
#define ZG_SYRK(TA, TRI, VV) syrk_kernel<T, TA, TRI, VV><<<tiles, SyrkCfg<T>::NT, 0, s>>>(p, tiles)
    if (vec) {
        if (lower) { if (trans) ZG_SYRK(true, 1, V); else ZG_SYRK(false, 1, V); }
        else { if (trans) ZG_SYRK(true, 2, V); else ZG_SYRK(false, 2, V); }
    } else {
        if (lower) { if (trans) ZG_SYRK(true, 1, 1); else ZG_SYRK(false, 1, 1); }
        else { if (trans) ZG_SYRK(true, 2, 1); else ZG_SYRK(false, 2, 1); }
    }
#undef ZG_SYRK
    return hipGetLastError();
}

// stored triangle of C <- W + beta * C (W = alpha * op(A) op(A)^T computed in
// full), or C <- beta * C when w is null (k == 0 or alpha == 0, exact 0 for
// beta == 0 as symmetric.zig:196)
template <typename T>
__global__ void syrk_commit_kernel(int n, int lower, const T* __restrict__ w, int64_t ldw, T beta, T* __restrict__ c,
                                   int64_t ldc) {
    const int i = blockIdx.x * 256 + threadIdx.x, j = blockIdx.y;
    if (i >= n || (lower ? i < j : i > j)) return;
    T* cp = c + (int64_t)j * ldc + i;
    const T s = (beta == T(0)) ? T(0) : beta * *cp;
    *cp = (w != nullptr) ? w[(int64_t)j * ldw + i] + s : s;
}

template <typename T>
size_t syrk_scratch_bytes(int n, int k) {
    if (n <= 0 || k <= 0) return 0;
    return syrk_plan<T>(n, k, kGemmScratchMax).scratch;
}

template <typename T>
int syrk_device(char uplo, bool trans, int n, int k, T alpha, const T* a, int64_t lda, T beta, T* c, int64_t ldc,
                hipStream_t s, int mode, int mode_param, T* part) {
    if (n <= 0) return ZYNUM_GPU_OK;
    const bool lower = (uplo == 'L');
    if (k <= 0 || alpha == T(0)) {
        // C = beta * C on the stored triangle only
        dim3 grid((n + 255) / 256, n);
        syrk_commit_kernel<T><<<grid, 256, 0, s>>>(n, lower, nullptr, 0, beta, c, ldc);
        return status_from_hip(hipGetLastError());
    }
    if (sizeof(T) == 8 && mode != ZYNUM_GPU_MODE_PLAIN) {
        if constexpr (sizeof(T) == 8) {
            T* w = nullptr;
            if (hipMalloc(&w, (size_t)n * n * sizeof(T)) != hipSuccess) {
                (void)hipGetLastError();
                return ZYNUM_GPU_DECLINE_ALLOC;
            }
            int st = ozaki_dgemm(trans, !trans, n, n, k, alpha, a, lda, a, lda, 0.0, w, n, s, mode, mode_param);
            if (st == ZYNUM_GPU_OK) {
                dim3 grid((n + 255) / 256, n);
                syrk_commit_kernel<T><<<grid, 256, 0, s>>>(n, lower, w, n, beta, c, ldc);
                st = status_from_hip(hipGetLastError());
                if (st == ZYNUM_GPU_OK) st = status_from_hip(hipStreamSynchronize(s));
            }
            (void)hipFree(w);
            return st;
        }
    }
    GemmArgs<T> p;
    p.m = n; p.n = n; p.k = k;
    p.lda = lda; p.ldb = lda; p.ldc = ldc;
    p.alpha = alpha; p.beta = beta;
    p.a = a; p.b = a; p.c = c;
    const int tn = (n + SyrkCfg<T>::BM - 1) / SyrkCfg<T>::BM;
    p.tiles_m = p.tiles_n = tn;
    p.group_m = 1;
    const int tiles = tn * (tn + 1) / 2;
    return status_from_hip(syrk_launch<T>(p, tiles, lower, trans, part, s));
}

// ---------------------------------------------------------------------------
// SYMM, TRMM, SYR2K on the GEMM core
// ---------------------------------------------------------------------------
inline int64_t ld_round(int64_t rows) { return (rows + 7) / 8 * 8; }
inline size_t bytes_round(size_t b) { return (b + 255) / 256 * 256; }

// S (n x n) <- the full symmetric matrix whose stored triangle is A's
// (symValue, access.zig:31-42).  One 32 x 32 tile per workgroup: the mirrored
// tile of A is read along its contiguous dimension and transposed in LDS.
template <typename T>
__global__ __launch_bounds__(256) void symm_fill_kernel(int n, int lower, const T* __restrict__ a, int64_t lda,
                                                        T* __restrict__ s, int64_t lds, int tiles) {
    __shared__ T t[32][33];
    const int bi = (int)(blockIdx.x % (unsigned)tiles), bj = (int)(blockIdx.x / (unsigned)tiles);
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
#pragma unroll
    for (int c = ty; c < 32; c += 8) {  // t[c][r] = A(bj*32 + r, bi*32 + c)
        const int r = bj * 32 + tx, cc = bi * 32 + c;
        if (r < n && cc < n) t[c][tx] = a[(int64_t)cc * lda + r];
    }
    __syncthreads();
#pragma unroll
    for (int c = ty; c < 32; c += 8) {  // S(i, j), i = bi*32 + tx, j = bj*32 + c
        const int i = bi * 32 + tx, j = bj * 32 + c;
        if (i < n && j < n) {
            const bool stored = lower ? (i >= j) : (i <= j);
            s[(int64_t)j * lds + i] = stored ? a[(int64_t)j * lda + i] : t[tx][c];
        }
    }
}

// Workgroups of trmm_fill_kernel, 256 rows of a column each: a column's, for
// as many columns beside each other as one launch takes (fewer than 2^32
// threads: 65536 columns of 65536 rows are refused).
inline unsigned trmm_fill_blocks(int n) {
    const int64_t rows = ((int64_t)n + 255) / 256;
    return (unsigned)(rows * std::min<int64_t>({n, 1 << 16, ((1 << 24) - 1) / rows}));
}

// T (n x n) <- the triangle of A, ones on a unit diagonal (triValue,
// access.zig:54-63, without the transpose), and zeros in the rest of the
// block x block blocks on the diagonal; nothing reads the others.
template <typename T>
__global__ __launch_bounds__(256) void trmm_fill_kernel(int n, int lower, int unit, int block, const T* __restrict__ a,
                                                        int64_t lda, T* __restrict__ t, int64_t ldt) {
    const int rows = (n + 255) / 256, i = (int)(blockIdx.x % (unsigned)rows) * 256 + threadIdx.x;
    for (int j = (int)(blockIdx.x / (unsigned)rows); j < n; j += gridDim.x / (unsigned)rows) {
        const bool stored = lower ? (i > j) : (i < j);
        if (i >= n || (!stored && i / block != j / block)) continue;
        T v = T(0);
        if (i == j) v = unit ? T(1) : a[(int64_t)j * lda + i];
        else if (stored) v = a[(int64_t)j * lda + i];
        t[(int64_t)j * ldt + i] = v;
    }
}

// FP64 triangular product in one launch: every output tile is multiplied over
// the K range where op(A) is not zero, the longest ranges first (the ranges
// differ, so the launch order is what balances the CUs: seven panel products,
// each with its own last round, took 420 us where this takes 270 at 2500^2).
// `grows`: the range is [0, end of the tile) along the triangle, else [start of
// the tile, K).
template <bool TA, bool TB, class CF>
__global__ __launch_bounds__(CF::NT) __attribute__((amdgpu_waves_per_eu(CF::OCC))) void trmm_dma_kernel(
    GemmArgs<double> p, int left, int grows) {
    __shared__ __attribute__((aligned(32))) double lds[CF::LDS];
    const int along = left ? p.tiles_m : p.tiles_n, across = left ? p.tiles_n : p.tiles_m;
    const int o = blockIdx.x / across, x = blockIdx.x % across, t = grows ? along - 1 - o : o;
    const int m0 = (left ? t : x) * CF::BM, n0 = (left ? x : t) * CF::BN, B = left ? CF::BM : CF::BN;
    const int k0 = grows ? 0 : t * B, k1 = grows ? min(p.k, (t + 1) * B) : p.k;
    GemmArgs<double> q = p;
    q.k = k1 - k0;
    q.a = TA ? p.a + k0 : p.a + (int64_t)k0 * p.lda;
    q.b = TB ? p.b + (int64_t)k0 * p.ldb : p.b + k0;
    gemm_tile_dma<TA, TB, CF>(q, m0, n0, lds);
}

template <class CF>
hipError_t trmm_dma_launch(GemmArgs<double> p, bool left, bool trans, bool grows, hipStream_t s) {
    p.tiles_m = (p.m + CF::BM - 1) / CF::BM;
    p.tiles_n = (p.n + CF::BN - 1) / CF::BN;
    const int grid = p.tiles_m * p.tiles_n;
    if (left) {
        if (trans) trmm_dma_kernel<true, false, CF><<<grid, CF::NT, 0, s>>>(p, 1, grows);
        else trmm_dma_kernel<false, false, CF><<<grid, CF::NT, 0, s>>>(p, 1, grows);
    } else {
        if (trans) trmm_dma_kernel<false, true, CF><<<grid, CF::NT, 0, s>>>(p, 0, grows);
        else trmm_dma_kernel<false, false, CF><<<grid, CF::NT, 0, s>>>(p, 0, grows);
    }
    return hipGetLastError();
}

// Estimated time of trmm_dma_launch with one tile size, as piece_plan's: the
// work spread evenly (longest first), at least the longest range alone.
inline double trmm_dma_us(int na, int across, int b_along, int b_across, double several, double one) {
    const double along = (na + b_along - 1) / b_along, tiles = along * ((across + b_across - 1) / b_across);
    const double flop = 2.0 * b_along * b_across / 0.307e6;
    const double mean = flop * ((along + 1) / 2 * b_along + 96.0);
    return std::max((tiles + kCus / 2) / kCus * mean / several, flop * (na + 96.0) / one);
}

// C = alpha * S * B + beta * C (side L, S m x m) or alpha * B * S + beta * C
// (side R, S n x n), S symmetric from the stored triangle of A.  The reference
// (symmetric.zig:56-70) forms each element as one sum over the full row of S;
// here S is expanded once into the workspace and the tuned GEMM runs on it.
// The reference has no alpha == 0 quick return (alpha * sum is formed, so a
// NaN or an infinity in S or B reaches C): neither has this product.
template <typename T>
int symm_device(char side, char uplo, int m, int n, T alpha, const T* a, int64_t lda, const T* b, int64_t ldb, T beta,
                T* c, int64_t ldc, hipStream_t s) {
    if (m <= 0 || n <= 0) return ZYNUM_GPU_OK;
    const bool left = (side == 'L');
    GemmDesc<T> d;
    d.m = m; d.n = n;
    d.alpha = alpha; d.beta = beta;
    d.c = c; d.ldc = ldc;
    const int na = left ? m : n;
    const int64_t lds = ld_round(na);
    d.k = na;
    d.a = d.b = b;
    const size_t sym_bytes = bytes_round((size_t)lds * na * sizeof(T));
    const size_t want = gemm_scratch_bytes<T>(d, true);  // partial sums of split tiles, behind S
    T* sym = static_cast<T*>(workspace_acquire(sym_bytes + want, s));
    if (!sym) return ZYNUM_GPU_DECLINE_ALLOC;
    const int tiles = (na + 31) / 32;
    const int64_t blocks = (int64_t)tiles * tiles;
    hipError_t e = hipSuccess;
    if (blocks > 0x7fffffff) e = hipErrorInvalidValue;
    if (e == hipSuccess) {
        symm_fill_kernel<T><<<(unsigned)blocks, 256, 0, s>>>(na, uplo == 'L', a, lda, sym, lds, tiles);
        e = hipGetLastError();
    }
    if (e == hipSuccess) {
        d.ta = false; d.tb = false;
        if (left) {
            d.a = sym; d.lda = lds; d.b = b; d.ldb = ldb;
        } else {
            d.a = b; d.lda = ldb; d.b = sym; d.ldb = lds;
        }
        e = want > 0 ? gemm_launch_scratch<T>(d, s, sym + sym_bytes / sizeof(T)) : gemm_launch_product<T>(d, s);
    }
    const int st = status_from_hip(e);
    workspace_release(s);
    return st;
}

// B = alpha * op(A) * B (side L) or alpha * B * op(A) (side R), A triangular.
// The triangle is expanded with zeros around its diagonal and B copied aside,
// then the product is formed over only the K range where op(A) is not zero, so
// the work is about half a full GEMM: one launch of output tiles in FP64, GEMMs
// over row (L) or column (R) panels of the result in FP32.
// triangular.zig:202-231 multiplies column by column (trmv) or row by row.
template <typename T>
int trmm_device(char side, char uplo, bool trans, char diag, int m, int n, T alpha, const T* a, int64_t lda, T* b,
                int64_t ldb, hipStream_t s) {
    if (m <= 0 || n <= 0) return ZYNUM_GPU_OK;
    if (alpha == T(0)) return status_from_hip(scale_launch<T>(m, n, T(0), b, ldb, s));
    const bool left = (side == 'L');
    const int na = left ? m : n;
    const int64_t ldt = ld_round(na), ldw = ld_round(m);
    const size_t t_bytes = bytes_round((size_t)ldt * na * sizeof(T));
    char* ws = static_cast<char*>(workspace_acquire(t_bytes + (size_t)ldw * n * sizeof(T), s));
    if (!ws) return ZYNUM_GPU_DECLINE_ALLOC;
    T* tri = reinterpret_cast<T*>(ws);
    T* b0 = reinterpret_cast<T*>(ws + t_bytes);
    const bool lower_eff = (uplo == 'L') != trans;  // op(A) lower triangular
    const int extent = left ? m : n;               // panels along this dimension
    int panel = (extent + 7) / 8;
    panel = std::max(256, (panel + 127) / 128 * 128);
    const unsigned blocks = trmm_fill_blocks(na);
    trmm_fill_kernel<T><<<blocks, 256, 0, s>>>(na, uplo == 'L', diag == 'U', sizeof(T) == 8 ? 128 : panel, a, lda, tri, ldt);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess)
        e = hipMemcpy2DAsync(b0, (size_t)ldw * sizeof(T), b, (size_t)ldb * sizeof(T), (size_t)m * sizeof(T), (size_t)n,
                             hipMemcpyDeviceToDevice, s);
    if constexpr (sizeof(T) == 8) {
        if (e == hipSuccess) {
            GemmArgs<double> p;
            p.m = m; p.n = n; p.k = na;
            p.alpha = alpha; p.beta = 0.0;
            p.a = left ? tri : b0; p.lda = left ? ldt : ldw;
            p.b = left ? b0 : tri; p.ldb = left ? ldw : ldt;
            p.c = b; p.ldc = ldb;
            p.group_m = 1;
            const bool grows = left == lower_eff;
            const int across = left ? n : m;
            const double us[3] = {trmm_dma_us(na, across, 128, 128, 0.94, 0.80), trmm_dma_us(na, across, 64, 128, 0.915, 0.75),
                                  trmm_dma_us(na, across, 64, 64, 0.87, 0.71)};
            if (us[0] <= us[1] && us[0] <= us[2]) e = trmm_dma_launch<Dma128x128>(p, left, trans, grows, s);
            else if (us[1] <= us[2]) e = left ? trmm_dma_launch<Dma64x128>(p, left, trans, grows, s)
                                              : trmm_dma_launch<Dma128x64>(p, left, trans, grows, s);
            else e = trmm_dma_launch<Dma64x64<double>>(p, left, trans, grows, s);
        }
        const int st = status_from_hip(e);
        workspace_release(s);
        return st;
    }
    for (int x0 = 0; e == hipSuccess && x0 < extent; x0 += panel) {
        const int x1 = std::min(extent, x0 + panel);
        GemmDesc<T> d;
        d.alpha = alpha;
        d.beta = T(0);
        if (left) {  // rows x0..x1 of op(A) are nonzero in columns [0, x1) (lower) or [x0, m) (upper)
            const int k0 = lower_eff ? 0 : x0, k1 = lower_eff ? x1 : m;
            d.m = x1 - x0; d.n = n; d.k = k1 - k0;
            d.ta = trans;
            d.a = trans ? tri + k0 + (int64_t)x0 * ldt : tri + x0 + (int64_t)k0 * ldt;
            d.lda = ldt;
            d.tb = false; d.b = b0 + k0; d.ldb = ldw;
            d.c = b + x0; d.ldc = ldb;
        } else {  // columns x0..x1 of op(A) are nonzero in rows [x0, n) (lower) or [0, x1) (upper)
            const int k0 = lower_eff ? x0 : 0, k1 = lower_eff ? n : x1;
            d.m = m; d.n = x1 - x0; d.k = k1 - k0;
            d.ta = false; d.a = b0 + (int64_t)k0 * ldw; d.lda = ldw;
            d.tb = trans;
            d.b = trans ? tri + x0 + (int64_t)k0 * ldt : tri + k0 + (int64_t)x0 * ldt;
            d.ldb = ldt;
            d.c = b + (int64_t)x0 * ldb; d.ldc = ldb;
        }
        e = gemm_launch<T>(d, s);
    }
    const int st = status_from_hip(e);
    workspace_release(s);
    return st;
}

// C_tri = alpha * (op(A) op(B)^T + op(B) op(A)^T) + beta * C_tri on the stored
// triangle (symmetric.zig:301-329): two launches of the triangle-tile kernel,
// the second adding alpha * op(B) op(A)^T to the first's result.
template <typename T>
int syr2k_device(char uplo, bool trans, int n, int k, T alpha, const T* a, int64_t lda, const T* b, int64_t ldb,
                 T beta, T* c, int64_t ldc, hipStream_t s, T* part) {
    if (n <= 0) return ZYNUM_GPU_OK;
    const bool lower = (uplo == 'L');
    if (k <= 0 || alpha == T(0)) {
        dim3 grid((n + 255) / 256, n);
        syrk_commit_kernel<T><<<grid, 256, 0, s>>>(n, lower, nullptr, 0, beta, c, ldc);
        return status_from_hip(hipGetLastError());
    }
    GemmArgs<T> p;
    p.m = n; p.n = n; p.k = k;
    p.ldc = ldc;
    p.alpha = alpha;
    p.c = c;
    const int tn = (n + SyrkCfg<T>::BM - 1) / SyrkCfg<T>::BM;
    p.tiles_m = p.tiles_n = tn;
    p.group_m = 1;
    const int tiles = tn * (tn + 1) / 2;
    hipError_t e = hipSuccess;
    for (int pass = 0; pass < 2 && e == hipSuccess; ++pass) {
        p.a = pass ? b : a;
        p.lda = pass ? ldb : lda;
        p.b = pass ? a : b;
        p.ldb = pass ? lda : ldb;
        p.beta = pass ? T(1) : beta;
        e = syrk_launch<T>(p, tiles, lower, trans, part, s);
    }
    return status_from_hip(e);
}

template size_t syrk_scratch_bytes<double>(int, int);
template size_t syrk_scratch_bytes<float>(int, int);
template int symm_device<double>(char, char, int, int, double, const double*, int64_t, const double*, int64_t, double,
                                 double*, int64_t, hipStream_t);
template int symm_device<float>(char, char, int, int, float, const float*, int64_t, const float*, int64_t, float,
                                float*, int64_t, hipStream_t);
template int trmm_device<double>(char, char, bool, char, int, int, double, const double*, int64_t, double*, int64_t,
                                 hipStream_t);
template int trmm_device<float>(char, char, bool, char, int, int, float, const float*, int64_t, float*, int64_t,
                                hipStream_t);
template int syr2k_device<double>(char, bool, int, int, double, const double*, int64_t, const double*, int64_t,
                                  double, double*, int64_t, hipStream_t, double*);
template int syr2k_device<float>(char, bool, int, int, float, const float*, int64_t, const float*, int64_t, float,
                                 float*, int64_t, hipStream_t, float*);
template size_t trsm_scratch_bytes<double>(char, char, bool, int, int, const double*, int64_t, double*, int64_t, int);
template size_t trsm_scratch_bytes<float>(char, char, bool, int, int, const float*, int64_t, float*, int64_t, int);
template int trsm_device<double>(char, char, bool, char, int, int, double, const double*, int64_t, double*, int64_t,
                                 hipStream_t, int, int, double*, size_t);
template int trsm_device<float>(char, char, bool, char, int, int, float, const float*, int64_t, float*, int64_t,
                                hipStream_t, int, int, float*, size_t);
template int syrk_device<double>(char, bool, int, int, double, const double*, int64_t, double, double*, int64_t,
                                 hipStream_t, int, int, double*);
template int syrk_device<float>(char, bool, int, int, float, const float*, int64_t, float, float*, int64_t,
                                hipStream_t, int, int, float*);

}  // namespace zg
