// The INT8 GEMM on a direct-to-LDS ring fed with whole 128-byte lines (included
// by ozaki.hip behind its MFMA wrappers and i8_store).
//
// 256x256 tiles of 8 waves, two per SIMD, each 128x64 in 16x16x64 MFMAs: 12
// fragment reads per 32 MFMAs against 8 per 16 for 16 waves of 64x64, whose
// reads alone take the LDS bandwidth at the MFMAs' peak rate.  The ring's 5
// slots of 64 k fill the LDS (160 KiB).  A line of 128 k is loaded as two
// halves one after the other, since a line's second half, loaded a slot later,
// is fetched from L2 again; a line's loads are issued 3 halves before the wait
// for them.  Per half: one barrier, then the next half's fragment reads and a
// line's direct loads between the MFMAs.  Half the distance (one barrier per
// line, its loads behind it) costs 11 %, so the loads' latency is what bounds
// it (the MFMAs are 75 % busy) next to the clock (1.73 GHz under this load).
//
// Fourteen products of 8192^3 (a split DGEMM): 5.7 ms, 2.7 POP/s, against 7.8 ms
// for the register-staged 16-wave tile; the whole call 8.46 -> 6.65 ms, 2048^3
// 298 -> 254 us, 1000 x 777 x 1301 115 -> 105.
// 4 waves of 128x128 (one per SIMD) spill: 7.95 ms.  Tile-order groups of 4 rows
// against 8: 6.91 and 7.04 ms (an XCD's 32 resident tiles are then 4 x 8).
//
// Results: the residue bytes go through LDS and leave as 256 consecutive rows
// of a column; straight from the MFMA layout a store instruction writes 4 bytes
// of 16 columns.
#pragma once

namespace zg {

struct RingCfg {
    using MF = I8Mfma<16>;
    static constexpr int BM = 256, BN = 256, WM = 2, WN = 4, NW = WM * WN, NT = 64 * NW;
    static constexpr int NS = 5;            // ring slots
    static constexpr int BK = 64;           // k bytes per slot
    static constexpr int SLOT = (BM + BN) * BK;
    static constexpr int LDS = NS * SLOT;   // 160 KiB
    static constexpr int FM = BM / WM / 16, FN = BN / WN / 16;
    static constexpr int LPW = (BM + BN) / 16 / NW;  // direct loads per slot, per wave
    static constexpr int CST = BM + 16;     // bytes per column of the result tile in LDS
};

// Position (of 4) of 16-byte chunk c of row r in its 64-byte LDS row: c ^
// ring_sw(r), which spreads the 16 rows of a fragment read over the banks.
__device__ __forceinline__ int ring_sw(int r) {
    const int g = (r >> 2) & 3;
    return (((g ^ (g >> 1)) & 1) << 1) | (g >> 1);
}

__global__ __launch_bounds__(RingCfg::NT) __attribute__((amdgpu_waves_per_eu(2))) void i8_ring_kernel(I8Args p) {
    using CF = RingCfg;
    using MF = CF::MF;
    constexpr int BM = CF::BM, BN = CF::BN, BK = CF::BK, FM = CF::FM, FN = CF::FN, NW = CF::NW, LPW = CF::LPW;
    extern __shared__ __attribute__((aligned(16))) int8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm0 = (wave % CF::WM) * (BM / CF::WM), wn0 = (wave / CF::WM) * (BN / CF::WN);
    int tm, tn;
    grouped_tile(xcd_remap(blockIdx.x, p.tiles_m * p.tiles_n), p.tiles_m, p.tiles_n, 4, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;
    const I8Out& out = p.outs[blockIdx.z];

    // Direct load l of this wave fills rows 16 q .. 16 q + 15 of a slot, q = wave
    // + NW l: lane i position i % 4 of row i / 4.  Rows past an edge repeat the
    // last one (their sums are not stored).
    uint32_t off[LPW];
#pragma unroll
    for (int l = 0; l < LPW; ++l) {
        const int q = wave + NW * l;
        const bool is_a = l < LPW / 2;
        const int r = (is_a ? q : q - BM / 16) * 16 + (lane >> 2);
        const int rows = is_a ? p.m - m0 : p.n - n0;
        off[l] = (uint32_t)min(r, rows - 1) * (uint32_t)p.kp + (uint32_t)(((lane & 3) ^ ring_sw(r)) * 16);
    }
    const int per = p.kp / BK;  // half-lines per plane row, even
    const int nh = per * out.npairs;
    const int8_t *src_a = nullptr, *src_b = nullptr;
    int iss = 0, pair = 0, wslot = 0;  // half-lines of the current planes issued, plane pair, slot to fill
    auto planes = [&](int i) {
        src_a = p.a + (int64_t)out.pairs[i].a * p.a_plane + (int64_t)m0 * p.kp;
        src_b = p.b + (int64_t)out.pairs[i].b * p.b_plane + (int64_t)n0 * p.kp;
    };
    auto load = [&](int l, int half, int slot) {
        __builtin_amdgcn_global_load_lds(
            (const void __attribute__((address_space(1)))*)((l < LPW / 2 ? src_a : src_b) + half * BK + off[l]),
            (void __attribute__((address_space(3)))*)(lds + slot + (wave + NW * l) * 1024), 16, 0, 0);
    };
    // operand `part` (0: A, 1: B) of a line's two halves, into the next two slots
    auto issue = [&](auto part) {
        const int s1 = wslot + CF::SLOT == CF::LDS ? 0 : wslot + CF::SLOT;
#pragma unroll
        for (int l = decltype(part)::value * LPW / 2; l < (decltype(part)::value + 1) * LPW / 2; ++l) {
            load(l, 0, wslot);
            load(l, 1, s1);
        }
    };
    using A = std::integral_constant<int, 0>;
    using B = std::integral_constant<int, 1>;
    // the next line, or the first of the next plane pair
    auto advance = [&]() {
        src_a += 2 * BK;
        src_b += 2 * BK;
        wslot += 2 * CF::SLOT;
        if (wslot >= CF::LDS) wslot -= CF::LDS;
        iss += 2;
        if (iss == per) {
            iss = 0;
            if (++pair < out.npairs) planes(pair);
        }
    };

    const int lr = lane & 15, lc = lane >> 4;
    const int fa0 = (wm0 + lr) * BK + ((lc ^ ring_sw(lr)) << 4);
    const int fb0 = BM * BK + (wn0 + lr) * BK + ((lc ^ ring_sw(lr)) << 4);
    struct Frag {
        v4i a[FM], b[FN];
    };
    auto read = [&](Frag& f, int slot) {
        const int8_t* base = lds + slot;
#pragma unroll
        for (int j = 0; j < FN; ++j) f.b[j] = *reinterpret_cast<const v4i*>(base + fb0 + j * 16 * BK);
#pragma unroll
        for (int i = 0; i < FM; ++i) f.a[i] = *reinterpret_cast<const v4i*>(base + fa0 + i * 16 * BK);
    };
    MF::acc_t acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = MF::zero();
    auto multiply = [&](const Frag& f) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[i][j] = MF::mma(f.a[i], f.b[j], acc[i][j]);
    };
    // every wave has read its fragments of the slot before, and every wave's
    // loads waited for so far are in LDS
    auto barrier = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };

    Frag f0, f1;
    if (nh > 0) {
        planes(0);
        issue(A{});
        issue(B{});
        advance();
        if (nh > 2) {
            issue(A{});
            issue(B{});
            advance();
            wait_vmcnt_max(2 * LPW);
        } else {
            wait_vmcnt_max(0);
        }
        barrier();
        read(f0, 0);
    }
    int rslot = CF::SLOT;  // slot of the next half-line's fragments
    auto next = [&]() { rslot = rslot + CF::SLOT == CF::LDS ? 0 : rslot + CF::SLOT; };
    // the reads first (the compiler keeps the direct loads, which write LDS, behind them)
    constexpr int kReads = FM + FN, kRest = (FM * FN - kReads) / (LPW + 1);
    auto schedule = [&](auto load_c) {
#pragma unroll
        for (int g = 0; g < kReads; ++g) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        if constexpr (decltype(load_c)::value) {
#pragma unroll
            for (int g = 0; g < LPW; ++g) {
                __builtin_amdgcn_sched_group_barrier(0x8, kRest, 0);
                __builtin_amdgcn_sched_group_barrier(0x20, 1, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto line = [&](auto load_c) {
        constexpr bool LOAD = decltype(load_c)::value;
        // half h (even): its line's other half is in LDS; the line after next is
        // loaded over the slots of halves h - 1 and h
        barrier();
        read(f1, rslot);
        if constexpr (LOAD) issue(A{});
        multiply(f0);
        schedule(load_c);
        next();
        // half h + 1: the next line has landed
        wait_vmcnt_max(LOAD ? LPW : 0);
        barrier();
        read(f0, rslot);  // (behind the last half a slot nobody writes, its values unused)
        if constexpr (LOAD) issue(B{});
        multiply(f1);
        schedule(load_c);
        next();
        if constexpr (LOAD) advance();
    };
    int h = 0;
    for (; h + 4 < nh; h += 2) line(std::true_type{});
    for (; h < nh; h += 2) line(std::false_type{});
    barrier();

    if (p.mode != 0) {
        i8_store<MF, FM, FN>(p, out, m0 + wm0, n0 + wn0, lane, [&](int i, int j, int r) { return (double)acc[i][j][r]; });
        return;
    }
    // u = y acc mod m: |y acc| < 2^40 is exact, and half a unit more keeps the
    // quotient's fraction in [1/2m, 1 - 1/2m], out of reach of its roundings.
    // The bytes go through LDS, so that a column's 256 rows are stored together.
    const double y = (double)out.y, md = (double)out.modulus, inv = out.inv_m, bias = 0.5 * out.inv_m;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            uint32_t word = 0;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const double v = y * (double)acc[i][j][r];
                word |= (uint32_t)__builtin_fma(-floor(__builtin_fma(v, inv, bias)), md, v) << (8 * r);
            }
            *reinterpret_cast<uint32_t*>(lds + (wn0 + j * 16 + lr) * CF::CST + wm0 + i * 16 + MF::group_row(lane, 0)) = word;
        }
    __syncthreads();
    uint8_t* u = p.u + (int64_t)blockIdx.z * p.u_plane;
    const int row = (tid & 31) * 8;
    if (m0 + row >= p.ldu) return;  // (ldu is a multiple of 4 at least: rows past it are not stored)
    for (int c = tid >> 5; c < BN && n0 + c < p.n; c += CF::NT / 32) {
        const uint2 w = *reinterpret_cast<const uint2*>(lds + c * CF::CST + row);
        uint8_t* d = u + (int64_t)(n0 + c) * p.ldu + m0 + row;
        *reinterpret_cast<uint32_t*>(d) = w.x;
        if (m0 + row + 4 < p.ldu) *reinterpret_cast<uint32_t*>(d + 4) = w.y;
    }
}

}  // namespace zg
