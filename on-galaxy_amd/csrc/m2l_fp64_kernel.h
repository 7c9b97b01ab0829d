// ============================================================================
// m2l_fp64_kernel.h -- M2L in FP64 on the matrix cores, one operator per set of
// mirrored offsets (M2LPlan of afmm_math.h).
//
//   L_t = sum_{c in V(t)} T[offset(t, c)] M_c  (AdaptiveFMM3D.hpp:82-86,
//   FmmExpansions3D.hpp:273-299)
//
// A slot is an offset with non-negative components on the reflected axes; the
// operators of its mirror images are D_m T D_m with diagonal signs. Per slot a
// target's up to four sources are combined by a Walsh-Hadamard transform (8
// additions per 4 sources and k step) and multiplied by T once: 84 products
// per target where its 189 offsets took one each. Bound by the matrix pipe:
// busy for 64% of the cycles at 1M bodies and p = 8, 1.08 of 1.58 ms at
// 2.2 GHz; the rest is gathers and transforms between the products. Time of
// the kernel with one product per offset and of this one, us: 16k Plummer p = 8
// 759 -> 420, 1M merger p = 8 2967 -> 1580, 300k p = 12 6935 -> 2900, 120k
// Hernquist p = 16 13292 -> 3100.
// ============================================================================
#pragma once

#include <stdexcept>

#include "m2l_common.h"

namespace afmm {
namespace {

template <int P>
__constant__ M2LPlan kPlan = make_m2l_plan(P);
template <int NX>
__constant__ M2LSymSlots<NX> kSymSlots = make_m2l_sym_slots<NX>();

// k steps per LDS chunk: the whole operator when two of it fit LDS (then one
// barrier per slot), else near-equal chunks of whole pairs, at most 60 KB.
constexpr int m2l_chunk_steps(int p) {
    const int nq = make_m2l_plan(p).nq, unit = 8 * m2l_step(p);
    if (2 * nq * unit <= 122 * 1024) return nq;
    const int most = 60 * 1024 / unit / 2 * 2, n = (nq + most - 1) / most;
    return ((nq + n - 1) / n + 1) / 2 * 2;
}

// The row blocks and quads of a role (of RS): near-equal runs of blocks, and
// each quad to the role with the least work so far (a block is four quads).
// Items are blocks (item < nb) and quads (nb + quad) of the plan, blocks first.
struct M2LRole {
    int nb = 0, n = 0;  // blocks, items
    signed char item[kPlanBlocks + kPlanQuads] = {};
    signed char turn[kPlanBlocks + kPlanQuads] = {};  // indices into item in the order of a step
};
constexpr M2LRole make_m2l_role(const M2LPlan& t, int rs, int role) {
    M2LRole r[4] = {};
    int cost[4] = {};
    for (int b = 0; b < t.nb; ++b) {
        const int k = b * rs / t.nb;
        r[k].item[r[k].n++] = (signed char)b;
        ++r[k].nb;
        cost[k] += 4;
    }
    for (int d = 0; d < t.nd; ++d) {
        int k = 0;
        for (int i = 1; i < rs; ++i)
            if (cost[i] < cost[k]) k = i;
        r[k].item[r[k].n++] = (signed char)(t.nb + d);
        ++cost[k];
    }
    // the order of a step: the quads spread between the blocks
    M2LRole x = r[role];
    int b = 0, d = x.nb, n = 0;
    while (b < x.nb || d < x.n)
        if (b < x.nb && (d >= x.n || b * (x.n - x.nb) <= (d - x.nb) * x.nb)) x.turn[n++] = (signed char)b++;
        else x.turn[n++] = (signed char)d++;
    return x;
}
constexpr int most_blocks(const M2LPlan& t, int rs) {
    int most = 0;
    for (int r = 0; r < rs; ++r) most = make_m2l_role(t, rs, r).nb > most ? make_m2l_role(t, rs, r).nb : most;
    return most;
}
constexpr int most_quads(const M2LPlan& t, int rs) {
    int most = 0;
    for (int r = 0; r < rs; ++r) {
        const M2LRole x = make_m2l_role(t, rs, r);
        most = x.n - x.nb > most ? x.n - x.nb : most;
    }
    return most;
}
template <int P, int RS>
struct M2LRoles {
    M2LRole r[RS];
    constexpr M2LRoles() : r{} {
        for (int k = 0; k < RS; ++k) r[k] = make_m2l_role(make_m2l_plan(P), RS, k);
    }
};
template <int P, int RS>
__constant__ M2LRoles<P, RS> kRoles = M2LRoles<P, RS>();

// Waves of a workgroup; its tile holds at most 16 kM2LWaves CB / RS targets.
constexpr int kM2LWaves = 8;
// Units of 16 bytes of an operator chunk per thread, and those it holds at once.
constexpr int m2l_stage_units(int p) {
    const int u = m2l_chunk_steps(p) * m2l_step(p) / 2, nt = kM2LWaves * 64;
    return (u + nt - 1) / nt;
}
constexpr int m2l_stage_regs(int p, int rs) { return rs > 1 ? m2l_stage_units(p) : (m2l_stage_units(p) + 1) / 2; }
// Pairs of k steps that a lane's source values are loaded ahead (a ring of
// registers): what the registers of a wave leave (256, or 128 with two
// workgroups per CU).
constexpr int m2l_depth(int p, int cb, int rs) {
    const M2LPlan t = make_m2l_plan(p);
    const int nm = 1 << m2l_axes(p);
    const int acc = cb * (8 * most_blocks(t, rs) + 2 * most_quads(t, rs));
    const int regs = m2l_workgroups(p) > 1 && rs <= 2 ? 96 : 200;
    const int left = (regs - acc - (4 + 3) * nm * cb - 4 * m2l_stage_regs(p, rs)) / (4 * nm * cb);
    const int d = left < 1 ? 1 : left > 4 ? 4 : left, np = (t.nq + 1) / 2;
    return d < np ? d : np;
}

// One workgroup per tile of targets of one octant group. A wave owns CB column
// blocks of 16 targets (the columns of v_mfma_f64_16x16x4_f64), or RS waves
// share one, each with its role's row blocks. The workgroup streams the
// operators of the slots present in its tile through LDS, double-buffered;
// each lane loads 16 bytes of every source D pairs of k steps ahead (four lanes
// one 64-byte run of a box; an absent source is the zero box np), combines
// them, passes the combinations through LDS into the matrix operand's lane
// order, and the wave runs the pair's matrix products. Loaded in that order
// directly, neighbouring lanes read different boxes, and the addresses of the
// 8-byte loads bound the kernel (39 cycles a load, 1.84 ms at 1M and p = 8).
// Operand layouts: 16x16x4: A[i][k] in lane i + 16 k, B[k][j]
// in lane j + 16 k, D[i][j] in lane j + 16 (i % 4), register i / 4; 4x4x4: the
// same B, A[i][k] in lanes i + 4 n + 16 k for n = 0..3 (its four column blocks
// take the same rows), D[i][j] in lane j + 16 i. Every row adds its
// slots and k steps in one order whatever the tile, CB and RS, and an absent
// source adds exact zeros: the same bits for all.
template <int P, int CB, int RS>
__global__ void __launch_bounds__(kM2LWaves * 64, 2 * (RS > 2 ? 1 : m2l_workgroups(P))) k_m2l_fp64(int np, int ntiles, const int* __restrict__ tstart,
                                                             const int* __restrict__ order,
                                                             const int* __restrict__ ic,
                                                             const int* __restrict__ srcT,
                                                             const int* __restrict__ present_g,
                                                             const double* __restrict__ A,
                                                             const double* __restrict__ Mp, double* __restrict__ L) {
    constexpr int S = nterms(P), NX = m2l_axes(P), NM = 1 << NX;
    constexpr M2LPlan PL = make_m2l_plan(P);
    constexpr int NQ = PL.nq, NB = PL.nb, QU = m2l_step(P), SP = m2l_pack(P);
    constexpr int NS = make_m2l_sym_slots<NX>().n;
    constexpr int GQ = m2l_chunk_steps(P), NC = (NQ + GQ - 1) / GQ;
    constexpr int NP = (NQ + 1) / 2, D = m2l_depth(P, CB, RS);
    constexpr int NPV = (NP + D - 1) / D * D;  // (pairs NP .. NPV - 1 do nothing)
    // the operator chunk goes to LDS through H registers of 16 bytes, in one or two halves
    constexpr int NT = kM2LWaves * 64, CHU = GQ * QU / 2, PER = m2l_stage_units(P), H = m2l_stage_regs(P, RS);
    constexpr int RBH = most_blocks(PL, RS), RDH = most_quads(PL, RS);
    static_assert(CB == 1 || RS == 1, "a wave owns several columns or shares one");
    __shared__ dbl2 abuf[2][CHU];
    __shared__ dbl2 turn[kM2LWaves][NM][64];  // per wave: from load order to operand order
    __shared__ unsigned char present[NS + 1];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int grp = wave / RS, role = wave % RS;
    const int j = lane & 15, kq = lane >> 4;        // operand order: column, k of a step
    const int dlane = (lane & 3) + 4 * kq;           // a quad's operand
    const int jl = lane >> 2, pl = lane & 3;         // load order
    const int put_at = 4 * jl + (pl ^ ((jl >> 2) & 3)), get_at = 4 * j + (kq ^ ((j >> 2) & 3));  // (spreads the banks)
    const int tile = xcd_item();
    if (tile >= ntiles) return;
    const int base = tstart[tile], end = tstart[tile + 1];
    // a tile's targets share their octant, hence the parities of their coordinates
    const int par = __builtin_amdgcn_readfirstlane(ic_parity(ic, order[base]));
    int rank[CB];  // of the target whose sources this lane loads (past the tile's end: its last one)
#pragma unroll
    for (int c = 0; c < CB; ++c) rank[c] = min(base + (grp * CB + c) * 16 + jl, end - 1);
    dbl4 acc[CB][RBH > 0 ? RBH : 1];
    double dacc[CB][RDH > 0 ? RDH : 1];
#pragma unroll
    for (int c = 0; c < CB; ++c) {
#pragma unroll
        for (int b = 0; b < RBH; ++b) acc[c][b] = dbl4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int r = 0; r < RDH; ++r) dacc[c][r] = 0.0;
    }
    for (int t = tid; t < NS; t += NT) present[t] = (unsigned char)present_g[(size_t)tile * NS + t];
    if (tid == 0) present[NS] = 1;  // sentinel
    __syncthreads();
    auto next_present = [&](int o) {
        ++o;
        while (!present[o]) ++o;
        return __builtin_amdgcn_readfirstlane(o);  // NS when none left
    };
    auto load_src = [&](int o, int (&src)[CB][NM]) {
        const short* rows = kSymSlots<NX>.row[par][o < NS ? o : 0];
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            const int* at = srcT + (size_t)(o < NS ? rows[m] : kSrcRows) * np;
#pragma unroll
            for (int c = 0; c < CB; ++c) src[c][m] = at[rank[c]];
        }
    };
    auto any_src = [&](const int (&src)[CB][NM]) {
        bool any = false;
#pragma unroll
        for (int c = 0; c < CB; ++c)
#pragma unroll
            for (int m = 0; m < NM; ++m) any |= src[c][m] != np;
        return __ballot(any) != 0ull;
    };
    // x[pair % D]: the values of a pair from every source
    dbl2 x[D][CB][NM];
    auto load_pair = [&](const int (&src)[CB][NM], auto tc) {
        constexpr int t = decltype(tc)::value;
#pragma unroll
        for (int c = 0; c < CB; ++c)
#pragma unroll
            for (int m = 0; m < NM; ++m)
                x[t % D][c][m] = *reinterpret_cast<const dbl2*>(Mp + (size_t)src[c][m] * SP + 8 * t + 2 * pl);
    };
    int o = next_present(-1), on;
    int scur[CB][NM], snext[CB][NM];
    bool has_cur, has_next;
    {
        const dbl2* a = reinterpret_cast<const dbl2*>(A + (size_t)min(o, NS - 1) * NQ * QU);
        for (int e = tid; e < CHU; e += NT) abuf[0][e] = a[e];
        load_src(o, scur);
        has_cur = any_src(scur);
        static_for<D>([&](auto t) { load_pair(scur, t); });
        on = o < NS ? next_present(o) : NS;
        load_src(on, snext);
    }
    __syncthreads();
    int buf = 0;
    // the k steps [T0, T1) of a chunk starting at step C0 (whole pairs), for one role
    auto products = [&](auto rc, auto cc, auto t0c, auto t1c) {
        constexpr int ROLE = decltype(rc)::value, C0 = decltype(cc)::value;
        constexpr int T0 = decltype(t0c)::value, T1 = decltype(t1c)::value;
        constexpr M2LRole R = make_m2l_role(PL, RS, ROLE);
        const double* ab = reinterpret_cast<const double*>(abuf[buf]);
        // the operator value of item k of the role at step q
        auto operand = [&](auto kc, int q) {
            constexpr int it = R.item[R.turn[decltype(kc)::value]];
            return ab[(q - C0) * QU + (it < NB ? it * 64 + lane : NB * 64 + (it - NB) * 16 + dlane)];
        };
        // operator values AD items ahead (over the steps T0 .. T1 - 1 as one sequence)
        constexpr int AD = 3, ITEMS = R.n * (T1 - T0);
        double ahead[AD];
        auto fetch_a = [&](auto gc) {
            constexpr int g = decltype(gc)::value;
            if constexpr (g < ITEMS) ahead[g % AD] = operand(std::integral_constant<int, g % (R.n > 0 ? R.n : 1)>{}, T0 + g / (R.n > 0 ? R.n : 1));
        };
        static_for<AD>(fetch_a);
        static_for<(T1 - T0 + 1) / 2>([&](auto tc) {
            constexpr int t = T0 / 2 + decltype(tc)::value;
            dbl2 w[CB][NM];
#pragma unroll
            for (int c = 0; c < CB; ++c) {
#pragma unroll
                for (int m = 0; m < NM; ++m) w[c][m] = x[t % D][c][m];
#pragma unroll
                for (int s = 1; s < NM; s <<= 1)
#pragma unroll
                    for (int m = 0; m < NM; ++m)
                        if (!(m & s)) {
                            const dbl2 u = w[c][m], v = w[c][m | s];
                            w[c][m] = u + v;
                            w[c][m | s] = u - v;
                        }
                // (a wave's LDS accesses complete in order)
#pragma unroll
                for (int m = 0; m < NM; ++m) turn[wave][m][put_at] = w[c][m];
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int m = 0; m < NM; ++m) w[c][m] = turn[wave][m][get_at];
                __builtin_amdgcn_wave_barrier();
            }
            if constexpr (t + D < NP) load_pair(scur, std::integral_constant<int, t + D>{});
            else if constexpr (t + D >= NPV) load_pair(snext, std::integral_constant<int, t + D - NPV>{});
            // the next slot's pairs that the idle pairs at the end would load
            if constexpr (t == NP - 1)
                static_for<NPV - NP>([&](auto v) {
                    load_pair(snext, std::integral_constant<int, NP + D - NPV + decltype(v)::value>{});
                });
            __builtin_amdgcn_sched_barrier(0);
            static_for<(2 * t + 1 < NQ ? 2 : 1)>([&](auto hc) {
                constexpr int h = decltype(hc)::value, q = 2 * t + h;
                static_for<R.n>([&](auto nc) {
                    constexpr int n = decltype(nc)::value, k = R.turn[n], it = R.item[k], g = (q - T0) * R.n + n;
                    constexpr int i = (it < NB ? PL.bcls[it] : PL.dcls[it < NB ? 0 : it - NB]) ^ PL.kcls[q];
                    const double a = ahead[g % AD];
                    fetch_a(std::integral_constant<int, g + AD>{});
#pragma unroll
                    for (int c = 0; c < CB; ++c) {
                        if constexpr (it < NB)
                            acc[c][k] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, w[c][i][h], acc[c][k], 0, 0, 0);
                        else
                            dacc[c][k - R.nb] =
                                __builtin_amdgcn_mfma_f64_4x4x4f64(a, w[c][i][h], dacc[c][k - R.nb], 0, 0, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);  // (keeps the loads where they are: registers)
                });
            });
        });
    };
    auto by_role = [&](auto cc, auto t0c, auto t1c) {
        static_assert(RS == 1 || RS == 2 || RS == 4, "row splits built");
        if constexpr (RS == 1) products(std::integral_constant<int, 0>{}, cc, t0c, t1c);
        else if constexpr (RS == 2) {
            if (role == 0) products(std::integral_constant<int, 0>{}, cc, t0c, t1c);
            else products(std::integral_constant<int, 1>{}, cc, t0c, t1c);
        } else {
            if (role == 0) products(std::integral_constant<int, 0>{}, cc, t0c, t1c);
            else if (role == 1) products(std::integral_constant<int, 1>{}, cc, t0c, t1c);
            else if (role == 2) products(std::integral_constant<int, 2>{}, cc, t0c, t1c);
            else products(std::integral_constant<int, 3>{}, cc, t0c, t1c);
        }
    };
    // chunk C of the current slot, staging the chunk after it
    auto chunk = [&](auto ci) {
        constexpr int C = decltype(ci)::value, C0 = C * GQ, C1 = C0 + GQ < NQ ? C0 + GQ : NQ;
        constexpr int CM = H < PER ? C0 + ((C1 - C0) / 2 + 1) / 2 * 2 : C1;
        constexpr int N0 = C + 1 < NC ? (C + 1) * GQ : 0;  // the staged chunk's steps
        constexpr int N1 = N0 + GQ < NQ ? N0 + GQ : NQ, UNITS = (N1 - N0) * QU / 2;
        const int so = C + 1 < NC ? o : min(on, NS - 1);  // (past the last slot: staged and not used)
        const dbl2* a = reinterpret_cast<const dbl2*>(A + ((size_t)so * NQ + N0) * QU);
        dbl2* dst = abuf[buf ^ 1];
        dbl2 pre[H];
        auto fetch = [&](auto h0) {
            static_for<H>([&](auto i) {
                constexpr int k = decltype(h0)::value + decltype(i)::value;
                if constexpr (k * NT < UNITS) pre[decltype(i)::value] = a[min(tid + NT * k, UNITS - 1)];
            });
        };
        auto put = [&](auto h0) {
            static_for<H>([&](auto i) {
                constexpr int k = decltype(h0)::value + decltype(i)::value;
                if constexpr (k * NT < UNITS) dst[min(tid + NT * k, UNITS - 1)] = pre[decltype(i)::value];
            });
        };
        constexpr std::integral_constant<int, 0> first{};
        constexpr std::integral_constant<int, H> second{};
        constexpr std::integral_constant<int, C0> c0{};
        constexpr std::integral_constant<int, CM> cm{};
        constexpr std::integral_constant<int, C1> c1{};
        fetch(first);
        if (has_cur) by_role(c0, c0, cm);
        put(first);
        if constexpr (H < PER) {
            fetch(second);
            if (has_cur) by_role(c0, cm, c1);
            put(second);
        }
        __syncthreads();
        buf ^= 1;
    };
    while (o < NS) {
        has_next = any_src(snext);
        static_for<NC>(chunk);
        if (!has_cur) static_for<D>([&](auto t) { load_pair(snext, t); });
        o = on;
        has_cur = has_next;
#pragma unroll
        for (int c = 0; c < CB; ++c)
#pragma unroll
            for (int m = 0; m < NM; ++m) scur[c][m] = snext[c][m];
        on = o < NS ? next_present(o) : NS;
        load_src(on, snext);
    }
    const M2LRole& mine = kRoles<P, RS>.r[role];
#pragma unroll
    for (int c = 0; c < CB; ++c) {
        const int at = base + (grp * CB + c) * 16 + j;
        if (at >= end) continue;
        double* __restrict__ out = L + (size_t)order[at] * S;
#pragma unroll
        for (int b = 0; b < RBH; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = b < mine.nb ? kPlan<P>.brow[16 * mine.item[b] + kq + 4 * r] : -1;
                if (row >= 0) out[row] = acc[c][b][r];
            }
#pragma unroll
        for (int d = 0; d < RDH; ++d) {
            const int row = mine.nb + d < mine.n ? kPlan<P>.drow[4 * (mine.item[mine.nb + d] - NB) + kq] : -1;
            if (row >= 0) out[row] = dacc[c][d];
        }
    }
}

}  // namespace

// Instantiated by the source files that include this header, a few orders each.
template <int P>
void m2l_fp64_launch(hipStream_t s, const M2LArgs& a) {
    const dim3 g(xcd_grid(a.ntiles)), b(kM2LWaves * 64);
    // Tiles of at most 64 and 32 targets share a column's rows over two and four
    // waves (shorter chains: the tree is too small to fill the CUs).
#define AFMM_M2L(CB, RS)                                                                                              \
    hipLaunchKernelGGL((k_m2l_fp64<P, CB, RS>), g, b, 0, s, a.np, a.ntiles, a.tstart, a.order, a.ic, a.srcT, a.present, \
                       a.A, a.Mp, a.L)
    if (a.tile <= 32) AFMM_M2L(1, 4);
    else if (a.tile <= 64) AFMM_M2L(1, 2);
    else if (a.tile <= 128) AFMM_M2L(1, 1);
    else if constexpr (m2l_columns(P) == 2) AFMM_M2L(2, 1);
    else throw std::runtime_error("M2L tile beyond the workgroup");
#undef AFMM_M2L
}

}  // namespace afmm
