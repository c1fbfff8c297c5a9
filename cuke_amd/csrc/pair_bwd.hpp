// Gradient tiles that evaluate every pair once (TransE, RotatE, TransH L1): included by score_bwd.hip.
//
// A workgroup owns TO negatives x 32 columns of one chunk and walks the chunk's positives (a range of them, `splits` workgroups
// share them), staged kKL at a time with their coefficients.  A thread holds four columns of RO negatives; per positive it adds
// the pair's gradient element to the negative's sum (registers) AND to the positive's, which the eight lane groups of a wave add up by
// lane exchanges and the waves through LDS.  bwd_tile_kernel's two orientations form the same element twice, and with it
// what the element costs: a sign or a reciprocal square root.
// The positives' sums are complete over the TO negatives of the workgroup only: one plane of [B, d] rows per tile of a launch's negatives,
// added up by bwd_pos_kernel; the negatives' rows likewise have one plane per range of positives, added up as the
// segmented reduction loads them.  Batches of many tiles take several launches, the later ones of which add to the planes.
#pragma once

#include <cmath>

#include "inspector_mid.hpp"
#include "tile_common.hpp"

namespace kge {

constexpr int kPairCols = 32;   // columns of the row per workgroup
constexpr int kPairKL = 16;     // positives staged per step
constexpr int kPairPitch = kPairCols + 4;
constexpr int kPairRO = 4, kPairWaves = 4;
constexpr int kPairOwners = kPairWaves * 8 * kPairRO;  // negatives of a workgroup whose waves all hold different ones

template <int MODEL>
struct PairShape {
    static constexpr bool kTH = MODEL == KGE_TRANSH;
    static constexpr int NPN = MODEL == KGE_ROTATE ? 2 : 1;  // planes of a negative's row and of its sums
    static constexpr int NPL = kTH ? 2 : NPN;                // planes of a positive's (TransH: the query and w) and of its sums
    static constexpr int NC = kTH ? 3 : 1;                   // coefficients of a pair
    static constexpr int PG = kPairOwners + 4;
    static constexpr int kRowFloats = NPL * kPairKL * kPairPitch, kCoefFloats = NC * kPairKL * PG;
    static constexpr int kSumFloats = kPairKL * kPairWaves * NPL * kPairCols;
    static constexpr int kLdsFloats = kRowFloats + kCoefFloats + kSumFloats + (kTH ? kPairKL : 0);
};

struct PairPlan {
    int phases;   // 1, 2 or 4: waves of a workgroup that share its negatives and take turns at the positives
    int tiles;    // tiles of negatives
    int planes;   // planes of the positives' sums: tiles of a launch
    int splits;   // ranges of positives: planes of the negatives' rows
    int per;      // positives of a range, a multiple of the step
};

struct PairArgs {
    PairPlan plan;
    int tile0;                 // first tile of the launch
    float *g0, *g1;            // [planes][B, d]; g1: TransH, the sums for w
    int64_t gplane;            // B * d
    float *occ_neg, *more_neg; // plane 0 of the negatives' rows [n_chunks * N, d]; planes 1 ... splits - 1
    int64_t nplane;            // n_chunks * N * d
};

__device__ __forceinline__ void swap_halves(float &a, float &b)  // upper 32 lanes of a <-> lower 32 lanes of b
{
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]), b = __uint_as_float(r[1]);
}
__device__ __forceinline__ void swap_rows(float &a, float &b)  // odd rows of 16 lanes of a <-> even rows of b
{
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]), b = __uint_as_float(r[1]);
}
__device__ __forceinline__ float add_ror8(float v)  // v + the value eight lanes on within the row of 16
{
    return v + __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), 0x128, 0xf, 0xf, true));
}

// Bound by vector-ALU issue (per wave instruction 2 clocks for subtractions and multiply-adds, 4 for the sign's v_med3, 8 for
// v_rsq): a RotatE element 26 clocks where two orientations took 52, a TransE L1 element 10 for 16, and two to four for the exchanges.
//   Gradient tiles, us, both orientations -> every pair once:  RotatE 1024 x 256 negatives x 1000 72 -> 55, 8192 x 256 x 500 in chunks of 1024
//   295 -> 184, 4278 x 300 x 426 in chunks of 31 245 -> 128;  TransE L1 30000 x 200 x 150 230 -> 158, 4096 x 1024 x 150 136 -> 87.
template <int MODEL, int P, int PH>
__global__ __launch_bounds__(kPairWaves *kWave, MODEL == KGE_TRANSE ? 4 : 3) void bwd_pair_kernel(TileArgs a, PairArgs pa, FusedInsp fi)
{
    using S = PairShape<MODEL>;
    constexpr bool kRot = MODEL == KGE_ROTATE, kTH = S::kTH, kSc = !kRot && P == 1, kL2 = !kRot && P == 2;
    static_assert(!kTH || P == 1, "TransH: L1 only");
    constexpr int RO = kPairRO, WAVES = kPairWaves, NPL = S::NPL, NPN = S::NPN, NC = S::NC, PG = S::PG, KL = kPairKL, TH = WAVES * kWave;
    constexpr int wo = WAVES / PH, TO = wo * 8 * RO;   // waves of different negatives; negatives of the tile
    constexpr int CPT = (KL * TO / 4 + TH - 1) / TH;   // coefficient quads per thread
    constexpr int NRAW = query_raw_count<MODEL>();
    extern __shared__ __align__(16) char dyn_smem[];
    if (fused_insp_block(fi, reinterpret_cast<uint32_t *>(dyn_smem))) return;
    float(*sL)[KL][kPairPitch] = reinterpret_cast<float(*)[KL][kPairPitch]>(dyn_smem);
    float(*sG)[KL][PG] = reinterpret_cast<float(*)[KL][PG]>(dyn_smem + sizeof(float) * S::kRowFloats);
    float *sR = reinterpret_cast<float *>(dyn_smem) + S::kRowFloats + S::kCoefFloats, *sA = sR + S::kSumFloats;

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), own_wave = wave % wo, phase = wave / wo;
    const int tx = lane & 7, ty = own_wave * 8 + (lane >> 3);
    const int d = a.d, half = d >> 1, klen = pair_len<MODEL>(d);
    int c, tile_y, tile_x;
    if (!xcd_tile((int)blockIdx.x - fi.blocks, (klen + kPairCols - 1) / kPairCols, pa.plan.planes * pa.plan.splits, a.n_chunks, c, tile_y, tile_x)) return;
    const int plane = tile_y / pa.plan.splits, split = tile_y - plane * pa.plan.splits;
    if (pa.tile0 + plane >= pa.plan.tiles) return;                        // (the last of several launches)
    const int k0 = (pa.tile0 + plane) * TO;                               // first negative
    const int b0 = split * pa.plan.per, b1 = min(a.C, b0 + pa.plan.per);  // positives of the chunk
    // (a quad of columns that would run past the row's end is moved back to end with it: see bwd_tile_body)
    const int lcol = tile_x * kPairCols + tx * 4, col = min(lcol, klen - 4), skip = lcol - col;

    // ---- negatives: registers ------------------------------------------------------------
    float4 own[NPN][RO], acc[NPN][RO];
#pragma unroll
    for (int o = 0; o < RO; ++o) {
        const float *pt = a.ent + a.neg[(int64_t)c * a.N + min(k0 + ty * RO + o, a.N - 1)] * (int64_t)d;
#pragma unroll
        for (int q = 0; q < NPN; ++q) {
            own[q][o] = load_quad(pt + q * half + col);
            acc[q][o] = zero4();
        }
    }
#pragma unroll
    for (int o = 0; o < RO; ++o)
#pragma unroll
        for (int q = 0; q < NPN; ++q) {
            if (k0 + ty * RO + o >= a.N) own[q][o] = zero4();
            if constexpr (kSc) own[q][o] = scale4(own[q][o], kSgnScale);
        }

    // ---- staging: rows by the first 8 KL threads, coefficients by all; requested a step ahead, ids two ------------
    const int srow = tid >> 3;
    const bool stager = tid < KL * 8;
    int64_t ih = 0, ir = 0;
    float4 rraw[NRAW], craw[CPT], sraw[kL2 ? CPT : 1], c1raw[kTH ? CPT : 1], c2raw[kTH ? CPT : 1];
    float ral = 0.0f;  // TransH: w . x of the staged positive
    auto load_idx = [&](int l0) {
        if (kRot || !stager) return;
        const int64_t b = (int64_t)c * a.C + min(l0 + srow, a.C - 1);
        ih = a.h[b], ir = a.r[b];
    };
    auto load_step = [&](auto stag, int l0) {
        constexpr int kEdge = decltype(stag)::value;  // 1: a quad of coefficients may straddle its row's end (see bwd_tile_body); 2: rows of fewer than four
        if (stager) {
            const float *pq = kRot ? a.query + ((int64_t)c * a.C + min(l0 + srow, a.C - 1)) * d : nullptr;
            load_query_raw<MODEL, true>(a.ent + ih * (int64_t)d, a.rel + ir * (int64_t)a.rel_dim, kTH ? a.aux + ir * (int64_t)d : nullptr, pq, col, klen, half, rraw);
            if constexpr (kTH) ral = a.side_pos[(int64_t)c * a.C + min(l0 + srow, a.C - 1)];
        }
        auto ld = [](const float *p, int kl, int lim) {
            if constexpr (kEdge == 1) return shift_quad(ld4_raw<true>(p, kl, lim), kl + 4 - lim);
            else return ld4_whole<kEdge == 0>(p, kl, lim);
        };
#pragma unroll
        for (int s = 0; s < CPT; ++s) {
            const int f = tid + TH * s, lrow = f / (TO / 4), kl = k0 + (f % (TO / 4)) * 4, bl = l0 + lrow;
            const bool inside = lrow < KL && bl < b1;
            const int64_t off = ((int64_t)c * a.C + (inside ? bl : 0)) * a.N;
            craw[s] = ld(a.dneg + off, kl, inside ? a.N : 0);
            if constexpr (kL2) sraw[s] = ld(a.sneg + off, kl, inside ? a.N : 0);
            if constexpr (kTH) {
                c1raw[s] = ld(a.side_neg + off, kl, inside ? a.N : 0);
                c2raw[s] = ld(a.side_neg + a.plane + off, kl, inside ? a.N : 0);
            }
        }
    };
    auto load_rows = [&](int l0) {
        if (a.N < 4) return load_step(std::integral_constant<int, 2>{}, l0);  // uniform
        if ((a.N & 3) && k0 + TO > a.N) return load_step(std::integral_constant<int, 1>{}, l0);
        load_step(std::integral_constant<int, 0>{}, l0);
    };
    auto store_step = [&](int l0) {
        if (stager) {
            float4 q0, q1;
            combine_query<MODEL, true>(rraw, ral, col, l0 + srow < b1 ? klen : 0, half, a.rsign, q0, q1);
            *reinterpret_cast<float4 *>(&sL[0][srow][tx * 4]) = kSc ? scale4(q0, kSgnScale) : q0;
            if constexpr (NPL == 2) *reinterpret_cast<float4 *>(&sL[1][srow][tx * 4]) = kSc ? scale4(q1, kSgnScale) : q1;
            if constexpr (kTH) {
                if (tx == 0) sA[srow] = ral;
            }
        }
#pragma unroll
        for (int s = 0; s < CPT; ++s) {
            const int f = tid + TH * s, lrow = f / (TO / 4);
            if (lrow >= KL) continue;
            float4 g = craw[s];
            if constexpr (kL2) {
                const float4 sc = sraw[s];
                g.x = sc.x > 0.0f ? g.x / sc.x : 0.0f;
                g.y = sc.y > 0.0f ? g.y / sc.y : 0.0f;
                g.z = sc.z > 0.0f ? g.z / sc.z : 0.0f;
                g.w = sc.w > 0.0f ? g.w / sc.w : 0.0f;
            }
            *reinterpret_cast<float4 *>(&sG[0][lrow][(f % (TO / 4)) * 4]) = g;
            if constexpr (kTH) {
                *reinterpret_cast<float4 *>(&sG[1][lrow][(f % (TO / 4)) * 4]) = c1raw[s];
                *reinterpret_cast<float4 *>(&sG[NC - 1][lrow][(f % (TO / 4)) * 4]) = mul4(scale4(g, -kSgnUnscale), c2raw[s]);  // multiplies scaled rows
            }
        }
    };

    load_idx(b0);
    load_rows(b0);
    load_idx(b0 + KL);
#pragma unroll 1
    for (int l0 = b0; l0 < b1; l0 += KL) {
        store_step(l0);
        __syncthreads();
        if (l0 + KL < b1) {
            load_rows(l0 + KL);
            load_idx(l0 + 2 * KL);
        }
        __builtin_amdgcn_sched_barrier(0);
        float4 sacc[NPN][RO];  // (a step's sums of their own: rounding grows with the steps, not the positives)
#pragma unroll
        for (int q = 0; q < NPN; ++q)
#pragma unroll
            for (int o = 0; o < RO; ++o) sacc[q][o] = zero4();
        // (TransH: the negatives' sums and those for w are formed with the opposite sign, which no operand has to carry, and change it when they leave)
        // (unrolled, the exchanges' registers and the next positive's operands spill)
#pragma unroll 1
        for (int l = phase; l < KL; l += PH) {
            float lv[NPL][4], sum[NPL][4];
#pragma unroll
            for (int q = 0; q < NPL; ++q) {
                const float4 v = *reinterpret_cast<const float4 *>(&sL[q][l][tx * 4]);
                lv[q][0] = v.x, lv[q][1] = v.y, lv[q][2] = v.z, lv[q][3] = v.w;
                sum[q][0] = sum[q][1] = sum[q][2] = sum[q][3] = 0.0f;
            }
            const float4 cf = *reinterpret_cast<const float4 *>(&sG[0][l][ty * RO]);
            float4 cp = zero4(), ep = zero4();
            float al = 0.0f;
            if constexpr (kTH) {
                cp = *reinterpret_cast<const float4 *>(&sG[1][l][ty * RO]), ep = *reinterpret_cast<const float4 *>(&sG[NC - 1][l][ty * RO]);
                al = sA[l];
            }
#pragma unroll
            for (int o = 0; o < RO; ++o) {
                const float g = reinterpret_cast<const float *>(&cf)[o];
                const float *t0 = reinterpret_cast<const float *>(&own[0][o]), *t1 = reinterpret_cast<const float *>(&own[NPN - 1][o]);
                float *n0 = reinterpret_cast<float *>(&sacc[0][o]), *n1 = reinterpret_cast<float *>(&sacc[NPN - 1][o]);
                const float cc = reinterpret_cast<const float *>(&cp)[o], ee = reinterpret_cast<const float *>(&ep)[o];
                const float gk = (al - cc) * g;  // times the sign: the pair's w . (x - t') part of minus w's gradient
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if constexpr (kRot) {
                        const float ur = lv[0][e] - t0[e], ui = lv[1][e] - t1[e];
                        // (the 1e-37: see bwd_tile_body)
                        const float k = g * __builtin_amdgcn_rsqf(fmaf(ur, ur, fmaf(ui, ui, 1e-37f)));
                        n0[e] = fmaf(k, ur, n0[e]), n1[e] = fmaf(k, ui, n1[e]);
                        sum[0][e] = fmaf(-k, ur, sum[0][e]), sum[1][e] = fmaf(-k, ui, sum[1][e]);
                    } else if constexpr (kTH) {
                        const float s = sgn_of_scaled(fmaf(cc, lv[1][e], lv[0][e] - t0[e]));
                        sum[0][e] = fmaf(g, s, sum[0][e]);
                        sum[1][e] = fmaf(ee, t0[e], fmaf(gk, s, sum[1][e]));
                        n0[e] = fmaf(ee, lv[1][e], fmaf(g, s, n0[e]));
                    } else {
                        const float u = lv[0][e] - t0[e];  // (P == 1: times 2^100)
                        const float s = P == 1 ? sgn_of_scaled(u) : u;
                        sum[0][e] = fmaf(g, s, sum[0][e]);
                        n0[e] = fmaf(-g, s, n0[e]);
                    }
                }
            }
            // The wave's eight lane groups: the values leave pairwise, so that each exchange halves what is carried.  A lane ends with column
            // 4 tx + i of one plane.
            float *red = sR + (l * WAVES + own_wave) * (NPL * kPairCols);
            const int rho = (lane >> 4) & 1, beta = (lane >> 3) & 1, hi = lane >> 5;
            if constexpr (NPL == 2) {
                float w[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    swap_halves(sum[0][i], sum[1][i]);
                    w[i] = sum[0][i] + sum[1][i];
                }
                swap_rows(w[0], w[2]);
                swap_rows(w[1], w[3]);
                const float y0 = add_ror8(w[0] + w[2]), y1 = add_ror8(w[1] + w[3]);
                red[hi * kPairCols + tx * 4 + 2 * rho + beta] = beta ? y1 : y0;
            } else {
                swap_halves(sum[0][0], sum[0][2]);
                swap_halves(sum[0][1], sum[0][3]);
                float z0 = sum[0][0] + sum[0][2], z1 = sum[0][1] + sum[0][3];
                swap_rows(z0, z1);
                const float y = add_ror8(z0 + z1);
                if (beta == 0) red[tx * 4 + 2 * hi + rho] = y;
            }
        }
#pragma unroll
        for (int q = 0; q < NPN; ++q)
#pragma unroll
            for (int o = 0; o < RO; ++o) acc[q][o] = add4(acc[q][o], sacc[q][o]);
        __syncthreads();
        // the waves' sums of this step's positives
#pragma unroll
        for (int s = 0; s < KL * NPL * kPairCols / TH; ++s) {
            const int v = tid + TH * s, l = v / (NPL * kPairCols), pc = v % (NPL * kPairCols), lc = pc % kPairCols;
            float x = sR[l * WAVES * (NPL * kPairCols) + pc];
#pragma unroll
            for (int w = 1; w < wo; ++w) x += sR[(l * WAVES + w) * (NPL * kPairCols) + pc];
            if (kTH && pc >= kPairCols) x = -x;
            const int jl = tile_x * kPairCols + (lc & ~3), j = min(jl, klen - 4);
            if (l0 + l < b1 && (lc & 3) >= jl - j) {
                float *to = (kTH && pc >= kPairCols ? pa.g1 : pa.g0) + plane * pa.gplane + ((int64_t)c * a.C + l0 + l) * d + (kRot && pc >= kPairCols ? half : 0) + j + (lc & 3);
                if (pa.tile0 > 0) x += *to;  // uniform
                *to = x;
            }
        }
    }

    if constexpr (PH > 1) {  // the phases' sums of the same negatives
        __syncthreads();
        float4 *sS = reinterpret_cast<float4 *>(dyn_smem);
        static_assert(sizeof(float4) * NPN * RO * TH * 3 / 4 <= sizeof(float) * S::kLdsFloats, "three of four phases pass through LDS");
        constexpr int slots = wo * kWave;
        const int slot = own_wave * kWave + lane;
        if (phase > 0) {
#pragma unroll
            for (int q = 0; q < NPN; ++q)
#pragma unroll
                for (int o = 0; o < RO; ++o) sS[((phase - 1) * NPN * RO + q * RO + o) * slots + slot] = acc[q][o];
        }
        __syncthreads();
        if (phase > 0) return;
        for (int p = 1; p < PH; ++p)
#pragma unroll
            for (int q = 0; q < NPN; ++q)
#pragma unroll
                for (int o = 0; o < RO; ++o) acc[q][o] = add4(acc[q][o], sS[((p - 1) * NPN * RO + q * RO + o) * slots + slot]);
    }
#pragma unroll
    for (int o = 0; o < RO; ++o) {
        const int kl = k0 + ty * RO + o;
        if (kl >= a.N) continue;
        float *dst = (split ? pa.more_neg + (split - 1) * pa.nplane : pa.occ_neg) + ((int64_t)c * a.N + kl) * d;
#pragma unroll
        for (int q = 0; q < NPN; ++q) {
            float *p = dst + q * half + col;
            const float4 v = kTH ? scale4(acc[q][o], -1.0f) : acc[q][o];
            if (skip == 0) {
                store_quad(p, v);
            } else {
                if (skip <= 1) p[1] = v.y;
                if (skip <= 2) p[2] = v.z;
                if (skip <= 3) p[3] = v.w;
            }
        }
    }
}

// Bytes of planes that a batch may have whatever its size (a larger one: as many again as it takes without them).
constexpr int64_t kPairRoom = 512 << 20;

inline PairPlan cut_pairs(int ph, int64_t tiles, int64_t planes, int64_t C, int64_t splits)
{
    const int64_t per = ceil_div(ceil_div(C, kPairKL), splits) * kPairKL;
    return PairPlan{ph, (int)tiles, (int)planes, (int)ceil_div(C, per), (int)per};
}

// A plan whose planes take no more than `room` bytes beyond the first of either side: fewer ranges, and the tiles in launches of `planes`
// each, by the rounds of workgroups that all launches take together (`resident` at a time; a round that is not full counts as 0.45 of one
// and the rest by its share, a launch 0.2 of one beside).  Both orientations / every plane at once / at most 512 MB of planes, tiles with the per-positive
// kernel and the reductions:
//   RotatE 1024 x 40943 negatives x 1000, one chunk     222 MB 14.20 ms    2347 MB 7.10 ms   734 MB 7.36 ms
//   RotatE 8192 x 8192 x 1000                           176    13.43       2470   10.18      569   11.99
//   RotatE 4096 x 14951 x 400                            57     5.73        985    4.19      473    4.60
//   TransE L1 4096 x 14951 x 400                         61     3.41        989    2.78      478    3.03
//   TransE L1 8192 x 4096 x 400 in chunks of 1024       128     1.67        796    1.56      639    1.53
// (256 MB: 7.96, 16.98, 5.05, 3.39 and 1.58 ms.  The planes' tiles taken one after the other by a workgroup: 20 registers more are spilled.)
inline PairPlan shrink_pairs(const PairPlan &full, int64_t C, int64_t cols, int64_t resident, int64_t plane_bytes, int64_t range_bytes, int64_t room)
{
    PairPlan best = cut_pairs(full.phases, full.tiles, 1, C, 1);
    double least = -1.0;
    for (int64_t launches = 1; launches <= full.tiles; launches = launches < 16 ? launches + 1 : 2 * launches) {
        const int64_t planes = ceil_div(full.tiles, launches);
        for (int64_t splits = 1; splits <= full.splits; splits = splits < 8 ? splits + 1 : splits + splits / 4) {
            const PairPlan p = cut_pairs(full.phases, full.tiles, planes, C, splits);
            if ((planes - 1) * plane_bytes + (p.splits - 1) * range_bytes > room) break;
            const double rounds = (double)(cols * planes * p.splits) / (double)resident, whole = floor(rounds), part = rounds - whole;
            const double cost = (double)(ceil_div(full.tiles, planes) * p.per) * (0.2 + whole + (whole < 1.0 ? 1.0 : (part > 0.0 ? 0.45 + 0.55 * part : 0.0)));
            if (least < 0.0 || cost < least) least = cost, best = p;
        }
    }
    return best;
}

// Whether a batch's gradient tiles evaluate every pair once, and how they are cut.  Both ways timed over 200 random shapes (256 ... 16384
// positives, chunks and negatives 16 ... 1024, widths 48 ... 1000; tiles, per-positive kernel and reductions together).
//   RotatE: always; 0.73 of the time in the mean, 1.06 at worst (874 x 77 negatives x 322 in chunks of 38).
//   TransE L1: 0.87 in the mean by the rule below.  A thread of the other tiles walks the longer side of a chunk; from 160 on that walk costs a
//   small batch more than the extra planes do.  A batch that fills the chip goes by the padded pairs of both forms.
//   TransH L1: a pair here is 10.3 vector instructions an element where both orientations take 12.6, and there are two planes a tile, so it pays where the
//   other tiles walk a long side with few workgroups, or pad.  By the walk times the 768 resident workgroups over the launch's own, and the
//   padded pairs of both forms, over 220 shapes of the same ranges: 0.87 in the mean, 1.03 at worst (always: 0.855 and 1.22).  Backward pass, us: 969 x 147
//   negatives x 96 in one chunk 102 -> 53, 1482 x 18 x 840 in chunks of 741 107 -> 54, 8575 x 222 x 280 in chunks of 25 397 -> 304; left as they
//   are 8192 x 256 x 200 in chunks of 256 (157, here 172) and 16384 x 1024 x 400 (1745, here 1793: 420 MB of planes).
//   TransE L2, where differences are summed (launch_tiles): no sign to save, so only the walk counts: 0.83 from 280 on, 1.0 below.
inline bool plan_pairs(const kge_tables *tab, const kge_batch *bat, int64_t room, PairPlan *out)
{
    if (!bat->neg || bat->chunk <= 0 || bat->n_neg <= 0 || bat->batch < bat->chunk || !rows_by_quads(tab)) return false;  // (rows by quads)
    if (tab->model != KGE_TRANSE && tab->model != KGE_ROTATE && !(tab->model == KGE_TRANSH && tab->norm_p == 1)) return false;
    const bool th = tab->model == KGE_TRANSH;
    const int64_t n_chunks = bat->batch / bat->chunk, C = bat->chunk, N = bat->n_neg, klen = tab->model == KGE_ROTATE ? tab->dim / 2 : tab->dim;
    const int64_t cols = ceil_div(klen, kPairCols) * n_chunks, steps = ceil_div(C, kPairKL), longer = C > N ? C : N;
    // Negatives of a workgroup: 128, or 64 / 32 by waves in two / four phases (5 / 20 % slower per pair), by what the last tile wastes and
    // what the planes cost (a plane of a batch beyond the caches as much as 17 negatives, else 6).  A launch that cannot fill the chip takes smaller ones.
    const int64_t plane = (bat->batch * tab->dim >= 4000000 ? 17 : 6) * (th ? 2 : 1);
    auto cost = [&](int ph) { return ceil_div(N, kPairOwners / ph) * (kPairOwners / ph * (ph == 1 ? 100 : ph == 2 ? 105 : 120) + plane * 100); };
    int ph = cost(1) <= cost(2) && cost(1) <= cost(4) ? 1 : (cost(2) <= cost(4) ? 2 : 4);
    while (ph < 4 && cols * ceil_div(N, kPairOwners / ph) * steps < 384) ph *= 2;
    const int64_t tiles = ceil_div(N, kPairOwners / ph);
    // Ranges of positives: 640 workgroups, and of long chunks at most 192 positives each (up to eight ranges).  RotatE 1024 x 256 x 1000, 128
    // workgroups a range: 2 / 4 / 6 / 8 ranges 71 / 57 / 60 / 55 us, and the reduction 2 us a plane.  A wave of the reduction reads its rows'
    // planes one after the other, 0.4 us each, a step takes 1.8 to 4.5 us: at most 2.5 times the root of the steps (TransE L1 16384 x 16
    // negatives x 96 in one chunk, 16 / 32 / 64 / 128 / 205 ranges: 149 / 104 / 91 / 105 / 128 us with the reduction).
    int64_t splits = ceil_div(640, cols * tiles);
    const int64_t by_length = ceil_div(C, 192) < 8 ? ceil_div(C, 192) : 8;
    splits = splits > by_length ? splits : by_length;
    const int64_t most = (int64_t)(2.5 * sqrt((double)steps)) + 1;
    splits = splits < most ? splits : most;
    splits = splits < steps ? splits : steps;
    *out = cut_pairs(ph, tiles, tiles, C, splits);
    const int64_t plane_bytes = 4 * bat->batch * tab->dim * (th ? 2 : 1), range_bytes = 4 * n_chunks * N * tab->dim;
    if ((tiles - 1) * plane_bytes + (out->splits - 1) * range_bytes > room)
        *out = shrink_pairs(*out, C, cols, tab->model == KGE_TRANSE ? 1024 : 768, plane_bytes, range_bytes, room);
    if (tab->model == KGE_ROTATE) return true;
    if (tab->norm_p == 2) return longer >= 280 && !transe_by_products(tab->dim, C, N, n_chunks);
    // clocks per wave: a padded pair of the other tiles 9.5 per orientation, one here 16
    const int64_t gx = ceil_div(klen, kTI), big = gx * (ceil_div(C, 64) + ceil_div(N, 64)) * n_chunks, to = big >= 1024 ? 64 : (big >= 512 ? 32 : 16);
    const double padded = (double)(ceil_div(C, to) * to * ceil_div(N, 32) * 32 + ceil_div(N, to) * to * ceil_div(C, 32) * 32);
    const double both = 9.5 * (double)(gx * kTI * n_chunks) * padded;
    if (th) {
        const int64_t wgs = gx * (ceil_div(C, to) + ceil_div(N, to)) * n_chunks, quarters = to == 64 && narrow_cols((int)klen) ? 4 * (klen / kTI) + 1 : 4 * gx;
        const double old_pairs = (double)(quarters * (kTI / 4) * n_chunks) * padded;
        const double pairs = (double)(cols * kPairCols * tiles) * ((double)(steps * kPairKL) * (kPairOwners / ph) * (ph == 1 ? 1.0 : ph == 2 ? 1.05 : 1.2) + 2.0 * (double)(plane * C));
        const double walk = 768.0 * (double)longer / (double)wgs, ratio = pairs / old_pairs;
        return walk > 620.0 || ratio < 0.5 || (walk > 100.0 && ratio < 0.6);
    }
    const double once = 16.0 * (double)(cols * kPairCols) * (double)(steps * kPairKL * (tiles * kPairOwners / ph) + plane * tiles * C);
    const bool fills = both > 1.5e10;  // (about 100 us)
    return once < both * (longer < 160 ? 0.8 : (fills ? 0.95 : 1.2));
}

template <int MODEL, int P>
static int launch_pairs(const TileArgs &a, PairArgs pa, const FusedInsp &fi, hipStream_t st)
{
    const int klen = MODEL == KGE_ROTATE ? a.d / 2 : a.d;
    const unsigned tiles = xcd_grid(ceil_div(klen, kPairCols), (int64_t)pa.plan.planes * pa.plan.splits, a.n_chunks);
    const auto kernel = pa.plan.phases == 1 ? bwd_pair_kernel<MODEL, P, 1> : (pa.plan.phases == 2 ? bwd_pair_kernel<MODEL, P, 2> : bwd_pair_kernel<MODEL, P, 4>);
    for (pa.tile0 = 0; pa.tile0 < pa.plan.tiles; pa.tile0 += pa.plan.planes) {
        const FusedInsp f = pa.tile0 == 0 ? fi : FusedInsp{};  // (the inspector's step rides once)
        size_t lds = sizeof(float) * PairShape<MODEL>::kLdsFloats;
        if (f.blocks > 0 && (size_t)f.lds_bytes > lds) lds = (size_t)f.lds_bytes;
        hipLaunchKernelGGL(kernel, dim3(tiles + (unsigned)f.blocks), dim3(kPairWaves * kWave), lds, st, a, pa, f);
    }
    KGE_CHECK_LAUNCH();
    return KGE_OK;
}

}  // namespace kge
