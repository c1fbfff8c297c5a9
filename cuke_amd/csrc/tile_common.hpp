// Pieces shared by the shared-negative tile kernels (forward and backward): guarded
// 128-bit row loads and the per-model "query" row a_b = f(h_b, r_b) that is formed on
// the fly while a tile is staged, so h and r are gathered inside the consuming kernel.
#pragma once

#include "common.hpp"

#ifndef KGE_TILE_OCC
#define KGE_TILE_OCC 3  // minimum workgroups per CU the tile kernels are compiled for
#endif

namespace kge {

// ---- quads of a row -----------------------------------------------------------------------------
// Rows (segments) of at least four floats are read 128 bits at a time whatever their width and alignment: the quad that
// would run past the end of the segment is moved back to end with it, so no address lies outside the row.  Its first
// elements belong to the quad before it as well: a sum over columns leaves them out (mask4), a result per column is
// formed twice and stored once.  `lim` is the segment's length, or 0 for a row outside the tile.
//   16-byte rows only (the rule before), everything else by single floats in 32 x 32 tiles: ComplEx, 512 queries
//   against 14951 candidates, 394 us at width 396 and 384 us at 402 beside 105 us at 400; one TransE step of 30000 x 150 x 200
//   negatives 466 us beside 374 us at width 152.
// v moved down by s elements, zeros from above (s <= 0: v; s >= 4: zeros)
__device__ __forceinline__ float4 shift_quad(float4 v, int s)
{
    const bool one = s == 1 || s == 3, two = s == 2 || s == 3, all = s >= 4;
    v = make_float4(one ? v.y : v.x, one ? v.z : v.y, one ? v.w : v.z, one ? 0.0f : v.w);
    v = make_float4(two ? v.z : v.x, two ? v.w : v.y, two ? 0.0f : v.z, two ? 0.0f : v.w);
    return make_float4(all ? 0.0f : v.x, all ? 0.0f : v.y, all ? 0.0f : v.z, all ? 0.0f : v.w);
}

// Four consecutive floats p[j .. j+3] (VEC: moved back to end with the row), zero where the element
// is not the quad's own.  Branch-free: an out-of-range request reads a valid address of the row and discards it, so the
// callers' loads sit in one basic block and the compiler can issue them back to back.
template <bool VEC>
__device__ __forceinline__ float4 ld4_raw(const float *p, int j, int lim);
template <bool VEC>
__device__ __forceinline__ float4 mask4(float4 v, int j, int lim);

template <bool VEC>
__device__ __forceinline__ float4 ld4(const float *p, int j, int lim)
{
    if constexpr (VEC) {
        return mask4<true>(ld4_raw<true>(p, j, lim), j, lim);
    } else {
        float4 q;
        const bool k0 = j + 0 < lim, k1 = j + 1 < lim, k2 = j + 2 < lim, k3 = j + 3 < lim;
        const float x0 = p[k0 ? j + 0 : 0], x1 = p[k1 ? j + 1 : 0], x2 = p[k2 ? j + 2 : 0], x3 = p[k3 ? j + 3 : 0];
        q.x = k0 ? x0 : 0.0f;
        q.y = k1 ? x1 : 0.0f;
        q.z = k2 ? x2 : 0.0f;
        q.w = k3 ? x3 : 0.0f;
        return q;
    }
}

// The same where a quad lies inside its row or outside it as a whole: lanes outside keep a zero and load nothing, so nothing
// touches the loaded register (a select on it would be waited for where it stands).
template <bool VEC>
__device__ __forceinline__ float4 ld4_whole(const float *p, int j, int lim)
{
    if constexpr (VEC) {
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (j < lim) v = load_quad(p + j);
        return v;
    } else {
        return ld4<false>(p, j, lim);
    }
}

__device__ __forceinline__ float4 zero4() { return make_float4(0.f, 0.f, 0.f, 0.f); }
__device__ __forceinline__ float4 mul4(float4 p, float4 q)
{
    return make_float4(p.x * q.x, p.y * q.y, p.z * q.z, p.w * q.w);
}
__device__ __forceinline__ float4 add4(float4 p, float4 q)
{
    return make_float4(p.x + q.x, p.y + q.y, p.z + q.z, p.w + q.w);
}

// sign(u) as a clamp: u * 2^100 clamped to [-1, 1] (exact 0 stays 0; |u| < 2^-100 would give a
// fraction, far below any fp32 residual that is not exactly zero).  The multiply is paid once per
// staged row element instead of once per pair element: scaling by a power of two commutes with
// every fp32 rounding (no overflow: table values times 2^100 stay far below 2^127), so a residual
// formed from rows that carry the factor 2^100 is exactly 2^100 times the residual of the plain
// rows, and its sign is one clamp away.  The L1 tile kernels of TransE / TransH stage their rows
// scaled; sums of |U| and of sign(U) * W are scaled back once per pair, and coefficients that
// multiply a scaled row carry 2^-100.
// Measured alternatives that did not pay (TransH, L1, 16384 x 1024 pairs x 400): clamping
// u * copysign(2^100, g) to [-|g|, |g|] to get g * sign(u) directly (forward 0.92 -> 1.10 ms, gradient
// tiles 1.74 -> 1.86 ms: v_med3_f32 and v_bfi_b32 issue at two thirds of the rate of add / mul / fmac);
// (sign(u) + 1) / 2 as ONE multiply-add with the output clamp, the coefficients' sums taken off once
// per step (one instruction fewer per element, same forward time, gradient tiles 1.74 -> 1.80 ms: a
// v_fma_f32 with a scalar-register operand issues at 60 % of the vector-operand rate, and with the
// factor in a vector register the per-pair bookkeeping ate the gain).
constexpr float kSgnScale = 0x1p100f, kSgnUnscale = 0x1p-100f;
__device__ __forceinline__ float sgn_of_scaled(float U) { return __builtin_amdgcn_fmed3f(U, -1.0f, 1.0f); }
__device__ __forceinline__ float4 scale4(float4 v, float s) { return make_float4(v.x * s, v.y * s, v.z * s, v.w * s); }

// reduction length of the pair kernels: complex pairs for RotatE, floats otherwise
template <int MODEL>
__device__ __forceinline__ int pair_len(int d)
{
    return MODEL == KGE_ROTATE ? d >> 1 : d;
}

// Four consecutive elements (index j .. j+3 of the reduction axis) of the query row.
//   DistMult  q0 = h*r                   ComplEx  q0 = (h o r) laid out [re | im]
//   TransE    q0 = h+r                   RotatE   q0 = Re(h e^{i theta}), q1 = Im(...) (from pq)
//   TransH    q0 = h + r - al*w (al = w.h), q1 = w
//   TransF    q0 = 2h + r: score = (h + r).t' + (t' - r).h = (2h + r).t' - r.h, a dot product with
//             the query plus a constant per positive
//   RESCAL    q0 = E[h] Proj[r], the projected row that the grouped forward pass left in pq:
//             score = (h M_r) . t' needs no projection of the negatives at all
// lim == 0 yields zeros (row outside the tile).
// RotatE takes its query rows from pq, the [B, d] buffer of rotated heads.
//
// Negatives that replace the HEAD use the same pair kernels: score(n, r, t) is the tail-mode
// function of (x, rho, n) with x = t and rho = -r (TransE, TransH, TransF), conj(r) (ComplEx), -theta
// (RotatE, already applied in pq) or r (DistMult).  The caller passes the tail row as `ph` and
// rs = -1; rs multiplies r (its imaginary half for ComplEx), which is exact, so rs = +1
// reproduces the tail-mode arithmetic bit for bit.
//
// Loading and forming are two steps.  A tile kernel that prefetches the next block of rows while it computes on the current one only
// overlaps the two if nothing touches the loaded registers before the compute: any arithmetic
// on them (h * r, the zero fill of a tail) makes the compiler wait for the loads where they are
// issued.  load_query_raw() therefore only loads -- clamped to a valid address, no select, no
// arithmetic -- and combine_query() forms the query row when the block is written to LDS.
template <bool VEC>
__device__ __forceinline__ float4 ld4_raw(const float *p, int j, int lim)
{
    if constexpr (VEC) {
        return load_quad(p + max(min(j, lim - 4), 0));
    } else {
        return make_float4(p[j + 0 < lim ? j + 0 : 0], p[j + 1 < lim ? j + 1 : 0], p[j + 2 < lim ? j + 2 : 0],
                           p[j + 3 < lim ? j + 3 : 0]);
    }
}

// the quad that ld4_raw(p, j, lim) loaded, zero where the element is not its own
template <bool VEC>
__device__ __forceinline__ float4 mask4(float4 v, int j, int lim)
{
    if constexpr (VEC) {
        const int skip = j + 4 - lim;  // elements that the quad before it has
        return make_float4(skip <= 0 ? v.x : 0.0f, skip <= 1 ? v.y : 0.0f, skip <= 2 ? v.z : 0.0f, skip <= 3 ? v.w : 0.0f);
    }
    return make_float4(j + 0 < lim ? v.x : 0.0f, j + 1 < lim ? v.y : 0.0f, j + 2 < lim ? v.z : 0.0f,
                       j + 3 < lim ? v.w : 0.0f);
}

template <int MODEL>
constexpr int query_raw_count()
{
    return MODEL == KGE_COMPLEX ? 4 : (MODEL == KGE_TRANSH ? 3 : 2);
}

template <int MODEL, bool VEC, int N>
__device__ __forceinline__ void load_query_raw(const float *ph, const float *pr, const float *pw, const float *pq,
                                               int j, int lim, int half, float4 (&raw)[N])
{
    static_assert(N == query_raw_count<MODEL>(), "raw operand count");
    if constexpr (MODEL == KGE_DISTMULT || MODEL == KGE_TRANSE || MODEL == KGE_TRANSF) {
        raw[0] = ld4_raw<VEC>(ph, j, lim);
        raw[1] = ld4_raw<VEC>(pr, j, lim);
    } else if constexpr (MODEL == KGE_COMPLEX) {
        if constexpr (VEC) {  // (a quad starts at a multiple of four of its half, see split_col)
            const int i = j < half ? j : j - half;
            const int l2 = lim ? half : 0;
            raw[0] = ld4_raw<true>(ph, i, l2), raw[1] = ld4_raw<true>(ph + half, i, l2);
            raw[2] = ld4_raw<true>(pr, i, l2), raw[3] = ld4_raw<true>(pr + half, i, l2);
        } else {
            float v[4][4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int jj = j + e;
                const int i = jj < lim ? (jj < half ? jj : jj - half) : 0;
                v[0][e] = ph[i], v[1][e] = ph[i + half], v[2][e] = pr[i], v[3][e] = pr[i + half];
            }
#pragma unroll
            for (int n = 0; n < 4; ++n) raw[n] = make_float4(v[n][0], v[n][1], v[n][2], v[n][3]);
        }
    } else if constexpr (MODEL == KGE_RESCAL) {
        raw[0] = ld4_raw<VEC>(pq, j, lim);
        raw[1] = raw[0];
    } else if constexpr (MODEL == KGE_ROTATE) {
        raw[0] = ld4_raw<VEC>(pq, j, lim);
        raw[1] = ld4_raw<VEC>(pq + half, j, lim);
    } else if constexpr (MODEL == KGE_TRANSH) {
        raw[0] = ld4_raw<VEC>(pw, j, lim);
        raw[1] = ld4_raw<VEC>(ph, j, lim);
        raw[2] = ld4_raw<VEC>(pr, j, lim);
    }
}

// The query row from its raw operands (same j, lim, half as load_query_raw).
template <int MODEL, bool VEC, int N>
__device__ __forceinline__ void combine_query(const float4 (&raw)[N], float al, int j, int lim, int half, float rs,
                                              float4 &q0, float4 &q1)
{
    q1 = zero4();
    if constexpr (MODEL == KGE_DISTMULT) {
        q0 = mask4<VEC>(mul4(raw[0], raw[1]), j, lim);
    } else if constexpr (MODEL == KGE_TRANSE) {
        const float4 vh = raw[0], vr = raw[1];
        q0 = mask4<VEC>(make_float4(fmaf(rs, vr.x, vh.x), fmaf(rs, vr.y, vh.y), fmaf(rs, vr.z, vh.z), fmaf(rs, vr.w, vh.w)),
                        j, lim);
    } else if constexpr (MODEL == KGE_TRANSF) {
        const float4 vh = raw[0], vr = raw[1];
        q0 = mask4<VEC>(make_float4(fmaf(rs, vr.x, 2.0f * vh.x), fmaf(rs, vr.y, 2.0f * vh.y), fmaf(rs, vr.z, 2.0f * vh.z),
                                    fmaf(rs, vr.w, 2.0f * vh.w)),
                        j, lim);
    } else if constexpr (MODEL == KGE_COMPLEX) {
        const float hr[4] = {raw[0].x, raw[0].y, raw[0].z, raw[0].w}, hi[4] = {raw[1].x, raw[1].y, raw[1].z, raw[1].w};
        const float rr[4] = {raw[2].x, raw[2].y, raw[2].z, raw[2].w};
        const float ri[4] = {rs * raw[3].x, rs * raw[3].y, rs * raw[3].z, rs * raw[3].w};
        float q[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int jj = VEC ? j : j + e;  // VEC: one side of the split for the whole quad
            const float v = jj < half ? hr[e] * rr[e] - hi[e] * ri[e] : hr[e] * ri[e] + hi[e] * rr[e];
            q[e] = VEC || jj < lim ? v : 0.0f;
        }
        q0 = make_float4(q[0], q[1], q[2], q[3]);
        if constexpr (VEC) q0 = mask4<true>(q0, j < half ? j : j - half, lim ? half : 0);
    } else if constexpr (MODEL == KGE_RESCAL) {
        q0 = mask4<VEC>(raw[0], j, lim);
    } else if constexpr (MODEL == KGE_ROTATE) {
        q0 = mask4<VEC>(raw[0], j, lim);
        q1 = mask4<VEC>(raw[1], j, lim);
    } else if constexpr (MODEL == KGE_TRANSH) {
        const float4 vw = raw[0], vh = raw[1], vr = raw[2];
        q1 = mask4<VEC>(vw, j, lim);
        q0 = mask4<VEC>(make_float4(fmaf(rs, vr.x, vh.x) - al * vw.x, fmaf(rs, vr.y, vh.y) - al * vw.y,
                                    fmaf(rs, vr.z, vh.z) - al * vw.z, fmaf(rs, vr.w, vh.w) - al * vw.w),
                        j, lim);
    } else {
        q0 = zero4();
    }
}

// Both steps at once.
template <int MODEL, bool VEC>
__device__ __forceinline__ void load_query(const float *ph, const float *pr, const float *pw, const float *pq, float al, int j, int lim,
                                           int half, float rs, float4 &q0, float4 &q1)
{
    float4 raw[query_raw_count<MODEL>()];
    load_query_raw<MODEL, VEC>(ph, pr, pw, pq, j, lim, half, raw);
    combine_query<MODEL, VEC>(raw, al, j, lim, half, rs, q0, q1);
}

// ComplEx rows are two segments of half floats, each walked in quads of its own: column jv of the padded row
// [re, padded to a multiple of four | im, padded] is column split_col(jv) of the row, and a quad that starts there belongs
// to one half.
__device__ __forceinline__ int split_col(int jv, int half)
{
    const int hp = (half + 3) & ~3;
    return jv < hp ? jv : jv - hp + half;
}
// a quad of a plain row, or of one half of a ComplEx row (VEC: j as split_col gives it)
template <int MODEL, bool VEC>
__device__ __forceinline__ float4 ld4_row_raw(const float *p, int j, int lim, int half)
{
    if constexpr (MODEL == KGE_COMPLEX && VEC) return ld4_raw<true>(p + (j < half ? 0 : half), j < half ? j : j - half, lim ? half : 0);
    else return ld4_raw<VEC>(p, j, lim);
}
template <int MODEL, bool VEC>
__device__ __forceinline__ float4 mask4_row(float4 v, int j, int lim, int half)
{
    if constexpr (MODEL == KGE_COMPLEX && VEC) return mask4<true>(v, j < half ? j : j - half, lim ? half : 0);
    else return mask4<VEC>(v, j, lim);
}

// XCD-aware tile placement.  The 256 CUs sit in 8 XCDs with one L2 each, and consecutive
// workgroup ids of a 1-D grid go to consecutive XCDs.  All tiles of one chunk share that
// chunk's positive and negative rows, so they are steered to one XCD: every gathered row is
// then fetched from HBM by a single L2 instead of by up to eight.  With fewer than 8 chunks a
// chunk's tiles are dealt round-robin to 8 / n_chunks XCDs so that no XCD stays idle.
// Returns false for the padding ids of the grid (see xcd_grid).
constexpr int kXcds = 8;
__host__ __device__ inline int xcd_split(int n_chunks) { return n_chunks >= kXcds ? 1 : kXcds / n_chunks; }
__device__ __forceinline__ bool xcd_tile(int lid, int tiles_x, int tiles_y, int n_chunks, int &c, int &ty, int &tx)
{
    const int per = tiles_x * tiles_y;
    const int split = xcd_split(n_chunks);
    const int per_v = (per + split - 1) / split;  // tiles of one virtual chunk
    const int xcd = lid % kXcds, k = lid / kXcds;
    const int vc = (k / per_v) * kXcds + xcd;      // virtual chunk = (chunk, residue of the tile id)
    c = vc / split;
    const int t = (k % per_v) * split + vc % split;
    ty = t / tiles_x;
    tx = t % tiles_x;
    return c < n_chunks && t < per;
}
inline unsigned xcd_grid(int64_t tiles_x, int64_t tiles_y, int64_t n_chunks)
{
    const int64_t split = xcd_split((int)n_chunks), per = tiles_x * tiles_y;
    return (unsigned)(kXcds * ceil_div(n_chunks * split, kXcds) * ceil_div(per, split));
}

// every row segment is a whole number of quads
template <int MODEL>
__host__ __device__ inline bool whole_quads(int d)
{
    return d % (MODEL == KGE_COMPLEX || MODEL == KGE_ROTATE ? 8 : 4) == 0;
}
// 128-bit row loads: every row segment (ComplEx, RotatE: each half) has at least four floats
inline bool rows_by_quads(const kge_tables *tab)
{
    const bool complex_rows = tab->model == KGE_COMPLEX || tab->model == KGE_ROTATE;
    return quad_row(complex_rows ? tab->dim / 2 : tab->dim);
}

}  // namespace kge
