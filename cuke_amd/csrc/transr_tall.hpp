// The grouped product of TransR / RESCAL in tiles of 64 triples x 128 columns, where want_tall says so (below): forward
// scores, the row list of the shared negatives, and dX; the forward pass with back rows keeps its 32-triple
// tiles.  This file is included by transr.hip (inside namespace kge).
//
// A relation's projection is read once per 64 of its triples instead of once per 32, a wave feeds four row blocks
// from every 128-byte piece it loads, and the left operand goes through LDS in slices of 64 columns (double buffered), so
// that two to four workgroups fit a CU whatever the row width is (whole rows in LDS left one at width 1024).
//   what bounds it: the matrix cores where groups are large (8192 x 1024 over 51 relations), the projections'
//   bytes where they are small (4096 x 512 over 237).  Whole RESCAL calls, 32-row tiles -> these, on one box: 8192 x 1024
//   over 51 relations (Zipf) 335 -> 236 us, 73 TFLOP/s; 4096 x 512 over 237 (Zipf) 107 -> 89 us; 512 x 1000 over 40
//   163 -> 61 us; one relation with 24576 rows of 1024 494 -> 478 us, 108 TFLOP/s.
// Tiles of fewer rows run one to three of the four 16-row blocks, so a tail costs what it holds.
//
// A superstep of the projection comes back after about two microseconds when the chip is busy, so what a CU holds in
// flight (three workgroups x three supersteps x 8 KB) sets the pace of what the matrix cores do not.

constexpr int kTallRows = 64;   // triples per tile
constexpr int kTallCols = 128;  // columns per workgroup at most: 32 per wave, two 16-column MFMA blocks
constexpr int kTallKC = 64;     // columns of the left operand staged at a time
constexpr int kTallPitch = kTallKC + 4;
constexpr int kTallRing = 4;    // supersteps (16 rows of k) of the projection in flight per wave, one of them in use
constexpr int kSplitRows = 32;    // tiles of more rows go by the bf16 matrix cores ...
constexpr int kSplitItems = 256;  // ... where a launch has more items than that
constexpr int kTallWgs = 4096;  // workgroups of a launch at most; they stride over the tiles

struct TallRows {  // what a tile knows about its rows (LDS, behind the staging buffers)
    global_f32 v[kTallRows], w[kTallRows];     // the rows the left operand is formed from
    int64_t t[kTallRows];                      // MODE 1: tail ids
    int b[kTallRows];
    float f[kTallRows], g[kTallRows];          // MODE 3: factor of the relation row, whether there is a t; MODE 2: coefficient, upstream gradient
    float sum[8][kTallRows];
};
// staging: two slices of the left operand, or (split tiles) one slice of both operands in three parts
constexpr size_t kTallStage = sizeof(__bf16) * kSplitPitch * (kTallRows + kTallCols);
static_assert(kTallStage >= sizeof(float) * 2 * kTallRows * kTallPitch && kTallStage % 16 == 0, "the row table stands behind both forms");
constexpr size_t kTallLds = kTallStage + sizeof(TallRows);

__host__ __device__ inline int tall_col_blocks(int d) { return (d + kTallCols - 1) / kTallCols; }
// columns of a block / of a wave: an even split, multiples of four / two
__host__ __device__ inline int tall_block_cols(int d) { return ((d + tall_col_blocks(d) - 1) / tall_col_blocks(d) + 3) & ~3; }

struct TallArgs {
    GemmArgs g;    // plan: tiles of kTallRows
    float *part;   // [column blocks][B] partial scores where there is more than one column block (pos set), else unused
    int64_t B;
};

// One superstep's B operands of a lane as they are loaded: at(e, s) = column e, k = 16 q + 4 kk + s.
template <int MODE>
struct TallSlot {
    floatx2 r[4];
    __device__ __forceinline__ float at(int e, int s) const { return r[s][e]; }
    __device__ __forceinline__ void keep(bool k)
    {
#pragma unroll
        for (int s = 0; s < 4; ++s) r[s] = k ? r[s] : floatx2{0.f, 0.f};
    }
};
template <>
struct TallSlot<2> {
    floatx4 r[2];
    __device__ __forceinline__ float at(int e, int s) const { return r[e][s]; }
    __device__ __forceinline__ void keep(bool k)
    {
#pragma unroll
        for (int e = 0; e < 2; ++e) r[e] = k ? r[e] : floatx4{0.f, 0.f, 0.f, 0.f};
    }
};

// Two B-operand values per k row for this lane: columns n0 + 2 li + {0, 1} of M (MODE 2: of M^T).  Addresses are the
// uniform base plus a 32-bit byte offset (a projection has at most 2^20 elements: no 64-bit address arithmetic on the
// vector ALUs, which would take issue slots from the matrix instructions); a k beyond the last row is clamped to
// it (the staged left operand is zero there, and tall_sweep() zeroes the clamped values too).
template <int MODE>
struct TallLoader {
    const char *M;
    uint32_t off[2], last, d4, k0;  // bytes
    __device__ __forceinline__ void init(const float *M_, int d_, int n0, int wcols, int li, int kk)
    {
        M = reinterpret_cast<const char *>(M_), d4 = 4u * (uint32_t)d_;
        const uint32_t col = (uint32_t)(n0 + (2 * li < wcols ? 2 * li : 0));
        if constexpr (MODE != 2) off[0] = 4u * (uint32_t)kk * d4 + 4u * col, last = ((uint32_t)d_ - 1) * d4 + 4u * col;
        else off[0] = col * d4, off[1] = off[0] + d4, last = d4 - 16, k0 = 16u * (uint32_t)kk;
    }
    __device__ __forceinline__ void load(int q, TallSlot<MODE> &dst) const
    {
        if constexpr (MODE != 2) {
            const uint32_t o = off[0] + 16u * (uint32_t)q * d4;
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const uint32_t f = o + s * d4;
                dst.r[s] = *reinterpret_cast<const floatx2 *>(M + (f < last ? f : last));
            }
        } else {
            const uint32_t k = k0 + 64u * (uint32_t)q, kc = k < last ? k : last;
#pragma unroll
            for (int e = 0; e < 2; ++e) dst.r[e] = *reinterpret_cast<const floatx4 *>(M + (off[e] + kc));
        }
    }
};

// RB row blocks of one tile against this wave's columns.  The next slice of the left operand is staged while this one
// is multiplied: fetch(i, c) requests row block i of slice c, put(i, c) writes it to LDS buffer c & 1.  Loads return in
// order, so the requests go out behind the first superstep's piece of the projection and the writes wait until the
// end of the slice, when everything in front of them has been used anyway.
template <int MODE, int RB, typename Fetch, typename Put>
__device__ __forceinline__ void tall_sweep(const TallLoader<MODE> &bl, int d, TallSlot<MODE> (&ring)[kTallRing], const float *lds, int li, int kk,
                                           Fetch fetch, Put put, floatx4 (&acc)[RB][2])
{
    static_assert(kTallRing == kTallKC / 16, "ring slot u is superstep u of every slice");
    const int nq = (d + 15) / 16, nc = (nq + kTallRing - 1) / kTallRing;
#pragma unroll 1
    for (int c = 0; c < nc; ++c) {
        const float *sX = lds + (c & 1) * (kTallRows * kTallPitch) + li * kTallPitch + 4 * kk;
        const int next = c + 1 < nc ? c + 1 : c;  // (past the end: the last slice once more, into the buffer nobody reads; no branch around a load)
#pragma unroll
        for (int u = 0; u < kTallRing; ++u) {
            const int q = kTallRing * c + u;
            bl.load(q + kTallRing - 1, ring[(u + kTallRing - 1) % kTallRing]);
            if (u == 0) {
#pragma unroll
                for (int i = 0; i < RB; ++i) fetch(i, next);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (q >= nq) continue;  // uniform
            if (16 * q + 16 > d) ring[u].keep(16 * q + 4 * kk < d);  // uniform: the last superstep of most widths; keeps 0 * inf out
            float4 a[RB];
#pragma unroll
            for (int m = 0; m < RB; ++m) a[m] = *reinterpret_cast<const float4 *>(sX + 16 * m * kTallPitch + 16 * u);
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int m = 0; m < RB; ++m) {
                    const float av = s == 0 ? a[m].x : s == 1 ? a[m].y : s == 2 ? a[m].z : a[m].w;
#pragma unroll
                    for (int e = 0; e < 2; ++e) acc[m][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, ring[u].at(e, s), acc[m][e], 0, 0, 0);
                }
        }
#pragma unroll
        for (int i = 0; i < RB; ++i) put(i, c + 1);
        __syncthreads();
    }
}

// threadIdx.x, opaque: what follows from it is formed anew per tile and not held across the forms of a tile that share a kernel
__device__ __forceinline__ int tile_tid()
{
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    return tid;
}

// fills the row table of the tile's `rows` rows from position p0 on (one thread per row; later rows repeat the first)
template <int MODE>
__device__ __forceinline__ void tall_rows(const GemmArgs &a, TallRows &R, int p0, int rows, bool array, bool derived)
{
    const int tid = threadIdx.x, d = a.d;
    if (tid < kTallRows) {
        const int p = p0 + (tid < rows ? tid : 0);
        int b;
        if constexpr (MODE == 3) b = p, R.f[tid] = a.rs[p];
        else b = (MODE == 2 && derived) ? a.src.perm[p] : (a.perm ? a.perm[p] : p);
        R.b[tid] = b;
        if constexpr (MODE == 2) {
            if (derived) {
                const RowMeta m = bwd_row_meta(a.src, p, d);
                R.f[tid] = m.coef, R.g[tid] = a.src.dpos ? a.src.dpos[b] : 0.0f;
                R.v[tid] = (global_f32)(bwd_qbase(a.src) + m.qoff), R.w[tid] = (global_f32)(a.src.resid + (int64_t)b * d);
            } else {
                R.v[tid] = (global_f32)(a.xs + (int64_t)p * d);
            }
        } else {
            const int64_t h = a.h[b], t = a.t[b];
            R.v[tid] = (global_f32)(array ? a.xs + (int64_t)p * d : a.ent + h * d);
            R.w[tid] = (global_f32)(a.ent + (MODE == 3 && t < 0 ? 0 : t) * d);  // (MODE 3, t = -1: no row; read and, in put(), dropped)
            if constexpr (MODE == 1) R.t[tid] = t;
            if constexpr (MODE == 3) R.g[tid] = t >= 0 ? 1.0f : 0.0f;
        }
    }
}

// MODE as in transr_gemm_body: 0 forward TransR, 1 forward RESCAL (or rows given as an array), 2 dX, 3 list rows.
// RB: 16-row blocks the tile runs (a template parameter: the staging and accumulator registers follow it).
template <int MODE, int RB>
__device__ __forceinline__ void tall_tile(const TallArgs &t, float *lds, int tile, int cb)
{
    const GemmArgs &a = t.g;
    const int d = a.d, ncb = tall_col_blocks(d);
    const int tid = tile_tid(), lane = tid & 63, wave = tid >> 6, li = lane & 15, kk = lane >> 4;
    // (uniform, but the compiler cannot know: the kernel also stores)
    const int p0 = __builtin_amdgcn_readfirstlane(a.plan.tile_p0[tile]), seg_end = __builtin_amdgcn_readfirstlane(a.plan.tile_end[tile]);
    const int64_t rid = __builtin_amdgcn_readfirstlane(a.plan.tile_rid[tile]);
    const int rows = seg_end - p0 < kTallRows ? seg_end - p0 : kTallRows;
    const float *M = a.proj + rid * (int64_t)d * d;

    const int bc = tall_block_cols(d), c0 = cb * bc, span = d - c0 < bc ? d - c0 : bc;
    const int cw = ((span + 3) / 4 + 1) & ~1;
    const int n0 = c0 + wave * cw;
    const int wcols = n0 >= c0 + span ? 0 : (c0 + span - n0 < cw ? c0 + span - n0 : cw);
    TallLoader<MODE> bl;
    TallSlot<MODE> ring[kTallRing];
    bl.init(M, d, wcols > 0 ? n0 : c0, wcols, li, kk);
#pragma unroll
    for (int u = 0; u + 1 < kTallRing; ++u) bl.load(u, ring[u]);  // the projection's first pieces fly during the index chain below
    __builtin_amdgcn_sched_barrier(0);

    TallRows &R = *reinterpret_cast<TallRows *>(reinterpret_cast<char *>(lds) + kTallStage);
    const bool array = a.xs != nullptr && (MODE == 1 || MODE == 2);
    const bool derived = MODE == 2 && !array;
    tall_rows<MODE>(a, R, p0, rows, array, derived);
    __syncthreads();

    // Staging: thread tid takes the quad tid % 16 of row tid / 16 of a row block.
    const int srow = tid >> 4, scol = (tid & 15) * 4;
    const bool l1 = derived && !a.src.rescal && a.src.norm_p == 1;
    const bool occ = derived && a.src.occ_v && cb == 0;
    constexpr bool kTwo = MODE == 0 || MODE == 3;
    float4 v[RB], w[RB];
    auto fetch = [&](int i, int c) {
        const int k4 = c * kTallKC + scol < d ? c * kTallKC + scol : 0;  // clamped: unconditional loads, masked in put()
        v[i] = load4g(R.v[16 * i + srow] + k4);
        if constexpr (kTwo) w[i] = load4g(R.w[16 * i + srow] + k4);
        else w[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        if constexpr (MODE == 2)
            if (occ) w[i] = load4g(R.w[16 * i + srow] + k4);
    };
    auto put = [&](int i, int c) {
        const int row = 16 * i + srow, col = c * kTallKC + scol;
        const bool colok = col < d;
        const float4 vv = v[i], ww = w[i];
        float4 x = vv;
        if constexpr (MODE == 0) x = make_float4(vv.x - ww.x, vv.y - ww.y, vv.z - ww.z, vv.w - ww.w);
        if constexpr (MODE == 3) {
            const bool keep = R.g[row] != 0.0f;
            x = make_float4(vv.x - (keep ? ww.x : 0.0f), vv.y - (keep ? ww.y : 0.0f), vv.z - (keep ? ww.z : 0.0f), vv.w - (keep ? ww.w : 0.0f));
        }
        if constexpr (MODE == 2) {
            if (derived) {
                x = scaled4(R.f[row], l1 ? sgn4(vv) : vv);
                if (occ && row < rows && colok)  // RESCAL: the tail's occurrence row g * (E[h] Proj[r])
                    *reinterpret_cast<float4 *>(a.src.occ_v + (int64_t)R.b[row] * d + col) = scaled4(R.g[row], ww);
            }
        }
        const bool ok = row < rows && colok;
        x = make_float4(ok ? x.x : 0.0f, ok ? x.y : 0.0f, ok ? x.z : 0.0f, ok ? x.w : 0.0f);
        *reinterpret_cast<float4 *>(&lds[(c & 1) * (kTallRows * kTallPitch) + row * kTallPitch + scol]) = x;
    };

    const bool colok = 2 * li < wcols;
    const int col = colok ? n0 + 2 * li : c0;
    float2 rv = make_float2(0.f, 0.f);  // the relation's row, for the epilogue
    if constexpr (MODE == 0 || MODE == 3) rv = *reinterpret_cast<const float2 *>(a.rel + rid * (int64_t)d + col);
    floatx4 acc[RB][2];
#pragma unroll
    for (int m = 0; m < RB; ++m) acc[m][0] = acc[m][1] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < RB; ++i) fetch(i, 0);
#pragma unroll
    for (int i = 0; i < RB; ++i) put(i, 0);
    __syncthreads();
    tall_sweep<MODE, RB>(bl, d, ring, lds, li, kk, fetch, put, acc);

    // Lane (li, kk) holds rows 16 m + 4 kk + r, columns n0 + 2 li + {0, 1}.  Everything is read before the first
    // store: a load between two stores makes the compiler wait for the stores in front of it.
    const bool want_pos = MODE < 2 && a.pos;
    int rb[RB][4];
    float2 y[RB][4];
#pragma unroll
    for (int m = 0; m < RB; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 16 * m + 4 * kk + r;
            rb[m][r] = R.b[row];
            y[m][r] = make_float2(acc[m][0][r], acc[m][1][r]);
            if constexpr (MODE == 0) y[m][r].x += rv.x, y[m][r].y += rv.y;
            if constexpr (MODE == 3) {
                const float f = R.f[row];  // +-1 or 0: exact products
                y[m][r].x += f * rv.x, y[m][r].y += f * rv.y;
            }
        }
    if constexpr (MODE < 2) {
        if (want_pos) {  // uniform
#pragma unroll
            for (int m0 = 0; m0 < RB; m0 += 2) {
            float2 tv[RB][4];
            if constexpr (MODE == 1) {  // the tails' rows, two blocks in one batch of loads
#pragma unroll
                for (int m = m0; m < RB && m < m0 + 2; ++m)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int row = 16 * m + 4 * kk + r;
                        tv[m][r] = *reinterpret_cast<const float2 *>(a.ent + R.t[row < rows ? row : 0] * (int64_t)d + col);
                    }
            }
#pragma unroll
            for (int m = m0; m < RB && m < m0 + 2; ++m)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float s;
                    if constexpr (MODE == 1) s = fmaf(y[m][r].x, tv[m][r].x, y[m][r].y * tv[m][r].y);
                    else s = a.norm_p == 1 ? fabsf(y[m][r].x) + fabsf(y[m][r].y) : fmaf(y[m][r].x, y[m][r].x, y[m][r].y * y[m][r].y);
                    s = row16_sum(colok ? s : 0.0f);
                    if (li == 0) R.sum[wave][16 * m + 4 * kk + r] = s;
                }
            }
        }
    }
    float *const out = MODE == 2 ? a.occ_h : a.resid;
    if (out && colok) {
#pragma unroll
        for (int m = 0; m < RB; ++m)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (16 * m + 4 * kk + r < rows) {
                    const int64_t o = (int64_t)rb[m][r] * d + col;
                    *reinterpret_cast<float2 *>(out + o) = y[m][r];
                    if constexpr (MODE == 2)
                        if (a.occ_t) *reinterpret_cast<float2 *>(a.occ_t + o) = make_float2(-y[m][r].x, -y[m][r].y);
                }
    }
    if constexpr (MODE < 2) {
        if (want_pos) {
            __syncthreads();
            if (tid < rows) {
                const float s = (R.sum[0][tid] + R.sum[1][tid]) + (R.sum[2][tid] + R.sum[3][tid]);
                if (ncb > 1) t.part[(int64_t)cb * t.B + R.b[tid]] = s;
                else a.pos[R.b[tid]] = (MODE == 0 && a.norm_p == 2) ? sqrtf(s) : s;
            }
        }
    }
}

// The same tile on the bf16 matrix cores (mfma_split.hpp), for tiles of more than kSplitRows rows: RB blocks of 32 rows, a wave takes all of them
// and 32 columns.  Both operands go through LDS in slices of 32, split once per slice; the projection's pieces are transposed on the way
// (a thread takes 4 x 4 elements: four rows of it are loaded, four columns written, 64 bytes of a row and 16 banks apart per two lanes).
//   What bounds it: the matrix cores and the slices' barriers where groups are large, else the projections' bytes.  Whole calls, fp32 tiles
//   -> these: RESCAL 8192 x 1024 over 51 relations (Zipf) 230 -> 184 us, 8192 x 512 over 11 82 -> 64; TransR 4096 x 512 over 60 64 -> 50,
//   over 237 91 -> 86 (bytes); the row list and dX of TransR against shared negatives, 4096 x 200 over 1345, 126 + 145 -> 122 + 107 us.
//   A launch of at most one item per CU runs every slice at its full latency and keeps the fp32 tiles' four supersteps in flight
//   (4096 x 128 over 20: 25 against 27 us).  Tiles of at most 32 rows do half of the work or less in fp32's 16-row blocks and keep more of the
//   projection in flight: score calls of 17 to 30 rows a relation (4096 to 7000 triples over 237, widths 400 and 512) TransR 80 to 100 us
//   split, 66 to 82 in fp32, RESCAL 82 to 97 and 67 to 79; split as one block of 32 rows 75 to 95.
template <int MODE, int RB>
__device__ __forceinline__ bool split_tile(const TallArgs &t, float *lds, int tile, int cb)
{
    const GemmArgs &a = t.g;
    const int d = a.d, ncb = tall_col_blocks(d);
    const int tid = tile_tid(), lane = tid & 63, wave = tid >> 6, fr = lane & 31, fg = lane >> 5;
    const int p0 = __builtin_amdgcn_readfirstlane(a.plan.tile_p0[tile]), seg_end = __builtin_amdgcn_readfirstlane(a.plan.tile_end[tile]);
    const int64_t rid = __builtin_amdgcn_readfirstlane(a.plan.tile_rid[tile]);
    const int rows = seg_end - p0 < kTallRows ? seg_end - p0 : kTallRows;
    const float *M = a.proj + rid * (int64_t)d * d;
    const int bc = tall_block_cols(d), c0 = cb * bc, span = d - c0 < bc ? d - c0 : bc;

    __bf16(*sX)[kSplitPitch] = reinterpret_cast<__bf16(*)[kSplitPitch]>(lds);
    __bf16(*sM)[kSplitPitch] = sX + kTallRows;  // by column of the product
    TallRows &R = *reinterpret_cast<TallRows *>(reinterpret_cast<char *>(lds) + kTallStage);
    auto put3 = [](__bf16 *at, float4 v) {
        bf16x4 p[kSplitParts];
        split_quad(v, p);
#pragma unroll
        for (int q = 0; q < kSplitParts; ++q) *reinterpret_cast<bf16x4 *>(at + q * kSplitK) = p[q];
    };

    // The projection: d % 4 == 0, so a quad lies inside a row or outside it; what lies outside is read from the last quad or row,
    // meets a left operand that is zero there (k) or is stored nowhere (columns).
    float4 m[4];
    const int kb = tid & 7, nb = tid >> 3;
    const char *base = reinterpret_cast<const char *>(M);
    const uint32_t d4 = 4u * (uint32_t)d;
    const uint32_t mcol = 4u * (uint32_t)min(c0 + 4 * nb, d - 4);  // bytes
    auto load_m = [&](int j0) {
        if constexpr (MODE != 2) {
#pragma unroll
            for (int i = 0; i < 4; ++i) m[i] = load_quad(reinterpret_cast<const float *>(base + ((uint32_t)min(j0 + 4 * kb + i, d - 1) * d4 + mcol)));
        } else {
            const uint32_t k = 4u * (uint32_t)min(j0 + 4 * kb, d - 4);
#pragma unroll
            for (int i = 0; i < 4; ++i) m[i] = load_quad(reinterpret_cast<const float *>(base + ((uint32_t)min(c0 + nb + 32 * i, d - 1) * d4 + k)));
        }
    };
    auto put_m = [&] {
        if constexpr (MODE != 2) {
            put3(&sM[4 * nb + 0][4 * kb], make_float4(m[0].x, m[1].x, m[2].x, m[3].x));
            put3(&sM[4 * nb + 1][4 * kb], make_float4(m[0].y, m[1].y, m[2].y, m[3].y));
            put3(&sM[4 * nb + 2][4 * kb], make_float4(m[0].z, m[1].z, m[2].z, m[3].z));
            put3(&sM[4 * nb + 3][4 * kb], make_float4(m[0].w, m[1].w, m[2].w, m[3].w));
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) put3(&sM[nb + 32 * i][4 * kb], m[i]);
        }
    };
    load_m(0);  // (flies during the index chain below)
    __builtin_amdgcn_sched_barrier(0);
    const bool array = a.xs != nullptr && (MODE == 1 || MODE == 2);
    const bool derived = MODE == 2 && !array;
    tall_rows<MODE>(a, R, p0, rows, array, derived);
    __syncthreads();

    // the left operand: thread tid stages the quad tid % 8 of row tid / 8 of a row block (as tall_tile's fetch and put)
    const bool l1 = derived && !a.src.rescal && a.src.norm_p == 1;
    const bool occ = derived && a.src.occ_v && cb == 0;
    constexpr bool kTwo = MODE == 0 || MODE == 3;
    float4 v[RB], w[RB];
    auto load_x = [&](int j0) {
        const int k4 = min(j0 + 4 * kb, d - 4);
#pragma unroll
        for (int i = 0; i < RB; ++i) {
            v[i] = load4g(R.v[32 * i + nb] + k4);
            if constexpr (kTwo) w[i] = load4g(R.w[32 * i + nb] + k4);
            else w[i] = make_float4(0.f, 0.f, 0.f, 0.f);
            if constexpr (MODE == 2)
                if (occ) w[i] = load4g(R.w[32 * i + nb] + k4);
        }
    };
    auto form_x = [&](int row, float4 vv, float4 ww) {
        float4 x = vv;
        if constexpr (MODE == 0) x = make_float4(vv.x - ww.x, vv.y - ww.y, vv.z - ww.z, vv.w - ww.w);
        if constexpr (MODE == 3) {
            const bool keep = R.g[row] != 0.0f;
            x = make_float4(vv.x - (keep ? ww.x : 0.0f), vv.y - (keep ? ww.y : 0.0f), vv.z - (keep ? ww.z : 0.0f), vv.w - (keep ? ww.w : 0.0f));
        }
        if constexpr (MODE == 2)
            if (derived) x = scaled4(R.f[row], l1 ? sgn4(vv) : vv);
        return x;
    };
    auto put_x = [&](int j0) {
        const int col = j0 + 4 * kb;
#pragma unroll
        for (int i = 0; i < RB; ++i) {
            const int row = 32 * i + nb;
            const bool ok = row < rows && col < d;
            const float4 x = form_x(row, v[i], w[i]);
            if constexpr (MODE == 2)
                if (occ && ok)  // RESCAL: the tail's occurrence row g * (E[h] Proj[r])
                    *reinterpret_cast<float4 *>(a.src.occ_v + (int64_t)R.b[row] * d + col) = scaled4(R.g[row], w[i]);
            put3(&sX[row][4 * kb], make_float4(ok ? x.x : 0.0f, ok ? x.y : 0.0f, ok ? x.z : 0.0f, ok ? x.w : 0.0f));
        }
    };

    floatx16 lead[RB], rest[RB];  // sums of the leading products / of the corrections
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) lead[i][e] = 0.0f, rest[i][e] = 0.0f;
    const bool active = 32 * wave < span;  // (uniform per wave)
    load_x(0);
#pragma unroll 1
    for (int j0 = 0; j0 < d; j0 += kSplitK) {
        put_x(j0);
        put_m();
        __syncthreads();
        if (j0 + kSplitK < d) load_x(j0 + kSplitK), load_m(j0 + kSplitK);
        __builtin_amdgcn_sched_barrier(0);  // (the requests go out before the products, not after them)
        if (active) {
#pragma unroll
            for (int u = 0; u < kSplitK / 16; ++u) {
                bf16x8 xv[RB][kSplitParts], mv[kSplitParts];
#pragma unroll
                for (int q = 0; q < kSplitParts; ++q) {
                    mv[q] = *reinterpret_cast<const bf16x8 *>(&sM[32 * wave + fr][q * kSplitK + 16 * u + 8 * fg]);
#pragma unroll
                    for (int i = 0; i < RB; ++i) xv[i][q] = *reinterpret_cast<const bf16x8 *>(&sX[32 * i + fr][q * kSplitK + 16 * u + 8 * fg]);
                }
#pragma unroll
                for (int q = 0; q < kSplitTerms; ++q)
#pragma unroll
                    for (int i = 0; i < RB; ++i) {
                        floatx16 &acc = q + 1 < kSplitTerms ? rest[i] : lead[i];
                        acc = mfma_bf16(xv[i][kTermA[q]], mv[kTermB[q]], acc);
                    }
            }
        }
        __syncthreads();
    }

    // A sum that is not finite (mfma_split.hpp): the caller forms the tile again in fp32.
    const bool colok = 32 * wave + fr < span;
    bool bad = false;
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) lead[i][e] += rest[i][e], bad = bad || (colok && not_finite(lead[i][e]));
    if (__syncthreads_or(bad)) return true;

    // Lane (fr, fg) holds rows 32 i + 8 (e / 4) + 4 fg + e % 4, column c0 + 32 wave + fr.
    const bool want_pos = MODE < 2 && a.pos;
    const int col = colok ? c0 + 32 * wave + fr : c0;
    float rv = 0.0f;  // the relation's row
    if constexpr (MODE == 0 || MODE == 3) rv = a.rel[rid * (int64_t)d + col];
    float *const out = MODE == 2 ? a.occ_h : a.resid;
    float tail[RB][16];  // RESCAL: the tails' rows, all requested before the first of them is waited for
    if (MODE == 1 && want_pos) {  // uniform
#pragma unroll
        for (int i = 0; i < RB; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int row = 32 * i + 8 * (e / 4) + 4 * fg + e % 4;
                tail[i][e] = a.ent[R.t[row < rows ? row : 0] * (int64_t)d + col];
            }
    }
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int e0 = 0; e0 < 16; e0 += 4) {
            const int row0 = 32 * i + 2 * e0 + 4 * fg;
            float y[4];
            int rb[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = row0 + e;
                y[e] = lead[i][e0 + e], rb[e] = R.b[row];
                if constexpr (MODE == 0) y[e] += rv;
                if constexpr (MODE == 3) y[e] += R.f[row] * rv;  // +-1 or 0: exact products
            }
            if constexpr (MODE < 2) {
                if (want_pos) {  // uniform
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        float s;
                        if constexpr (MODE == 1) s = y[e] * tail[i][e0 + e];
                        else s = a.norm_p == 1 ? fabsf(y[e]) : y[e] * y[e];
                        s = row16_sum(colok ? s : 0.0f);
                        if ((fr & 15) == 0) R.sum[2 * wave + (fr >> 4)][row0 + e] = s;
                    }
                }
            }
            if (out && colok) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (row0 + e < rows) {
                        const int64_t o = (int64_t)rb[e] * d + col;
                        out[o] = y[e];
                        if constexpr (MODE == 2)
                            if (a.occ_t) a.occ_t[o] = -y[e];
                    }
            }
        }
    if constexpr (MODE < 2) {
        if (want_pos) {
            __syncthreads();
            if (tid < rows) {
                float s = 0.0f;
#pragma unroll
                for (int q = 0; q < 8; ++q) s += R.sum[q][tid];
                if (ncb > 1) t.part[(int64_t)cb * t.B + R.b[tid]] = s;
                else a.pos[R.b[tid]] = (MODE == 0 && a.norm_p == 2) ? sqrtf(s) : s;
            }
        }
    }
    return false;
}

// SPLIT: launches that may hold more than kSplitItems items (tall_may_split); the others leave the split tiles' code out.
// Two loops over the workgroup's items, not two branches in one: side by side in a loop the two forms' invariants are held at once.
template <int MODE, bool SPLIT>
__global__ __launch_bounds__(256, 3) void transr_tall_kernel(TallArgs t, FusedInsp fi)
{
    extern __shared__ __align__(16) float lds[];
    if (fused_insp_block(fi, reinterpret_cast<uint32_t *>(lds))) return;
    const int ncb = tall_col_blocks(t.g.d), n = t.g.plan.num_tiles[0] * ncb, step = (int)gridDim.x - fi.blocks, first = (int)blockIdx.x - fi.blocks;
    const int split_rows = SPLIT && n > kSplitItems ? kSplitRows : kTallRows;  // tiles of more rows are split
    uint64_t again = 0;  // items (by turn; launch_tall gives a workgroup at most 64) whose sums were not all finite
    auto rows_of = [&](int it) { return t.g.plan.tile_end[it / ncb] - t.g.plan.tile_p0[it / ncb]; };
    if constexpr (SPLIT) {
        for (int it = first, turn = 0; it < n; it += step, ++turn)
            if (rows_of(it) > split_rows) {
                if (split_tile<MODE, 2>(t, lds, it / ncb, it % ncb)) again |= uint64_t(1) << turn;
                __syncthreads();  // the next tile reuses the staging buffers
            }
    }
    for (int it = first, turn = 0; it < n; it += step, ++turn) {
        const int tile = it / ncb, cb = it % ncb, rows = rows_of(it);
        if (SPLIT && rows > split_rows && !((again >> turn) & 1)) continue;
        if (rows > 48) tall_tile<MODE, 4>(t, lds, tile, cb);
        else if (rows > 32) tall_tile<MODE, 3>(t, lds, tile, cb);
        else if (rows > 16) tall_tile<MODE, 2>(t, lds, tile, cb);
        else tall_tile<MODE, 1>(t, lds, tile, cb);
        __syncthreads();
    }
}

// Scores from the column blocks' partial sums, in block order.
__global__ __launch_bounds__(256) void tall_finish_kernel(const float *part, int ncb, int64_t B, int root, float *pos)
{
    const int64_t b = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (b >= B) return;
    float s = 0.0f;
    for (int q = 0; q < ncb; ++q) s += part[q * B + b];
    pos[b] = root ? sqrtf(s) : s;
}

// Whether a launch may hold more than kSplitItems items: by the tiles that groups make on average, the last of each half full.  (A
// kernel with the split tiles' code is slower even where none is split: RESCAL score calls of 6400 triples over 20 relations, width 64
// 8.7 -> 12.0 us, width 200 16.2 -> 21.0.)
static bool tall_may_split(int64_t d, int64_t rows, int64_t groups)
{
    return (rows / kTallRows + groups / 2) * tall_col_blocks((int)d) > kSplitItems;
}

// Whether a batch of `rows` rows in at most n_rel groups goes by these tiles rather than by 32-row tiles and streamed
// small groups (transr_gemm_kernel).  The rule sees the counts, not the distribution.  Both sides measured over 64 to
// 1000 columns, 20 to 1600 groups, 2 to 32 rows per group on average, uniform and Zipf (1.0, 1.2), 64-row time / 32-row
// time of a TransR score call and of its backward, geometric means (extremes):
//   up to 128 columns   one column block: a projection is read half as often.  0.86 (0.67 to 1.09) and 0.92 where these
//                       tiles are taken; at two rows per group and more than 256 tiles 0.92 (0.77 to 1.07)
//   up to 256           two column blocks stage every row twice: only where the 32-row tiles leave compute units idle.
//                       Up to 200 tiles 1.00 (0.79 to 1.17) and 0.94; 201 to 256 tiles 1.17 (1.00 to 1.41) and 0.97;
//                       above 1.17 (0.84 to 1.56) and 0.95.  Groups that fill their tiles' 64 rows on average (from 32 rows per
//                       relation on) go by the bf16 matrix cores there, if the launch has the items for it: score calls 0.73 to 0.98
//                       (8192 triples over 3 to 237 relations, width 132 / 200 / 256), RESCAL's at width 132 1.00 to 1.09; TransR's row
//                       list of 90000 rows over 588 relations below; at 8 rows per relation 0.95 to 1.14, at 2 1.1 to 1.3.  With
//                       fewer items (4000 to 7400 triples over 3 to 100 relations, fp32 tiles) TransR 0.86 to 1.04, mean 0.96, from width
//                       160 on and 1.00 below; RESCAL, whose scores of two column blocks take a kernel more, 0.92 to 1.12, mean 1.03
//   above               a 32-row tile is one workgroup however wide its rows are: few groups leave the chip idle.
//                       0.76 (0.24 to 1.33) and 0.78; where streaming is taken (many groups of a few rows, bound by
//                       reading the projections) 0.95 (0.70 to 1.28) and 0.89
static bool want_tall(int model, int64_t d, int64_t rows, int64_t n_rel)
{
    const int64_t groups = rows < n_rel ? rows : n_rel, short_tiles = groups + rows / 32;
    if (d <= kTallCols) return short_tiles <= 256 || rows >= 4 * n_rel;
    if (d <= 2 * kTallCols) return short_tiles <= 200 || (rows >= 32 * n_rel && (tall_may_split(d, rows, groups) || (model == KGE_TRANSR && d >= 160)));
    return groups <= 256 || rows >= 16 * n_rel;
}

static int64_t tall_tiles(int64_t groups, int64_t rows) { return groups + rows / kTallRows + 1; }
static size_t tall_part_floats(int64_t d, int64_t B) { return tall_col_blocks((int)d) > 1 ? (size_t)tall_col_blocks((int)d) * (size_t)B : 0; }

// max_tiles: upper bound of the plan's tiles (a.plan holds tiles of kTallRows).  part: tall_part_floats() where a.pos is set.
static int launch_tall(int mode, const GemmArgs &a, int64_t max_tiles, bool split, float *part, int64_t B, const FusedInsp &fi, hipStream_t st)
{
    const int ncb = tall_col_blocks(a.d);
    if (a.pos && ncb > 1 && !part) return KGE_EWORKSPACE;
    const TallArgs t{a, part, B};
    const int64_t items = max_tiles * ncb;
    const int64_t wgs = items / 64 + 1 > kTallWgs ? items / 64 + 1 : kTallWgs;  // (at most 64 items each: transr_tall_kernel)
    const dim3 grid((unsigned)((items < wgs ? items : wgs) + fi.blocks)), block(256);
    const size_t lds = fi.blocks > 0 && (size_t)fi.lds_bytes > kTallLds ? (size_t)fi.lds_bytes : kTallLds;
    auto launch = [&](auto plain_kernel, auto split_kernel) { hipLaunchKernelGGL(split ? split_kernel : plain_kernel, grid, block, lds, st, t, fi); };
    switch (mode) {
    case 0: launch(transr_tall_kernel<0, false>, transr_tall_kernel<0, true>); break;
    case 1: launch(transr_tall_kernel<1, false>, transr_tall_kernel<1, true>); break;
    case 2: launch(transr_tall_kernel<2, false>, transr_tall_kernel<2, true>); break;
    default: launch(transr_tall_kernel<3, false>, transr_tall_kernel<3, true>);
    }
    if (a.pos && ncb > 1)
        hipLaunchKernelGGL(tall_finish_kernel, dim3((unsigned)ceil_div(B, 256)), dim3(256), 0, st, part, ncb, B,
                           mode == 0 && a.norm_p == 2 ? 1 : 0, a.pos);
    KGE_CHECK_LAUNCH();
    return KGE_OK;
}
