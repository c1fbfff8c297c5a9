// TransR with shared negatives: every negative is projected once per (relation, chunk) group.
//
// The reference defines the shared-negative TransR score on the flattened batch * blocksize
// triples (apps/examples/examples.py:1447-1480: the views of vh, vt, vr, mr are all expanded to
// output_size rows before bvm), i.e. one vector x matrix product per (positive, negative) pair.
// With x_b the entity the positive keeps (the head; the tail when the negatives replace heads),
// sigma = +1 / -1 and n_k the chunk's negatives, the pair residual splits into two projections,
//     (x_b - n_k) M_r + R_r   =   a_b - P_(g,k),      a_b = x_b M_r + sigma R_r,   P_(g,k) = n_k M_r
// (head mode: (n_k - x_b) M_r + R_r = -(a_b - P_(g,k)), same norm), and P only depends on the
// GROUP g = (relation, chunk) of the positive.  So the batch is turned into one list of rows to
// project, ordered by relation,
//     relation u :  [ positives' own rows (h - t) | their a rows | N rows per group of u ]
// which the grouped matrix-core kernels of transr.hip project in ONE pass (list mode), and small
// per-pair kernels form the scores ||a_b - P_(g(b),k)|| and, backward, the gradients with respect
// to the a and P rows; the chain through the projections (dX = Q M^T, dM = X^T Q) is again one
// grouped pass over the same list.  The matrix-core work drops from B (1 + N) rows to
// 2 B + G N rows, G = number of distinct (relation, chunk) pairs of the batch.
//
// This file is included by transr.hip (inside namespace kge) below the grouped kernels.

constexpr int kNegSeg = 8;  // sorted positions per wave of the P-row gradient sum

struct NegShape {
    int64_t B, N, C, n_chunks, NN, d, U_cap, G_cap, L_cap;
    int64_t dslots;
    PlanSizes plans;
    bool dm_split;
};

static NegShape neg_shape(const kge_tables *tab, const kge_batch *bat)
{
    NegShape s{};
    s.B = bat->batch, s.N = bat->n_neg, s.C = bat->chunk, s.d = tab->dim;
    s.n_chunks = s.C > 0 ? s.B / s.C : 0;
    s.NN = s.n_chunks * s.N;
    s.U_cap = s.B < tab->n_rel ? s.B : tab->n_rel;
    const int64_t pairs = tab->n_rel * s.n_chunks;
    s.G_cap = s.B < pairs ? s.B : pairs;
    s.L_cap = 2 * s.B + s.G_cap * s.N;
    s.plans = PlanSizes{0, s.U_cap + s.L_cap / kDmChunk + 1, s.L_cap / kDmChunk + 1, 0, s.d, tall_may_split(s.d, s.L_cap, s.U_cap)};
    if (want_tall(tab->model, s.d, s.L_cap, tab->n_rel)) s.plans.tall = tall_tiles(s.U_cap, s.L_cap);
    else s.plans.tiles = s.U_cap + s.L_cap / kTM + 1;
    s.dslots = 2 * (s.L_cap / kDmChunk) + 2;
    // dM by items of 128 x 128 where there can be one for each resident workgroup: below that the fp32 items, four to seven times as many,
    // spread a chunk's walk over more of the chip (1024 triples x 128, 50 relations, N = 16: 17.5 us against 28.7; 4096 x 152, 10
    // relations, N = 64: 28.4 against 28.5).  Groups of fewer negatives are a slice or two, all index chain and epilogue (1024 x 200, 500
    // relations, N = 40: 55 against 60), and those of at most kDmSmall rows one workgroup's work in both, three a CU with the fp32 kernel
    // (2048 x 100, 1345 relations, N = 20: 27 against 32).  Above: 4096 x 200, 1345 relations, N = 64 151 -> 123; x 256, 200 relations
    // 262 -> 166; x 48, 2000 relations 98 -> 68; 2048 x 128, 300 relations, N = 48 48 -> 32; 512 x 64, 2000 relations, N = 64 21 -> 17.
    const int64_t nt = dm_split_tiles((int)s.d);
    s.dm_split = s.N >= 48 && s.plans.dtiles * nt * nt >= kDmSplitWgs;
    return s;
}

// forward workspace: the groups, the row list, both tile plans and the projected rows;
// kge_score_bwd finds them through kge_saved.fwd_workspace
struct NegFwdLayout {
    size_t knum, kseg, kinv, ksseg;
    size_t gstart, segl, rowpos, rowa, rowp, hl, tl, rsl, plans, y, total;
};

static NegFwdLayout neg_fwd_layout(const NegShape &s)
{
    NegFwdLayout l{};
    size_t o = 0;
    auto take = [&](size_t bytes) {
        const size_t at = o;
        o += up256(bytes > 0 ? bytes : 1);
        return at;
    };
    l.knum = take(sizeof(int32_t));
    l.kseg = take(sizeof(int32_t) * (s.B + 1));
    l.kinv = take(sizeof(int32_t) * s.B);
    l.ksseg = take(sizeof(int32_t) * s.B);
    l.gstart = take(sizeof(int32_t) * (s.U_cap + 1));
    l.segl = take(sizeof(int32_t) * (s.U_cap + 1));
    l.rowpos = take(sizeof(int32_t) * s.B);
    l.rowa = take(sizeof(int32_t) * s.B);
    l.rowp = take(sizeof(int32_t) * s.G_cap);
    l.hl = take(sizeof(int64_t) * s.L_cap);
    l.tl = take(sizeof(int64_t) * s.L_cap);
    l.rsl = take(sizeof(float) * s.L_cap);
    l.plans = take(plans_bytes(s.plans));
    l.y = take(sizeof(float) * (size_t)(s.L_cap * s.d));
    l.total = o;
    return l;
}

struct NegBwdLayout {
    size_t zero, ql, dxl, occ, qr, glist, gcount, ppart, part_e, part_r, dpart, total;
};

static NegBwdLayout neg_bwd_layout(const NegShape &s)
{
    NegBwdLayout l{};
    size_t o = 0;
    auto take = [&](size_t bytes) {
        const size_t at = o;
        o += up256(bytes > 0 ? bytes : 1);
        return at;
    };
    const size_t rows = sizeof(float) * (size_t)(s.L_cap * s.d);
    l.zero = take(sizeof(float) * ((size_t)s.d + kDmTickets)), l.ql = take(rows), l.dxl = take(rows);
    l.occ = take(sizeof(float) * (size_t)((2 * s.B + s.NN) * s.d));
    l.qr = take(sizeof(float) * (size_t)(s.B * s.d));
    l.glist = take(sizeof(int32_t) * s.B);
    l.gcount = take(sizeof(int32_t) * s.n_chunks);
    l.ppart = take(sizeof(float) * (size_t)(ceil_div(s.B, kNegSeg) * s.N * 2 * s.d));
    l.part_e = take(sizeof(float) * (size_t)seg_partial_floats(2 * s.B + s.NN, s.d));
    l.part_r = take(sizeof(float) * (size_t)seg_partial_floats(s.B, s.d));
    l.dpart = take(sizeof(float) * (size_t)(s.dslots * s.d * s.d));
    l.total = o;
    return l;
}

// Everything the small kernels index with (device pointers into the forward workspace).
struct NegIdx {
    const int64_t *h, *r, *t, *neg;
    // inspection of the relation ids (the caller's rel_insp)
    const int32_t *r_num, *r_seg, *r_perm, *r_inv, *r_sseg;
    const int64_t *r_uniq;
    // the groups (relation, chunk), in relation order: their number, segments of the positions, group of a positive / of a position
    int32_t *k_num, *k_seg, *k_inv, *k_sseg;
    int32_t *gstart, *segl, *rowpos, *rowa, *rowp;
    int64_t *hl, *tl;
    float *rsl;
    int64_t B, N, C, n_chunks, G_cap;
    int d, head;
};

// The groups of positives that share relation and chunk.  The relation inspection's order is stable, so within a relation the positives, and
// with them their chunks, ascend: a group begins where either changes, and its first position holds its smallest positive.  A workgroup
// owns kGroupPos positions and counts the groups that begin before them itself (8 bytes a position), so it waits for no other; four workgroups'
// positions at a time, since the last workgroup of 131072 positions goes through 31.
//   gstart[u]: relation u's first group; segl[u]: its first list row = 2 per positive of the smaller relations + N per group
// (The groups as an inspection of keys relation * n_chunks + chunk, with a kernel for the keys and one for the starts, took 26 us of
// launches at 4096 positives; this one 8.  With the row list and the plan behind it, us, groups before a workgroup one position range at a time / four:
// 32768 positives 33 / 25, 65536 50 / 32, 131072 85 / 47; with the inspection 64, 42 and 74.)
constexpr int kGroupThreads = 1024, kGroupPos = 4 * kGroupThreads;
__global__ __launch_bounds__(kGroupThreads) void tneg_groups_kernel(NegIdx x)
{
    __shared__ int s_wave[kGroupThreads / kWave], s_before[kGroupThreads / kWave];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, B = (int)x.B;
    const uint32_t C = (uint32_t)x.C;
    int b[4], u[4];
    int heads, rel_heads;  // bit i: position p + i begins a group / a relation
    auto look = [&](int p) {  // (unconditional loads: positions past the end read the last one)
        const int pp = min(max(p - 1, 0), B - 1);
        int b0 = x.r_perm[pp], u0 = x.r_sseg[pp];
#pragma unroll
        for (int i = 0; i < 4; ++i) b[i] = x.r_perm[min(p + i, B - 1)], u[i] = x.r_sseg[min(p + i, B - 1)];
        uint32_t c0 = (uint32_t)b0 / C;
        heads = rel_heads = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t c = (uint32_t)b[i] / C;
            const bool first = p + i == 0, rel = first || u[i] != u0;
            if (p + i < B && rel) rel_heads |= 1 << i;
            if (p + i < B && (rel || c != c0)) heads |= 1 << i;
            c0 = c, u0 = u[i];
        }
    };
    const int start = (int)blockIdx.x * kGroupPos;
    int before = 0;
    constexpr int kFly = 4;
    for (int q = 0; q < start; q += kFly * kGroupPos) {
        int eb[kFly][5], eu[kFly][5];
#pragma unroll
        for (int v = 0; v < kFly; ++v) {
            const int at = q + v * kGroupPos < start ? q + v * kGroupPos + 4 * tid : 4 * tid;  // (in front of `start`, or not counted)
#pragma unroll
            for (int i = 0; i < 5; ++i) eb[v][i] = x.r_perm[max(at + i - 1, 0)], eu[v][i] = x.r_sseg[max(at + i - 1, 0)];
        }
#pragma unroll
        for (int v = 0; v < kFly; ++v) {
            int n = q + v * kGroupPos + 4 * tid == 0 ? 1 : 0;  // (position 0 begins a group; its neighbour in front is itself here)
#pragma unroll
            for (int i = 0; i < 4; ++i) n += eu[v][i + 1] != eu[v][i] || (uint32_t)eb[v][i + 1] / C != (uint32_t)eb[v][i] / C ? 1 : 0;
            before += q + v * kGroupPos < start ? n : 0;
        }
    }
    before = wave_sum_i(before);
    const int p = start + 4 * tid;
    look(p);
    int scan = __popc(heads);  // inclusive over the wave
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const int v = __shfl_up(scan, o, kWave);
        if (lane >= o) scan += v;
    }
    if (lane == kWave - 1) s_wave[wave] = scan;
    if (lane == 0) s_before[wave] = before;
    __syncthreads();
    int g = scan - __popc(heads) - 1;  // the group of the position in front of this thread's
    for (int w = 0; w < kGroupThreads / kWave; ++w) g += s_before[w] + (w < wave ? s_wave[w] : 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (p + i >= B) break;
        if (heads >> i & 1) x.k_seg[++g] = p + i;
        x.k_sseg[p + i] = g, x.k_inv[b[i]] = g;
        if (rel_heads >> i & 1) x.gstart[u[i]] = g, x.segl[u[i]] = (int32_t)(2 * (int64_t)(p + i) + x.N * g);
        if (p + i == B - 1) {
            x.k_num[0] = g + 1, x.k_seg[g + 1] = B;
            x.gstart[u[i] + 1] = g + 1, x.segl[u[i] + 1] = (int32_t)(2 * x.B + x.N * (g + 1));
        }
    }
}

// The tile plan of the list product, which needs of the list no more than where the relations' rows start (the first workgroup), beside
// the list rows (entity to project, entity to subtract or -1, factor of the relation row) and where
// each positive's and each group's rows sit.  (The list, then both plans: 5 + 19 us at 90000 rows; the plan of dM, the longer one,
// rides with tneg_pair_fwd_kernel.)
__global__ __launch_bounds__(1024) void tneg_list_kernel(NegIdx x, TilePlan plan, int tile)
{
    __shared__ int s_tot[2][96];
    if (blockIdx.x == 0) return plan_body<false>(x.r_num, x.segl, x.r_uniq, plan, tile, 0, 0, s_tot);
    const int64_t total = x.B + x.G_cap * x.N;
    const int G = x.k_num[0];
    for (int64_t i = ((int64_t)blockIdx.x - 1) * blockDim.x + threadIdx.x; i < total; i += ((int64_t)gridDim.x - 1) * blockDim.x) {
        if (i < x.B) {
            const int p = (int)i;  // position in relation order
            const int u = x.r_sseg[p], s0 = x.r_seg[u], n_u = x.r_seg[u + 1] - s0, j = p - s0;
            const int b = x.r_perm[p];
            const int base = x.segl[u];
            const int64_t hb = x.h[b], tb = x.t[b];
            x.hl[base + j] = hb, x.tl[base + j] = tb, x.rsl[base + j] = 1.0f;
            x.rowpos[b] = base + j;
            const int ra = base + n_u + j;
            x.hl[ra] = x.head ? tb : hb, x.tl[ra] = -1, x.rsl[ra] = x.head ? -1.0f : 1.0f;
            x.rowa[b] = ra;
        } else {
            const int64_t q = i - x.B;
            const int g = (int)(q / x.N), k = (int)(q % x.N);
            if (g >= G) continue;
            const int brep = x.r_perm[x.k_seg[g]];  // any positive of the group names its relation and chunk
            const int u = x.r_inv[brep];
            const int64_t c = brep / x.C;
            const int n_u = x.r_seg[u + 1] - x.r_seg[u];
            const int base = x.segl[u] + 2 * n_u + (g - x.gstart[u]) * (int)x.N;
            x.hl[base + k] = x.neg[c * x.N + k], x.tl[base + k] = -1, x.rsl[base + k] = 0.0f;
            if (k == 0) x.rowp[g] = base;
        }
    }
}

// For chunk c: the first list row of every group that has a positive in the chunk, in the order of the groups' first positives
// (glist[c * C + i], i < gcount[c]).  The first one also clears the row that dM subtracts from list rows without a second
// entity.  A workgroup of 256 threads of tneg_pair_bwd_p2_kernel's launch, which needs none of it (as a launch of its own, a wave a chunk, 11 us).
struct ChunkGroups {
    int32_t *glist, *gcount;
    float *zero_row;
};
__device__ __forceinline__ void tneg_chunk_groups(const NegIdx &x, const ChunkGroups &o, int64_t c)
{
    __shared__ int s_cnt[2][4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (c == 0)
        for (int i = tid; i < x.d + kDmTickets; i += 256) o.zero_row[i] = 0.0f;  // (and the counters behind it)
    int count = 0, turn = 0;
    for (int64_t i0 = 0; i0 < x.C; i0 += 256, turn ^= 1) {
        const int64_t i = i0 + tid;
        const int64_t b = c * x.C + (i < x.C ? i : x.C - 1);
        const int g = x.k_inv[b];
        const bool rep = i < x.C && x.r_perm[x.k_seg[g]] == (int32_t)b;
        const uint64_t m = __ballot(rep);
        if (lane == 0) s_cnt[turn][wave] = __popcll(m);
        __syncthreads();  // (one a turn: the counts alternate between two places)
        int at = count;
        for (int w = 0; w < 4; ++w) {
            if (w < wave) at += s_cnt[turn][w];
            count += s_cnt[turn][w];
        }
        if (rep) o.glist[c * x.C + at + __popcll(m & ((1ull << lane) - 1))] = x.rowp[g];
    }
    if (tid == 0) o.gcount[c] = count;
}

// A row held by a wave: NQ float4 per lane (NQ = ceil(dim / 256) <= 4, a template parameter of
// the kernels so that narrow rows issue no idle loads).
template <int NQ>
struct NegRow {
    float4 v[NQ];
};

template <int NQ>
__device__ __forceinline__ NegRow<NQ> neg_load_row(const float *p, int d, int lane)
{
    NegRow<NQ> r;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int j = q * 256 + lane * 4;
        const float4 v = *reinterpret_cast<const float4 *>(p + (j < d ? j : 0));  // clamped: unconditional load
        r.v[q] = j < d ? v : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    return r;
}

template <int NQ>
__device__ __forceinline__ void neg_store_row(float *p, int d, int lane, const NegRow<NQ> &r)
{
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int j = q * 256 + lane * 4;
        if (j < d) *reinterpret_cast<float4 *>(p + j) = r.v[q];
    }
}

template <int P, int NQ>
__device__ __forceinline__ float neg_norm_partial(const NegRow<NQ> &a, const NegRow<NQ> &p)
{
    float s = 0.0f;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const float u0 = a.v[q].x - p.v[q].x, u1 = a.v[q].y - p.v[q].y, u2 = a.v[q].z - p.v[q].z, u3 = a.v[q].w - p.v[q].w;
        if constexpr (P == 1) s += (fabsf(u0) + fabsf(u1)) + (fabsf(u2) + fabsf(u3));
        else s = fmaf(u0, u0, fmaf(u1, u1, fmaf(u2, u2, fmaf(u3, u3, s))));
    }
    return s;
}

struct NegPairArgs {
    const float *ent;
    const float *y;         // projected list rows [L, d]
    float *pos, *neg;       // forward outputs (pos nullable)
    float *resid;           // forward: positives' residual rows [B, d] (nullable)
    const float *dpos, *dneg, *spos, *sneg;  // backward inputs (dpos / dneg nullable)
    float *ql, *qr;         // backward: upstream rows of the list, per-positive relation rows
};

// One wave per positive: pos[b] = ||y_pos||, neg[b][k] = ||a_b - P_(g(b),k)||.  The first workgroups make the plan of the backward pass's dM (one alone
// took longer than all the pairs: 36 us against 25).
struct DmPlanArgs {
    TilePlan plan;
    int chunk, nib, small_max;
};
constexpr int kPairFwdWaves = 16;
template <int P, int NQ>
__global__ __launch_bounds__(kWave *kPairFwdWaves) void tneg_pair_fwd_kernel(NegIdx x, NegPairArgs a, DmPlanArgs dm)
{
    __shared__ int s_tot[2][96];
    if (blockIdx.x < kPlanShares) return plan_body<true>(x.r_num, x.segl, x.r_uniq, dm.plan, dm.chunk, dm.nib, dm.small_max, s_tot, (int)blockIdx.x);
    const int lane = threadIdx.x & 63;
    const int64_t b = ((int64_t)blockIdx.x - kPlanShares) * kPairFwdWaves + (threadIdx.x >> 6);
    if (b >= x.B) return;
    const int d = x.d;
    const int N = (int)x.N;
    const NegRow<NQ> ya = neg_load_row<NQ>(a.y + (int64_t)x.rowa[b] * d, d, lane);
    const float *pg = a.y + (int64_t)x.rowp[x.k_inv[b]] * d;
    if (a.pos || a.resid) {
        const NegRow<NQ> yp = neg_load_row<NQ>(a.y + (int64_t)x.rowpos[b] * d, d, lane);
        NegRow<NQ> z;
#pragma unroll
        for (int q = 0; q < NQ; ++q) z.v[q] = make_float4(0.f, 0.f, 0.f, 0.f);
        const float s = wave_sum(neg_norm_partial<P, NQ>(yp, z));
        if (a.pos && lane == 0) a.pos[b] = P == 2 ? sqrtf(s) : s;
        if (a.resid) neg_store_row(a.resid + b * (int64_t)d, d, lane, yp);
    }
    for (int k0 = 0; k0 < N; k0 += 4) {  // four rows in flight
        NegRow<NQ> p[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) p[u] = neg_load_row<NQ>(pg + (int64_t)(k0 + u < N ? k0 + u : N - 1) * d, d, lane);
        float s[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) s[u] = neg_norm_partial<P, NQ>(ya, p[u]);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1)
#pragma unroll
            for (int u = 0; u < 4; ++u) s[u] += __shfl_xor(s[u], o, kWave);
        if (lane < 4 && k0 + lane < N) {
            const float v = lane == 0 ? s[0] : (lane == 1 ? s[1] : (lane == 2 ? s[2] : s[3]));
            a.neg[b * (int64_t)N + k0 + lane] = P == 2 ? sqrtf(v) : v;
        }
    }
}

// Backward of the pairs, one pass.  A workgroup owns kNegSeg consecutive positions of the key order, in which the positives of a group sit
// next to each other, and 256 columns of the rows, a lane one of them.  It holds the group's P rows (KN negatives) in registers beside their
// sums and walks its positives: a pair element is formed once and goes into both
//   the a row's upstream gradient   ga_b = sum over k of c_bk phi(a_b - P_k)       (whole in one lane: no sum across lanes), and
//   the P row's                     Q_k  = - sum over the group's b of the same.
// A group that lies wholly inside the block leaves its Q rows final, one that began in an earlier block goes to partial slot 0 of the
// block, one that continues past it to slot 1 (the scheme of seg_reduce.hip); tneg_pair_bwd_p2_kernel adds those up.  The order of
// every sum is fixed by the sorted order.  The positives' own rows (upstream rows of both list rows, the row that goes to the
// relation table) are finished here as well.
//   Bound by the rows it reads (P rows once per block and group, 90 MB at 4096 x 64 x 200) and the stores behind them.  As two kernels, a wave
//   per positive over its group's P rows and a wave per (eight positions, negative) over both rows of every pair, it was 600 MB out of the
//   L2 and 144 us; now 55 us (4096 positives x 64 negatives x 200, 1270 groups).
template <int P, int KN>
__global__ __launch_bounds__(256) void tneg_pair_bwd_kernel(NegIdx x, NegPairArgs a, float *partial)
{
    __shared__ float s_c[kNegSeg][kWave];   // the pairs' coefficients, KN negatives at a time
    __shared__ float s_ga[kNegSeg][256];
    __shared__ int s_b[kNegSeg], s_g[kNegSeg], s_pa[kNegSeg], s_pp[kNegSeg];
    const int tid = threadIdx.x, lane = tid & 63, d = x.d, N = (int)x.N;
    const int64_t j = blockIdx.x, p0 = j * kNegSeg;
    const int cnt = (int)(x.B - p0 < kNegSeg ? x.B - p0 : kNegSeg);
    const int col = (int)blockIdx.y * 256 + tid;
    const bool colok = col < d;
    const int cc = colok ? col : d - 1;  // clamped: unconditional loads
    if (tid < kNegSeg) {
        const int64_t pc = p0 + (tid < cnt ? tid : cnt - 1);
        const int b = x.r_perm[pc], g = x.k_sseg[pc];
        s_b[tid] = b, s_g[tid] = g, s_pa[tid] = x.rowa[b], s_pp[tid] = x.rowp[g];
    }
    const int g_before = p0 > 0 ? x.k_sseg[p0 - 1] : -1, g_after = p0 + cnt < x.B ? x.k_sseg[p0 + cnt] : -1;
#pragma unroll
    for (int q = 0; q < kNegSeg; ++q) s_ga[q][tid] = 0.0f;
    __syncthreads();
    if (a.dneg) {  // uniform
        for (int k0 = 0; k0 < N; k0 += KN) {
            const int kn = N - k0 < KN ? N - k0 : KN;
            for (int i = tid; i < kNegSeg * KN; i += 256) {
                const int q = i / KN, k = i % KN;
                float c = 0.0f;
                if (q < cnt && k < kn) {
                    const int64_t o = s_b[q] * (int64_t)N + k0 + k;
                    c = a.dneg[o];
                    if constexpr (P == 2) {
                        const float s = a.sneg[o];
                        c = s > 0.0f ? c / s : 0.0f;
                    }
                }
                s_c[q][k] = c;
            }
            __syncthreads();
            float pr[KN], sum[KN];
            int g = -1;
            auto flush = [&] {
                if (!colok) return;
                float *dst;
                int64_t stride = d;
                if (g == g_before) dst = partial + ((j * N + k0) * 2 + 0) * (int64_t)d, stride = 2 * d;
                else if (g == g_after) dst = partial + ((j * N + k0) * 2 + 1) * (int64_t)d, stride = 2 * d;
                else dst = a.ql + ((int64_t)x.rowp[g] + k0) * d;
#pragma unroll
                for (int k = 0; k < KN; ++k)
                    if (k < kn) dst[k * stride + col] = sum[k];
            };
            float ya = a.y[(int64_t)s_pa[0] * d + cc];
#pragma unroll 1
            for (int q = 0; q < cnt; ++q) {
                if (s_g[q] != g) {  // uniform
                    if (g >= 0) flush();
                    g = s_g[q];
                    const float *src = a.y + ((int64_t)s_pp[q] + k0) * d + cc;
#pragma unroll
                    for (int k = 0; k < KN; ++k) pr[k] = src[(k < kn ? k : kn - 1) * (int64_t)d], sum[k] = 0.0f;
                }
                const float next = a.y[(int64_t)s_pa[q + 1 < cnt ? q + 1 : q] * d + cc];
                const float cv = s_c[q][lane & (KN - 1)];
                float ga = 0.0f;
#pragma unroll
                for (int k = 0; k < KN; ++k) {
                    const float c = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cv), k));
                    const float u = ya - pr[k], ph = P == 1 ? sgn(u) : u;
                    ga = fmaf(c, ph, ga);
                    sum[k] = fmaf(-c, ph, sum[k]);
                }
                s_ga[q][tid] += ga;
                ya = next;
            }
            flush();
            __syncthreads();  // the next turn's coefficients
        }
    } else {
        // no upstream gradient for the pairs: zero rows, by the blocks in which a group starts
        for (int q = 0; q < cnt && colok; ++q)
            if (p0 + q == x.k_seg[s_g[q]])
                for (int k = 0; k < N; ++k) a.ql[((int64_t)s_pp[q] + k) * d + col] = 0.0f;
        for (int k = 0; k < N && colok; ++k) partial[((j * N + k) * 2 + 0) * (int64_t)d + col] = 0.0f, partial[((j * N + k) * 2 + 1) * (int64_t)d + col] = 0.0f;
    }
    if (!colok) return;  // (no barrier below)
    const float sg = x.head ? -1.0f : 1.0f;
#pragma unroll 2
    for (int q = 0; q < cnt; ++q) {
        const int b = s_b[q], ra = s_pa[q], rp = x.rowpos[b];
        const float yp = a.y[(int64_t)rp * d + col];
        float gs = a.dpos ? a.dpos[b] : 0.0f;
        if constexpr (P == 2) {
            const float s = a.spos[b];
            gs = s > 0.0f ? gs / s : 0.0f;
        }
        const float qp = gs * (P == 1 ? sgn(yp) : yp), ga = s_ga[q][tid];
        a.ql[(int64_t)rp * d + col] = qp;
        a.ql[(int64_t)ra * d + col] = ga;
        a.qr[b * (int64_t)d + col] = fmaf(sg, ga, qp);
    }
}

template <int NQ>
__global__ __launch_bounds__(256) void tneg_pair_bwd_p2_kernel(NegIdx x, const float *partial, float *ql, ChunkGroups chunks)
{
    if ((int64_t)blockIdx.x < x.n_chunks) return tneg_chunk_groups(x, chunks, blockIdx.x);
    const int lane = threadIdx.x & 63;
    const int64_t w = ((int64_t)blockIdx.x - x.n_chunks) * 4 + (threadIdx.x >> 6);
    const int N = (int)x.N, d = x.d;
    const int64_t j = w / N;
    const int k = (int)(w % N);
    const int64_t p0 = j * kNegSeg;
    if (p0 >= x.B) return;
    const int64_t p1 = p0 + kNegSeg < x.B ? p0 + kNegSeg : x.B;
    const int g = x.k_sseg[p1 - 1];
    const int s0 = x.k_seg[g], s1 = x.k_seg[g + 1];
    if (s1 <= p0 + kNegSeg || s0 < p0) return;  // no group starts here and continues
    const int64_t je = (s1 - 1) / kNegSeg;
    NegRow<NQ> acc = neg_load_row<NQ>(partial + ((j * N + k) * 2 + 1) * (int64_t)d, d, lane);
    constexpr int kFly = NQ == 1 ? 8 : (NQ == 2 ? 4 : 2);
    for (int64_t jj = j + 1; jj <= je; jj += kFly) {
        NegRow<NQ> t[kFly];
#pragma unroll
        for (int u = 0; u < kFly; ++u) t[u] = neg_load_row<NQ>(partial + (((jj + u <= je ? jj + u : je) * N + k) * 2) * (int64_t)d, d, lane);
#pragma unroll
        for (int u = 0; u < kFly; ++u)
            if (jj + u <= je) {
#pragma unroll
                for (int e = 0; e < NQ; ++e)
                    acc.v[e] = make_float4(acc.v[e].x + t[u].v[e].x, acc.v[e].y + t[u].v[e].y, acc.v[e].z + t[u].v[e].z,
                                           acc.v[e].w + t[u].v[e].w);
            }
    }
    neg_store_row(ql + (int64_t)(x.rowp[g] + k) * d, d, lane, acc);
}

// Occurrence rows in the order of the entity inspection, concat(h, t, neg): the list's dX rows are
// added up per positive (own row and a row: one wave each, the first workgroups) and per
// (chunk, negative) over the chunk's groups (one workgroup each: its waves take the groups i = wave, wave + occ_waves(), ... and
// their sums are added in wave order through LDS).  Bound by the chain of round trips per wave: 159 groups a chunk in four waves 34 us,
// in sixteen 21 us (65 MB).
template <int NQ>
constexpr int occ_waves() { return NQ == 1 ? 16 : 8; }  // (wider rows: registers for eight rows in flight)
template <int NQ>
__global__ __launch_bounds__(kWave * occ_waves<NQ>()) void tneg_occ_kernel(NegIdx x, const float *dxl, const int32_t *glist,
                                                       const int32_t *gcount, float *occ)
{
    constexpr int kOccWaves = occ_waves<NQ>();
    __shared__ float4 s_part[kOccWaves - 1][NQ * kWave];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int d = x.d;
    const int64_t pos_blocks = ceil_div(x.B, kOccWaves);
    if ((int64_t)blockIdx.x < pos_blocks) {
        const int64_t w = (int64_t)blockIdx.x * kOccWaves + wave;
        if (w >= x.B) return;
        const NegRow<NQ> dp = neg_load_row<NQ>(dxl + (int64_t)x.rowpos[w] * d, d, lane), da = neg_load_row<NQ>(dxl + (int64_t)x.rowa[w] * d, d, lane);
        NegRow<NQ> oh, ot;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const float4 p = dp.v[q], v = da.v[q];
            if (x.head) {
                oh.v[q] = p;
                ot.v[q] = make_float4(v.x - p.x, v.y - p.y, v.z - p.z, v.w - p.w);
            } else {
                oh.v[q] = make_float4(p.x + v.x, p.y + v.y, p.z + v.z, p.w + v.w);
                ot.v[q] = make_float4(-p.x, -p.y, -p.z, -p.w);
            }
        }
        neg_store_row(occ + w * (int64_t)d, d, lane, oh);
        neg_store_row(occ + (x.B + w) * (int64_t)d, d, lane, ot);
        return;
    }
    const int64_t q = (int64_t)blockIdx.x - pos_blocks;  // (chunk, negative); uniform for the workgroup
    if (q >= x.n_chunks * x.N) return;
    const int64_t c = q / x.N;
    const int k = (int)(q % x.N);
    const int cnt = gcount[c];
    NegRow<NQ> acc;
#pragma unroll
    for (int e = 0; e < NQ; ++e) acc.v[e] = make_float4(0.f, 0.f, 0.f, 0.f);
    constexpr int kFly = NQ == 1 ? 8 : (NQ == 2 ? 4 : 2);  // groups in flight per wave
    for (int i = wave; i < cnt; i += kOccWaves * kFly) {
        NegRow<NQ> r[kFly];
#pragma unroll
        for (int u = 0; u < kFly; ++u) {
            const int iu = i + kOccWaves * u;
            r[u] = neg_load_row<NQ>(dxl + (int64_t)(glist[c * x.C + (iu < cnt ? iu : i)] + k) * d, d, lane);
        }
#pragma unroll
        for (int u = 0; u < kFly; ++u)
            if (i + kOccWaves * u < cnt) {
#pragma unroll
                for (int e = 0; e < NQ; ++e)
                    acc.v[e] = make_float4(acc.v[e].x + r[u].v[e].x, acc.v[e].y + r[u].v[e].y, acc.v[e].z + r[u].v[e].z,
                                           acc.v[e].w + r[u].v[e].w);
            }
    }
    if (wave > 0) {
#pragma unroll
        for (int e = 0; e < NQ; ++e) s_part[wave - 1][e * kWave + lane] = acc.v[e];
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
        for (int e = 0; e < NQ; ++e)
            for (int w = 0; w + 1 < kOccWaves; ++w) {
                const float4 p = s_part[w][e * kWave + lane];
                acc.v[e] = make_float4(acc.v[e].x + p.x, acc.v[e].y + p.y, acc.v[e].z + p.z, acc.v[e].w + p.w);
            }
        neg_store_row(occ + (2 * x.B + q) * (int64_t)d, d, lane, acc);
    }
}

// ---- host side --------------------------------------------------------------------------------
// launch `stmt` with NQ_ = float4 per lane of a row (dim <= 1024: 1..4)
#define TNEG_BY_WIDTH(d_, stmt)            \
    do {                                   \
        const int nq_ = ((d_) + 255) / 256; \
        if (nq_ <= 1) {                    \
            constexpr int NQ_ = 1;         \
            stmt;                          \
        } else if (nq_ == 2) {             \
            constexpr int NQ_ = 2;         \
            stmt;                          \
        } else if (nq_ == 3) {             \
            constexpr int NQ_ = 3;         \
            stmt;                          \
        } else {                           \
            constexpr int NQ_ = 4;         \
            stmt;                          \
        }                                  \
    } while (0)
#define TNEG_BY_NORM(p_, kern, W_, grid_, ...)                                                          \
    do {                                                                                            \
        if ((p_) == 1) hipLaunchKernelGGL((kern<1, W_>), grid_, dim3(256), 0, st, __VA_ARGS__);    \
        else hipLaunchKernelGGL((kern<2, W_>), grid_, dim3(256), 0, st, __VA_ARGS__);              \
    } while (0)
// The workspaces are sized for the worst case G = min(B, n_rel * n_chunks) groups (the count is only known on
// the device): about four arrays of (2 B + G N) * dim floats, with many relations about four times the
// B * N * dim floats of the flattened triples.  Above this many bytes (forward + backward) the path declines and
// the caller scores the flattened triples (or sees the shape in the error), instead of running out of memory.
constexpr size_t kNegWorkspaceCap = size_t(24) << 30;

static bool transr_neg_path_ok(const kge_tables *tab, const kge_batch *bat)
{
    if (tab->model != KGE_TRANSR || !bat->neg || !bat->rel_insp) return false;
    if (!mfma_path_ok(tab, bat) || gemm_lds_bytes((int)tab->dim) > kMaxGemmLds) return false;
    const NegShape s = neg_shape(tab, bat);
    if (!(s.n_chunks > 0 && tab->n_rel * s.n_chunks < (int64_t(1) << 31) && s.L_cap < (int64_t(1) << 31) &&
          s.L_cap * s.d < (int64_t(1) << 36)))
        return false;
    return neg_fwd_layout(s).total + neg_bwd_layout(s).total <= kNegWorkspaceCap;
}

size_t transr_neg_fwd_workspace(const kge_tables *tab, const kge_batch *bat)
{
    if (!transr_neg_path_ok(tab, bat)) return 0;
    return neg_fwd_layout(neg_shape(tab, bat)).total;
}

size_t transr_neg_bwd_workspace(const kge_tables *tab, const kge_batch *bat)
{
    if (!transr_neg_path_ok(tab, bat)) return 0;
    return neg_bwd_layout(neg_shape(tab, bat)).total;
}

static NegIdx neg_idx(const kge_tables *tab, const kge_batch *bat, const NegShape &s, const NegFwdLayout &l, char *ws)
{
    const kge_inspection *ri = bat->rel_insp;
    NegIdx x{};
    x.h = bat->h, x.r = bat->r, x.t = bat->t, x.neg = bat->neg;
    x.r_num = ri->num_unique, x.r_seg = ri->seg_offsets, x.r_perm = ri->perm, x.r_inv = ri->inverse, x.r_sseg = ri->sorted_seg;
    x.r_uniq = ri->unique_ids;
    x.k_num = reinterpret_cast<int32_t *>(ws + l.knum);
    x.k_seg = reinterpret_cast<int32_t *>(ws + l.kseg);
    x.k_inv = reinterpret_cast<int32_t *>(ws + l.kinv);
    x.k_sseg = reinterpret_cast<int32_t *>(ws + l.ksseg);
    x.gstart = reinterpret_cast<int32_t *>(ws + l.gstart);
    x.segl = reinterpret_cast<int32_t *>(ws + l.segl);
    x.rowpos = reinterpret_cast<int32_t *>(ws + l.rowpos);
    x.rowa = reinterpret_cast<int32_t *>(ws + l.rowa);
    x.rowp = reinterpret_cast<int32_t *>(ws + l.rowp);
    x.hl = reinterpret_cast<int64_t *>(ws + l.hl);
    x.tl = reinterpret_cast<int64_t *>(ws + l.tl);
    x.rsl = reinterpret_cast<float *>(ws + l.rsl);
    x.B = s.B, x.N = s.N, x.C = s.C, x.n_chunks = s.n_chunks, x.G_cap = s.G_cap;
    x.d = (int)tab->dim, x.head = bat->neg_mode == KGE_NEG_HEAD ? 1 : 0;
    return x;
}

int launch_transr_neg_fwd(const kge_tables *tab, const kge_batch *bat, float *pos, float *neg, float *resid, void *workspace,
                          size_t workspace_bytes, hipStream_t st)
{
    if (!transr_neg_path_ok(tab, bat)) return KGE_EUNSUPPORTED;
    if (bat->fuse_inspection) return KGE_EINVAL;  // no kernel of this path hosts the inspector's workgroups
    if (!neg) return KGE_EINVAL;
    const NegShape s = neg_shape(tab, bat);
    const NegFwdLayout l = neg_fwd_layout(s);
    if (!workspace || workspace_bytes < l.total || !aligned16(workspace)) return KGE_EWORKSPACE;
    char *ws = static_cast<char *>(workspace);
    const NegIdx x = neg_idx(tab, bat, s, l, ws);
    const kge_inspection *ri = bat->rel_insp;
    const int d = (int)tab->dim;

    // the groups, the list and its tile plans
    hipLaunchKernelGGL(tneg_groups_kernel, dim3((unsigned)ceil_div(s.B, kGroupPos)), dim3(kGroupThreads), 0, st, x);
    const int64_t list_threads = s.B + s.G_cap * s.N;
    const int64_t list_blocks = ceil_div(list_threads, 1024);
    const Plans plans = plans_at(ws + l.plans, s.plans);
    hipLaunchKernelGGL(tneg_list_kernel, dim3((unsigned)(list_blocks < 2048 ? list_blocks : 2048) + 1), dim3(1024), 0, st, x,
                       s.plans.tall ? plans.tall : plans.tiles, s.plans.tall ? kTallRows : kTM);
    timeline_mark(bat->timeline, st, "groups + row list + plan");

    // one grouped pass projects every list row
    float *y = reinterpret_cast<float *>(ws + l.y);
    GemmArgs ga{tab->ent, tab->rel, tab->aux, x.hl, nullptr, x.tl, nullptr, x.segl, ri->num_unique, ri->unique_ids,
                TilePlan{}, nullptr, x.rsl, nullptr, y, nullptr, nullptr, d, tab->norm_p, 0, 0, BwdSrc{}};
    if (const int rc = launch_product(3, ga, plans, s.plans, s.U_cap, nullptr, s.B, FusedInsp{}, st)) return rc;
    timeline_mark(bat->timeline, st, s.plans.tall ? "transr_tall_kernel<list>" : "transr_gemm_kernel<list>");

    NegPairArgs pa{};
    pa.ent = tab->ent, pa.y = y, pa.pos = pos, pa.neg = neg, pa.resid = resid;
    const DmPlanArgs dm{plans.dm, kDmChunk, dm_nib(d, s.dm_split), dm_small_max(d)};
    const dim3 pgrid((unsigned)ceil_div(s.B, kPairFwdWaves) + kPlanShares), pblock(kWave * kPairFwdWaves);
    TNEG_BY_WIDTH(d, hipLaunchKernelGGL((tab->norm_p == 1 ? tneg_pair_fwd_kernel<1, NQ_> : tneg_pair_fwd_kernel<2, NQ_>), pgrid, pblock, 0, st, x, pa, dm));
    timeline_mark(bat->timeline, st, "tneg_pair_fwd_kernel");
    KGE_CHECK_LAUNCH();
    return KGE_OK;
}

int launch_transr_neg_bwd(const kge_tables *tab, const kge_batch *bat, const kge_saved *saved, const float *dpos,
                          const float *dneg, const kge_grads *grads, void *workspace, size_t workspace_bytes, hipStream_t st)
{
    if (!transr_neg_path_ok(tab, bat)) return KGE_EUNSUPPORTED;
    if (bat->fuse_inspection) return KGE_EINVAL;
    const NegShape s = neg_shape(tab, bat);
    const NegFwdLayout fl = neg_fwd_layout(s);
    const NegBwdLayout l = neg_bwd_layout(s);
    // the forward call's workspace holds the groups, the list, the plans and the projected rows
    if (!saved->fwd_workspace || saved->fwd_workspace_bytes < fl.total) return KGE_EINVAL;
    if (!workspace || workspace_bytes < l.total || !aligned16(workspace)) return KGE_EWORKSPACE;
    if (!grads->ent_rows || !grads->rel_rows || !grads->aux_rows) return KGE_EINVAL;
    // the per-positive kernel reads the positive scores whenever the norm is L2 (dpos == NULL stands for
    // zeros, not for "skip"), so they are required as in launch_transr_bwd
    if (tab->norm_p == 2 && (!saved->pos || (dneg && !saved->neg))) return KGE_EINVAL;
    if (!bat->ent_insp || bat->ent_insp->n != 2 * s.B + s.NN) return KGE_ESHAPE;
    char *fws = static_cast<char *>(const_cast<void *>(saved->fwd_workspace)), *ws = static_cast<char *>(workspace);
    const NegIdx x = neg_idx(tab, bat, s, fl, fws);
    const kge_inspection *ri = bat->rel_insp;
    const int d = (int)tab->dim;
    float *y = reinterpret_cast<float *>(fws + fl.y);
    float *zero_row = reinterpret_cast<float *>(ws + l.zero), *ql = reinterpret_cast<float *>(ws + l.ql);
    float *dxl = reinterpret_cast<float *>(ws + l.dxl), *occ = reinterpret_cast<float *>(ws + l.occ);
    float *qr = reinterpret_cast<float *>(ws + l.qr);
    int32_t *glist = reinterpret_cast<int32_t *>(ws + l.glist), *gcount = reinterpret_cast<int32_t *>(ws + l.gcount);
    const Plans plans = plans_at(fws + fl.plans, s.plans);

    NegPairArgs pa{};
    pa.ent = tab->ent, pa.y = y, pa.dpos = dpos, pa.dneg = dneg, pa.spos = saved->pos, pa.sneg = saved->neg;
    pa.ql = ql, pa.qr = qr;
    float *ppart = reinterpret_cast<float *>(ws + l.ppart);
    const dim3 bgrid((unsigned)ceil_div(s.B, kNegSeg), (unsigned)ceil_div(d, 256));
    if (s.N <= 16) TNEG_BY_NORM(tab->norm_p, tneg_pair_bwd_kernel, 16, bgrid, x, pa, ppart);
    else if (s.N <= 32) TNEG_BY_NORM(tab->norm_p, tneg_pair_bwd_kernel, 32, bgrid, x, pa, ppart);
    else TNEG_BY_NORM(tab->norm_p, tneg_pair_bwd_kernel, 64, bgrid, x, pa, ppart);
    const dim3 sgrid((unsigned)(ceil_div(ceil_div(s.B, kNegSeg) * s.N, 4) + s.n_chunks));
    const ChunkGroups chunks{glist, gcount, zero_row};
    TNEG_BY_WIDTH(d, hipLaunchKernelGGL(tneg_pair_bwd_p2_kernel<NQ_>, sgrid, dim3(256), 0, st, x, ppart, ql, chunks));
    timeline_mark(bat->timeline, st, "tneg_pair_bwd kernels");

    // dX = Q M^T over the list (rows stay in list order), dM = X^T Q per relation
    GemmArgs ga{tab->ent, tab->rel, tab->aux, x.hl, nullptr, x.tl, nullptr, x.segl, ri->num_unique, ri->unique_ids,
                TilePlan{}, ql, nullptr, nullptr, nullptr, dxl, nullptr, d, tab->norm_p, 0, 0, BwdSrc{}};
    if (const int rc = launch_product(2, ga, plans, s.plans, s.U_cap, nullptr, s.B, FusedInsp{}, st)) return rc;
    timeline_mark(bat->timeline, st, s.plans.tall ? "transr_tall_kernel<dX>" : "transr_gemm_kernel<dX>");
    DmArgs da{nullptr, ql, x.segl, plans.dm, grads->aux_rows, reinterpret_cast<float *>(ws + l.dpart), d, ri->num_unique,
              BwdSrc{}, nullptr, nullptr, 0, tab->ent, x.hl, x.tl, zero_row, reinterpret_cast<int32_t *>(zero_row + d)};
    if (s.dm_split) hipLaunchKernelGGL(transr_dm_split_kernel, dim3((unsigned)kDmSplitWgs), dim3(256), dm_split_lds_bytes(d), st, da);
    else hipLaunchKernelGGL(transr_dm_kernel, dim3((unsigned)kDmWgs), dim3(256), dm_lds_bytes(d), st, da, FusedInsp{}, SegL1Rider{});
    timeline_mark(bat->timeline, st, s.dm_split ? "transr_dm_split_kernel" : "transr_dm_kernel");
    TNEG_BY_WIDTH(d, hipLaunchKernelGGL(tneg_occ_kernel<NQ_>, dim3((unsigned)(ceil_div(s.B, occ_waves<NQ_>()) + s.NN)), dim3(kWave * occ_waves<NQ_>()), 0, st, x, dxl,
                                        glist, gcount, occ));
    timeline_mark(bat->timeline, st, "tneg_occ_kernel");
    KGE_CHECK_LAUNCH();
    if (bat->insp_ready && hipStreamWaitEvent(st, reinterpret_cast<hipEvent_t>(bat->insp_ready), 0) != hipSuccess)
        return KGE_ELAUNCH;
    const SegJob jobs[2] = {{occ, bat->ent_insp, d, grads->ent_rows, reinterpret_cast<float *>(ws + l.part_e), false},
                            {qr, ri, d, grads->rel_rows, reinterpret_cast<float *>(ws + l.part_r), false}};
    const SumRider finish = dm_finish_rider(da, s.plans.dsplit);  // the split groups' partial matrices
    return launch_seg_reduce_jobs(jobs, 2, st, bat->timeline, &finish, false, bat->loss_total);
}
