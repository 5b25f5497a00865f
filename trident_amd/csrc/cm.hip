// Cluster-major exact scan (mode 10) on the matrix cores, for gfx950.
//
// The reference's CM-FP32 (src/trident_v4_kernels.cu:268-374) gives every (query, cluster) pair
// one block that walks the cluster's float32 rows with one warp per row, and keeps a per-pair
// top-K in shared memory.  Here a work unit is one slice of a cluster (whole 64-vector blocks)
// and up to 128 (past 256 dims 64) of the queries that probe it (the batched route's units), so
// each row block is read from HBM once per unit, and the query x vector products are dense 16 x 16
// tiles: queries are the A rows (held in registers), vectors the B columns (read from LDS), on
// v_mfma_f32_16x16x32_bf16 over three-part bfloat16 operands, past 256 dims on
// v_mfma_f32_16x16x4f32.
//
// Exactness.  For float32 vectors q, x (exact reals), d = |q - x|^2 = nq + nx - 2 q.x with
// nq = |q|^2, nx = |x|^2:
//   s   = the matrix-core dot product in any association, |s - q.x| <= kappa sum |q_d x_d| <=
//         kappa |q| |x|, each product and addition taken with relative error <= 2^-23 (round to
//         nearest gives 2^-24; the factor two also covers truncation):
//         * float32 products (past 256 dims): kappa = (D_pad + 8) 2^-23 (1 + 2^-10), recursive
//           summation over at most D_pad + 8 roundings on any path, first order plus its rest;
//         * three-part bfloat16 operands x = h + m + l + r, |m| <= 2^-8 (1 + 2^-8) |x|, |l| <= 2^-16
//           (1 + 2^-7) |x|, |r| <= 2^-24 |x| (up to 256 dims): the h h products pass through at
//           most D_pad + 4 additions; h m, m h, h l, m m, l h (together <= 2^-7 (1 + 2^-5) |q_d x_d|)
//           share an accumulator, at most 5 D_pad + 4 additions; the dropped terms are <= 4.2 *
//           2^-24 |q_d x_d|: kappa = (D_pad + 4) 2^-23 (1 + 2^-7) + (5 D_pad + 4) 2^-30 (1 + 2^-5)
//           + 4.2 * 2^-24.  Parts or products below 2^-126 that the matrix cores flush add at
//           most 6 D_pad 2^-126 (1 + |q| + |x|) absolutely, which E carries as D_pad 2^-100 (the
//           rest is far inside its 2^-20 S).
//   nq, nx are float64 sums of exact float64 squares (relative error <= D_pad 2^-53 < 2^-43),
//         rounded to float32 (2^-24 more);
//   base = (nq + nx) - 2 s in float32: two roundings, <= 2^-24 (nq + nx) + 2^-24 |base|;
//   the canonical float64 distance d64 of the refine is within 2^-43 d of d.
// With S = nq + nx + 2 |s| (>= |base|, >= d) these add up to <= 2 kappa |q|^ |x|^ + 2^-21 S
// (|.|^ the norms rounded up).  E = (2 kappa |q|^ |x|^ + 2^-20 S) (1 + 2^-20), computed in
// float32, also covers its own roundings and those of base - E and base + E (each <= 2^-24
// (S + E)), so lb = max(base - E, 0) <= d64 <= base + E = ub.
//
// Threshold.  Per query, ub_best holds a float32 value t such that at least K distinct probed
// rows have ub <= t (so the K-th smallest d64 is <= t).  Each lane keeps, for each of its query
// rows, the smallest ub of its column over the unit so far (column j of every tile: distinct
// vectors); when at least K of a row's 16 column minima are below the query's current t, t drops
// to their K-th smallest (atomicMin on the float bits, which order like the values for
// non-negative floats).  After such a drop only K - 1 minima are below t, so the selection runs
// again only when another column's minimum falls below t.  A row is listed iff its lb
// is <= the query's t at that moment; every row of the exact top-K (ties included) qualifies,
// because lb <= d64 <= the K-th smallest d64 <= t.  The listed (lb, ub) keys then give tau = the
// K-th smallest listed ub (fine_tau_kernel), and the refine computes the canonical distance of
// the listed rows whose lb <= tau only.
//
// K > 16.  Sixteen column minima cannot certify K rows, so the in-scan selection never fires;
// instead the warm-up launch over the first probes lists every row, and cm_seed_kernel sets
// ub_best to the K-th smallest listed ub (K distinct probed rows have ub <= it) and empties the
// lists before the main launch, which lists against that fixed threshold.
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"

namespace trident {

typedef float v4f __attribute__((ext_vector_type(4)));

namespace {

typedef float v2f __attribute__((ext_vector_type(2)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

constexpr int kCmBV = 64;      // vectors per LDS block
constexpr int kCmQW = 16;      // queries per matrix tile
constexpr int kCmQueue = 256;  // listed rows a wave queues before it appends them

// Loads n floats of src (n <= 4, 16-byte aligned when n == 4 and vec) into v, zero beyond n.
__device__ __forceinline__ float4 load_upto4(const float* src, int n, bool vec) {
    if (n >= 4 && vec) return *reinterpret_cast<const float4*>(src);
    float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (n > 0) v.x = src[0];
    if (n > 1) v.y = src[1];
    if (n > 2) v.z = src[2];
    if (n > 3) v.w = src[3];
    return v;
}

// x, formed anew at each use: lane addresses hoisted out of the unit loop would not fit the registers.
__device__ __forceinline__ int opaque(int x) {
    asm volatile("" : "+v"(x));
    return x;
}

// The same where vec rows are whole float4s up to their end (D % 4 == 0): n is then never 1, 2 or 3.
__device__ __forceinline__ float4 load4(const float* src, int n, bool vec) {
    float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (vec) {
        if (n > 0) v = *reinterpret_cast<const float4*>(src);
    } else {
        if (n > 0) v.x = src[0];
        if (n > 1) v.y = src[1];
        if (n > 2) v.z = src[2];
        if (n > 3) v.w = src[3];
    }
    return v;
}

// The wave's query rows as one lane sees them: rows 4 g + r of its 16-query group.
struct CmRows {
    int rq[4];       // query ids (-1: no query)
    float t_row[4];  // thresholds (-1: never listed)
    float nq_r[4];   // |q| rounded up
    float qn_r[4];   // |q|^2 in float32
    float cmin[4];   // the smallest ub of this lane's column over the unit so far
};

// One 16-vector tile's bounds, thresholds and listing, from its float32 dot products sv (rows
// 4 g + r, column j = lane & 15 = block row bi): lb <= d64 <= ub by the error band above, the
// query's threshold lowered to the K-th smallest of its 16 column minima when at least K are
// below it (K <= 16), and the rows with lb <= threshold listed as (lb, ub) keys.
__device__ __forceinline__ void cm_tile_epilogue(const BatchArgs& a, const v4f sv, int bi, int nvb,
                                                 const float* s_xn, const float* s_nx, float kap2,
                                                 CmRows& Q, int row0,
                                                 unsigned long long& st_surv) {
    const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
    const int K = a.K;
    const bool vv = bi < nvb;
    const float xn = s_xn[bi], nx = s_nx[bi];
    float lbf[4], ubf[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const float sd = sv[r];
        const float base = (Q.qn_r[r] + xn) - 2.0f * sd;
        const float S = (Q.qn_r[r] + xn) + 2.0f * fabsf(sd);
        const float E = fmaf(kap2 * Q.nq_r[r], nx, 0x1p-20f * S) * (1.0f + 0x1p-20f);
        float lb = fmaxf(base - E, 0.0f), ub = base + E;
        if (!(ub < INFINITY)) {  // overflow or NaN: no bound
            lb = 0.0f;
            ub = INFINITY;
        }
        lbf[r] = vv ? lb : INFINITY;
        ubf[r] = vv ? ub : INFINITY;
        Q.cmin[r] = fminf(Q.cmin[r], ubf[r]);
    }
    // ---- thresholds: the K-th smallest column minimum per query row, when at least K of the
    // row's 16 are below the query's t ----
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const uint64_t bm = __ballot(Q.cmin[r] < Q.t_row[r]);
        const int cg = __popcll((bm >> (16 * g)) & 0xffffull);
        if (__ballot(cg >= K) == 0ull) continue;
        const float my = Q.cmin[r];
        int rank = 0;
#pragma unroll 1
        for (int o = 1; o < 16; ++o) {  // rare: kept rolled (no hoisted lane maps)
            const float ot = __shfl_xor(my, o, kWave);
            rank += (ot < my || (ot == my && (j ^ o) < j)) ? 1 : 0;
        }
        float kth = rank == K - 1 ? my : 0.0f;
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) kth = fmaxf(kth, __shfl_xor(kth, o, kWave));
        if (cg >= K && Q.rq[r] >= 0 && kth < Q.t_row[r]) {
            Q.t_row[r] = kth;
            if (j == 0) atomicMin(&a.ub_best[Q.rq[r]], __float_as_uint(kth));
        }
    }
    // ---- list the rows with lb <= t: one atomic per (row, lane group); the warm-up pass
    // (cm_emit = 0) only sets thresholds ----
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        if (!a.cm_emit) break;
        // vv explicitly: a query without a threshold yet has t = +inf, and the +inf keys of
        // columns past the slice would compare <= it
        const bool ps = vv && lbf[r] <= Q.t_row[r];
        const uint64_t m = __ballot(ps);
        if (m == 0ull) continue;
        const uint32_t gm = (uint32_t)(m >> (16 * g)) & 0xffffu;
        const int rk = __popc(gm & ((1u << j) - 1u));
        const int leader = gm ? __ffs(gm) - 1 : 0;
        int base = 0;
        if (ps && rk == 0) base = atomicAdd(&a.cand_cnt[Q.rq[r]], __popc(gm));
        base = __shfl(base, 16 * g + leader, kWave);
        if (ps) {
            const int slot = base + rk;
            if (slot < a.cap) {
                const size_t o = (size_t)Q.rq[r] * a.cap + slot;
                a.cand_key[o] = ((uint64_t)__float_as_uint(lbf[r]) << 32) | __float_as_uint(ubf[r]);
                a.cand_id[o] = row0 + bi;
            }
            ++st_surv;
        }
    }
}

}  // namespace

// How many of the other fifteen values of this lane's group of sixteen are smaller (EQ: equal).
template <bool EQ>
__device__ __forceinline__ int rank16(uint32_t v) {
    int rank = 0;
    auto one = [&](auto o_c) __attribute__((always_inline)) {
        constexpr int kRowRor = 0x120;  // DPP: rotate within the 16-lane row
        const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kRowRor + decltype(o_c)::value, 0xf, 0xf, false);
        rank += (EQ ? o == v : o < v) ? 1 : 0;
    };
    one(std::integral_constant<int, 1>{});
    one(std::integral_constant<int, 2>{});
    one(std::integral_constant<int, 3>{});
    one(std::integral_constant<int, 4>{});
    one(std::integral_constant<int, 5>{});
    one(std::integral_constant<int, 6>{});
    one(std::integral_constant<int, 7>{});
    one(std::integral_constant<int, 8>{});
    one(std::integral_constant<int, 9>{});
    one(std::integral_constant<int, 10>{});
    one(std::integral_constant<int, 11>{});
    one(std::integral_constant<int, 12>{});
    one(std::integral_constant<int, 13>{});
    one(std::integral_constant<int, 14>{});
    one(std::integral_constant<int, 15>{});
    return rank;
}

// x = h + m + l + r, each part rounded to nearest even (|r| <= 2^-24 |x|; the differences are exact),
// of 2 N values; part p of values 2 i, 2 i + 1 in part[p][i].  A value that rounds to infinity makes
// its products, and with them the row's bounds, infinite or NaN: the row is then listed without a
// bound and refined.
template <int N>
__device__ __forceinline__ void split3(const float (&x)[2 * N], uint32_t (&part)[3][N]) {
    float v[2 * N];
#pragma unroll
    for (int i = 0; i < 2 * N; ++i) v[i] = x[i];
#pragma unroll
    for (int p = 0; p < 3; ++p) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const v2bf h = __builtin_convertvector(v2f{v[2 * i], v[2 * i + 1]}, v2bf);
            const uint32_t w = __builtin_bit_cast(uint32_t, h);
            part[p][i] = w;
            if (p < 2) {
                v[2 * i] -= __uint_as_float(w << 16);
                v[2 * i + 1] -= __uint_as_float(w & 0xffff0000u);
            }
        }
    }
}

// The narrow layout (D_pad = 4 D4 <= 256), eight waves.  A unit's queries (16 a wave: A rows, in
// registers) meet 64-row blocks of its slice (B columns) as three-part bfloat16 operands, six
// products a dimension on v_mfma_f32_16x16x32_bf16: the dot products are as close as float32 matrix
// products (the parts hold 24 bits) at 16 / 6 of their rate.  Per block each wave converts the eight
// rows it loaded while the previous block was computed (whole 128-byte lines, eight lanes a row: the
// float64 norms need no second pass), and the waves read the four tiles from LDS in operand order.
//
// What was between the products bound the float32 form of this kernel (0.11 of its matrix peak at
// 4000 queries, nlist 1024, nprobe 32, K = 10, D = 128): one returning global atomic per listed run of
// rows, loads waited for where they were issued, and some 20 operations a pair.  Here a pair costs six
// operations until it passes a test that every listed row passes (base against t plus a bound of
// E), listed rows are queued in LDS and appended with one atomic per query and flush, and the
// thresholds are read a block ahead and selected once a block: 1957 us -> 817 there (warm-up and main
// pass), 275 -> 178 for 40 queries on 1e6 rows (nprobe 64).
//
// What bounds it now (10,000 queries, nprobe 64, counters): the vector unit issues in 0.56 of the slots
// (conversion, first test, norms), the matrix cores are busy for 0.36 (828 TFLOP/s, padding of tiles
// included), waves wait for half of their cycles at the two barriers of a block and its loads.  The 40
// queries read 480 MB at 2.7 TB/s, half of a copy's rate: with one 16-query tile the eight waves share a
// block's four tiles, so half of them only convert.
template <int D4>
__global__ __launch_bounds__(kCmThreads, D4 <= 32 ? 4 : 2) void cm_scan_kernel(BatchArgs a) {
    constexpr int DP = 4 * D4;  // D_pad
    constexpr int NS = DP / 32;
    constexpr int NW = kCmThreads / kWave;
    static_assert(D4 % 8 == 0 && D4 <= 64, "D_pad a multiple of 32, at most 256");
    static_assert(NW * 8 == kCmBV && NW * kCmQW == kCmUnitQ, "a wave converts 8 rows, holds 16 queries");
    __shared__ v4u s_b[kCmBV / 16][NS][3][kWave];
    __shared__ float s_xn[kCmBV], s_nx[kCmBV];  // |x|^2, |x| rounded up
    __shared__ float s_kx[kCmBV], s_xk[kCmBV];  // the rows' part of the first test
    __shared__ __align__(16) float s_qn[NW][kCmQW];  // |q|^2
    __shared__ __align__(16) float s_nq[NW][kCmQW];  // |q| rounded up
    __shared__ __align__(16) float s_t[NW][kCmQW];   // thresholds (-inf: no query)
    __shared__ __align__(16) float s_a[NW][kCmQW];   // the queries' part of the first test
    __shared__ int s_qid[NW][kCmQW];                 // -1: no query
    __shared__ int s_cnt[NW][kCmQW];
    __shared__ uint64_t s_key[NW][kCmQueue];
    __shared__ uint32_t s_ent[NW][kCmQueue];         // query slot << 27 | row of the unit
    __shared__ int s_unit[2];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int D = a.D, K = a.K;
    const int u0 = a.unit_off[a.unit_beg], u1 = min(a.unit_off[a.unit_end], a.max_units);
    // kappa of the six-product sums (hh in one accumulator, the rest in another; see the head)
    const float kap2 = (float)(2.0 * ((DP + 4) * 0x1p-23 * (1.0 + 0x1p-7) +
                                      (5 * DP + 4) * 0x1p-30 * (1.0 + 0x1p-5) + 4.2 * 0x1p-24));
    const float kabs = DP * 0x1p-100f;
    // First test of a pair: every row with lb <= t has
    //     -2 s <= t - (nq + nx) + kap2 |q| |x| + 2^-18 (nq + nx) + 2 kabs,
    // since E's S is at most 2 (nq + nx) (1 + 2^-10) and the doubled constants cover the roundings (t
    // <= 4 (nq + nx), else -2 s is far below the right side); halved and split into a query's part a =
    // ((1 - 2^-18) nq - t) / 2 and a row's parts kx, xk it is s >= fma(kx, |q|, a) + xk, written so
    // that a NaN passes.
    auto query_part = [&](float qn, float t) { return 0.5f * ((qn - 0x1p-18f * qn) - t); };
    const bool xvec = (D & 3) == 0 && (reinterpret_cast<uintptr_t>(a.xb) & 15) == 0;
    const bool qvec = (D & 3) == 0 && (reinterpret_cast<uintptr_t>(a.xq) & 15) == 0;
    unsigned long long st_cand = 0, st_surv = 0;

    // work units from one counter (slot (it + 1) & 1 is written while slot it & 1 is read; the
    // previous read of the written slot happened before this iteration's first barrier)
    if (tid == 0) s_unit[0] = atomicAdd(a.ctr, 1);
    for (int it = 0;; ++it) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __syncthreads();
        const int ui = __builtin_amdgcn_readfirstlane(s_unit[it & 1]) + u0;
        if (ui < u0 || ui >= u1) break;
        if (tid == 0) s_unit[(it + 1) & 1] = atomicAdd(a.ctr, 1);
        const int4 un = a.units[ui];
        const int cid = un.x & 0xfffff, cnt = un.x >> 20, start = un.y, vb = un.z, ve = un.w;
        const int v0 = a.vec_off[cid];
        const int G = (cnt + kCmQW - 1) / kCmQW;  // 16-query groups (1..8)
        const int R = NW / G;                     // waves sharing a group split its tiles
        const int gq = wid / R, rr = wid - gq * R;
        const bool active = gq < G;
        const int nq = active ? min(kCmQW, cnt - gq * kCmQW) : 0;
        // rows this unit reads from a host-mapped base: its slice, once
        if (a.host_rows && a.xb_host && tid == 0) atomicAdd(a.host_rows, (unsigned long long)(ve - vb));

        // the lane's share of a block's rows: float4 chunks 8 s + lane / 8 of row 8 wid + lane % 8
        float4 pre[NS];
        auto load_rows = [&](int blk0) __attribute__((always_inline)) {
            const int l = opaque(lane);
            const int row = min(blk0 + 8 * wid + (l & 7), ve - 1);  // past the slice: its last row again
            const int d0 = 4 * (l >> 3);
            const float* xr = a.xb + (size_t)(v0 + row) * D + d0;
            if (xvec) {
#pragma unroll
                for (int s = 0; s < NS; ++s)  // D % 4 == 0: whole or past the row's end
                    pre[s] = d0 + 32 * s < D ? *reinterpret_cast<const float4*>(xr + 32 * s)
                                             : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            } else {
#pragma unroll
                for (int s = 0; s < NS; ++s) pre[s] = load4(xr + 32 * s, D - d0 - 32 * s, false);
            }
        };
        load_rows(vb);

        // ---- this wave's queries: A operands (row j, dims 32 s + 8 g .. + 7) and norms ----
        bf8 qa[NS][3];
        float cmin[4];  // the smallest ub of this lane's column over the unit so far, rows 4 g + r
#pragma unroll
        for (int r = 0; r < 4; ++r) cmin[r] = INFINITY;
        {
            const int l = opaque(lane), j = l & 15, g = l >> 4;
            const bool qv = j < nq;
            const int qid = qv ? a.pair_qid[start + gq * kCmQW + j] : 0;
            const float* qp = a.xq + (size_t)qid * D;
            double qn = 0.0;
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                const int d = 32 * s + 8 * g;
                const float4 u = load4(qp + d, qv ? D - d : 0, qvec);
                const float4 v = load4(qp + d + 4, qv ? D - d - 4 : 0, qvec);
                const float x[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
#pragma unroll
                for (int i = 0; i < 8; ++i) qn = fma((double)x[i], (double)x[i], qn);
                uint32_t part[3][4];
                split3<4>(x, part);
#pragma unroll
                for (int p = 0; p < 3; ++p)
                    qa[s][p] = __builtin_bit_cast(bf8, v4u{part[p][0], part[p][1], part[p][2], part[p][3]});
            }
            qn += shfl_f64(qn, l ^ 16);
            qn += shfl_f64(qn, l ^ 32);
            if (g == 0) {
                s_qn[wid][j] = (float)qn;
                s_nq[wid][j] = __double2float_ru(sqrt(qn) * (1.0 + 0x1p-40));
                s_qid[wid][j] = qv ? qid : -1;
                const float t = qv ? __uint_as_float(a.ub_best[qid]) : -INFINITY;
                s_t[wid][j] = t;
                s_a[wid][j] = query_part((float)qn, t);
                s_cnt[wid][j] = 0;
            }
        }
        wave_sync();
        // the query this lane keeps the threshold of (lanes past the wave's queries: none)
        const int tq = lane < nq ? s_qid[wid][opaque(lane)] : -1;

        // appends the queued rows to their queries' lists
        int nque = 0;
        auto flush = [&]() __attribute__((always_inline)) {
            wave_sync();
            const int fl = opaque(lane);
            int rank[kCmQueue / kWave];
#pragma unroll
            for (int i = 0; i < kCmQueue / kWave; ++i) {
                const int e = i * kWave + fl;
                rank[i] = e < nque ? atomicAdd(&s_cnt[wid][s_ent[wid][e] >> 27], 1) : 0;
            }
            wave_sync();
            if (tq >= 0) {
                const int c = s_cnt[wid][fl];
                if (c > 0) s_cnt[wid][fl] = atomicAdd(&a.cand_cnt[tq], c);
            }
            wave_sync();
#pragma unroll
            for (int i = 0; i < kCmQueue / kWave; ++i) {
                const int e = i * kWave + fl;
                if (e < nque) {
                    const uint32_t en = s_ent[wid][e];
                    const int at = s_cnt[wid][en >> 27] + rank[i];
                    if (at < a.cap) {
                        const size_t o = (size_t)s_qid[wid][en >> 27] * a.cap + at;
                        a.cand_key[o] = s_key[wid][e];
                        a.cand_id[o] = v0 + vb + (int)(en & 0x7ffffffu);
                    }
                }
            }
            wave_sync();
            if (lane < kCmQW) s_cnt[wid][fl] = 0;
            wave_sync();
            nque = 0;
        };

        bool lower = false;  // a column minimum fell below its query's threshold since the last selection
        for (int blk0 = vb; blk0 < ve; blk0 += kCmBV) {
            const int nvb = min(kCmBV, ve - blk0);
            // ---- the loaded rows into operand order, and their norms ----
            {
                const int l = opaque(lane);
                const int row = 8 * wid + (l & 7), x8 = l >> 3;
                double xn = 0.0;
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    const float x[4] = {pre[s].x, pre[s].y, pre[s].z, pre[s].w};
#pragma unroll
                    for (int i = 0; i < 4; ++i) xn = fma((double)x[i], (double)x[i], xn);
                    // dims 4 x8 .. + 3 of step s: lane group x8 / 2, half x8 % 2 of its 16 bytes
                    uint32_t part[3][2];
                    split3<2>(x, part);
#pragma unroll
                    for (int p = 0; p < 3; ++p)
                        reinterpret_cast<v2u*>(&s_b[wid >> 1][s][p][(row & 15) + 16 * (x8 >> 1)])[x8 & 1] =
                            v2u{part[p][0], part[p][1]};
                }
                xn += shfl_f64(xn, l ^ 8);
                xn += shfl_f64(xn, l ^ 16);
                xn += shfl_f64(xn, l ^ 32);
                if (x8 == 0) {
                    const float n2 = (float)xn, n = __double2float_ru(sqrt(xn) * (1.0 + 0x1p-40));
                    s_xn[row] = n2;
                    s_nx[row] = n;
                    s_kx[row] = -0.5f * (kap2 * n * (1.0f + 0x1p-20f));
                    s_xk[row] = 0.5f * (n2 - fmaf(0x1p-18f, n2, 2.0f * kabs));
                }
            }
            __syncthreads();
            if (blk0 + kCmBV < ve) load_rows(blk0 + kCmBV);
            // thresholds other units lowered, used from the next block on
            const uint32_t tb = tq >= 0 ? a.ub_best[tq] : 0u;
            if (active) {
                // ---- the wave's tiles: rr, rr + R, ... (16 vectors each) ----
#pragma unroll 1
                for (int tl = rr; tl < kCmBV / 16 && 16 * tl < nvb; tl += R) {
                    v4f hh = {0.0f, 0.0f, 0.0f, 0.0f}, rest = hh;
                    const int lane_b = opaque(lane);
                    bf8 b[3];
#pragma unroll
                    for (int p = 0; p < 3; ++p) b[p] = __builtin_bit_cast(bf8, s_b[tl][0][p][lane_b]);
#pragma unroll
                    for (int s = 0; s < NS; ++s) {
                        // one step's operands in flight ahead of the matrix cores, no more: all of
                        // them hoisted would not fit the registers
                        bf8 n[3];
#pragma unroll
                        for (int p = 0; p < 3; ++p)
                            n[p] = __builtin_bit_cast(bf8, s_b[tl][s + 1 < NS ? s + 1 : s][p][lane_b]);
                        const bf8(&q)[3] = qa[s];
                        hh = __builtin_amdgcn_mfma_f32_16x16x32_bf16(q[0], b[0], hh, 0, 0, 0);
                        rest = __builtin_amdgcn_mfma_f32_16x16x32_bf16(q[0], b[1], rest, 0, 0, 0);
                        rest = __builtin_amdgcn_mfma_f32_16x16x32_bf16(q[1], b[0], rest, 0, 0, 0);
                        rest = __builtin_amdgcn_mfma_f32_16x16x32_bf16(q[0], b[2], rest, 0, 0, 0);
                        rest = __builtin_amdgcn_mfma_f32_16x16x32_bf16(q[1], b[1], rest, 0, 0, 0);
                        rest = __builtin_amdgcn_mfma_f32_16x16x32_bf16(q[2], b[0], rest, 0, 0, 0);
#pragma unroll
                        for (int p = 0; p < 3; ++p) b[p] = n[p];
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    // constants from LDS after each tile's products (the barrier keeps them out of
                    // the registers meanwhile)
                    asm volatile("" ::: "memory");
                    const int l = opaque(lane), j = l & 15, g = l >> 4;
                    const int bi = 16 * tl + j;
                    const v4f sv = hh + rest;
                    const float4 a4 = *reinterpret_cast<const float4*>(&s_a[wid][4 * g]);
                    const float4 nq4 = *reinterpret_cast<const float4*>(&s_nq[wid][4 * g]);
                    const float av[4] = {a4.x, a4.y, a4.z, a4.w};
                    const float nqv[4] = {nq4.x, nq4.y, nq4.z, nq4.w};
                    const float kx = s_kx[bi], xk = s_xk[bi];
                    bool ps[4];
                    uint64_t pm[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        ps[r] = !(sv[r] < fmaf(kx, nqv[r], av[r]) + xk);
                        pm[r] = __ballot(ps[r]);
                    }
                    if ((pm[0] | pm[1] | pm[2] | pm[3]) == 0ull) continue;
                    const float xn = s_xn[bi], nx = s_nx[bi];
                    const float4 qn4 = *reinterpret_cast<const float4*>(&s_qn[wid][4 * g]);
                    const float4 t4 = *reinterpret_cast<const float4*>(&s_t[wid][4 * g]);
                    const float qnv[4] = {qn4.x, qn4.y, qn4.z, qn4.w};
                    const float tv[4] = {t4.x, t4.y, t4.z, t4.w};
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        if ((r & 1) == 0 && nque > kCmQueue - 2 * kWave) flush();  // room for two rows' lanes
                        if (pm[r] == 0ull) continue;
                        const float w = qnv[r] + xn;
                        const float base = w - 2.0f * sv[r], S = w + 2.0f * fabsf(sv[r]);
                        const float E = fmaf(kap2 * nqv[r], nx, fmaf(0x1p-20f, S, kabs)) * (1.0f + 0x1p-20f);
                        float lb = fmaxf(base - E, 0.0f), ub = base + E;
                        if (!(ub < INFINITY)) {  // overflow or NaN: no bound
                            lb = 0.0f;
                            ub = INFINITY;
                        }
                        // columns past the slice and rows without a query (t = -inf) never pass
                        const bool in = ps[r] && bi < nvb && lb <= tv[r];
                        if (in && ub < cmin[r]) {
                            cmin[r] = ub;
                            lower |= ub < tv[r];
                        }
                        const uint64_t m = __ballot(in);
                        if (m == 0ull || !a.cm_emit) continue;
                        if (in) {
                            const int at = nque + mask_rank(m);
                            s_key[wid][at] = ((uint64_t)__float_as_uint(lb) << 32) | __float_as_uint(ub);
                            s_ent[wid][at] = (uint32_t)(4 * g + r) << 27 | (uint32_t)(blk0 - vb + bi);
                        }
                        nque += __popcll(m);
                        st_surv += __popcll(m);
                    }
                }
                // ---- thresholds: where at least K of a query row's 16 column minima are below its
                // t, the K-th smallest becomes t (the warm-up, which lists nothing, selects after its
                // last block only).  Each lane ranks its minimum among the row's sixteen by fifteen
                // lane rotations. ----
                if (K <= kCmQW && __ballot(lower) != 0ull && (a.cm_emit || blk0 + kCmBV >= ve)) {
                    lower = false;
                    const int g = opaque(lane) >> 4;
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int slot = 4 * g + r;
                        const uint32_t my = __float_as_uint(cmin[r]);
                        const bool below = my < 0x7f800000u && __uint_as_float(my) < s_t[wid][slot];
                        const uint64_t bm = __ballot(below);
                        const bool enough = __popc((uint32_t)(bm >> (16 * g)) & 0xffffu) >= K;
                        if (__ballot(enough) == 0ull) continue;
                        const int lt = rank16<false>(my);
                        bool kth = below && lt == K - 1;
                        const uint64_t km = __ballot(kth);
                        // a tie at the K-th leaves no lane with that rank: the lanes that tie store it
                        if (__ballot(enough && ((uint32_t)(km >> (16 * g)) & 0xffffu) == 0u) != 0ull)
                            kth = below && lt < K && lt + rank16<true>(my) >= K - 1;
                        if (kth) {
                            s_t[wid][slot] = __uint_as_float(my);
                            atomicMin(&a.ub_best[s_qid[wid][slot]], my);
                        }
                    }
                }
                wave_sync();
                if (tq >= 0) {
                    const int l = opaque(lane);
                    const float t = fminf(s_t[wid][l], __uint_as_float(tb));
                    s_t[wid][l] = t;
                    s_a[wid][l] = query_part(s_qn[wid][l], t);
                }
                wave_sync();
                if (a.stats && rr == 0) st_cand += (unsigned long long)nq * nvb;
            }
            __syncthreads();  // the next block overwrites s_b, s_xn, s_nx
        }
        if (nque > 0) flush();
    }

    if (a.stats) {
        if (lane == 0) {
            const int slot = (int)(blockIdx.x % kStatSlots) * 4;
            atomicAdd(&a.stats[slot + 0], st_cand);
            atomicAdd(&a.stats[slot + 1], st_cand * (unsigned long long)DP);
            atomicAdd(&a.stats[slot + 2], st_surv);
        }
    }
}

// Wide layout (D_pad > 256, up to 1024): a query row no longer fits in registers, so the
// dimensions are walked in chunks of kCmWC dims.  Per 64-row block and chunk the block's rows
// are staged in LDS (64 x kCmWC floats, 33 KB: four workgroups per CU) and each wave reloads its
// 16 query rows' chunk (kCmWC / 4 floats a lane, from L2); every tile of the wave keeps one
// accumulator chain across the chunks (the wave's up to four tiles are independent chains for
// the matrix core).  The float64 row norms add up chunk by chunk in LDS.  Bounds, thresholds and
// listing are those of the narrow kernel, with kappa over the padded dimensions.
constexpr int kCmWC = 128;

__global__ __launch_bounds__(256) void cm_scan_wide_kernel(BatchArgs a) {
    constexpr int C4 = kCmWC / 4;  // floats per lane per chunk
    constexpr int RS = kCmWC + 4;  // LDS row stride: an odd number of 16-byte chunks
    __shared__ __align__(16) float s_x[kCmBV * RS];
    __shared__ double s_xd[kCmBV];
    __shared__ float s_xn[kCmBV];
    __shared__ float s_nx[kCmBV];
    __shared__ double s_qn[kWavesPerBlock][kCmQW];
    __shared__ float s_nq[kWavesPerBlock][kCmQW];
    __shared__ int s_qid[kWavesPerBlock][kCmQW];
    __shared__ int s_unit[2];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 15, g = lane >> 4;
    const int D = a.D;
    const int nch = (a.D_pad + kCmWC - 1) / kCmWC;  // chunks; dims past D are zero
    const int u0 = a.unit_off[a.unit_beg], u1 = min(a.unit_off[a.unit_end], a.max_units);
    const float kap2 = (float)(2.0 * (double)(nch * kCmWC + 8) * 0x1p-23 * (1.0 + 0x1p-10));
    const bool xvec = (D & 3) == 0 && (reinterpret_cast<uintptr_t>(a.xb) & 15) == 0;
    const bool qvec = (D & 3) == 0 && (reinterpret_cast<uintptr_t>(a.xq) & 15) == 0;
    unsigned long long st_cand = 0, st_surv = 0;

    if (tid == 0) s_unit[0] = atomicAdd(a.ctr, 1);
    for (int it = 0;; ++it) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __syncthreads();
        const int ui = __builtin_amdgcn_readfirstlane(s_unit[it & 1]) + u0;
        if (ui < u0 || ui >= u1) break;
        if (tid == 0) s_unit[(it + 1) & 1] = atomicAdd(a.ctr, 1);
        const int4 un = a.units[ui];
        const int cid = un.x & 0xfffff, cnt = un.x >> 20, start = un.y, vb = un.z, ve = un.w;
        const int v0 = a.vec_off[cid];
        const int G = (cnt + kCmQW - 1) / kCmQW;  // 16-query groups (1..4)
        const int R = kWavesPerBlock / G;         // waves sharing a group split its tiles
        const int gq = wid / R, rr = wid - gq * R;
        const bool active = gq < G;
        const int nq = active ? min(kCmQW, cnt - gq * kCmQW) : 0;
        // rows this unit reads from a host-mapped base: its slice, once
        if (a.host_rows && a.xb_host && tid == 0) atomicAdd(a.host_rows, (unsigned long long)(ve - vb));
        const bool qv = j < nq;
        const int qid = active && qv ? a.pair_qid[start + gq * kCmQW + j] : 0;
        const float* qrow = a.xq + (size_t)qid * D;

        // ---- this wave's query rows: norms over all dims (lane (j, g): dims c kCmWC + g C4
        // .. + C4 - 1 of query j, for every chunk c) ----
        CmRows qs;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            qs.rq[r] = -1;
            qs.t_row[r] = -1.0f;
            qs.nq_r[r] = qs.qn_r[r] = 0.0f;
            qs.cmin[r] = INFINITY;
        }
        if (active) {
            double qn = 0.0;
            for (int c = 0; c < nch; ++c) {
#pragma unroll
                for (int k = 0; k < C4 / 4; ++k) {
                    const int d0 = c * kCmWC + g * C4 + 4 * k;
                    const float4 v = load_upto4(qrow + d0, qv ? D - d0 : 0, qvec);
                    qn = fma((double)v.x, (double)v.x, qn);
                    qn = fma((double)v.y, (double)v.y, qn);
                    qn = fma((double)v.z, (double)v.z, qn);
                    qn = fma((double)v.w, (double)v.w, qn);
                }
            }
            qn += shfl_f64(qn, lane ^ 16);
            qn += shfl_f64(qn, lane ^ 32);
            if (g == 0) {
                s_qn[wid][j] = qn;
                s_nq[wid][j] = __double2float_ru(sqrt(qn) * (1.0 + 0x1p-40));
                s_qid[wid][j] = qv ? qid : -1;
            }
            wave_sync();
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = 4 * g + r;
                qs.rq[r] = row < nq ? s_qid[wid][row] : -1;
                qs.qn_r[r] = (float)s_qn[wid][row];
                qs.nq_r[r] = s_nq[wid][row];
                qs.t_row[r] = qs.rq[r] >= 0 ? __uint_as_float(a.ub_best[qs.rq[r]]) : -1.0f;
            }
        }

        for (int blk0 = vb; blk0 < ve; blk0 += kCmBV) {
            const int nvb = min(kCmBV, ve - blk0);
            // the wave's tiles rr, rr + R, ... inside the block (1 to 4, wave-uniform), one
            // accumulator chain each
            int nt = 0;
#pragma unroll
            for (int t = 0; t < 4; ++t) nt += t * R < kWavesPerBlock && 16 * (rr + t * R) < nvb ? 1 : 0;
            v4f acc[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) acc[t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
            for (int c = 0; c < nch; ++c) {
                const int cb = c * kCmWC;
                // ---- stage the block's rows, dims [cb, cb + kCmWC) (zero past D): 64 x 32
                // float4 chunks, eight per thread, in two halves whose loads are all issued
                // before their LDS stores ----
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    float4 v[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const int i = tid + kBlock * (4 * h + k);
                        const int r = i / (kCmWC / 4), c4 = i - r * (kCmWC / 4);
                        const int d0 = cb + 4 * c4;
                        v[k] = load_upto4(a.xb + (size_t)(v0 + blk0 + min(r, nvb - 1)) * D + d0,
                                          min(r < nvb ? D - d0 : 0, 4), xvec);
                    }
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const int i = tid + kBlock * (4 * h + k);
                        const int r = i / (kCmWC / 4), c4 = i - r * (kCmWC / 4);
                        *reinterpret_cast<float4*>(s_x + r * RS + 4 * c4) = v[k];
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                // ---- this chunk's query values (A operands; a lane's dims lie wholly inside
                // or outside D when D % 4 == 0, the vector path) ----
                float qa[C4];
                if (active) {
#pragma unroll
                    for (int k = 0; k < C4 / 4; ++k) {
                        const int d0 = cb + g * C4 + 4 * k;
                        const int left = qv ? D - d0 : 0;
                        float4 v;
                        if (qvec) v = left > 0 ? *reinterpret_cast<const float4*>(qrow + d0)
                                               : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                        else v = load_upto4(qrow + d0, left, false);
                        qa[4 * k] = v.x;
                        qa[4 * k + 1] = v.y;
                        qa[4 * k + 2] = v.z;
                        qa[4 * k + 3] = v.w;
                    }
                }
                __syncthreads();
                __builtin_amdgcn_sched_barrier(0);
                // ---- the chunk's share of the row norms: 4 threads a row ----
                {
                    const int r = tid >> 2, p = tid & 3;
                    const float* xr = s_x + r * RS + p * C4;
                    double xn = 0.0;
#pragma unroll 8
                    for (int d = 0; d < C4; ++d) xn = fma((double)xr[d], (double)xr[d], xn);
                    xn += shfl_f64(xn, lane ^ 1);
                    xn += shfl_f64(xn, lane ^ 2);
                    if (p == 0) s_xd[r] = (c == 0 ? 0.0 : s_xd[r]) + xn;
                }
                __builtin_amdgcn_sched_barrier(0);
                if (active) {
                    // NT tiles (rows 16 (rr + t R) ..), straight-line per 4-dim step
                    auto mma = [&](auto nt_c) __attribute__((always_inline)) {
                        constexpr int NT = decltype(nt_c)::value;
#pragma unroll
                        for (int s4 = 0; s4 < C4 / 4; ++s4) {
                            float4 b[NT];
#pragma unroll
                            for (int t = 0; t < NT; ++t)
                                b[t] = *reinterpret_cast<const float4*>(
                                    s_x + (16 * (rr + t * R) + j) * RS + g * C4 + 4 * s4);
#pragma unroll
                            for (int t = 0; t < NT; ++t) {
                                acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[4 * s4], b[t].x, acc[t], 0, 0, 0);
                                acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[4 * s4 + 1], b[t].y, acc[t], 0, 0, 0);
                                acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[4 * s4 + 2], b[t].z, acc[t], 0, 0, 0);
                                acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[4 * s4 + 3], b[t].w, acc[t], 0, 0, 0);
                            }
                            // one step's LDS reads at a time: hoisting every step's reads ahead
                            // of the matrix cores would hold them all in registers
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    };
                    switch (nt) {
                        case 1: mma(std::integral_constant<int, 1>{}); break;
                        case 2: mma(std::integral_constant<int, 2>{}); break;
                        case 3: mma(std::integral_constant<int, 3>{}); break;
                        default: mma(std::integral_constant<int, 4>{}); break;
                    }
                }
                __syncthreads();  // the next chunk overwrites s_x; s_xd complete after the last
            }
            if (tid < kCmBV) {
                const double xn = s_xd[tid];
                s_xn[tid] = (float)xn;
                s_nx[tid] = __double2float_ru(sqrt(xn) * (1.0 + 0x1p-40));
            }
            __syncthreads();
            if (active) {
                uint32_t tb[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) tb[r] = a.ub_best[max(qs.rq[r], 0)];
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (qs.rq[r] >= 0) qs.t_row[r] = fminf(qs.t_row[r], __uint_as_float(tb[r]));
                // VALU reads of matrix-core results: wait states fenced from the scheduler
                __builtin_amdgcn_sched_barrier(0);
                asm volatile("s_nop 7\n\ts_nop 7");
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    if (t >= nt) break;
                    cm_tile_epilogue(a, acc[t], 16 * (rr + t * R) + j, nvb, s_xn, s_nx, kap2, qs,
                                     v0 + blk0, st_surv);
                }
                if (a.stats && rr == 0 && lane == 0) st_cand += (unsigned long long)nq * nvb;
            }
            __syncthreads();  // the next block overwrites s_xd, s_xn, s_nx
        }
    }

    if (a.stats) {
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) st_surv += __shfl_xor(st_surv, o, kWave);
        if (lane == 0) {
            const int slot = (int)(blockIdx.x % kStatSlots) * 4;
            atomicAdd(&a.stats[slot + 0], st_cand);
            atomicAdd(&a.stats[slot + 1], st_cand * (unsigned long long)a.D_pad);
            atomicAdd(&a.stats[slot + 2], st_surv);
        }
    }
}

template __global__ void cm_scan_kernel<8>(BatchArgs);
template __global__ void cm_scan_kernel<16>(BatchArgs);
template __global__ void cm_scan_kernel<24>(BatchArgs);
template __global__ void cm_scan_kernel<32>(BatchArgs);
template __global__ void cm_scan_kernel<40>(BatchArgs);
template __global__ void cm_scan_kernel<48>(BatchArgs);
template __global__ void cm_scan_kernel<56>(BatchArgs);
template __global__ void cm_scan_kernel<64>(BatchArgs);

}  // namespace trident
