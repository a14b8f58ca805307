// Exact k nearest neighbours, up to kKnnWaveMax entries per query, by one
// wavefront for kKnnGroup consecutive queries (Morton order): the queries
// share the list of buckets around them (pair_cell.h), each then takes the
// points within an FP32 radius from it, ranks them by (FP64 squared distance,
// caller's index) and certifies its k-th entry against the points left out,
// as knn_select_row (common.h) does.  A query whose radius does not settle in
// kKnnTries tries (many copies) is left to the list path of Engine::knn_exact.
#pragma once

#include "common.h"

namespace vgc {

constexpr int kKnnWaveMax = 96;
constexpr int kKnnGroup = 8;
// radii tried per query: enough to close in from too few and too many where a
// lone point's ball touches a dense cluster (200k points, k = 16, 1000 of them
// around the cluster of the others: with 8 tries and no bracket the queries
// left to the lists took 192 ms, now 0.84 ms in all; 20k queries far from 100k
// points 1.56 -> 0.43 ms)
constexpr int kKnnTries = 16;

struct alignas(16) KnnLds {
    uint64_t cand[kCandCap];
    union {
        int front[2][kFrontCap];
        uint64_t cand_b[kCandCap];
    };
    int bucket[kBucketCap];
    int near_list[kNearCap];
    double d[kCandCap];
    int id[kCandCap];
};

struct KnnParams {
    ClipParams C;       // pts, orig, pf, nodes, IL
    const pt4* qp;      // queries, FP64 and FP32, Morton order
    const pf4* qf;
    const int* qpos;    // Morton place of each query among the points (nullptr: itself)
    const int* qrow;    // output row
    int nq, kk, n;      // queries, entries per query, points
    int self_rule;
    double e;           // knn_vec_err
    int* out_idx;
    double* out_d2;
    int* fail;          // queries left to the list path, and their number
    unsigned* nfail;
};

VGC_HD void knn_fail(const KnnParams& K, int t) {
#if defined(VGC_EMU)
    K.fail[__atomic_fetch_add(K.nfail, 1u, __ATOMIC_RELAXED)] = t;
#else
    if (lane0()) K.fail[atomicAdd(K.nfail, 1u)] = t;
#endif
}

// The distance of a query to the box of the points.
VGC_HD float knn_box_distance(const KnnParams& K, const pf4& q) {
    const bnode b = K.C.nodes[K.C.IL.t0[0] + 1];
    const float x = fmaxf(fmaxf(b.lo[0] - q.x, q.x - b.hi[0]), 0.0f);
    const float y = fmaxf(fmaxf(b.lo[1] - q.y, q.y - b.hi[1]), 0.0f);
    const float z = fmaxf(fmaxf(b.lo[2] - q.z, q.z - b.hi[2]), 0.0f);
    return sqrtf(x * x + y * y + z * z);
}

// Query t; N: the wave's bucket list, r2: the first squared radius to try,
// last2: the one that served the wave's last query far from its points (0:
// none yet).
VGC_HD void knn_wave_query(const KnnParams& K, KnnLds& L, const NearList& N, int t, float r2,
                           float& last2) {
    const LI lane = lane_id_here();
    const pf4 q = K.qf[t];
    const pt4 p = K.qp[t];
    float lo2 = 0.0f, hi2 = INFINITY;  // too few and too many points
    bool far = false;
    int n = 0;
    for (int it = 0; it < kKnnTries; ++it) {
        if (uni(N.inst >= 0 && r2 <= N.r2)) {
            int none;
            near_scan(K.C, L, N, -1, -1, q, q, -1.0f, r2, 0.0f, -1.0f, n, none);
        } else {
            PowerFilter F{};
            n = gather_ring(K.C, L, -1, 0, q.x, q.y, q.z, -1.0f, r2, F);
        }
        if (n < 0 || n > kCandCap) {
            const float f = n < 0 ? 0.5f : cbrtf((0.5f * (kCandCap + K.kk)) / float(n));
            hi2 = uni(fminf(hi2, r2));
            r2 = uni(r2 * f * f);
            if (!(r2 > lo2)) r2 = uni(sqrtf(lo2) * sqrtf(hi2));
            continue;
        }
        if (n < K.kk && n < K.n) {
            const float f = cbrtf((1.2f * K.kk + 4.0f) / float(n > 0 ? n : 1));
            lo2 = r2;
            r2 = uni(r2 * f * f);
            if (4 * n < K.kk) {
                if (!far) {
                    const float d = knn_box_distance(K, q);
                    lo2 = uni(fmaxf(lo2, 0.99999f * d * d));
                    r2 = uni(fmaxf(r2, (d + sqrtf(r2)) * (d + sqrtf(r2))));
                }
                far = true;
                r2 = uni(fmaxf(r2, last2));
            }
            if (!(r2 < hi2)) r2 = uni(sqrtf(lo2) * sqrtf(hi2));
            continue;
        }
        if (far) last2 = r2;
        // FP64 distances and caller's indices of the listed points
        LD d[2];
        LI id[2], rank[2] = {LI(0), LI(0)};
        const bool two = n > kWave;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            d[s] = LD(INFINITY);
            id[s] = LI(0x7FFFFFFF);
            if (s == 1 && !two) continue;
            const LI k = lane + kWave * s;
            const LB ok = k < n;
            const LI m = cvt<int>(cvt<uint32_t>(lds_ld(L.cand, select(ok, k, LI(0)))));
            const Lane<pt4> x = gld(K.C.pts, m, ok);
            const LD dx = pt_x(x) - p.x, dy = pt_y(x) - p.y, dz = pt_z(x) - p.z;
            d[s] = select(ok, dx * dx + dy * dy + dz * dz, LD(INFINITY));
            id[s] = gld(K.C.orig, m, ok);
            lds_st(L.d, select(ok, k, LI(0)), d[s], ok);
            lds_st(L.id, select(ok, k, LI(0)), id[s], ok);
        }
        wave_sync();
        for (int i = 0; i < n; ++i) {
            const LD di = lds_ld(L.d, LI(i));
            const LI ii = lds_ld(L.id, LI(i));
            rank[0] = rank[0] + select((di < d[0]) | ((di == d[0]) & (ii < id[0])), LI(1), LI(0));
            if (two) rank[1] = rank[1] + select((di < d[1]) | ((di == d[1]) & (ii < id[1])), LI(1), LI(0));
        }
        wave_sync();
        const LB in0 = (lane < n) & (rank[0] < K.kk), in1 = (lane + kWave < n) & (rank[1] < K.kk);
        if (n < K.n) {
            // no point left out may be nearer than the last entry
            const double lim = knn_outside_bound(r2, K.e);
            if (ballot((in0 & !(d[0] < lim)) | (in1 & !(d[1] < lim)))) {
                r2 = uni(knn_list_radius(1.15f * r2, K.e));
                continue;
            }
        }
        const int row = K.qrow[t];
        const int kout = K.self_rule ? K.kk - 1 : K.kk;
        int skip = 0;
        bool empty = false;
        if (K.self_rule) {
            // the point itself and its copies come first, at distance 0
            const LB z0 = in0 & (d[0] == 0.0), z1 = in1 & (d[1] == 0.0);
            skip = popc64(ballot(z0)) + popc64(ballot(z1));
            empty = ballot((z0 & (id[0] < row)) | (z1 & (id[1] < row))) != 0;
        }
        const Lane<long long> base = Lane<long long>((long long)row * kout);
        const LB w0 = in0 & (rank[0] >= skip) & LB(!empty), w1 = in1 & (rank[1] >= skip) & LB(!empty);
        const Lane<long long> a0 = base + cvt<long long>(rank[0] - skip), a1 = base + cvt<long long>(rank[1] - skip);
        gst(K.out_idx, a0, id[0], w0);
        gst(K.out_d2, a0, d[0], w0);
        if (two) {
            gst(K.out_idx, a1, id[1], w1);
            gst(K.out_d2, a1, d[1], w1);
        }
        const int have = empty ? 0 : K.kk - skip;
        if (have < kout) {
            for (int k0 = 0; k0 < kout; k0 += kWave) {
                const LI k = lane + k0;
                const LB pad = (k >= have) & (k < kout);
                gst(K.out_idx, base + cvt<long long>(k), LI(-1), pad);
                gst(K.out_d2, base + cvt<long long>(k), LD(-1.0), pad);
            }
        }
        return;
    }
    knn_fail(K, t);
}

// Queries first .. first + count - 1 (at most kKnnGroup).
VGC_HD void process_knn(const KnnParams& K, int first, int count, KnnLds& L) {
    const LI lane = lane_id();
    const LB has = lane < count;
    const LI t = first + select(has, lane, LI(0));
    const int c0 = K.qpos ? K.qpos[first] : first;
    const float d4 = uni(near_spacing(K.C, c0, 0, 1));
    // kNearRing spacings hold about 60 points; a quarter more than wanted, and
    // within the candidate buffer
    const float want = fminf(1.25f * K.kk + 8.0f, 108.0f);
    const float r = kNearRing * d4 * cbrtf(want * (1.0f / 60.0f));
    NearList N;
    N.inst = 0;
    N.r2 = (1.25f * r) * (1.25f * r);
    N.n = d4 > 0.0f ? near_buckets(K.C, L, 0, lane_seed(K.qf, t, has), has, N.r2) : -1;
    if (N.n < 0) N.inst = -1;
    float r2 = r * r;
    if (!(d4 > 0.0f)) {
        // a bucket of copies, or of fewer than five points: the whole tree's
        // box over the point count
        const bnode b = K.C.nodes[K.C.IL.t0[0] + 1];
        const float x = b.hi[0] - b.lo[0], y = b.hi[1] - b.lo[1], z = b.hi[2] - b.lo[2];
        const float f = cbrtf((1.25f * K.kk + 8.0f) / float(K.n));
        r2 = (x * x + y * y + z * z) * f * f + 1e-30f;
    }
    r2 = uni(r2);
    float last2 = 0.0f;
    for (int k = 0; k < count; ++k) knn_wave_query(K, L, N, first + k, r2, last2);
}

}  // namespace vgc
