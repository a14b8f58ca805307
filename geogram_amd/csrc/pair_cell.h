// The first clipping pass: two Voronoi / Laguerre cells per 64-lane wavefront,
// one per half, with FP32 corner state (clip_cell.h describes the cell, its
// certified signs and the FP64 rebuild of the corners).
//
// Why halves.  A cell holds about 21 live corners and forms 4 new ones per
// cut, so a whole wavefront per cell leaves two lanes of three idle; the
// kernel is bound by VALU issue, so two cells that share every instruction
// cost little more than one.  Corner c of a cell is slot c / 32 of lane
// c % 32 of its half: 64 corners per cell in two register slots, the second
// touched only while a cell of the pair has more than 32 corners (branches
// on the wave-uniform masks).  Corner ids, the order of the new corners and
// the order of every sum are those of the one-cell-per-wave kernels, so the
// outputs are the same bits.
//
// Wave-uniform state is kept in 64-bit lane masks (low word: the lower
// half's cell, high word: the upper half's), so per-cell decisions are scalar
// instructions.  The neighbour search of a half runs on the whole wave (the
// walks of clip_cell.h); its sorted candidates are staged in LDS as FP32
// plane rows, which both halves read by broadcast, 32 lanes one row.  A half
// that meets a plane that cuts waits until the other half has one too (or is
// done), so both halves clip together.
//
// FP32 rows are scaled by a power of two s per cell (e s, h s^2; box planes
// n, h s) chosen from the first ring, so that the rows of near seeds are of
// order one whatever the units, and corner magnitudes stay far from FP32
// underflow.  The scale changes no mantissa: signs, degenerate corners and
// bounds are those of the unscaled rows.
//
// A cell that needs anything rare (a sign or corner that FP32 cannot certify,
// more than 64 corners or planes, a coincident earlier seed, a walk that
// outgrows its buffers) is flagged CELL_UNCERTAIN without outputs; the FP64
// first pass redoes it from the start.  One that uses up its rings goes to the
// second gather.
#pragma once

#include "clip_cell.h"

namespace vgc {

constexpr int kPairPlanes = 64;   // plane rows per cell
constexpr int kStageCap = kWave;  // candidates of a ring, sorted and staged
constexpr int kNearCap = 256;     // buckets around a wave's cells
// corner magnitudes |D|_abs and max|N|_abs outside these bounds are left to
// the FP64 pass: (|N|_abs)^2, D^2 and the products of the sign bound then
// neither overflow nor underflow
constexpr float kPairDabsMin = 1e-12f, kPairDabsMax = 1e12f, kPairNMax = 1e15f;
constexpr float kPairE1Min = 1e-6f, kPairE1Max = 1e6f, kPairHMax = 1e12f;

struct alignas(16) PairHalf {
    float pe[kPairPlanes][4];      // e.x e.y e.z h (scaled)
    int pg[kPairPlanes];           // Morton position of the neighbour, -1 for the box
    uint8_t st_tab[kPairPlanes];   // new corner whose first plane is p
    uint8_t en_tab[kPairPlanes];   // new corner whose second plane is p
    uint32_t job[64];              // new corners: a | b << 8 | across << 16
    uint64_t key[kStageCap];       // the ring's candidates, sorted
};
// FP32 rows of the next candidates of a half
struct alignas(16) PairStage {
    float row[kStageCap][4];       // e.x e.y e.z h (scaled)
    float aux[kStageCap][2];       // security-radius value, |e|_1
};
// what a half's neighbour search keeps between rings
struct PairCtl {
    int c, inst;
    float rlo2, rhi2, all2, scale, inv;
    int nfilt, ct_on;
};
struct alignas(16) PairInt {
    double row[kPairPlanes][4];    // FP64 plane rows
    double q[64][3];               // corner points
    uint32_t cpl[64];              // corner planes
    uint32_t cadj[64];             // corner adjacency
    int v2t[kPairPlanes];          // first corner of each face
};
struct alignas(16) PairLds {
    union {
        struct {
            PairHalf h[2];
            PairCtl ctl[2];
            // unsorted candidates of the ring being gathered
            uint64_t cand[kCandCap];
            union {
                struct {
                    union {
                        int front[2][kFrontCap];
                        uint64_t cand_b[kCandCap];  // those of the upper half's cell
                    };
                    int bucket[kBucketCap];
                };
                PairStage stage[2];
            };
        };
        PairInt in[2];
    };
    int near_list[kNearCap];  // buckets around the wave's cells
};
static_assert(sizeof(PairLds) <= 10240, "16 wavefronts per CU");

// ---------------------------------------------------------------- helpers

constexpr uint64_t kLoHalf = 0xFFFFFFFFull, kHiHalf = ~kLoHalf;
VGC_HD uint64_t half_mask(int h) { return h ? kHiHalf : kLoHalf; }
// the halves (all their lanes) in which m has a lane
VGC_HD uint64_t halves(uint64_t m) {
    return (uint32_t(m) ? kLoHalf : 0ull) | (uint32_t(m >> 32) ? kHiHalf : 0ull);
}
VGC_HD int popc_half(uint64_t m, int h) { return popc32(h ? uint32_t(m >> 32) : uint32_t(m)); }
// the half's word of m per lane
VGC_HD LU half_word(uint64_t m, const LB& up) {
    return select(up, LU(uint32_t(m >> 32)), LU(uint32_t(m)));
}

struct RowLanes {
    LF x, y, z, w;
};
VGC_HD RowLanes lds_row(const float* p, const LI& idx) {
    RowLanes r;
#if defined(VGC_EMU)
    for (int l = 0; l < kWave; ++l) {
        const float* q = p + 4 * idx[l];
        r.x[l] = q[0];
        r.y[l] = q[1];
        r.z[l] = q[2];
        r.w[l] = q[3];
    }
#else
    const float4 v = reinterpret_cast<const float4*>(p)[idx];
    r.x = v.x;
    r.y = v.y;
    r.z = v.z;
    r.w = v.w;
#endif
    return r;
}
VGC_HD void lds_pair(const float* p, const LI& idx, LF& a, LF& b) {
#if defined(VGC_EMU)
    for (int l = 0; l < kWave; ++l) {
        a[l] = p[2 * idx[l]];
        b[l] = p[2 * idx[l] + 1];
    }
#else
    const float2 v = reinterpret_cast<const float2*>(p)[idx];
    a = v.x;
    b = v.y;
#endif
}
VGC_HD void lds_st_row(float* p, const LI& idx, const LF& x, const LF& y, const LF& z, const LF& w,
                       const LB& m) {
#if defined(VGC_EMU)
    for (int l = 0; l < kWave; ++l)
        if (m[l]) {
            float* q = p + 4 * idx[l];
            q[0] = x[l];
            q[1] = y[l];
            q[2] = z[l];
            q[3] = w[l];
        }
#else
    if (m) reinterpret_cast<float4*>(p)[idx] = make_float4(x, y, z, w);
#endif
}
// masked store to global memory at a per-lane index
template <class T>
VGC_HD void gst(T* p, const Lane<long long>& idx, const Lane<T>& v, const LB& m) {
#if defined(VGC_EMU)
    for (int l = 0; l < kWave; ++l)
        if (m[l]) p[idx[l]] = v[l];
#else
    if (m) p[idx] = v;
#endif
}

#if defined(VGC_EMU)
#define VGC_PT_FIELD(F)                               \
    inline LD pt_##F(const Lane<pt4>& q) {            \
        LD r;                                         \
        for (int l = 0; l < kWave; ++l) r[l] = q[l].F; \
        return r;                                     \
    }
#else
#define VGC_PT_FIELD(F) \
    VGC_HD double pt_##F(const pt4& q) { return q.F; }
#endif
VGC_PT_FIELD(x)
VGC_PT_FIELD(y)
VGC_PT_FIELD(z)
VGC_PT_FIELD(w)
#undef VGC_PT_FIELD

// the power of two s with 1 <= s^2 x < 4 (x > 0, normal)
VGC_HD LF pow2_inv_sqrt(const LF& x) {
    const LI e = (cvt<int>(fbits(x) >> LU(23)) & 0xFF) - 127;
    return from_bits(cvt<uint32_t>(127 - (e >> 1)) << LU(23));
}

// Corner of three scaled FP32 rows (make_corner's formulas), with the bounds
// premultiplied for the tests: gn = gamma9 max|N|abs, gd = gamma9 |D|abs, and
// num / den2 the upper bound of 4.1 times its squared distance (make_corner's
// FP32 radius bound without the division).
struct PairCorner {
    LF nx, ny, nz, d, gn, gd, num, den2;
    LB bad;
};
VGC_HD PairCorner pair_corner(const RowLanes& a, const RowLanes& b, const RowLanes& c) {
    constexpr float G = Prec<float>::gamma9;
    PairCorner C;
    const LF bcx = vfma(b.y, c.z, -(b.z * c.y)), bcy = vfma(b.z, c.x, -(b.x * c.z)),
             bcz = vfma(b.x, c.y, -(b.y * c.x));
    const LF cax = vfma(c.y, a.z, -(c.z * a.y)), cay = vfma(c.z, a.x, -(c.x * a.z)),
             caz = vfma(c.x, a.y, -(c.y * a.x));
    const LF abx = vfma(a.y, b.z, -(a.z * b.y)), aby = vfma(a.z, b.x, -(a.x * b.z)),
             abz = vfma(a.x, b.y, -(a.y * b.x));
    const LF Aax = vabs(a.x), Aay = vabs(a.y), Aaz = vabs(a.z), Aah = vabs(a.w);
    const LF Abx = vabs(b.x), Aby = vabs(b.y), Abz = vabs(b.z), Abh = vabs(b.w);
    const LF Acx = vabs(c.x), Acy = vabs(c.y), Acz = vabs(c.z), Ach = vabs(c.w);
    const LF mbcx = vfma(Aby, Acz, Abz * Acy), mbcy = vfma(Abz, Acx, Abx * Acz),
             mbcz = vfma(Abx, Acy, Aby * Acx);
    const LF mcax = vfma(Acy, Aaz, Acz * Aay), mcay = vfma(Acz, Aax, Acx * Aaz),
             mcaz = vfma(Acx, Aay, Acy * Aax);
    const LF mabx = vfma(Aay, Abz, Aaz * Aby), maby = vfma(Aaz, Abx, Aax * Abz),
             mabz = vfma(Aax, Aby, Aay * Abx);
    C.nx = vfma(a.w, bcx, vfma(b.w, cax, c.w * abx));
    C.ny = vfma(a.w, bcy, vfma(b.w, cay, c.w * aby));
    C.nz = vfma(a.w, bcz, vfma(b.w, caz, c.w * abz));
    C.d = vfma(a.x, bcx, vfma(a.y, bcy, a.z * bcz));
    const LF nax = vfma(Aah, mbcx, vfma(Abh, mcax, Ach * mabx));
    const LF nay = vfma(Aah, mbcy, vfma(Abh, mcay, Ach * maby));
    const LF naz = vfma(Aah, mbcz, vfma(Abh, mcaz, Ach * mabz));
    const LF nmax = vmax(nax, vmax(nay, naz));
    const LF dabs = vfma(Aax, mbcx, vfma(Aay, mbcy, Aaz * mbcz));
    C.bad = !(C.d > Prec<float>::gamma5 * dabs) | !(dabs >= kPairDabsMin) | !(dabs < kPairDabsMax) |
            !(nmax < kPairNMax);
    C.gn = G * nmax;
    C.gd = G * dabs;
    const LF e = 1.8f * C.gn;
    const LF m = vmax(vabs(C.nx), vmax(vabs(C.ny), vabs(C.nz)));
    C.num = (vfma(C.nx, C.nx, vfma(C.ny, C.ny, C.nz * C.nz)) + e * vfma(LF(3.47f), m, e)) *
            (4.1f * 1.00001f);
    const LF den = C.d - C.gd;
    C.den2 = den * den;
    return C;
}

// Corner state of the pair; slot s of lane l is corner 32 s + l % 32 of the
// cell of lane l's half
struct PairState {
    LF nx[2], ny[2], nz[2], d[2], gn[2], gd[2], num[2], den2[2];
    LU pl[2], adj[2];
    uint64_t valid[2];
};

// algorithmic work of the two cells (VGC_COUNT_WORK)
struct PairWork {
    uint64_t nclip[2], ntest[2], nlive[2], nnew[2];
};

// Is bit idx (a corner id of the lane's own cell) set?  w0 / w1: the cell's
// words of slots 0 and 1.
VGC_HD LB pair_bit(const LU& w0, const LU& w1, const LU& idx, bool two) {
    if (!two) return ((w0 >> (idx & LU(31u))) & LU(1u)) != LU(0u);
    return ((select(idx < LU(32u), w0, w1) >> (idx & LU(31u))) & LU(1u)) != LU(0u);
}

// byte k of w replaced by the low byte of v
VGC_HD LU set_byte(const LU& w, int k, const LU& v) {
#if defined(VGC_EMU)
    return (w & ~LU(0xFFu << (8 * k))) | ((v & LU(0xFFu)) << LU(8 * k));
#else
    // selector bytes 4..7 take from w, 0..3 from v
    return __builtin_amdgcn_perm(w, v, k == 0 ? 0x07060500u : k == 1 ? 0x07060004u : 0x07000504u);
#endif
}

// a | b << 8 | y << 16 from bytes k and k + 1 (of three) of pl and byte k of
// adj
VGC_HD LU pack_job(const LU& pl, const LU& adj, int k) {
#if defined(VGC_EMU)
    return byte_of(pl, k) | (byte_of(pl, (k + 1) % 3) << LU(8)) | (byte_of(adj, k) << LU(16));
#else
    // bytes 4..7 of the selector's source are pl, 0..3 adj; 0x0c: zero
    const uint32_t sel = k == 0 ? 0x0c000504u : k == 1 ? 0x0c010605u : 0x0c020406u;
    return __builtin_amdgcn_perm(pl, adj, sel);
#endif
}

// ranks of the lanes of m within their half, counted from a (lower half) or
// b (upper half)
VGC_HD LI half_rank(uint64_t m, int a, int b, const LB& up) {
#if defined(VGC_EMU)
    LI r = mbcnt(m);
    for (int l = 0; l < kWave; ++l) r[l] += up[l] ? b - popc_half(m, 0) : a;
    return r;
#else
    const int base = select(up, b - popc_half(m, 0), a);
    return __builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32),
                                     __builtin_amdgcn_mbcnt_lo(uint32_t(m), uint32_t(base)));
#endif
}

// The planes of the halves in `pend`, whose rows are r (with neighbour j and
// conflict masks cf), cut their cells (np planes so far).  Returns the halves
// whose cell cannot go on here (plane or corner capacity, a corner not
// certified); `empty` receives those whose cell vanished.
template <bool COUNT>
VGC_HD uint64_t pair_cut(PairState& st, PairLds& L, LI& np, const RowLanes& r, const LI& j,
                         uint64_t pend, const uint64_t (&cf)[2], const LB& up, const LI& hl,
                         PairWork& work, uint64_t& empty) {
    uint64_t c0 = cf[0] & pend, c1 = cf[1] & pend;
    // every corner in conflict: the cell is empty
    empty = pend & ~halves((st.valid[0] & ~c0) | (st.valid[1] & ~c1));
    pend &= ~empty;
    uint64_t fail = pend & ballot(np >= kPairPlanes);
    pend &= ~fail;
    c0 &= pend;
    c1 &= pend;
    const bool two = st.valid[1] != 0;
    const LU w0 = half_word(c0, up), w1 = two ? half_word(c1, up) : LU(0u);
    const LI hoff = select(up, LI(int(sizeof(PairHalf))), LI(0));
    {
        const LB m = mask_bit(pend) & (hl == 0);
        lds_st_row(&L.h[0].pe[0][0], (hoff >> 4) + np, r.x, r.y, r.z, r.w, m);
        lds_st(L.h[0].pg, (hoff >> 2) + np, j, m);
    }
    // neighbours in conflict across each edge: border edges of conflicting
    // corners have none, kept corners with one are re-linked below
    const uint64_t k0 = st.valid[0] & ~c0 & pend, k1 = st.valid[1] & ~c1 & pend;
    uint64_t nb0[3], nb1[3];
    int ta = 0, tb = 0;  // new corners of each half
    int ba[6], bb[6];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        nb0[k] = ballot(pair_bit(w0, w1, byte_of(st.adj[0], k), two));
        nb1[k] = two ? ballot(pair_bit(w0, w1, byte_of(st.adj[1], k), two)) : 0ull;
        ba[2 * k] = ta;
        bb[2 * k] = tb;
        ta += popc_half(c0 & ~nb0[k], 0);
        tb += popc_half(c0 & ~nb0[k], 1);
        ba[2 * k + 1] = ta;
        bb[2 * k + 1] = tb;
        ta += popc_half(c1 & ~nb1[k], 0);
        tb += popc_half(c1 & ~nb1[k], 1);
    }
    const uint64_t f0 = pend & ~k0, f1 = pend & ~k1;
    if (ta > popc_half(f0, 0) + popc_half(f1, 0)) fail |= pend & kLoHalf;
    if (tb > popc_half(f0, 1) + popc_half(f1, 1)) fail |= pend & kHiHalf;
    pend &= ~fail;
    if (pend == 0) return fail;
    if (COUNT) {
        work.nnew[0] += (pend & kLoHalf) ? ta : 0;
        work.nnew[1] += (pend & kHiHalf) ? tb : 0;
    }
    // jobs in (edge, corner) order
    const LI joff = hoff >> 2;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const uint64_t m0 = c0 & ~nb0[k] & pend;
        lds_st(L.h[0].job, joff + half_rank(m0, ba[2 * k], bb[2 * k], up),
               pack_job(st.pl[0], st.adj[0], k), mask_bit(m0));
        if (two) {
            const uint64_t m1 = c1 & ~nb1[k] & pend;
            lds_st(L.h[0].job, joff + half_rank(m1, ba[2 * k + 1], bb[2 * k + 1], up),
                   pack_job(st.pl[1], st.adj[1], k), mask_bit(m1));
        }
    }
    wave_sync();
    // targets: the first free corner slots
    const LI total = select(up, LI(tb), LI(ta));
    uint64_t t0, t1 = 0, bad = 0;
    LI cid0 = hl, rank1 = LI(0);
    auto target = [&](int s, const LI& rank, uint64_t tm) {
        const LB is_t = mask_bit(tm);
        const LU jb = lds_ld(L.h[0].job, joff + select(is_t, rank, LI(0)));
        const LI a = cvt<int>(jb & LU(0xFFu)) & (kPairPlanes - 1);
        const LI b = cvt<int>((jb >> LU(8)) & LU(0xFFu)) & (kPairPlanes - 1);
        const RowLanes ra = lds_row(&L.h[0].pe[0][0], (hoff >> 4) + a);
        const RowLanes rb = lds_row(&L.h[0].pe[0][0], (hoff >> 4) + b);
        const PairCorner C = pair_corner(ra, rb, r);
        bad |= ballot(is_t & C.bad);
        st.nx[s] = select(is_t, C.nx, st.nx[s]);
        st.ny[s] = select(is_t, C.ny, st.ny[s]);
        st.nz[s] = select(is_t, C.nz, st.nz[s]);
        st.d[s] = select(is_t, C.d, st.d[s]);
        st.gn[s] = select(is_t, C.gn, st.gn[s]);
        st.gd[s] = select(is_t, C.gd, st.gd[s]);
        st.num[s] = select(is_t, C.num, st.num[s]);
        st.den2[s] = select(is_t, C.den2, st.den2[s]);
        st.pl[s] = select(is_t, (jb & LU(0xFFFFu)) | (cvt<uint32_t>(np) << LU(16)), st.pl[s]);
        st.adj[s] = select(is_t, jb >> LU(16), st.adj[s]);
        const Lane<uint8_t> id = cvt<uint8_t>(hl + 32 * s);
        lds_st(L.h[0].st_tab, hoff + a, id, is_t);
        lds_st(L.h[0].en_tab, hoff + b, id, is_t);
    };
    {
        const LI rank = half_rank(f0, 0, 0, up);
        t0 = ballot(mask_bit(f0 & pend) & (rank < total));
        target(0, rank, t0);
    }
    const int fa = popc_half(f0, 0), fb = popc_half(f0, 1);
    if (ta > fa || tb > fb) {
        rank1 = half_rank(f1, fa, fb, up);
        t1 = ballot(mask_bit(f1 & pend) & (rank1 < total));
        if (t1) target(1, rank1, t1);
    }
    // (uniform again: the branches above join where lanes' stores do)
    t1 = uni(t1);
    bad = uni(bad);
    wave_sync();
    // link the new corners around the new face; kept corners re-point to them
    auto link = [&](int s, uint64_t tm, const uint64_t (&nb)[3], uint64_t keep) {
        const LB is_t = mask_bit(tm);
        const LU a = st.pl[s] & LU(kPairPlanes - 1), b = (st.pl[s] >> LU(8)) & LU(kPairPlanes - 1);
        const Lane<uint8_t> n1 = lds_ld(L.h[0].st_tab, hoff + cvt<int>(b));
        const Lane<uint8_t> n2 = lds_ld(L.h[0].en_tab, hoff + cvt<int>(a));
        const LU lk = (st.adj[s] & LU(0xFFu)) | (cvt<uint32_t>(n1) << LU(8)) |
                      (cvt<uint32_t>(n2) << LU(16));
        st.adj[s] = select(is_t, lk, st.adj[s]);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const uint64_t hit = keep & nb[k];
            if (hit) {
                const LI v = cvt<int>(byte_of(st.pl[s], (k + 1) % 3)) & (kPairPlanes - 1);
                const Lane<uint8_t> z = lds_ld(L.h[0].st_tab, hoff + v);
                st.adj[s] = select(mask_bit(hit), set_byte(st.adj[s], k, cvt<uint32_t>(z)), st.adj[s]);
            }
        }
    };
    link(0, t0, nb0, k0 & pend);
    if (two || t1) link(1, t1, nb1, k1 & pend);
    st.valid[0] = (st.valid[0] & ~pend) | (k0 & pend) | t0;
    st.valid[1] = (st.valid[1] & ~pend) | (k1 & pend) | t1;
    np = np + select(mask_bit(pend), LI(1), LI(0));
    wave_sync();
    return fail | halves(bad);
}

// The cnt <= kStageCap sorted candidates of half h as FP32 rows; returns the
// number staged.  A candidate with the position and weight of the one before
// it gives the same plane and is not staged: its id takes the other's place
// (under the exact tie rule the copy takes over the face of the first one).
// A candidate at the position of the seed c itself is not staged either if it
// comes later in the caller's order (consider's rule).  -1 when a candidate
// needs the general kernel: an earlier one at the seed's position, or a row out
// of the range of the FP32 bounds.
template <bool W>
VGC_HD int pair_stage(const ClipParams& P, PairLds& L, int h, int c, float scale, const pt4& pc,
                      double cw, int cnt) {
    const LI lane = lane_id();
    const LB ok = lane < cnt;
    const LU64 key = lds_ld(L.h[h].key, select(ok, lane, LI(0)));
    const LI j = cvt<int>(cvt<uint32_t>(key));
    const Lane<pt4> q = gld(P.pts, j, ok);
    const LD s = LD(double(scale));
    const LD ex = pt_x(q) - pc.x, ey = pt_y(q) - pc.y, ez = pt_z(q) - pc.z;
    const LD d2 = ex * ex + ey * ey + ez * ez;
    LD h2 = 0.5 * d2;
    LD rho = d2;
    if constexpr (W) {
        h2 = 0.5 * (d2 + (pc.w - pt_w(q)));
        const LD sd = d2 + cw;
        // no corner can be out of reach while sd <= 0
        rho = select(sd > 0.0, sd * (sd / d2), LD(-1.0)) * (1.0 - 1e-6);
    }
    const LF fx = cvt<float>(ex * s), fy = cvt<float>(ey * s), fz = cvt<float>(ez * s);
    const LF fh = cvt<float>(h2 * s * s), fr = cvt<float>(rho * s * s);
    const LF e1 = vabs(fx) + vabs(fy) + vabs(fz);
    float* row = &L.stage[h].row[0][0];
    float* aux = &L.stage[h].aux[0][0];
    wave_sync();  // the previous ring is consumed
    lds_st_row(row, lane, fx, fy, fz, fh, ok);
    lds_st(aux, lane * 2, fr, ok);
    lds_st(aux, lane * 2 + 1, e1, ok);
    wave_sync();
    const LB out = ok & (!(d2 > 0.0) | !(e1 >= kPairE1Min) | !(e1 <= kPairE1Max) | !(vabs(fh) <= kPairHMax));
    const uint64_t om = ballot(out);
    uint64_t zm = 0;  // at the seed
    if (om) {
        zm = ballot(ok & (d2 == 0.0));
        if (om & ~zm) return -1;
        const LI oj = gld(P.orig, select(mask_bit(zm), j, LI(0)), mask_bit(zm));
        if (ballot(mask_bit(zm) & (oj < P.orig[c]))) return -1;
    }
    // copies follow one another in the sorted order, at one FP32 distance
    const LU64 kp = lds_ld(L.h[h].key, select(ok & (lane > 0), lane - 1, LI(0)));
    const LB same = ok & (lane > 0) & ((kp >> LU64(32)) == (key >> LU64(32)));
    if (ballot(same) == 0 && zm == 0) return cnt;
    const LI jp = cvt<int>(cvt<uint32_t>(kp));
    const Lane<pt4> qp = gld(P.pts, jp, same);
    const uint64_t dm = ballot(same & (pt_x(qp) == pt_x(q)) & (pt_y(qp) == pt_y(q)) &
                               (pt_z(qp) == pt_z(q)) & (pt_w(qp) == pt_w(q)));
    if ((dm | zm) == 0) return cnt;
    const uint64_t okm = ballot(ok) & ~zm, keep = okm & ~dm, last = okm & ~((dm & ~zm) >> 1);
    const LI at = mbcnt(keep) - select(mask_bit(keep), LI(0), LI(1));
    wave_sync();
    lds_st_row(row, at, fx, fy, fz, fh, mask_bit(keep));
    lds_st(aux, at * 2, fr, mask_bit(keep));
    lds_st(aux, at * 2 + 1, e1, mask_bit(keep));
    lds_st(L.h[h].key, at, key, mask_bit(last));
    wave_sync();
    return popc64(keep);
}

// A half's corner values by corner id over the whole wave.
VGC_HD LF pair_to_wave(const LF& x0, const LF& x1, int h) {
    const LI lane = lane_id();
    const LI src = (lane & 31) + 32 * h;
    return select(lane < 32, shfl(x0, src), shfl(x1, src));
}

// ---------------------------------------------------- neighbour search
//
// A wave's cells are consecutive in Morton order, so they share one walk of
// the tree: the buckets within a radius r of the box of their seeds go to
// L.near_list once, and each cell's first ring (and its next ones, while
// they stay within r) is a scan of those buckets.  A walk per cell and the
// repeats of rings that had come out too large cost 40 % of the pass.

// The wave's shared bucket list: complete for every seed of instance inst
// within sqrt(r2) of the wave's seeds.
struct NearList {
    int inst;  // -1: no list (each cell walks the tree)
    int n;
    float r2;
};
// radius of the list and of a first ring over the mean 4th nearest distance
// among bucket mates
constexpr float kNearList = 2.3f, kNearRing = 1.95f;

// Mean distance to the 4th nearest bucket mate of 4 * passes seeds of the
// bucket of seed c (0: none has four).
VGC_HD float near_spacing(const ClipParams& P, int c, int inst, int passes) {
    const LI lane = lane_id();
    const int p0 = P.IL.p0[inst], n = P.IL.n[inst];
    const int m0 = c - ((c - p0) & (kBucket - 1));
    float sum = 0.0f, cnt = 0.0f;
    const LI m = m0 + (lane & (kBucket - 1));
    const LB in = m < p0 + n;
    const SeedLanes q = lane_seed(P.pf, select(in, m, LI(m0)), in);
    for (int k = 0; k < passes; ++k) {
        // row r of 16 lanes takes seed 4 (k + c / 4) + r of the bucket
        const LI s = m0 + ((((c - m0) & ~3) + 4 * k + (lane >> 4)) & (kBucket - 1));
        const LB sin = s < p0 + n;
        const SeedLanes p = lane_seed(P.pf, select(sin, s, LI(m0)), sin);
        const LF dx = q.x - p.x, dy = q.y - p.y, dz = q.z - p.z;
        const LB ok = in & sin & (m != s);
        const LF d2 = select(ok, dx * dx + dy * dy + dz * dz, LF(INFINITY));
        LI below = LI(0);
#pragma unroll
        for (int i = 1; i < kBucket; ++i) below = below + select(row_ror(d2, i) < d2, LI(1), LI(0));
        uint64_t fourth = ballot((below == 3) & (d2 < INFINITY));
        for (int r = 0; r < 4; ++r) {
            const uint64_t f = fourth & (0xFFFFull << (16 * r));
            if (!f) continue;
            const float d = readlane(d2, ffs64(f));
            sum += sqrtf(d);
            cnt += 1.0f;
        }
    }
    return cnt > 0.0f ? sum / cnt : 0.0f;
}

// The buckets of instance inst within sqrt(r2) of the box of the points p of
// the lanes in `has` into L.near_list; returns their number, -1 when they or
// the walk overflow.
template <class LDS>
VGC_HD int near_buckets(const ClipParams& P, LDS& L, int inst, const SeedLanes& p, const LB& has,
                        float r2) {
    const LI lane = lane_id();
    const float hx = wave_maxf(select(has, p.x, LF(-INFINITY))), lx = -wave_maxf(select(has, -p.x, LF(-INFINITY)));
    const float hy = wave_maxf(select(has, p.y, LF(-INFINITY))), ly = -wave_maxf(select(has, -p.y, LF(-INFINITY)));
    const float hz = wave_maxf(select(has, p.z, LF(-INFINITY))), lz = -wave_maxf(select(has, -p.z, LF(-INFINITY)));
    const int nb = P.IL.nb[inst], Lv = P.IL.L[inst];
    const bnode* T = P.nodes + P.IL.t0[inst];
    int nf = walk_start(L, Lv), cur = 0, nbk = 0;
    while (nf > 0) {
        int nn = 0;
        for (int base = 0; base < nf; base += kWave) {
            const LI idx = base + lane;
            const LB in = idx < nf;
            const LI node = lds_ld(&L.front[cur][0], select(in, idx, LI(0)));
            const BoxLanes B = load_box(T, node, in);
            const LF dx = vmaxf(vmaxf(B.lx - hx, lx - B.hx), 0.0f);
            const LF dy = vmaxf(vmaxf(B.ly - hy, ly - B.hy), 0.0f);
            const LF dz = vmaxf(vmaxf(B.lz - hz, lz - B.hz), 0.0f);
            // (the margin covers the rounding of a seed's own distances)
            const LB hit = in & ((dx * dx + dy * dy + dz * dz) * 0.99999f <= r2);
            const LB internal = node < Lv;
            const LB push = hit & internal;
            const LB leaf = hit & !internal & (node - Lv < nb);
            const LB deep = push & (2 * node < Lv);
            const uint64_t mp = ballot(push), md = ballot(deep), ml = ballot(leaf);
            const LI rp = nn + 2 * mbcnt(mp) + 2 * mbcnt(md);
            const LI first = select(deep, 4 * node, 2 * node);
            const LB okp = push & (rp + select(deep, LI(3), LI(1)) < kFrontCap);
            lds_st(&L.front[cur ^ 1][0], select(okp, rp, LI(0)), first, okp);
            lds_st(&L.front[cur ^ 1][0], select(okp, rp + 1, LI(0)), first + 1, okp);
            const LB okd = okp & deep;
            lds_st(&L.front[cur ^ 1][0], select(okd, rp + 2, LI(0)), first + 2, okd);
            lds_st(&L.front[cur ^ 1][0], select(okd, rp + 3, LI(0)), first + 3, okd);
            const LI rl = nbk + mbcnt(ml);
            lds_st(L.near_list, select(rl < kNearCap, rl, LI(0)), node - Lv, leaf & (rl < kNearCap));
            nn += 2 * popc64(mp) + 2 * popc64(md);
            nbk += popc64(ml);
        }
        wave_sync();
        if (nn > kFrontCap || nbk > kNearCap) return -1;
        nf = nn;
        cur ^= 1;
    }
    return nbk;
}

// The listed seeds q with lo < d2 <= hi of the cells of the two halves
// (seeds ca, cb at a, b; hi < 0: none wanted) into L.cand and L.cand_b as
// (d2 bits << 32 | q), unsorted.  na, nb receive their numbers (only the
// first kCandCap are stored).
template <class LDS>
VGC_HD void near_scan(const ClipParams& P, LDS& L, const NearList& N, int ca, int cb, const pf4& a,
                      const pf4& b, float loa, float hia, float lob, float hib, int& na, int& nb) {
    const LI lane = lane_id();
    const int p0 = P.IL.p0[N.inst], n = P.IL.n[N.inst], Lv = P.IL.L[N.inst];
    const bnode* T = P.nodes + P.IL.t0[N.inst];
    int nbk = 0;
    for (int base = 0; base < N.n; base += kWave) {
        const LI idx = base + lane;
        const LB in = idx < N.n;
        const LI bk = lds_ld(L.near_list, select(in, idx, LI(0)));
        const BoxLanes B = load_box(T, bk + Lv, in);
        const LF ax = vmaxf(vmaxf(B.lx - a.x, a.x - B.hx), 0.0f);
        const LF ay = vmaxf(vmaxf(B.ly - a.y, a.y - B.hy), 0.0f);
        const LF az = vmaxf(vmaxf(B.lz - a.z, a.z - B.hz), 0.0f);
        const LF bx = vmaxf(vmaxf(B.lx - b.x, b.x - B.hx), 0.0f);
        const LF by = vmaxf(vmaxf(B.ly - b.y, b.y - B.hy), 0.0f);
        const LF bz = vmaxf(vmaxf(B.lz - b.z, b.z - B.hz), 0.0f);
        const LB hit = in & ((ax * ax + ay * ay + az * az <= hia) | (bx * bx + by * by + bz * bz <= hib));
        const uint64_t m = ballot(hit);
        const LI r = nbk + mbcnt(m);
        lds_st(L.bucket, select(hit, r, LI(0)) & (kBucketCap - 1), bk, hit & (r < kBucketCap));
        nbk += popc64(m);
    }
    wave_sync();
    if (nbk > kBucketCap) {
        // more than kBucketCap buckets around one cell: more seeds than a
        // ring holds
        na = nb = kBucketCap * kBucket;
        return;
    }
    na = nb = 0;
    for (int base = 0; base < nbk; base += kWave / kBucket) {
        const LI bi = base + (lane >> 4);
        const LB inb = bi < nbk;
        const LI m = p0 + lds_ld(L.bucket, select(inb, bi, LI(0))) * kBucket + (lane & (kBucket - 1));
        const LB ok = inb & (m < p0 + n);
        const SeedLanes q = lane_seed(P.pf, select(ok, m, LI(p0)), ok);
        const LF ax = q.x - a.x, ay = q.y - a.y, az = q.z - a.z;
        const LF bx = q.x - b.x, by = q.y - b.y, bz = q.z - b.z;
        const LF da = ax * ax + ay * ay + az * az, db = bx * bx + by * by + bz * bz;
        const uint64_t ta = ballot(ok & (da > loa) & (da <= hia) & (m != ca));
        const uint64_t tb = ballot(ok & (db > lob) & (db <= hib) & (m != cb));
        const LU64 id = cvt<uint64_t>(cvt<uint32_t>(m));
        const LI ra = na + mbcnt(ta), rb = nb + mbcnt(tb);
        lds_st(L.cand, ra & (kCandCap - 1), (cvt<uint64_t>(fbits(da)) << LU64(32)) | id,
               mask_bit(ta) & (ra < kCandCap));
        lds_st(L.cand_b, rb & (kCandCap - 1), (cvt<uint64_t>(fbits(db)) << LU64(32)) | id,
               mask_bit(tb) & (rb < kCandCap));
        na += popc64(ta);
        nb += popc64(tb);
    }
    wave_sync();
}

// The nearest of the ring's n <= kCandCap unsorted candidates src into out in
// ascending order, at most kStageCap: of more, those within a lowered bound
// that keeps 52 .. kStageCap of them where the distances allow (the others are
// gathered again if the cell still needs them; from 40, 48 or 58 on: within
// 0.5 % on 2000 to 2M seeds).  rhi2 is lowered to that
// bound; returns the count, -1 when more than kStageCap share one distance.
// Sorted by counting: a lane's rank is the number of keys below its own (two
// instructions per key, against 21 rounds of compares and LDS traffic of a
// bitonic network).
VGC_HD int ring_sort(uint64_t* src, int n, float& rhi2, uint64_t* out) {
    const LI lane = lane_id();
    const LB in0 = lane < n;
    LU64 a = lds_ld(src, select(in0, lane, LI(0)));
    if (n > kStageCap) {
        const LB in1 = lane + kWave < n;
        const LU64 b = lds_ld(src, select(in1, lane + kWave, LI(0)));
        const LF da = from_bits(cvt<uint32_t>(a >> LU64(32))), db = from_bits(cvt<uint32_t>(b >> LU64(32)));
        float lo = 0.0f, hi = rhi2, best = 0.0f;
        int keep = 0;
        for (int it = 0; it < 32; ++it) {
            const float t = it == 0 ? hi * (0.4f + 0.6f * 58.0f / float(n)) : 0.5f * (lo + hi);
            const int k = popc64(ballot(in0 & (da <= t))) + popc64(ballot(in1 & (db <= t)));
            if (k > kStageCap) {
                hi = t;
                continue;
            }
            lo = t;
            if (k > keep) {
                keep = k;
                best = t;
            }
            if (k >= 52) break;
        }
        if (keep == 0) return -1;
        rhi2 = uni(best);
        // the kept ones together (every key read before the first write)
        const LB ka = in0 & (da <= rhi2), kb = in1 & (db <= rhi2);
        const uint64_t ma = ballot(ka), mb = ballot(kb);
        wave_sync();
        lds_st(src, select(ka, mbcnt(ma), LI(0)), a, ka);
        lds_st(src, select(kb, popc64(ma) + mbcnt(mb), LI(0)), b, kb);
        wave_sync();
        n = keep;
        a = lds_ld(src, select(lane < n, lane, LI(0)));
    }
    LI rank = LI(0);
    for (int i = 0; i < n; ++i) rank = rank + select(lds_ld(src, LI(i)) < a, LI(1), LI(0));
    lds_st(out, select(lane < n, rank, LI(0)), a, lane < n);
    wave_sync();
    return n;
}

// ------------------------------------------------------------- the pair

// The next ring of half h, gathered and sorted into L.h[h].key (c: the seed;
// first: no ring yet).  Returns the candidate count, -1 when the cell is
// complete, -2 when the cell is left to the FP64 pass, -3 when it has used up
// its rings.
template <bool W>
VGC_HD int pair_ring(const ClipParams& P, PairLds& L, const PairState& st, const NearList& N, int h,
                     bool first) {
    PairCtl& K = L.ctl[h];
    const int c = uni(K.c), inst = uni(K.inst);
    float rlo2 = uni(K.rlo2), rhi2 = uni(K.rhi2);
    int nfilt = uni(K.nfilt);
    bool ct_on = uni(K.ct_on) != 0;
    const pf4 pq = P.pf[c];
    PowerFilter F{};
    CornerTab CT;
    CT.live = 0;
    if (!first) {
        // ring exhausted: can a seed beyond rhi2 still cut the cell?
        const float all2 = uni(K.all2), inv = uni(K.inv);
        const pt4 pc = P.pts[c];
        const uint64_t hm = half_mask(h);
        LF r2 = select(mask_bit(st.valid[0] & hm), st.num[0] / st.den2[0], LF(0.0f));
        if (st.valid[1] & hm)
            r2 = vmax(r2, select(mask_bit(st.valid[1] & hm), st.num[1] / st.den2[1], LF(0.0f)));
        // num carries the factor 4.1 of the security radius
        const double r2now =
            double(wave_maxf(r2)) * ((1.0 / 4.1) * (1.0 + 1e-6)) * double(inv) * double(inv);
        const float need2 = radius_for(r2now, pc.w, W ? P.wmax[inst] : 0.0, W);
        if (uni(need2 <= rhi2 || rhi2 >= all2)) return -1;
        rlo2 = rhi2;
        rhi2 = need2 < all2 ? need2 : all2;
        if (uni(inst == N.inst && rhi2 <= N.r2)) {
            int n, none;
            near_scan(P, L, N, c, c, pq, pq, rlo2, rhi2, 0.0f, -1.0f, n, none);
            if (n <= kCandCap) {
                n = ring_sort(L.cand, n, rhi2, L.h[h].key);
                K.rlo2 = rlo2;
                K.rhi2 = rhi2;
                wave_sync();
                return n < 0 ? -2 : n;
            }
        }
        // filter of the partial cell: its corners by id over the wave
        CellRun<1, float> R;
        R.pc = pc;
        R.wi = pc.w;
        R.box = P.box + 6 * inst;
        const float g = 1.000001f / Prec<float>::gamma9;
        R.st.nx[0] = pair_to_wave(st.nx[0], st.nx[1], h) * inv;
        R.st.ny[0] = pair_to_wave(st.ny[0], st.ny[1], h) * inv;
        R.st.nz[0] = pair_to_wave(st.nz[0], st.nz[1], h) * inv;
        R.st.d[0] = pair_to_wave(st.d[0], st.d[1], h);
        R.st.nmax[0] = pair_to_wave(st.gn[0], st.gn[1], h) * (inv * g);
        R.st.dabs[0] = pair_to_wave(st.gd[0], st.gd[1], h) * g;
        R.st.valid[0] = h ? (st.valid[0] >> 32) | (st.valid[1] & kHiHalf)
                          : (st.valid[0] & kLoHalf) | (st.valid[1] << 32);
        if (!make_filter<1, W>(R, F, CT)) {
            F.on = 0;
            CT.live = 0;
        }
    }
    int n;
    while (true) {
        n = first ? gather_ring(P, L, c, inst, pq.x, pq.y, pq.z, rlo2, rhi2, F)
                  : gather_dfs<W>(P, L, c, inst, pq.x, pq.y, pq.z, rlo2, rhi2, F, CT, ct_on);
        if (F.on && ++nfilt > P.pair_rings) return -3;
        if (n >= 0 && n <= kCandCap) break;
        // too many seeds (or tree nodes): narrow the ring, same shell-volume
        // fraction in r^3, and gather again
        const float lo = rlo2 > 0.0f ? rlo2 : 0.0f;
        const float r3lo = lo * sqrtf(lo), r3hi = rhi2 * sqrtf(rhi2);
        const float frac = n < 0 ? 0.125f : 0.75f * kCandCap / float(n);
        float nh = cbrtf(r3lo + (r3hi - r3lo) * frac);
        nh = nh * nh;
        if (uni(!(nh > lo * 1.000001f) || !(nh < rhi2))) return -2;
        rhi2 = nh;
    }
    n = ring_sort(L.cand, n, rhi2, L.h[h].key);
    K.rlo2 = rlo2;
    K.rhi2 = rhi2;
    K.nfilt = nfilt;
    K.ct_on = ct_on;
    wave_sync();
    return n < 0 ? -2 : n;
}

// Items item0 and item0 + 1 (the second only if below end); near2: squared
// radius of the first ring (0: unknown).
template <bool W, bool COUNT>
VGC_HD void process_pair(const ClipParams& P, int item0, int end, PairLds& L, const NearList& N,
                         float near2) {
    const LI lane = lane_id_here();
    const LB up = lane >= 32;
    const LI hl = lane & 31;
    wave_sync();  // the previous pair of this wave is done with the LDS
    // a cell's scalars are held by every lane of its half
    const LI item = select(up, LI(item0 + 1), LI(item0));
    const LB have = item < end;
    const LI items = select(have, item, LI(item0));
    const LI c = P.items ? gld(P.items, items, LB(true)) : items;
    const LI inst = P.inst_of ? gld(P.inst_of, c, LB(true)) : LI(0);
    const LI oc = gld(P.orig, c, LB(true));
    LB on = have;
    if (P.abort_flag) on = on & !flag_up(P.abort_flag, inst);
    if (P.n_real > 0) {
        // an image of a seed across the period: a candidate only
        const LB image = on & (oc >= P.n_real);
        gst(P.flags, cvt<long long>(c), LU(uint32_t(CELL_DONE)), image & (hl == 0));
        on = on & !image;
    }
    uint64_t live = ballot(on);
    if (live == 0) return;

    // the first ring: the radius of the wave's bucket list (or, without one,
    // the radius that holds about 60 seeds of a cloud spread over the box)
    LF scale;
    {
        const LI n = gld(P.IL.n, inst, LB(true));
        const LI b6 = inst * 6;
        const LF bx = cvt<float>(gld(P.box, b6 + 3, LB(true)) - gld(P.box, b6 + 0, LB(true)));
        const LF by = cvt<float>(gld(P.box, b6 + 4, LB(true)) - gld(P.box, b6 + 1, LB(true)));
        const LF bz = cvt<float>(gld(P.box, b6 + 5, LB(true)) - gld(P.box, b6 + 2, LB(true)));
        const LF all2 = (bx * bx + by * by + bz * bz) * 1.0002f;
        const LF nf = cvt<float>(n);
        const LF rhi2 = near2 > 0.0f ? LF(near2) : 1.9f * all2 / vcbrtf(nf * nf);
        // the power of two that brings the ring's radius to 1 .. 2
        scale = pow2_inv_sqrt(rhi2);
        const LB m0l = hl == 0;
        const LI ko = select(up, LI(int(sizeof(PairCtl)) / 4), LI(0));
        lds_st(&L.ctl[0].c, ko, c, m0l);
        lds_st(&L.ctl[0].inst, ko, inst, m0l);
        lds_st(&L.ctl[0].rlo2, ko, LF(-1.0f), m0l);
        lds_st(&L.ctl[0].rhi2, ko, rhi2, m0l);
        lds_st(&L.ctl[0].all2, ko, all2, m0l);
        lds_st(&L.ctl[0].scale, ko, scale, m0l);
        lds_st(&L.ctl[0].inv, ko, 1.0f / scale, m0l);
        lds_st(&L.ctl[0].nfilt, ko, LI(0), m0l);
        lds_st(&L.ctl[0].ct_on, ko, LI(0), m0l);
    }

    // the box: planes 0..5 and corners in the first 8 lanes, as init_box
    PairState st;
    LI np = LI(6);
    {
        const Lane<pt4> pc = gld(P.pts, c, LB(true));
        const LI axis = hl >> 1;
        const LB neg = (hl & 1) != 0, m6 = hl < 6;
        const LD pcoord = select(axis == 0, pt_x(pc), select(axis == 1, pt_y(pc), pt_z(pc)));
        const LD face = gld(P.box, inst * 6 + select(neg, axis, axis + 3), m6);
        const LF hf = cvt<float>(select(neg, pcoord - face, face - pcoord) * cvt<double>(scale));
        const LF sg = select(neg, LF(-1.0f), LF(1.0f));
        const LI hoff = select(up, LI(int(sizeof(PairHalf))), LI(0));
        lds_st_row(&L.h[0].pe[0][0], (hoff >> 4) + hl, select(axis == 0, sg, LF(0.0f)),
                   select(axis == 1, sg, LF(0.0f)), select(axis == 2, sg, LF(0.0f)), hf, m6);
        lds_st(L.h[0].pg, (hoff >> 2) + hl, LI(-1), m6);
        wave_sync();
        const LI sx = hl & 1, sy = (hl >> 1) & 1, sz = (hl >> 2) & 1;
        const LI X = 1 - sx, Y = 3 - sy, Z = 5 - sz;
        const LB pos = ((sx + sy + sz) & 1) != 0;
        const LI a = select(pos, X, Y), b = select(pos, Y, X), l8 = hl & 7;
        const RowLanes ra = lds_row(&L.h[0].pe[0][0], (hoff >> 4) + a);
        const RowLanes rb = lds_row(&L.h[0].pe[0][0], (hoff >> 4) + b);
        const RowLanes rc = lds_row(&L.h[0].pe[0][0], (hoff >> 4) + Z);
        const PairCorner C = pair_corner(ra, rb, rc);
        st.nx[0] = C.nx;
        st.ny[0] = C.ny;
        st.nz[0] = C.nz;
        st.d[0] = C.d;
        st.gn[0] = C.gn;
        st.gd[0] = C.gd;
        st.num[0] = C.num;
        st.den2[0] = C.den2;
        st.pl[0] = cvt<uint32_t>(a) | (cvt<uint32_t>(b) << LU(8)) | (cvt<uint32_t>(Z) << LU(16));
        const LI a1 = select(pos, l8 ^ 1, l8 ^ 2), a2 = select(pos, l8 ^ 2, l8 ^ 1);
        st.adj[0] = cvt<uint32_t>(l8 ^ 4) | (cvt<uint32_t>(a1) << LU(8)) | (cvt<uint32_t>(a2) << LU(16));
        st.nx[1] = st.ny[1] = st.nz[1] = LF(0.0f);
        st.d[1] = LF(1.0f);
        st.gn[1] = st.gd[1] = st.num[1] = LF(0.0f);
        st.den2[1] = LF(1.0f);
        st.pl[1] = st.adj[1] = LU(0u);
        st.valid[0] = 0x000000FF000000FFull & live;
        st.valid[1] = 0;
        // a box corner out of the FP32 range
        live &= ~halves(ballot(C.bad) & st.valid[0]);
    }

    // ------------------------------------------------ security-radius loop
    const uint64_t have_m = halves(st.valid[0]);
    uint64_t done = 0, empty = 0;  // halves finished; the others of have_m fail
    uint64_t rings = 0;            // of those: out of rings
    LI cnt = LI(0);                // candidates of the ring
    uint64_t first = kLoHalf | kHiHalf, more = kLoHalf | kHiHalf;
    PairWork work{};
    const LI soff4 = select(up, LI(int(sizeof(PairStage)) / 16), LI(0));
    const LI soff2 = select(up, LI(int(sizeof(PairStage)) / 8), LI(0));
    const LI koff = select(up, LI(int(sizeof(PairHalf)) / 8), LI(0));
    if (N.inst >= 0 && ballot(inst != N.inst) == 0) {
        // both first rings in one scan of the wave's buckets
        const int ca = uni(L.ctl[0].c), cb = uni(L.ctl[1].c);
        int n2[2];
        near_scan(P, L, N, ca, cb, P.pf[ca], P.pf[cb], -1.0f, (live & kLoHalf) ? near2 : -1.0f, -1.0f,
                  (live & kHiHalf) ? near2 : -1.0f, n2[0], n2[1]);
#pragma unroll 1
        for (int h = 0; h < 2; ++h) {
            if (!(live & half_mask(h))) continue;
            float r2 = near2;
            if (n2[h] > kCandCap) {
                // too many: once more within the radius that holds about 64
                const float f = cbrtf(64.0f / float(n2[h]));
                r2 *= f * f;
                int none;
                const int ch = h ? cb : ca;
                near_scan(P, L, N, ch, ch, P.pf[ch], P.pf[ch], -1.0f, h ? -1.0f : r2, -1.0f,
                          h ? r2 : -1.0f, h ? none : n2[h], h ? n2[h] : none);
                // (copies without an end: the cell's own walk)
                if (n2[h] > kCandCap) continue;
            }
            const int k = ring_sort(h ? L.cand_b : L.cand, n2[h], r2, L.h[h].key);
            L.ctl[h].rhi2 = r2;
            if (k < 0) continue;
            first &= ~half_mask(h);
            more &= ~half_mask(h);
            cnt = select(mask_bit(half_mask(h)), LI(k), cnt);
        }
        wave_sync();
    }
    while (live) {
        // the next ring of every live half
#pragma unroll 1
        for (int h = 0; h < 2; ++h) {
            const uint64_t hm = half_mask(h);
            if (!(live & more & hm)) continue;
            const int n = pair_ring<W>(P, L, st, N, h, (first & hm) != 0);
            first &= ~hm;
            if (n < 0) {
                live &= ~hm;
                if (n == -1) done |= hm;
                if (n == -3) rings |= hm;
            }
            cnt = select(mask_bit(hm), LI(n), cnt);
        }
        more = kLoHalf | kHiHalf;
        LI n = LI(0);  // staged now
#pragma unroll 1
        for (int h = 0; h < 2; ++h) {
            const uint64_t hm = half_mask(h);
            if (!(live & hm)) continue;
            const int ch = uni(L.ctl[h].c);
            const pt4 pc = P.pts[ch];
            const int k = pair_stage<W>(P, L, h, ch, uni(L.ctl[h].scale), pc,
                                        W ? pc.w - P.wmax[uni(L.ctl[h].inst)] : 0.0,
                                        readlane(cnt, 32 * h));
            if (k < 0) live &= ~hm;
            n = select(mask_bit(hm), LI(k), n);
        }
        // the staged candidates, nearest first
        uint64_t run = live, pend = 0, cf[2] = {0, 0};
        LI k = LI(0);
        while (true) {
            const LI ks = select(k < n, k, LI(0));
            const RowLanes r = lds_row(&L.stage[0].row[0][0], soff4 + ks);
            LF rho, e1;
            lds_pair(&L.stage[0].aux[0][0], soff2 + ks, rho, e1);
            const LF ah = vabs(r.w);
            const LF t0 = vfma(r.x, st.nx[0], vfma(r.y, st.ny[0], vfma(r.z, st.nz[0], -(r.w * st.d[0]))));
            const LF b0 = vfma(e1, st.gn[0], ah * st.gd[0]);
            uint64_t cc0 = ballot(t0 >= 0.0f) & st.valid[0];
            uint64_t uu = ~ballot(vabs(t0) > b0) & st.valid[0];
            uint64_t ss = ballot(st.num[0] >= rho * st.den2[0]) & st.valid[0];
            uint64_t cc1 = 0;
            if (st.valid[1]) {
                const LF t1 = vfma(r.x, st.nx[1], vfma(r.y, st.ny[1], vfma(r.z, st.nz[1], -(r.w * st.d[1]))));
                const LF b1 = vfma(e1, st.gn[1], ah * st.gd[1]);
                cc1 = ballot(t1 >= 0.0f) & st.valid[1];
                uu |= ~ballot(vabs(t1) > b1) & st.valid[1];
                ss |= ballot(st.num[1] >= rho * st.den2[1]) & st.valid[1];
            }
            // ring at its end, security radius reached, sign not certified,
            // plane cuts: in this order
            uint64_t rem = run & ballot(k < n);
            const uint64_t reach = rem & ~halves(ss);
            rem &= ~reach;
            if (COUNT) {
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    if (rem & half_mask(h)) {
                        work.ntest[h]++;
                        work.nlive[h] += popc_half(st.valid[0], h) + popc_half(st.valid[1], h);
                    }
            }
            const uint64_t unc = rem & halves(uu);
            rem &= ~unc;
            const uint64_t cut = rem & halves(cc0 | cc1);
            done |= reach;
            live &= ~(reach | unc);
            cf[0] = (cf[0] & ~cut) | (cc0 & cut);
            cf[1] = (cf[1] & ~cut) | (cc1 & cut);
            pend |= cut;
            run = rem & ~cut;
            k = k + select(mask_bit(run), LI(1), LI(0));
            if (run) continue;
            if (pend == 0) break;
            const LI j = cvt<int>(cvt<uint32_t>(lds_ld(&L.h[0].key[0], koff + ks)));
            if (COUNT) {
                if (pend & kLoHalf) work.nclip[0]++;
                if (pend & kHiHalf) work.nclip[1]++;
            }
            uint64_t gone = 0;
            const uint64_t bad = pair_cut<COUNT>(st, L, np, r, j, pend, cf, up, hl, work, gone);
            empty |= gone;
            live &= ~(gone | bad);
            st.valid[0] = uni(st.valid[0]);
            st.valid[1] = uni(st.valid[1]);
            live = uni(live);
            run = uni(pend & live);
            k = k + select(mask_bit(run), LI(1), LI(0));
            pend = 0;
            if (run == 0) break;
        }
    }

    if (COUNT && lane0()) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            atomic_add_u64(P.counters + 0, work.nclip[h]);
            atomic_add_u64(P.counters + 1, work.ntest[h]);
            atomic_add_u64(P.counters + 2, work.nlive[h]);
            atomic_add_u64(P.counters + 3, work.nnew[h]);
        }
    }
    const Lane<long long> cl = cvt<long long>(c), ocl = cvt<long long>(oc);
    const LB lead = hl == 0;
    {
        const LB failed = mask_bit(have_m & ~(done | empty)) & lead;
        gst(P.flags, cl,
            select(mask_bit(rings), LU(uint32_t(CELL_NEED_K | CELL_WHY_RINGS)), LU(uint32_t(CELL_UNCERTAIN))),
            failed);
        const LB em = mask_bit(empty) & lead;
        gst(P.r2, cl, LD(0.0), failed | em);
        if (empty) {
            if (P.abort_flag) flag_set(P.abort_flag, inst, em);
            gst(P.vol, ocl, LD(0.0), em);
            for (int a = 0; a < 3; ++a) gst(P.mg, ocl * 3ll + (long long)a, LD(0.0), em);
            gst(P.nbr_cnt, ocl, LI(0), em);
            if (P.e2) gst(P.e2, ocl, LD(0.0), em);
            gst(P.flags, cl, LU(uint32_t(CELL_EMPTY | CELL_DONE)), em);
        }
    }
    const uint64_t fin = done;
    if (fin == 0) return;

    // ------------------------------------------------------ integration
    // FP64 rows of the planes (as the FP64 pass forms them); the planes'
    // neighbours move to registers, the LDS changes its use
    const LB finl = mask_bit(fin);
    np = select(finl, np, LI(0));
    LI pgv[2];
#pragma unroll
    for (int s = 0; s < 2; ++s)
        pgv[s] = lds_ld(L.h[0].pg, select(up, LI(int(sizeof(PairHalf)) / 4), LI(0)) + hl + 32 * s);
    wave_sync();
    const Lane<pt4> pc = gld(P.pts, c, LB(true));
    const LI o8 = select(up, LI(int(sizeof(PairInt)) / 8), LI(0));
    const LI o4 = select(up, LI(int(sizeof(PairInt)) / 4), LI(0));
    const bool many = ballot(np > 32) != 0;  // a cell with over 32 planes
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        if (s == 1 && !many) continue;
        const LI f = hl + 32 * s;
        const LB in = f < np;
        const LB seed = in & (f >= 6);
        const Lane<pt4> q = gld(P.pts, select(seed, pgv[s], LI(0)), seed);
        LD ex = pt_x(q) - pt_x(pc), ey = pt_y(q) - pt_y(pc), ez = pt_z(q) - pt_z(pc);
        const LD d2 = ex * ex + ey * ey + ez * ez;
        LD hh = W ? 0.5 * (d2 + (pt_w(pc) - pt_w(q))) : 0.5 * d2;
        if (s == 0) {
            const LI axis = f >> 1;
            const LB neg = (f & 1) != 0, bx = f < 6;
            const LD sg = select(neg, LD(-1.0), LD(1.0));
            const LD pcoord = select(axis == 0, pt_x(pc), select(axis == 1, pt_y(pc), pt_z(pc)));
            const LD face = gld(P.box, inst * 6 + select(neg, axis, axis + 3), bx);
            hh = select(bx, select(neg, pcoord - face, face - pcoord), hh);
            ex = select(bx, select(axis == 0, sg, LD(0.0)), ex);
            ey = select(bx, select(axis == 1, sg, LD(0.0)), ey);
            ez = select(bx, select(axis == 2, sg, LD(0.0)), ez);
        }
        double* row = &L.in[0].row[0][0];
        const LI fo = o8 + f * 4;
        lds_st(row, fo + 0, ex, in);
        lds_st(row, fo + 1, ey, in);
        lds_st(row, fo + 2, ez, in);
        lds_st(row, fo + 3, hh, in);
        lds_st(L.in[0].v2t, o4 + f, LI(0x7FFFFFFF), in);
    }
    wave_sync();
    const uint64_t vf[2] = {st.valid[0] & fin, st.valid[1] & fin};
    LD r2f = LD(0.0);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        if (vf[s] == 0) continue;
        const LB vs = mask_bit(vf[s]);
        const LI cid = hl + 32 * s;
        LI p3[3];
        LD e[3][4];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            p3[k] = select(vs, cvt<int>(byte_of(st.pl[s], k)) & (kPairPlanes - 1), LI(0));
#pragma unroll
            for (int a = 0; a < 4; ++a) e[k][a] = lds_ld(&L.in[0].row[0][0], o8 + p3[k] * 4 + a);
        }
        // N and D as make_corner forms them (FP32 certified that the corner
        // is not degenerate: no magnitudes here, and one division)
        const LD bcx = vfma(e[1][1], e[2][2], -(e[1][2] * e[2][1])),
                 bcy = vfma(e[1][2], e[2][0], -(e[1][0] * e[2][2])),
                 bcz = vfma(e[1][0], e[2][1], -(e[1][1] * e[2][0]));
        const LD cax = vfma(e[2][1], e[0][2], -(e[2][2] * e[0][1])),
                 cay = vfma(e[2][2], e[0][0], -(e[2][0] * e[0][2])),
                 caz = vfma(e[2][0], e[0][1], -(e[2][1] * e[0][0]));
        const LD abx = vfma(e[0][1], e[1][2], -(e[0][2] * e[1][1])),
                 aby = vfma(e[0][2], e[1][0], -(e[0][0] * e[1][2])),
                 abz = vfma(e[0][0], e[1][1], -(e[0][1] * e[1][0]));
        const LD nx = vfma(e[0][3], bcx, vfma(e[1][3], cax, e[2][3] * abx));
        const LD ny = vfma(e[0][3], bcy, vfma(e[1][3], cay, e[2][3] * aby));
        const LD nz = vfma(e[0][3], bcz, vfma(e[1][3], caz, e[2][3] * abz));
        const LD inv = 1.0 / vfma(e[0][0], bcx, vfma(e[0][1], bcy, e[0][2] * bcz));
        const LD qx = nx * inv, qy = ny * inv, qz = nz * inv;
        r2f = vmax(r2f, select(vs, vfma(qx, qx, vfma(qy, qy, qz * qz)), LD(0.0)));
        lds_st(&L.in[0].q[0][0], o8 + cid * 3 + 0, qx, vs);
        lds_st(&L.in[0].q[0][0], o8 + cid * 3 + 1, qy, vs);
        lds_st(&L.in[0].q[0][0], o8 + cid * 3 + 2, qz, vs);
        lds_st(L.in[0].cpl, o4 + cid, st.pl[s], vs);
        lds_st(L.in[0].cadj, o4 + cid, st.adj[s], vs);
#pragma unroll
        for (int k = 0; k < 3; ++k) lds_min(L.in[0].v2t, o4 + p3[k], cid, vs);
    }
    gst(P.r2, cl, half_max(r2f), finl & lead);
    wave_sync();
    // the fan's apex: the first live corner
    const uint64_t a0 = vf[0] & kLoHalf, a1 = vf[1] & kLoHalf, b0 = vf[0] >> 32, b1 = vf[1] >> 32;
    const int apex_a = a0 ? ffs64(a0) : a1 ? ffs64(a1) + 32 : 0;
    const int apex_b = b0 ? ffs64(b0) : b1 ? ffs64(b1) + 32 : 0;
    const LI apex = select(up, LI(apex_b), LI(apex_a));
    const double* Q = &L.in[0].q[0][0];
    const LD ox = lds_ld(Q, o8 + apex * 3 + 0), oy = lds_ld(Q, o8 + apex * 3 + 1),
             oz = lds_ld(Q, o8 + apex * 3 + 2);
    LD vacc = LD(0.0), mxa = LD(0.0), mya = LD(0.0), mza = LD(0.0), e2a = LD(0.0);
    LI ntet = LI(0);
    int nface[2] = {0, 0}, out[2] = {0, 0};
    const Lane<long long> obase = ocl * (long long)P.face_stride;
#pragma unroll 1
    for (int s = 0; s < 2; ++s) {
        if (s == 1 && !many) continue;
        const LI f = hl + 32 * s;
        const LB inr = f < np;
        const LI fs = select(inr, f, LI(0));
        LI t0 = lds_ld(L.in[0].v2t, o4 + fs);
        const LB act = finl & inr & (t0 != LI(0x7FFFFFFF));
        // (lanes without a face walk from the apex, adding zeros: every point
        // they read is one of the cell)
        t0 = select(act, t0, apex) & 63;
        const LU fu = cvt<uint32_t>(fs);
        auto nxt = [&](const LI& t) -> LI {
            const LU plt = lds_ld(L.in[0].cpl, o4 + t);
            const LU adt = lds_ld(L.in[0].cadj, o4 + t);
            const LI sh = select(byte_of(plt, 0) == fu, LI(16), select(byte_of(plt, 1) == fu, LI(0), LI(8)));
            return cvt<int>(adt >> cvt<uint32_t>(sh)) & 63;
        };
        const LD q0x = lds_ld(Q, o8 + t0 * 3 + 0), q0y = lds_ld(Q, o8 + t0 * 3 + 1),
                 q0z = lds_ld(Q, o8 + t0 * 3 + 2);
        const LI t1 = nxt(t0);
        LI t = nxt(t1);
        LD q1x = lds_ld(Q, o8 + t1 * 3 + 0), q1y = lds_ld(Q, o8 + t1 * 3 + 1),
           q1z = lds_ld(Q, o8 + t1 * 3 + 2);
        LD area = LD(0.0), fv = LD(0.0), fmx = LD(0.0), fmy = LD(0.0), fmz = LD(0.0), fe = LD(0.0);
        const LD oq0 = (ox * ox + oy * oy + oz * oz) + (q0x * q0x + q0y * q0y + q0z * q0z);
        const LD ux = q0x - ox, uy = q0y - oy, uz = q0z - oz;
        const LD rx = ox + q0x, ry = oy + q0y, rz = oz + q0z;
        LD vx = q1x - ox, vy = q1y - oy, vz = q1z - oz;
        LD ax = q1x - q0x, ay = q1y - q0y, az = q1z - q0z;
        LB go = act & (t != t0);
        for (int guard = 0; guard < 64 && any(go); ++guard) {
            const LD qx = lds_ld(Q, o8 + t * 3 + 0), qy = lds_ld(Q, o8 + t * 3 + 1),
                     qz = lds_ld(Q, o8 + t * 3 + 2);
            // tetrahedron and triangle terms exactly as in process_cell, the
            // differences of the previous point carried along; a lane whose
            // face is done adds zeros
            const LD wx = qx - ox, wy = qy - oy, wz = qz - oz;
            const LD cx = uy * vz - uz * vy, cy = uz * vx - ux * vz, cz = ux * vy - uy * vx;
            const LD tv = select(go, vabs(cx * wx + cy * wy + cz * wz) * (1.0 / 6.0), LD(0.0));
            if (COUNT) ntet = ntet + select(go, LI(1), LI(0));
            fv = fv + tv;
            const LD sx = rx + q1x + qx, sy = ry + q1y + qy, sz = rz + q1z + qz;
            fmx = fmx + tv * sx / 4.0;
            fmy = fmy + tv * sy / 4.0;
            fmz = fmz + tv * sz / 4.0;
            if (P.e2) {
                const LD nn = oq0 + (q1x * q1x + q1y * q1y + q1z * q1z) + (qx * qx + qy * qy + qz * qz) +
                              (sx * sx + sy * sy + sz * sz);
                fe = fe + tv * nn * (1.0 / 20.0);
            }
            if (P.faces) {
                const LD bx = qx - q0x, by = qy - q0y, bz = qz - q0z;
                const LD wx2 = ay * bz - az * by, wy2 = az * bx - ax * bz, wz2 = ax * by - ay * bx;
                const LD ta = 0.5 * vsqrt(wx2 * wx2 + wy2 * wy2 + wz2 * wz2);
                area = area + select(go, ta, LD(0.0));
                ax = bx;
                ay = by;
                az = bz;
            }
            q1x = qx;
            q1y = qy;
            q1z = qz;
            vx = wx;
            vy = wy;
            vz = wz;
            const LI tn = nxt(t);
            t = select(go, tn, t);
            go = go & (t != t0);
        }
        vacc = vacc + fv;
        e2a = e2a + fe;
        mxa = mxa + fmx;
        mya = mya + fmy;
        mza = mza + fmz;
        if (COUNT) {
            const uint64_t am = ballot(act);
            nface[0] += popc_half(am, 0);
            nface[1] += popc_half(am, 1);
        }
        const LI pg = s == 0 ? pgv[0] : pgv[1];
        const LB outm = act & (pg >= 0);
        const uint64_t om = ballot(outm);
        if (P.faces) {
            const LI rank = half_rank(om, out[0], out[1], up);
            const LI oj0 = gld(P.orig, select(outm, pg, LI(0)), outm);
            const LI oj = P.src ? gld(P.src, select(outm, oj0, LI(0)), outm) : oj0;
            const Lane<long long> at = obase + cvt<long long>(rank);
            gst(P.nbr_tmp, at, oj, outm);
            gst(P.area_tmp, at, area, outm);
        }
        out[0] += popc_half(om, 0);
        out[1] += popc_half(om, 1);
    }
    const LD V = half_sum(vacc);
    const LD Mx = half_sum(mxa), My = half_sum(mya), Mz = half_sum(mza);
    if (COUNT) {
        const LD nt = half_sum(cvt<double>(ntet));
        const unsigned long long ta = (unsigned long long)readlane(nt, 0);
        const unsigned long long tb = (unsigned long long)readlane(nt, 32);
        if (lane0()) {
            atomic_add_u64(P.counters + 4, ta + tb);
            atomic_add_u64(P.counters + 5, (unsigned long long)(nface[0] + nface[1]));
        }
    }
    const LB w0 = finl & lead;
    gst(P.vol, ocl, V, w0);
    gst(P.mg, ocl * 3ll + 0ll, Mx + V * pt_x(pc), w0);
    gst(P.mg, ocl * 3ll + 1ll, My + V * pt_y(pc), w0);
    gst(P.mg, ocl * 3ll + 2ll, Mz + V * pt_z(pc), w0);
    gst(P.nbr_cnt, ocl, select(up, LI(out[1]), LI(out[0])), w0);
    gst(P.flags, cl, LU(uint32_t(CELL_DONE)), w0);
    if (P.e2) gst(P.e2, ocl, half_sum(e2a), w0);
}

// Items first .. first + count - 1 (at most 8), two at a time, by one
// wavefront.
template <bool W, bool COUNT>
VGC_HD void process_pairs(const ClipParams& P, int first, int count, PairLds& L) {
    wave_sync();  // the previous cells of this wave are done with the LDS
    NearList N;
    const LI lane = lane_id();
    const LB has = lane < count;
    const LI item = first + select(has, lane, LI(0));
    const LI c = P.items ? gld(P.items, item, LB(true)) : item;
    const int c0 = readlane(c, 0);
    const int inst = P.inst_of ? P.inst_of[c0] : 0;
    N.inst = inst;
    const float d4 = uni(near_spacing(P, c0, inst, count > 2 ? kBucket / 4 : 1));
    const float ring2 = (kNearRing * d4) * (kNearRing * d4);
    N.r2 = (kNearList * d4) * (kNearList * d4);
    bool one = d4 > 0.0f;
    if (P.inst_of) one = one && ballot(gld(P.inst_of, c, LB(true)) != inst) == 0;
    N.n = one ? near_buckets(P, L, inst, lane_seed(P.pf, c, has), has, N.r2) : -1;
    if (N.n < 0) N.inst = -1;
    for (int k = 0; k < count; k += 2) process_pair<W, COUNT>(P, first + k, first + count, L, N, ring2);
}

// Cells per wavefront of k_pair: 8, which share one walk of the tree, once
// that leaves enough wavefronts for the 4096 resident ones to even out,
// else 4 or 2; 1 where the chip stays half empty anyway and the time is that
// of one wavefront.  Whole calls with 1 / 2 / 4 / 8 cells, in ms, uniform
// seeds: 4096 0.41 / 0.41 / 0.48 / 0.60, 30k 0.85 / 0.74 / 0.76 / 0.85, 150k
// 2.86 / 2.41 / 1.92 / 2.04, 400k 7.25 / 5.44 / 5.06 / 4.81, 1M 17.0 / 12.1 /
// 11.3 / 11.0; 16-Gaussian ones: 4096 1.10 / 1.29 / 1.66 / 1.91, 60k 3.33 /
// 2.99 / 3.37 / 3.76, 200k 10.2 / 9.3 / 9.0 / 9.3, 600k 14.0 / 11.3 / 10.2 /
// 10.2 (up to 10k clustered seeds, 1 is 15 % faster still).
static inline int pair_group(int n) { return n >= 400000 ? 8 : n >= 150000 ? 4 : n > 4096 ? 2 : 1; }

}  // namespace vgc
