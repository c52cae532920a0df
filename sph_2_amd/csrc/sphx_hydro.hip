// Bucketed SPH pair passes for the mixed-precision path: smoothing-length
// iteration, density + EOS, velocity divergence/curl, hydro acceleration +
// du/dt.  The particles come in 64-particle Morton buckets; a group (one
// wavefront) takes a bucket or a part of one, culls super-bucket and bucket
// AABBs in FP64 and walks the candidates of its run: the smoothing lengths
// count them, the list walk records every particle's neighbours.  Which
// particles are neighbours is decided by the oracle's FP64 distance (screened
// in FP32).  Density, div/curl and hydro then sum over the lists; kernel
// values and pair sums run in FP32 with Kahan-compensated accumulation.
//
// Reference kernels replaced (11_Dec_2022/GPU_sph/Important_Test_Simulations/
// Evrard_collapse/myCppSPHLibs_v2.h): smoothing_h 7-64, getDensity 69-114,
// div_curlVel 247-322, acc_sph 327-417, get_dU 634-719,
// getPressure_Adiabatic/getCsound_Adiabatic 766-789.
#include "sphx_internal.h"

#include <algorithm>

namespace {

// Walk the candidate buckets, in increasing order, of a group of particles of
// run `r` with bounding box ib (xl, xh, yl, yh, zl, zh).  `reach_s(S)` and
// `reach_b(J)` give the reach against super S and bucket J; `body(J)` is
// called once per surviving bucket with the whole wavefront converged.
template <class ReachS, class ReachB, class Body>
__device__ __forceinline__ void for_candidates(const Tables &t, int r, const double *ib, int lane,
                                               ReachS reach_s, ReachB reach_b, Body body) {
    double axl = ib[0], axh = ib[1], ayl = ib[2], ayh = ib[3], azl = ib[4], azh = ib[5];
    int s0 = t.r_sbeg[r], s1 = t.r_send[r];
    for (int sb = s0; sb < s1; sb += 64) {
        int S = sb + lane;
        bool sp = false;
        if (S < s1) {
            double d2 = sphx_box_d2(axl, axh, ayl, ayh, azl, azh, t.sxl[S], t.sxh[S], t.syl[S],
                                    t.syh[S], t.szl[S], t.szh[S]);
            sp = sphx_within(d2, reach_s(S));
        }
        uint64_t smask = __ballot(sp);
        while (smask) {
            int S2 = sb + __builtin_ctzll(smask);
            smask &= smask - 1;
            int j0 = t.s_bbeg[S2], j1 = t.s_bend[S2];
            int J = j0 + lane;
            bool bp = false;
            if (J < j1) {
                double d2 = sphx_box_d2(axl, axh, ayl, ayh, azl, azh, t.bxl[J], t.bxh[J],
                                        t.byl[J], t.byh[J], t.bzl[J], t.bzh[J]);
                bp = sphx_within(d2, reach_b(J));
            }
            uint64_t bmask = __ballot(bp);
            while (bmask) {
                int J2 = j0 + __builtin_ctzll(bmask);
                bmask &= bmask - 1;
                body(J2);
            }
        }
    }
}

// for_candidates with the candidate loads run ahead: `load(J, beg, cnt)`
// issues the reads `body(J, v)` needs of bucket J (lane q: particle beg + q,
// q < cnt) and is called for the next surviving bucket before `body` runs on
// the current one, so a walk no longer waits on each bucket's loads.  The
// buckets' first particle and count come with the bucket culling, one bucket
// per lane, and reach the loads by readlane.  Buckets are met in the same
// order as by for_candidates.
template <class ReachS, class ReachB, class Load, class Body>
__device__ __forceinline__ void for_candidates_pf(const Tables &t, int r, const double *ib, int lane,
                                                  ReachS reach_s, ReachB reach_b, Load load,
                                                  Body body) {
    double axl = ib[0], axh = ib[1], ayl = ib[2], ayh = ib[3], azl = ib[4], azh = ib[5];
    int s0 = t.r_sbeg[r], s1 = t.r_send[r];
    decltype(load(0, 0, 0)) cur{};
    int Jc = -1;
    for (int sb = s0; sb < s1; sb += 64) {
        int S = sb + lane;
        bool sp = false;
        if (S < s1) {
            double d2 = sphx_box_d2(axl, axh, ayl, ayh, azl, azh, t.sxl[S], t.sxh[S], t.syl[S],
                                    t.syh[S], t.szl[S], t.szh[S]);
            sp = sphx_within(d2, reach_s(S));
        }
        uint64_t smask = __ballot(sp);
        while (smask) {
            int S2 = sb + __builtin_ctzll(smask);
            smask &= smask - 1;
            int j0 = t.s_bbeg[S2], j1 = t.s_bend[S2];
            int J = j0 + lane;
            bool bp = false;
            int vbeg = 0, vcnt = 0;
            if (J < j1) {
                double d2 = sphx_box_d2(axl, axh, ayl, ayh, azl, azh, t.bxl[J], t.bxh[J],
                                        t.byl[J], t.byh[J], t.bzl[J], t.bzh[J]);
                bp = sphx_within(d2, reach_b(J));
                vbeg = t.b_beg[J];
                vcnt = t.b_cnt[J];
            }
            uint64_t bmask = __ballot(bp);
            while (bmask) {
                int q = __builtin_ctzll(bmask);
                bmask &= bmask - 1;
                auto nxt = load(j0 + q, __builtin_amdgcn_readlane(vbeg, q),
                                __builtin_amdgcn_readlane(vcnt, q));
                if (Jc >= 0) body(Jc, cur);
                cur = nxt;
                Jc = j0 + q;
            }
        }
    }
    if (Jc >= 0) body(Jc, cur);
}

// Segments of a bucket.  64 consecutive Morton-sorted particles usually fill
// one compact cell, but where the curve jumps between distant cells their
// bounding box spans much of the run and would make every bucket of that
// region a candidate.  A bucket is therefore cut wherever two consecutive
// particles lie in different cells of Morton level t.r_lcut[run]; each
// segment walks the candidates of its own box and only its lanes accumulate.
// Candidates are still met in increasing order, so every sum is unchanged.
// Returns the ballot of lanes that start a segment (lane 0 never set).
__device__ __forceinline__ uint64_t bucket_cuts(const Tables &t, int r, int i, bool ok, int lane) {
    bool cut = false;
    if (t.keys && ok && lane > 0) {
        uint64_t x = t.keys[i] ^ t.keys[i - 1];
        if (x) {
            int hb = 63 - __builtin_clzll(x);
            int lev = t.mbits - 1 - hb / 3;  // Morton level of the cell boundary crossed
            cut = lev <= t.r_lcut[r];
        }
    }
    return __ballot(cut);
}

// End (exclusive) of the segment that starts at lane s0.
__device__ __forceinline__ int seg_end(uint64_t cuts, int s0, int cnt) {
    uint64_t rest = s0 >= 63 ? 0ull : cuts & (~0ull << (s0 + 1));
    int s1 = rest ? __builtin_ctzll(rest) : cnt;
    return s1 < cnt ? s1 : cnt;
}

// Bounding box and max h of the lanes with `mine` set.
__device__ __forceinline__ void seg_box(bool mine, double x, double y, double z, double h,
                                        double *box, double *hmax) {
    box[0] = wave_min_d(mine ? x : INFINITY);
    box[1] = wave_max_d(mine ? x : -INFINITY);
    box[2] = wave_min_d(mine ? y : INFINITY);
    box[3] = wave_max_d(mine ? y : -INFINITY);
    box[4] = wave_min_d(mine ? z : INFINITY);
    box[5] = wave_max_d(mine ? z : -INFINITY);
    *hmax = wave_max_d(mine ? h : 0.0);
}

// The particles a walk group takes: a whole bucket (P = 1) or, in runs too
// small to fill the device with one wave per bucket, a half, a quarter or an
// eighth of one, so that there are P times the groups and each meets fewer candidates.
// A group holds T = 64 / P targets, lane L the target L mod T; its P lanes per
// target are slices that take a P-th of every batch of candidates each.  A
// part walks the candidates of its own box, exactly as a segment does, so every
// particle still meets its candidates in increasing order.
struct WalkSlot {
    int b;      // bucket
    int cnt;    // targets of the group
    int first;  // first particle
    int bl0;    // bucket lane of target 0
    int part;
};
template <int P>
__device__ __forceinline__ WalkSlot walk_slot(const Tables &t) {
    const int g = xcd_block(blockIdx.x, gridDim.x);
    WalkSlot w;
    w.b = t.boff + g / P;
    w.part = g % P;
    w.bl0 = (64 / P) * w.part;
    const int c = t.b_cnt[w.b] - w.bl0;
    w.cnt = c < 0 ? 0 : (c > 64 / P ? 64 / P : c);
    w.first = t.b_beg[w.b] + w.bl0;
    return w;
}

// Sum of v over the P slices of a target.
template <int P>
__device__ __forceinline__ int slice_sum(int v) {
    for (int o = 64 / P; o < 64; o <<= 1) v += __shfl_xor(v, o, 64);
    return v;
}
// Exclusive prefix of v over the slices of a target, and the total.
template <int P>
__device__ __forceinline__ int slice_scan(int v, int lane, int *total) {
    if (P == 1) {
        *total = v;
        return 0;
    }
    int pre = 0, tot = 0;
    for (int k = 0; k < P; ++k) {
        const int u = __shfl(v, (lane & (64 / P - 1)) + k * (64 / P), 64);
        if (k < lane / (64 / P)) pre += u;
        tot += u;
    }
    *total = tot;
    return pre;
}

// ---------------------------------------------------------------------------
// Tile walk.  The candidates of a group's box are gathered bucket by bucket
// (each lane one particle), the ones in reach compacted in order into LDS as
// FP32 coordinates relative to the box's centre, and tested 64 at a time: a
// batch costs each lane 8 FP32 instructions a candidate (the sign of
// r^2 - s^2 shifted into a mask) where the FP64 test of one candidate at a
// time took 11 FP64 ones (four cycles each against two), three 8-byte LDS
// broadcasts and, a bucket keeping about eight of its 64 particles, the loop's
// overhead for every handful.  The decision stays the FP64 one: the FP32 value
// is trusted only outside a band that bounds its error (walk_band), and a batch
// with a value inside it (about one in a thousand) is tested again in FP64.
// Bound: each wave's chain of gather, compaction, LDS round trip and batch.  At
// 1,048,576 particles the list walk issues 0.20 VALU and 0.016 LDS instructions a
// SIMD-cycle with three waves resident and 17 % of their cycles waiting.
constexpr int TW_LIST = 192;       // surviving buckets collected at a time
constexpr float TW_FAR = 1.0e18f;  // relative coordinate of what is never in reach

template <bool HH>
struct WalkLds {
    float x[128], y[128], z[128];
    float h[HH ? 128 : 1];
    int32_t j[128];
    int2 bl[TW_LIST];
};

// Frame of a group: centre and half extents of its box, scaled by a power of
// two that brings the search radius near one, so that FP32 neither over- nor
// underflows at any scale of the run.  A radius whose square comes near the
// ends of the FP64 range (below 2^-480, above 2^500), where r^2 itself is
// rounded coarsely, and a box or radius that is not finite leave sc = 0: every
// candidate is then tested in FP64, a bucket at a time.
struct WalkFrame {
    double ox, oy, oz, sc;
    float ex, ey, ez;
};
__device__ __forceinline__ WalkFrame walk_frame(const double *gb, double reach) {
    WalkFrame f;
    f.ox = 0.5 * (gb[0] + gb[1]);
    f.oy = 0.5 * (gb[2] + gb[3]);
    f.oz = 0.5 * (gb[4] + gb[5]);
    const int be = (int)(((unsigned long long)__double_as_longlong(reach) >> 52) & 0x7ffull);
    const bool fine = reach > 0.0 && be >= 543 && be <= 1523;
    f.sc = fine ? __longlong_as_double((long long)(2046 - be) << 52) : 0.0;
    // from the centre as it was rounded: far from the origin it is off the box's
    // middle by as much as the particles' own spacing there
    f.ex = __double2float_ru(fmax(gb[1] - f.ox, f.ox - gb[0]) * f.sc * (1.0 + 0x1p-40));
    f.ey = __double2float_ru(fmax(gb[3] - f.oy, f.oy - gb[2]) * f.sc * (1.0 + 0x1p-40));
    f.ez = __double2float_ru(fmax(gb[5] - f.oz, f.oz - gb[4]) * f.sc * (1.0 + 0x1p-40));
    if (!(f.ex < INFINITY && f.ey < INFINITY && f.ez < INFINITY)) {
        f.sc = f.ox = f.oy = f.oz = 0.0;
        f.ex = f.ey = f.ez = 0.0f;
    }
    return f;
}
// Bound on |r^2 - S^2| below which the FP32 value may have the wrong sign:
// coordinates up to M rounded to 24 bits move r^2 near S^2 by at most 2^-24
// (4 sqrt(3) S M + 2 sqrt(3) S^2), the additions and S^2 itself (or the
// rounded t = h_i + h_j squared) by under 2^-24 12 S^2; twice that.  Where S is
// so small against M that larger r could be misjudged too, every value is.
__device__ __forceinline__ float walk_band(double S, double M) {
    if (!(S * 1.0e4 > M)) return INFINITY;
    return __double2float_ru(0x1p-23 * (8.0 * S * M + 20.0 * S * S));
}

// Calls the sink for the candidates of the group's box gb within `reach` (HH:
// reach + h_j), in increasing order.  Sink: chunk(hc, exact) before the candidates
// of a chunk (hc: their largest h; exact: every batch is to be tested in FP64),
// cand(x, y, z, h) for each candidate of the lane's slice of a batch, batch(L,
// base, n) after it.  Returns the number of candidate buckets.
template <int P, bool HH, class Sink>
__device__ __forceinline__ int tile_walk(const Tables &t, const Soa &s, WalkLds<HH> &L, int r,
                                         int lane, const double *gb, double reach,
                                         const WalkFrame &f, Sink &sink) {
    constexpr int Q = 64 / P;  // candidates of a batch per slice
    const uint64_t lt = (1ull << lane) - 1ull;
    const int q0 = (lane / Q) * Q;  // Q targets, Q candidates: slice = lane / Q
    int ncand = 0, nl = 0;
    double hc = 0.0;  // largest h of the collected buckets (this lane's)
    auto walk = [&]() {
        double hmax = 0.0;
        if (HH) hmax = wave_max_d(hc);
        hc = 0.0;
        // |relative coordinate| of a particle in reach is at most e + reach; its
        // rounding and that of the distance widen the test by 2^-20
        const float rr = __double2float_ru((reach + hmax) * f.sc);
        // a candidate's h so far above the group's own that squares in FP32 come
        // near its range, or the far coordinate, is decided in FP64 as well
        const bool exact = !(f.sc > 0.0 && rr < 1.0e15f);
        sink.chunk(hmax, exact);
        if (exact) {  // (inside the compaction it cost k_lists 2-4 %, here nothing)
            for (int k = 0; k < nl; ++k) {
                const int2 e = L.bl[k];
                L.j[lane] = e.x + lane;
                __builtin_amdgcn_wave_barrier();
                sink.begin();
                sink.batch(L, 0, e.y, q0);
                __builtin_amdgcn_wave_barrier();
            }
            nl = 0;
            return;
        }
        const float mx = f.ex + 0x1p-20f * (f.ex + rr), my = f.ey + 0x1p-20f * (f.ey + rr),
                    mz = f.ez + 0x1p-20f * (f.ez + rr);
        struct Cand {
            double x, y, z, h;
            int beg, n;
        };
        auto load = [&](int k) {
            Cand c{0.0, 0.0, 0.0, 0.0, 0, 0};
            if (k < nl) {
                const int2 e = L.bl[k];
                c.beg = __builtin_amdgcn_readfirstlane(e.x);
                c.n = __builtin_amdgcn_readfirstlane(e.y);
                if (lane < c.n) {
                    c.x = s.x[c.beg + lane];
                    c.y = s.y[c.beg + lane];
                    c.z = s.z[c.beg + lane];
                    if (HH) c.h = s.h[c.beg + lane];
                }
            }
            return c;
        };
        int tail = 0;
        auto batch = [&](int base, int n) {
            __builtin_amdgcn_wave_barrier();
            sink.begin();
#pragma unroll 8
            for (int k = 0; k < Q; ++k) {
                if (P == 1 && k == 32) sink.word();
                const int q = base + q0 + k;
                sink.cand(L.x[q], L.y[q], L.z[q], HH ? L.h[HH ? q : 0] : 0.0f);
            }
            sink.batch(L, base, n, q0);
            __builtin_amdgcn_wave_barrier();
        };
        // two buckets' loads are in flight while a third is compacted
        Cand c0 = load(0), c1 = load(1);
        int lim = nl;
        for (int k = 0; k < lim; ++k) {
            const Cand c2 = load(k + 2);
            const float rx = (float)((c0.x - f.ox) * f.sc), ry = (float)((c0.y - f.oy) * f.sc),
                        rz = (float)((c0.z - f.oz) * f.sc);
            const float dx = fmaxf(fabsf(rx) - mx, 0.0f), dy = fmaxf(fabsf(ry) - my, 0.0f),
                        dz = fmaxf(fabsf(rz) - mz, 0.0f);
            float hj = 0.0f, ra = rr;
            if (HH) {
                hj = (float)(c0.h * f.sc);
                ra = (float)((reach + c0.h) * f.sc);
            }
            ra = ra * (1.0f + 0x1p-20f);
            // a NaN coordinate fails here as it fails every distance test
            const bool finite = fabsf(rx) < INFINITY && fabsf(ry) < INFINITY && fabsf(rz) < INFINITY;
            const bool keep = lane < c0.n && finite && (dx * dx + dy * dy) + dz * dz <= ra * ra;
            const uint64_t m = __ballot(keep);
            if (m) {
                if (keep) {
                    const int at = (tail + __popcll(m & lt)) & 127;
                    L.x[at] = rx;
                    L.y[at] = ry;
                    L.z[at] = rz;
                    if (HH) L.h[HH ? at : 0] = hj;
                    L.j[at] = c0.beg + lane;
                }
                const int nt = tail + __popcll(m);
                if ((nt ^ tail) & 64) {
                    batch(tail & 64, 64);
                    lim = sink.full() ? 0 : lim;
                }
                tail = nt & 127;
            }
            c0 = c1;
            c1 = c2;
        }
        const int n = tail & 63, base = tail & 64;
        if (n) {
            if (lane >= n) {
                L.x[base + lane] = TW_FAR;
                L.y[base + lane] = TW_FAR;
                L.z[base + lane] = TW_FAR;
                if (HH) L.h[HH ? base + lane : 0] = 0.0f;
            }
            batch(base, n);
        }
        nl = 0;
    };
    const int s0 = t.r_sbeg[r], s1 = t.r_send[r];
    for (int sb = s0; sb < s1; sb += 64) {
        const int S = sb + lane;
        bool sp = S < s1;
        // with few supers their test costs more than the bucket tests it saves
        if (sp && s1 - s0 > 2) {
            const double d2 = sphx_box_d2(gb[0], gb[1], gb[2], gb[3], gb[4], gb[5], t.sxl[S], t.sxh[S],
                                          t.syl[S], t.syh[S], t.szl[S], t.szh[S]);
            sp = sphx_within(d2, HH ? reach + t.shmax[S] : reach);
        }
        uint64_t smask = __ballot(sp);
        while (smask) {
            const int S2 = sb + __builtin_ctzll(smask);
            smask &= smask - 1;
            const int j0 = t.s_bbeg[S2], J = j0 + lane;
            bool bp = false;
            double hb = 0.0;
            int2 e = make_int2(0, 0);
            if (J < t.s_bend[S2]) {
                const double d2 = sphx_box_d2(gb[0], gb[1], gb[2], gb[3], gb[4], gb[5], t.bxl[J],
                                              t.bxh[J], t.byl[J], t.byh[J], t.bzl[J], t.bzh[J]);
                if (HH) hb = t.bhmax[J];
                bp = sphx_within(d2, HH ? reach + hb : reach);
                e = make_int2(t.b_beg[J], t.b_cnt[J]);
            }
            const uint64_t bmask = __ballot(bp);
            if (bp) {
                L.bl[nl + __popcll(bmask & lt)] = e;
                if (HH) hc = fmax(hc, hb);
            }
            nl += __popcll(bmask);
            ncand += __popcll(bmask);
            __builtin_amdgcn_wave_barrier();
            if (nl > TW_LIST - 64) walk();
            if (sink.full()) return ncand;
        }
    }
    if (nl) walk();
    return ncand;
}

// What the sinks share: a lane's target in the frame, and the in-reach masks
// of the current batch.  Bit 31 - k of word w (bit Q - 1 - k with fewer than 32
// candidates per slice) is candidate q0 + 32 w + k.
struct WalkTarget {
    float x, y, z;
    __device__ __forceinline__ void set(const WalkFrame &f, bool act, double xi, double yi, double zi) {
        // an idle lane sits where nothing is in reach
        x = act ? (float)((xi - f.ox) * f.sc) : -TW_FAR;
        y = act ? (float)((yi - f.oy) * f.sc) : -TW_FAR;
        z = act ? (float)((zi - f.oz) * f.sc) : -TW_FAR;
    }
};
__device__ __forceinline__ uint32_t sign_in(uint32_t m, float d) {
    return __builtin_amdgcn_alignbit(m, __float_as_uint(d), 31);  // m << 1 | sign of d
}

// Count of the candidates for which `exact(j)`, known to hold exactly when
// r^2 <= S^2 up to FP64 rounding at S, does.
template <int P, class Exact>
struct CountSink {
    WalkTarget p;
    float nS2, band;
    Exact exact;
    int kc;
    uint32_t m0, m1;
    float amin;
    __device__ __forceinline__ CountSink(const WalkFrame &f, bool act, double xi, double yi, double zi,
                                         double S, Exact ex)
        : exact(ex), kc(0) {
        p.set(f, act, xi, yi, zi);
        const double Ss = S * f.sc, M = fmax(fmax(f.ex, f.ey), f.ez) + 2.0;
        nS2 = act ? -(float)(Ss * Ss) : 1.0f;
        band = f.sc > 0.0 ? (act ? walk_band(Ss, M) : -1.0f) : INFINITY;
    }
    __device__ __forceinline__ void chunk(double, bool) {}
    __device__ __forceinline__ bool full() const { return false; }
    __device__ __forceinline__ void begin() { m0 = m1 = 0u; amin = INFINITY; }
    __device__ __forceinline__ void word() { m0 = m1; m1 = 0u; }
    __device__ __forceinline__ void cand(float cx, float cy, float cz, float) {
        const float dx = cx - p.x, dy = cy - p.y, dz = cz - p.z;
        const float d = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, __builtin_fmaf(dz, dz, nS2)));
        m1 = sign_in(m1, d);
        amin = fminf(amin, fabsf(d));
    }
    template <class LDS>
    __device__ __forceinline__ void batch(const LDS &L, int base, int n, int q0) {
        if (__any(amin <= band)) {
            int c = 0;
            for (int k = 0; k < 64 / P; ++k)
                if (q0 + k < n && !(nS2 > 0.0f) && exact(L.j[base + q0 + k])) ++c;
            kc += c;
        } else {
            kc += __popc(m0) + __popc(m1);
        }
    }
};

// Candidate filter: lane q holds particle q of a staged candidate bucket and
// keeps it when it may lie within `reach` of the target group's box (the same
// conservative FP64 test as the bucket culling).  A dropped particle is out of
// reach of every target particle, so the kept ones, compacted in their
// original order, give exactly the sums of the unfiltered loop.
struct Kept {
    int n, slot;
};
__device__ __forceinline__ Kept keep_mask(bool keep, int lane) {
    uint64_t m = __ballot(keep);
    Kept k;
    k.n = __popcll(m);
    k.slot = __popcll(m & ((1ull << lane) - 1ull));
    return k;
}

__device__ __forceinline__ bool near_box(const double *bx, double x, double y, double z,
                                         double reach) {
    return sphx_within(sphx_box_d2(bx[0], bx[1], bx[2], bx[3], bx[4], bx[5], x, x, y, y, z, z),
                       reach);
}

struct SmoothArgs {
    int32_t nngb, ndown, nup, max_iter;
    int32_t predictor;
    const RunParams *rp;
    int32_t *h_iters;  // per particle, nullable
    int64_t *counters;
    double hstep;      // RULE 2: the step as a fraction of h_prev (2 x the reference's coeff)
    double hmin;       // RULE 5: the floor on h after eleven steps (0: none)
    // step rules: the counts that a window's ends are aimed at and the slack
    // either side of them (hwin 0: no window holds this band)
    int32_t hwin, wlo, whi, wslack;
};

// One walk over the candidates of the group's active targets: for each segment
// with some, make(frame, mine) gives the sink of its targets (mine: the lanes of
// those), done(sink, mine) takes it back.  Once some targets have settled, the
// walk culls against the box of those still active.
template <int P, class Make, class Done>
__device__ __forceinline__ void smooth_walk(const Tables &t, const Soa &s, WalkLds<false> &L, int r,
                                            int lane, int cnt, bool ok, uint64_t cuts, double xi,
                                            double yi, double zi, bool active, double reach,
                                            Make make, Done done) {
    const int tl = lane & (64 / P - 1);
    for (int g0 = 0; g0 < cnt;) {
        const int g1 = seg_end(cuts, g0, cnt);
        const bool mine = active && tl >= g0 && tl < g1;
        g0 = g1;
        const double R = wave_max_d(mine ? reach : 0.0);
        if (!(R > 0.0)) continue;  // no active target in this segment
        double gb[6], hdummy;
        seg_box(mine, xi, yi, zi, 0.0, gb, &hdummy);
        const WalkFrame f = walk_frame(gb, R);
        auto sink = make(f, mine);
        tile_walk<P, false>(t, s, L, r, lane, gb, R, f, sink);
        done(sink, mine);
    }
}

// Counts of passes of a group, for the counters.
__device__ __forceinline__ void smooth_counters(const SmoothArgs &a, int lane, bool ok, int it) {
    int itmax = wave_max_i(ok ? it : 0);
    unsigned long long itsum = 0;
    {
        int v = ok ? it : 0;
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
        itsum = (unsigned long long)v;
    }
    if (lane == 0) {
        atomicMax((unsigned long long *)&a.counters[CNT_H_ITERS_MAX], (unsigned long long)itmax);
        atomicAdd((unsigned long long *)&a.counters[CNT_H_ITERS_SUM], itsum);
    }
}

// The count-band iteration: a log-space Newton step, kept inside the bracket
// by bisection.
template <int P>
__global__ __launch_bounds__(64) void k_smoothing(Tables t, Soa s, SmoothArgs a) {
    __shared__ WalkLds<false> L;
    const WalkSlot ws = walk_slot<P>(t);
    const int lane = threadIdx.x, tl = lane & (64 / P - 1);
    const int cnt = ws.cnt;
    const int i = ws.first + tl;
    const bool ok = tl < cnt;
    const int r = t.b_run[ws.b];
    const int64_t nrun = (int64_t)t.r_pend[r] - t.r_pbeg[r];
    const double xi = ok ? s.x[i] : 0.0, yi = ok ? s.y[i] : 0.0, zi = ok ? s.z[i] : 0.0;
    const double hprev = ok ? s.h[i] : 0.0;
    const uint64_t cuts = bucket_cuts(t, r, i, ok && lane < 64 / P, lane);
    const bool whole = fabs(xi) < INFINITY && fabs(yi) < INFINITY && fabs(zi) < INFINITY;
    double sr;
    {
#pragma clang fp contract(off)
        sr = 2.0 * hprev;
        if (a.predictor && ok) {
            double dt = a.rp[r].dt;
            double f = sphx_h_factor(a.nngb, s.k[i]);
            double t1 = 0.5 * hprev;
            double t2 = 1.0 + f;
            double t3 = t1 * t2;
            double u = hprev * s.divv[i];
            u = u * dt;
            double t6 = u / 3.0;
            double sp = 2.0 * (t3 + t6);
            if (sp > 0.0 && sp < INFINITY) sr = sp;
        }
    }
    double lo = 0.0, hi = 0.0;
    int klo = 0, khi = 0, kfin = 0;
    bool have_lo = false, have_hi = false, done = !ok, conv = false;
    int it = 0;
    while (true) {
        bool active = ok && !done;
        if (!__any(active)) break;
        const double s2 = sphx_sq(sr);
        int kc = 0;
        auto in = [&](int j) { return sphx_r2(xi - s.x[j], yi - s.y[j], zi - s.z[j]) <= s2; };
        smooth_walk<P>(
            t, s, L, r, lane, cnt, ok, cuts, xi, yi, zi, active, sr,
            [&](const WalkFrame &f, bool mine) {
                return CountSink<P, decltype(in)>(f, mine && whole, xi, yi, zi, sr, in);
            },
            [&](const CountSink<P, decltype(in)> &c, bool mine) { kc = mine ? c.kc : kc; });
        kc = slice_sum<P>(kc);
        if (active) {
#pragma clang fp contract(off)
            ++it;
            if (kc >= a.ndown && kc <= a.nup) {
                done = true;
                conv = true;
                kfin = kc;
            } else {
                if (kc < a.ndown) {
                    lo = sr; klo = kc; have_lo = true;
                    if ((int64_t)kc >= nrun) done = true;
                } else {
                    hi = sr; khi = kc; have_hi = true;
                }
                if (!done) {
                    double snew = sr * sphx_h_factor(a.nngb, kc);
                    if (have_lo && have_hi) {
                        if (!(snew > lo && snew < hi)) snew = 0.5 * (lo + hi);
                        if (!(snew > lo && snew < hi)) done = true;
                    }
                    if (!done) {
                        sr = snew;
                        if (it >= a.max_iter) done = true;
                    }
                }
            }
        }
    }
    if (ok) {
        if (!conv) {
            if (have_hi) { sr = hi; kfin = khi; }
            else { sr = lo; kfin = klo; }
            if (lane < 64 / P) atomicAdd((unsigned long long *)&a.counters[CNT_H_CAPPED], 1ull);
        }
        if (lane < 64 / P) {
            s.h[i] = 0.5 * sr;
            s.k[i] = kfin;
            if (a.h_iters) a.h_iters[i] = it;
        }
    }
    smooth_counters(a, lane, ok && lane < 64 / P, it);
}

// A lane of the step rules (RULES 2, 4, 5; see k_smoothing_steps) and one pass
// of its rule after a count kc at the radius sr.  Only kc's place against the
// band moves the radius; its value is what kfin returns.
template <int RULE>
struct StepIter {
    double sr, hprev;
    double coef;   // RULES 2, 4: the step over h_prev (RULE 4 halves it)
    double smax;   // RULE 2: the largest radius tried
    double sc;     // the radius of the last count
    int kpre;      // RULE 4: the previous pass's count
    int it, kfin;
    bool done, conv;

    __device__ __forceinline__ void pass(int kc, const SmoothArgs &a) {
#pragma clang fp contract(off)
        ++it;
        sc = sr;
        if (RULE == 4 && kc > a.nup) kc = a.nup + 1;  // LIBV7 stops counting there
        const bool in_band = kc >= a.ndown && kc <= a.nup;
        // LIBSX:1226-1228: after the eleventh step an h under the floor is
        // set to it and ends the iteration, in the band or not
        const bool floor_h = RULE == 5 && a.hmin > 0.0 && it > 11 && 0.5 * sr < a.hmin;
        if (RULE == 4 && ((kc < a.ndown && kpre > a.nup) || (kc > a.nup && kpre < a.ndown)))
            coef = 0.5 * coef;  // a jump across the band
        if (RULE == 5) {
            const double hc = 0.5 * sr;
            if (kc < a.ndown) sr = 2.0 * (hc + 0.003 * hc);
            if (kc > a.nup) sr = 2.0 * (hc - 0.003 * hc);
        } else {
            if (kc < a.ndown) sr = sr + coef * hprev;
            if (kc > a.nup) sr = sr - coef * hprev;
        }
        if (sr > smax) smax = sr;
        kpre = kc;
        kfin = kc;
        if (floor_h) {
            sr = 2.0 * a.hmin;
            done = true;
            conv = true;
        } else if (in_band) {  // before the pass limit, as the reference tests
            done = true;
            conv = true;
        } else if (it > (RULE == 4 ? SPHX_H4_PASSES : (RULE == 5 ? SPHX_H5_PASSES : a.max_iter))) {
            // the pass limit: RULE 2 takes the largest radius, RULES 4, 5 the last
            if (RULE == 2) sr = smax;
            done = true;
        }
    }
    // whether a particle at distance d is counted at radius rad
    static __device__ __forceinline__ bool counts(double d, double rad) {
        return RULE == 5 ? d < rad : d <= rad;
    }
};

// The step rules ask of a pass only on which side of the band its count lies,
// and the distances that decide it are the few about the band's radii.  So a
// target first finds a window (w0, w1] of radii with fewer than ndown particles
// up to w0 and more than nup (or the whole run) up to w1, keeping the window's
// distances in LDS, and then passes without walking: a count is the particles
// up to w0 plus the window's, and between two crossings of the band all passes
// fall on one side, decided by one distance.
//
// Bound: the walks, which every pass took before.  Now there are two or three a
// group, whatever the passes: the first pass's count, and windows whose ends are
// aimed, from the counts at the last ones, at the band and a quarter of the spare
// slots beyond it on either side (45 and 83 neighbours for the band 59 to 69), or
// halved in between.  A window takes nup - ndown + 2 distances at least, of
// HW_CAP.  Walks of a target on an Evrard sphere of 16,384, from 1.3 times the
// length (102 passes for all of these): 2.03 on average and 4 at most for the band
// 59 to 69, 2.41 and 5 for 44 to 84, 3.4 and 9 for 36 to 92 (and from a third of
// the length to three times it 2.7 and 7 for the first); with both ends
// scaled together about the middle of the band they were passes and 16 walks
// more for most targets from bands of 41 counts on.  A wider band, a target left
// without a window (more than 64 particles at one distance, a start that is not a
// positive number) is walked pass by pass.  The slots take 512 B a target.
constexpr int HW_CAP = 64;
constexpr int HW_WALKS = 8;
constexpr int HW_SPARE = 4;  // with fewer slots to spare the search takes too long

// Collects the window: base counts r^2 <= W0, the indices of the candidates
// with W0 < r^2 <= W1 go to the target's column (the first HW_CAP of them).
template <int P>
struct WindowSink {
    WalkTarget p;
    float nW1, dW, band;
    double xi, yi, zi, W0, W1;
    const Soa *s;
    double *col;
    int lane, base, inw;
    uint32_t a0, a1, b0, b1;  // masks of r^2 <= W1 and <= W0
    float amin;
    __device__ __forceinline__ WindowSink(const WalkFrame &f, bool act, double x, double y, double z,
                                          double w0, double w1, double W0_, double W1_, const Soa *s_,
                                          double *col_, int lane_)
        : xi(x), yi(y), zi(z), W0(W0_), W1(W1_), s(s_), col(col_), lane(lane_), base(0), inw(0) {
        p.set(f, act, x, y, z);
        const double M = fmax(fmax(f.ex, f.ey), f.ez) + 2.0;
        const double s1 = w1 * f.sc, s0 = W0 < 0.0 ? 0.0 : w0 * f.sc;
        nW1 = act ? -(float)(s1 * s1) : 1.0f;
        // r^2 = 0 is inside a window from 0, where the band cannot be trusted to
        // tell: every value within it is tested in FP64
        dW = (float)(s1 * s1 - s0 * s0);
        band = f.sc > 0.0 ? (act ? walk_band(s1, M) : -1.0f) : INFINITY;
    }
    __device__ __forceinline__ void chunk(double, bool) {}
    __device__ __forceinline__ bool full() const { return false; }
    __device__ __forceinline__ void begin() { a0 = a1 = b0 = b1 = 0u; amin = INFINITY; }
    __device__ __forceinline__ void word() { a0 = a1; b0 = b1; a1 = b1 = 0u; }
    __device__ __forceinline__ void cand(float cx, float cy, float cz, float) {
        const float dx = cx - p.x, dy = cy - p.y, dz = cz - p.z;
        const float d = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, __builtin_fmaf(dz, dz, nW1)));
        const float e = d + dW;
        a1 = sign_in(a1, d);
        b1 = sign_in(b1, e);
        amin = fminf(amin, fminf(fabsf(d), fabsf(e)));
    }
    template <class LDS>
    __device__ __forceinline__ void batch(const LDS &L, int base_, int n, int q0) {
        constexpr int Q = 64 / P;
        if (__any(amin <= band)) {
            a0 = a1 = b0 = b1 = 0u;
            for (int k = 0; k < Q; ++k) {
                if (P == 1 && k == 32) word();
                a1 <<= 1;
                b1 <<= 1;
                if (!(nW1 > 0.0f) && q0 + k < n) {
                    const int j = L.j[base_ + q0 + k];
                    const double r2 = sphx_r2(xi - s->x[j], yi - s->y[j], zi - s->z[j]);
                    a1 |= r2 <= W1 ? 1u : 0u;
                    b1 |= r2 <= W0 ? 1u : 0u;
                }
            }
        }
        base += __popc(b0) + __popc(b1);
        uint32_t w[2] = {a0 & ~b0, a1 & ~b1};
        int tot;
        int at = inw + slice_scan<P>(__popc(w[0]) + __popc(w[1]), lane, &tot);
#pragma unroll
        for (int v = 0; v < 2; ++v) {
            if (P > 1 && v == 0) continue;
            const int first = P == 1 ? 32 * v : 0, bits = P == 1 ? 32 : Q;
            while (w[v]) {
                const int k = 31 - __builtin_clz(w[v]);
                w[v] &= ~(1u << k);
                if (at < HW_CAP)
                    reinterpret_cast<int32_t *>(&col[at * Q])[0] = L.j[base_ + q0 + first + bits - 1 - k];
                ++at;
            }
        }
        inw += tot;
    }
};

// The reference's own rules.  RULE 2: LIBSX3:947-1006, LIBV2:7-64
// (do_smoothingX4 with ten times the step): fixed steps of a.hstep h_prev
// (0.002 or 0.02) from 2 h_prev (or the eq. 31 start, in the reference's order
// of operations), counts by sqrt(r^2) <= s as the reference tests, the largest
// radius taken after max_iter + 1 passes.  RULE 4: the LIBV7 driver's rule
// (LIBV7:255-328): steps of 0.01 h_prev, halved on every jump across the band,
// the last radius after 501 passes, counts that stop at nup + 1.  RULE 5:
// h_smooth_fast (LIBSX:1133-1184): from h_prev with no predictor, h -+= 0.003 h
// on the current h, the count strict (sqrt(r^2) < 2h), the last h after
// SPHX_H5_PASSES passes.
template <int RULE, int P>
__global__ __launch_bounds__(64) void k_smoothing_steps(Tables t, Soa s, SmoothArgs a) {
    constexpr int T = 64 / P;
    __shared__ WalkLds<false> L;
    __shared__ double hw[HW_CAP * T];
    const WalkSlot ws = walk_slot<P>(t);
    const int lane = threadIdx.x, tl = lane & (T - 1), slice = lane / T;
    const int cnt = ws.cnt;
    const int i = ws.first + tl;
    const bool ok = tl < cnt;
    const int r = t.b_run[ws.b];
    const int64_t nrun = (int64_t)t.r_pend[r] - t.r_pbeg[r];
    const double xi = ok ? s.x[i] : 0.0, yi = ok ? s.y[i] : 0.0, zi = ok ? s.z[i] : 0.0;
    const double hprev = ok ? s.h[i] : 0.0;
    const uint64_t cuts = bucket_cuts(t, r, i, ok && lane < T, lane);
    const bool fin = fabs(xi) < INFINITY && fabs(yi) < INFINITY && fabs(zi) < INFINITY;
    double sr;
    {
#pragma clang fp contract(off)
        sr = 2.0 * hprev;
        if (RULE != 5 && a.predictor && ok) {
            double dt = a.rp[r].dt;
            double f = sphx_h_factor(a.nngb, s.k[i]);
            double t1 = 0.5 * hprev;
            double t2 = 1.0 + f;
            double t3 = t1 * t2;
            double t6;
            if (RULE == 4) {  // LIBV7:265-266: ((1/3 h) divV) dt
                double u = (1.0 / 3.0) * hprev;
                u = u * s.divv[i];
                t6 = u * dt;
            } else {          // LIBSX3:961: (1/3 (h divV)) dt
                double u = hprev * s.divv[i];
                u = (1.0 / 3.0) * u;
                t6 = u * dt;
            }
            double sp = 2.0 * (t3 + t6);
            if (sp > 0.0 && sp < INFINITY) sr = sp;
        }
    }
    using Iter = StepIter<RULE>;
    Iter q{sr, hprev, a.hstep, sr, sr, a.nup, 0, 0, !ok, false};

    auto count = [&](bool active, double rad) {
        int kc = 0;
        auto in = [&](int j) {
            return Iter::counts(sqrt(sphx_r2(xi - s.x[j], yi - s.y[j], zi - s.z[j])), rad);
        };
        smooth_walk<P>(
            t, s, L, r, lane, cnt, ok, cuts, xi, yi, zi, active, rad,
            [&](const WalkFrame &f, bool mine) {
                return CountSink<P, decltype(in)>(f, mine && fin, xi, yi, zi, rad, in);
            },
            [&](const CountSink<P, decltype(in)> &c, bool mine) { kc = mine ? c.kc : kc; });
        return slice_sum<P>(kc);
    };

    // the first pass settles most targets of a run in progress, and tells the
    // others where the band is
    const int k0 = count(ok, sr);
    double w0 = 0.0, w1 = 0.0;
    if (ok) {
        q.pass(k0, a);
        const double c0 = sr * sphx_h_factor(a.nngb, k0);
        w0 = a.wlo > 0 ? c0 * sphx_h_factor(a.wlo, a.nngb) : 0.0;
        w1 = c0 * sphx_h_factor(a.whi, a.nngb);
    }

    // the window
    double *col = hw + tl;
    double lo = 0.0, hi = INFINITY;  // radii known to hold < ndown, and > nup (or the run)
    double u = INFINITY, v = 0.0;    // and the next ones known not to
    int base = 0, inw = 0;
    bool sel = false, whole = false;
    bool open = a.hwin && ok && !q.done && fin && sr > 0.0 && sr < INFINITY && w1 < INFINITY;
    for (int walk = 0; walk < HW_WALKS && __any(open); ++walk) {
        // r^2 bounds of the window; 0 itself is inside a window from 0
        const double W0 = w0 > 0.0 ? sphx_sq(w0) : -1.0, W1 = sphx_sq(w1);
        smooth_walk<P>(
            t, s, L, r, lane, cnt, ok, cuts, xi, yi, zi, open, w1,
            [&](const WalkFrame &f, bool mine) {
                return WindowSink<P>(f, mine, xi, yi, zi, w0, w1, W0, W1, &s, col, lane);
            },
            [&](const WindowSink<P> &c, bool mine) {
                base = mine ? c.base : base;
                inw = mine ? c.inw : inw;
            });
        const int bs = slice_sum<P>(base);
        if (open) {
            base = bs;
            const int tot = base + inw;
            const bool lo_ok = base < a.ndown;
            whole = (int64_t)tot >= nrun;
            const bool hi_ok = tot > a.nup || whole;
            if (lo_ok && w0 > lo) lo = w0;
            if (base > a.nup && w0 < hi) hi = w0;
            if (hi_ok && w1 < hi) hi = w1;
            if (tot < a.ndown && !whole && w1 > lo) lo = w1;
            if (!lo_ok && w0 < u) u = w0;
            if (!hi_ok && w1 > v) v = w1;
            if (lo_ok && hi_ok && inw <= HW_CAP) {
                sel = true;
                open = false;
            } else {
                // an end that is not near enough: the middle of the radii between
                // which it must lie, once both are known (at last the one that
                // is known to do), before that aimed anew from its own count (the
                // lower one from the upper's where its own says too little)
                double nw0 = w0, nw1 = w1;
                if (!lo_ok || base < a.wlo - a.wslack) {
                    nw0 = 2 * (int64_t)base > a.wlo ? w0 * sphx_h_factor(a.wlo, base)
                                                    : w1 * sphx_h_factor(a.wlo, tot);
                    if (lo > 0.0 && u < INFINITY) nw0 = walk >= 4 && !lo_ok ? lo : 0.5 * (lo + u);
                }
                if (!hi_ok || tot - a.wslack > a.whi) {
                    nw1 = w1 * sphx_h_factor(a.whi, tot);
                    if (v > 0.0 && hi < INFINITY) nw1 = walk >= 4 && !hi_ok ? hi : 0.5 * (v + hi);
                }
                if (a.wlo == 0) nw0 = 0.0;
                w0 = fmax(lo, nw0);
                w1 = fmin(hi, nw1);
                if (!(w0 < w1) && lo < hi && hi < INFINITY) {  // both in one gap
                    w0 = lo + (hi - lo) / 3.0;
                    w1 = hi - (hi - lo) / 3.0;
                }
                open = w0 < w1 && w1 < INFINITY;
                if (open) base = inw = 0;
            }
        }
    }

    // the passes of the targets that have a window, on its distances; a
    // target's slices share the scans of its column
    bool recount = false;
    if (__any(sel)) {
        const int mw = wave_max_i(sel ? inw : 0);
        if (!sel) inw = 0;
        for (int k = slice; k < mw; k += P) {
            const int at = (k < inw ? k : 0) * T;
            if (k < inw) {
                const int j = reinterpret_cast<const int32_t *>(&col[at])[0];
                col[at] = sqrt(sphx_r2(xi - s.x[j], yi - s.y[j], zi - s.z[j]));
            }
        }
        __syncthreads();
        auto count_at = [&](double rad) {
            int c = 0;
#pragma unroll 4
            for (int k = slice; k < mw; k += P)
                c += (k < inw && Iter::counts(col[(k < inw ? k : 0) * T], rad)) ? 1 : 0;
            return base + slice_sum<P>(c);
        };
        bool run = sel;
        while (__any(run)) {
            const int kc = count_at(q.sr);
            const bool low = kc < a.ndown;
            const double s0 = q.sr;
            int need = 0;  // distances to cross until the band's side changes
            if (run) {
                q.pass(kc, a);
                run = !q.done;
                need = run ? (low ? a.ndown - kc : kc - a.nup) : 0;
            }
            // the need-th distance beyond s0 in the direction of travel: upwards
            // among those not counted at s0, downwards among the counted
            double edge = -INFINITY;  // of +-distance, increasing
            int got = 0;
            bool more = got < need;
            while (__any(more)) {
                double best = INFINITY;
                int mult = 0;
#pragma unroll 4
                for (int k = slice; k < mw; k += P) {
                    const double d = col[(k < inw ? k : 0) * T];
                    const double v = low ? d : -d;
                    const bool in = k < inw && Iter::counts(d, s0) != low && v > edge && v <= best;
                    mult = in ? (v < best ? 1 : mult + 1) : mult;
                    best = in ? v : best;
                }
                for (int o = T; o < 64; o <<= 1) {
                    const double ob = __shfl_xor(best, o, 64);
                    const int om = __shfl_xor(mult, o, 64);
                    mult = ob < best ? om : (ob == best ? mult + om : mult);
                    best = fmin(best, ob);
                }
                if (more) {
                    edge = best;  // +inf: none left (the whole run is in the window)
                    got += mult;
                    more = mult > 0 && got < need;
                }
            }
            if (!low) edge = -edge;
            // passes on the same side of the band
            while (run && (low ? !Iter::counts(edge, q.sr) : Iter::counts(edge, q.sr))) {
                q.pass(low ? a.ndown - 1 : a.nup + 1, a);
                run = !q.done;
            }
        }
        // the count that the last pass was made on
        const int kc = count_at(q.sc);
        if (sel) {
            q.kfin = RULE == 4 && kc > a.nup ? a.nup + 1 : kc;
            // exact inside the window (RULE 4 stops counting above the band)
            const bool above = whole || q.sc < w1 || (RULE == 4 && kc > a.nup);
            recount = !(q.sc > w0 && above);
        }
    }

    // the others pass by pass, and one count for those that ended outside
    // their window
    while (true) {
        const bool active = ok && (sel ? recount : !q.done);
        if (!__any(active)) break;
        const int kc = count(active, sel ? q.sc : q.sr);
        if (active) {
            if (sel) {
                q.kfin = RULE == 4 && kc > a.nup ? a.nup + 1 : kc;
                recount = false;
            } else {
                q.pass(kc, a);
            }
        }
    }
    if (ok && lane < T) {
        if (!q.conv) atomicAdd((unsigned long long *)&a.counters[CNT_H_CAPPED], 1ull);
        s.h[i] = 0.5 * q.sr;
        s.k[i] = q.kfin;
        if (a.h_iters) a.h_iters[i] = q.it;
    }
    smooth_counters(a, lane, ok && lane < T, q.it);
}

// Cubic spline W / (sigma / h^3) and grad-W factor F / (sigma / h^5) in FP32.
// q = r / h; the pair terms' fused multiply-adds are written out (see below).
__device__ __forceinline__ float w_shape(float r, float hinv, float q) {
    // both pieces, then a select: the lanes of a wave straddle q = 1, so a
    // branch would run both anyway and add the exec-mask bookkeeping
#pragma clang fp contract(off)
    float w1 = __builtin_fmaf(q, 0.75f * q * q, __builtin_fmaf(q, -1.5f * q, 1.0f));
    float w = fmaxf(__builtin_fmaf(-r, hinv, 2.0f), 0.0f);
    float w2 = 0.25f * w * w * w;
    return q <= 1.0f ? w1 : w2;
}
__device__ __forceinline__ float f_shape(float q) {
#pragma clang fp contract(off)
    float f1 = __builtin_fmaf(2.25f, q, -3.0f);
    float w = fmaxf(2.0f - q, 0.0f);
    float f2 = -0.75f * w * w * __builtin_amdgcn_rcpf(q);
    return q <= 1.0f ? f1 : f2;
}

struct PairGeom {
    float dx, dy, dz, r2, hinv, r, q;
};

__device__ __forceinline__ PairGeom pair_geom(double dx, double dy, double dz, double r2,
                                              double t) {
#pragma clang fp contract(off)
    PairGeom g;
    g.dx = (float)dx;
    g.dy = (float)dy;
    g.dz = (float)dz;
    g.r2 = (float)r2;
    float hij = 0.5f * (float)t;
    g.hinv = __builtin_amdgcn_rcpf(hij);
    g.r = __builtin_amdgcn_sqrtf(g.r2);
    g.q = g.r * g.hinv;
    return g;
}

// The pair terms of the div/curl and hydro passes, shared by the candidate
// walks and the neighbour-list passes so that both evaluate every pair with
// the same instructions (the list passes are then bit-identical to the walks).
// Their fused multiply-adds are written out: left to the compiler, which
// products it fuses depends on the loop around them.
struct Terms4 {
    float a, b, c, d;
};
__device__ __forceinline__ Terms4 divcurl_terms(double vxi, double vyi, double vzi, double vxj,
                                                double vyj, double vzj, float mj,
                                                const PairGeom &g) {
#pragma clang fp contract(off)
    float h5 = g.hinv * g.hinv;
    h5 = h5 * h5 * g.hinv;
    float F = SPHX_SIGMA_F * h5 * f_shape(g.q) * mj;
    float vx = (float)(vxi - vxj), vy = (float)(vyi - vyj), vz = (float)(vzi - vzj);
    return {F * __builtin_fmaf(vz, g.dz, __builtin_fmaf(vx, g.dx, vy * g.dy)),
            F * __builtin_fmaf(vy, g.dz, -(vz * g.dy)), F * __builtin_fmaf(vz, g.dx, -(vx * g.dz)),
            F * __builtin_fmaf(vx, g.dy, -(vy * g.dx))};
}
__device__ __forceinline__ void divcurl_pair(double vxi, double vyi, double vzi, double vxj,
                                             double vyj, double vzj, float mj, double dx,
                                             double dy, double dz, double r2, double tt,
                                             KahanF &kd, KahanF &kx, KahanF &ky, KahanF &kz) {
    const Terms4 t = divcurl_terms(vxi, vyi, vzi, vxj, vyj, vzj, mj, pair_geom(dx, dy, dz, r2, tt));
    kd.add(t.a);
    kx.add(t.b);
    ky.add(t.c);
    kz.add(t.d);
}

struct HydroArgs {
    float alpha, beta, eta2, w_eps;
    int32_t av_form, balsara;
};

// Particle i's side of the hydro pair terms.
struct HydroI {
    double vx, vy, vz;
    float rho, pr, c, f;  // rho, P / rho^2, sound speed, Balsara factor
};

__device__ __forceinline__ Terms4 hydro_terms(const HydroArgs &a, const HydroI &I, double vxj,
                                              double vyj, double vzj, float mj, float rhoj, float prj,
                                              float cj, float fj, double tt, const PairGeom &g) {
#pragma clang fp contract(off)
    float h5 = g.hinv * g.hinv;
    h5 = h5 * h5 * g.hinv;
    float F = SPHX_SIGMA_F * h5 * f_shape(g.q);
    float vx = (float)(I.vx - vxj), vy = (float)(I.vy - vyj), vz = (float)(I.vz - vzj);
    float vr = __builtin_fmaf(vz, g.dz, __builtin_fmaf(vx, g.dx, vy * g.dy));
    float pij = 0.0f;
    if (vr <= 0.0f) {
        float rhob = 0.5f * (I.rho + rhoj);
        float hij = 0.5f * (float)tt;
        if (a.av_form == 0) {
            float mu = hij * vr / __builtin_fmaf(hij * hij, a.eta2, g.r2);
            pij = __builtin_fmaf(a.beta * mu, mu, -(a.alpha * 0.5f * (I.c + cj) * mu)) / rhob;
        } else {
            float w = vr / (g.r + a.w_eps);
            pij = -0.5f * a.alpha * __builtin_fmaf(-3.0f, w, I.c + cj) * w / rhob;
        }
        pij *= 0.5f * (I.f + fj);
    }
    float mF = mj * F;
    float sc_ = mF * (I.pr + prj + pij);
    return {-sc_ * g.dx, -sc_ * g.dy, -sc_ * g.dz, mF * __builtin_fmaf(0.5f, pij, I.pr) * vr};
}
__device__ __forceinline__ void hydro_pair(const HydroArgs &a, const HydroI &I, double vxj,
                                           double vyj, double vzj, float mj, float rhoj,
                                           float prj, float cj, float fj, double dx, double dy,
                                           double dz, double r2, double tt, KahanF &kx,
                                           KahanF &ky, KahanF &kz, KahanF &kdu) {
    const Terms4 t = hydro_terms(a, I, vxj, vyj, vzj, mj, rhoj, prj, cj, fj, tt,
                                 pair_geom(dx, dy, dz, r2, tt));
    kx.add(t.a);
    ky.add(t.b);
    kz.add(t.c);
    kdu.add(t.d);
}

__device__ __forceinline__ double balsara_f(double dv, double cv, double c, double h) {
    double a = fabs(dv);
    return a / (a + cv + 0.0001 * c / h);
}

// Position of entry k of lane L in its bucket's list block: lanes hold their
// entries in runs of 8 (32 bytes), the runs of the 64 lanes side by side, so
// that a lane fills its own 32-byte piece as it accepts neighbours (four lanes
// complete a 128-byte line together) and iteration k of a list pass reads
// 64 runs that iterations k + 1 .. k + 7 read again.
__device__ __forceinline__ int64_t nbr_slot(int k, int lane) {
    return ((int64_t)(k >> 3) * 64 + lane) * 8 + (k & 7);
}

// Calls f(rec) for entries 0 .. len-1 of this lane's list, every lane on its
// own entry k at once (maxlen: the wave's longest list), rec = load(j) issued
// one entry ahead and each 8-entry run (two 16-byte loads) one run ahead: with
// one record in flight a lane waited out an L2 trip for every neighbour.
template <class Load, class F>
__device__ __forceinline__ void for_list(const int32_t *lp, int lane, int len, int maxlen, int self,
                                         Load load, F f) {
    if (maxlen <= 0) return;
    auto run = [&](int k0, int4 &a, int4 &c) {
        a = c = make_int4(self, self, self, self);
        if (k0 < len) {
            const int4 *p = reinterpret_cast<const int4 *>(lp + nbr_slot(k0, lane));
            a = p[0];
            c = p[1];
        }
    };
    int4 a, c, na, nc;
    run(0, a, c);
    auto nxt = load(len > 0 ? a.x : self);
    for (int k0 = 0; k0 < maxlen; k0 += 8) {
        run(k0 + 8, na, nc);
#pragma unroll 2
        for (int q = 0; q < 8; ++q) {
            if (k0 + q >= maxlen) break;
            a.x = a.y; a.y = a.z; a.z = a.w; a.w = c.x;
            c.x = c.y; c.y = c.z; c.z = c.w; c.w = na.x;
            const auto cur = nxt;
            nxt = load(k0 + q + 1 < len ? a.x : self);  // entries past len are not indices
            if (k0 + q < len) f(cur);
        }
        a = na;
        c = nc;
    }
}

struct DensArgs {
    double gamma;
    int32_t *nsym;        // symmetric neighbour count, nullable
    int64_t *counters;
    // neighbour lists for the div/curl and hydro passes (all null: none written)
    int32_t *lst;         // [bucket][entry < SPHX_NBR_MAX][lane]: accepted j in walk order
    PairRec *rec;         // per particle: the j-side values of the pair passes
    int32_t *ovf;         // eight per bucket (eighths): 1 when a list did not fit
};

// The density term of a pair, shared by the walk and the list pass.
__device__ __forceinline__ float density_term(float mj, double dx, double dy, double dz, double r2,
                                              double tt) {
#pragma clang fp contract(off)
    PairGeom g = pair_geom(dx, dy, dz, r2, tt);
    float h3 = g.hinv * g.hinv * g.hinv;
    return mj * (SPHX_SIGMA_F * h3 * w_shape(g.r, g.hinv, g.q));
}

// Sums of the softened pairs' gravity (sphx_soft_factor), without G.
struct SoftSum {
    KahanF x, y, z;
    __device__ __forceinline__ void init() { x.init(); y.init(); z.init(); }
    static __device__ __forceinline__ float factor(float mj, double r2, double hi, double hj) {
#pragma clang fp contract(off)
        return -mj * sphx_soft_factor((float)r2, (float)hi + (float)hj);
    }
    __device__ __forceinline__ void add(float mj, double dx, double dy, double dz, double r2, double hi,
                                        double hj) {
#pragma clang fp contract(off)
        const float s = factor(mj, r2, hi, hj);
        x.add(s * (float)dx);
        y.add(s * (float)dy);
        z.add(s * (float)dz);
    }
    __device__ __forceinline__ void store(const Soa &s, int i) const {
        s.gx[i] = x.value();
        s.gy[i] = y.value();
        s.gz[i] = z.value();
    }
};

// rho and EOS of particle i, and what the pair passes stage of them for a
// neighbour.
__device__ __forceinline__ void density_store(const Soa &s, const DensArgs &a, int i,
                                              const KahanF &acc) {
    double rho = acc.value();
    double u = s.u[i];
    double P = (a.gamma - 1.0) * rho * u;
    double c = sqrt(a.gamma * (a.gamma - 1.0) * u);
    s.rho[i] = rho;
    s.P[i] = P;
    s.c[i] = c;
    if (a.rec) {
        a.rec[i].rho = (float)rho;
        a.rec[i].pr = (float)(P / (rho * rho));
        a.rec[i].c = (float)c;
    }
}

// Density and EOS of the particles of bucket b by the candidate walk.
template <bool SOFT>
__device__ __forceinline__ void density_bucket(const Tables &t, const Soa &s, const DensArgs &a,
                                               int b) {
    __shared__ double sx[64], sy[64], sz[64], sh[64];
    __shared__ float sm[64];
    int lane = threadIdx.x;
    int cnt = t.b_cnt[b];
    int i = t.b_beg[b] + lane;
    bool ok = lane < cnt;
    double xi = ok ? s.x[i] : 0.0, yi = ok ? s.y[i] : 0.0, zi = ok ? s.z[i] : 0.0;
    double hi = ok ? s.h[i] : 0.0;
    double hI = t.bhmax[b];
    const double ib[6] = {t.bxl[b], t.bxh[b], t.byl[b], t.byh[b], t.bzl[b], t.bzh[b]};
    KahanF acc;
    acc.init();
    SoftSum soft;
    soft.init();
    int nn = 0;
    int ncand = 0;
    const int r = t.b_run[b];
    const uint64_t cuts = bucket_cuts(t, r, i, ok, lane);
    for (int g0 = 0; g0 < cnt;) {
      const int g1 = seg_end(cuts, g0, cnt);
      const bool mine = lane >= g0 && lane < g1;
      double gb[6], hS;
      if (cuts) {
          seg_box(ok && mine, xi, yi, zi, hi, gb, &hS);
      } else {
          for (int k = 0; k < 6; ++k) gb[k] = ib[k];
          hS = hI;
      }
      g0 = g1;
      struct Cand {
          double x, y, z, h, m;
          int n;
      };
      for_candidates_pf(
        t, r, gb, lane, [&](int S) { return hS + t.shmax[S]; }, [&](int J) { return hS + t.bhmax[J]; },
        [&](int, int jb, int jc) {
            Cand c{0.0, 0.0, 0.0, 0.0, 0.0, jc};
            if (lane < jc) {
                c.x = s.x[jb + lane];
                c.y = s.y[jb + lane];
                c.z = s.z[jb + lane];
                c.h = s.h[jb + lane];
                c.m = s.m[jb + lane];
            }
            return c;
        },
        [&](int, const Cand &c) {
            ++ncand;
            double xj = c.x, yj = c.y, zj = c.z, hj = c.h;
            bool keep = false;
            if (lane < c.n) keep = near_box(gb, xj, yj, zj, hS + hj);
            Kept k = keep_mask(keep, lane);
            if (k.n == 0) return;
            __syncthreads();
            if (keep) {
                sx[k.slot] = xj;
                sy[k.slot] = yj;
                sz[k.slot] = zj;
                sh[k.slot] = hj;
                sm[k.slot] = (float)c.m;
            }
            __syncthreads();
            // candidates four at a time, their LDS loads issued before the tests
            // (each pair is met in the same order as one at a time)
            auto pair = [&](int q, double dx, double dy, double dz, double r2, double tt, double hj) {
                    acc.add(density_term(sm[q], dx, dy, dz, r2, tt));
                    if (SOFT) soft.add(sm[q], dx, dy, dz, r2, hi, hj);
                    ++nn;
                };
            int q0 = 0;
            for (; q0 + 4 <= k.n; q0 += 4) {
                double cx[4], cy[4], cz[4], ch[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    cx[u] = sx[q0 + u]; cy[u] = sy[q0 + u]; cz[u] = sz[q0 + u]; ch[u] = sh[q0 + u];
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    double dx = xi - cx[u], dy = yi - cy[u], dz = zi - cz[u];
                    double r2 = sphx_r2(dx, dy, dz);
                    double tt = hi + ch[u];
                    if (mine && r2 <= sphx_sq(tt)) pair(q0 + u, dx, dy, dz, r2, tt, ch[u]);
                }
            }
            for (int q = q0; q < k.n; ++q) {
                double dx = xi - sx[q], dy = yi - sy[q], dz = zi - sz[q];
                double r2 = sphx_r2(dx, dy, dz);
                double tt = hi + sh[q];
                if (mine && r2 <= sphx_sq(tt)) pair(q, dx, dy, dz, r2, tt, sh[q]);
            }
        });
    }
    if (ok) {
        density_store(s, a, i, acc);
        if (SOFT) soft.store(s, i);
        if (a.nsym) a.nsym[i] = nn;
    }
    if (lane == 0 && a.counters)
        atomicAdd((unsigned long long *)&a.counters[CNT_CAND], (unsigned long long)ncand);
}

template <bool SOFT>
__global__ __launch_bounds__(64) void k_density(Tables t, Soa s, DensArgs a) {
    density_bucket<SOFT>(t, s, a, t.boff + xcd_block(blockIdx.x, gridDim.x));
}

// Neighbour lists: the candidates with r_ij^2 <= (h_i + h_j)^2 of every
// particle, in increasing order, and the geometric half of its PairRec.  The
// density, div/curl and hydro sums iterate these lists, one lane a particle: in
// the walk a pair's terms ran across the wave for every candidate that any of
// its 64 lanes accepted (about 600 for the 64 to 80 neighbours of a lane).
// Bound as the tile walk is, and by the list stores.
template <int P>
struct ListSink {
    WalkTarget p;
    float fh, band;
    double xi, yi, zi, hi, hS, sc, e;
    const Soa *s;
    int32_t *lst;  // the target's first run of the block: entry k at nbr_slot(k, 0)
    int lane, nn;
    bool act;
    uint32_t m0, m1;
    float amin;
    __device__ __forceinline__ bool full() const { return __any(nn > SPHX_NBR_MAX); }
    __device__ __forceinline__ ListSink(const WalkFrame &f, bool act_, double x, double y, double z,
                                        double h, double hS_, const Soa *s_, int32_t *lst_, int lane_,
                                        int nn_)
        : fh(act_ ? (float)(h * f.sc) : 0.0f), xi(x), yi(y), zi(z), hi(h), hS(hS_), sc(f.sc),
          e(fmax(fmax(f.ex, f.ey), f.ez)), s(s_), lst(lst_), lane(lane_), nn(nn_), act(act_) {
        p.set(f, act, x, y, z);
    }
    __device__ __forceinline__ void chunk(double hc, bool ex) {
        const double S = (hi + hc) * sc, M = e + 1.001 * (hS + hc) * sc;
        band = ex ? INFINITY : (act ? walk_band(S, M) : -1.0f);
    }
    __device__ __forceinline__ void begin() { m0 = m1 = 0u; amin = INFINITY; }
    __device__ __forceinline__ void word() { m0 = m1; m1 = 0u; }
    __device__ __forceinline__ void cand(float cx, float cy, float cz, float ch) {
        const float dx = cx - p.x, dy = cy - p.y, dz = cz - p.z, tt = ch + fh;
        const float r2 = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz));
        const float d = __builtin_fmaf(-tt, tt, r2);
        m1 = sign_in(m1, d);
        amin = fminf(amin, fabsf(d));
    }
    template <class LDS>
    __device__ __forceinline__ void batch(const LDS &L, int base, int n, int q0) {
        constexpr int Q = 64 / P;
        if (__any(amin <= band)) {
            m0 = m1 = 0u;
            for (int k = 0; k < Q; ++k) {
                if (P == 1 && k == 32) word();
                m1 <<= 1;
                if (act && q0 + k < n) {
                    const int j = L.j[base + q0 + k];
                    const double r2 = sphx_r2(xi - s->x[j], yi - s->y[j], zi - s->z[j]);
                    m1 |= r2 <= sphx_sq(hi + s->h[j]) ? 1u : 0u;
                }
            }
        }
        uint32_t w[2] = {m0, m1};
        int tot;
        int at = nn + slice_scan<P>(__popc(m0) + __popc(m1), lane, &tot);
#pragma unroll
        for (int v = P == 1 ? 0 : 1; v < 2; ++v) {
            const int last = P == 1 ? 32 * v + 31 : Q - 1;
            while (w[v]) {
                const int k = 31 - __builtin_clz(w[v]);
                w[v] &= ~(1u << k);
                if (at < SPHX_NBR_MAX) lst[((at >> 3) << 9) | (at & 7)] = L.j[base + q0 + last - k];
                ++at;
            }
        }
        nn += tot;
    }
};

template <int P>
__global__ __launch_bounds__(64) void k_lists(Tables t, Soa s, DensArgs a) {
    constexpr int T = 64 / P;
    __shared__ WalkLds<true> L;
    const WalkSlot ws = walk_slot<P>(t);
    const int lane = threadIdx.x, tl = lane & (T - 1);
    const int b = ws.b, cnt = ws.cnt;
    const int i = ws.first + tl;
    const bool ok = tl < cnt;
    const double xi = ok ? s.x[i] : 0.0, yi = ok ? s.y[i] : 0.0, zi = ok ? s.z[i] : 0.0;
    const double hi = ok ? s.h[i] : 0.0;
    const int r = t.b_run[b];
    const uint64_t cuts = bucket_cuts(t, r, i, ok && lane < T, lane);
    const bool fin = fabs(xi) < INFINITY && fabs(yi) < INFINITY && fabs(zi) < INFINITY && hi == hi;
    int32_t *lst = a.lst + (int64_t)b * SPHX_NBR_MAX * 64 + (ws.bl0 + tl) * 8;
    int nn = 0, ncand = 0;
    for (int g0 = 0; g0 < cnt;) {
        const int g1 = seg_end(cuts, g0, cnt);
        const bool mine = ok && tl >= g0 && tl < g1;
        g0 = g1;
        double gb[6], hS;
        seg_box(mine, xi, yi, zi, hi, gb, &hS);
        const WalkFrame f = walk_frame(gb, hS);
        ListSink<P> sink(f, mine && fin, xi, yi, zi, hi, hS, &s, lst, lane, 0);
        ncand += tile_walk<P, true>(t, s, L, r, lane, gb, hS, f, sink);
        if (mine) nn = sink.nn;
    }
    if (ok && lane < T) {
        if (a.nsym) a.nsym[i] = nn;
        PairRec *q = a.rec + i;
        q->x = xi; q->y = yi; q->z = zi; q->h = hi;
        q->vx = s.vx[i]; q->vy = s.vy[i]; q->vz = s.vz[i];
        q->m = (float)s.m[i];
        q->len = nn;
        q->pad = 0;
    }
    // eight flags per bucket, one per eighth
    const uint64_t o = __ballot(ok && nn > SPHX_NBR_MAX);
    if (lane < 8 / P) a.ovf[8 * b + (8 / P) * ws.part + lane] = o ? 1 : 0;
    if (lane == 0 && a.counters)
        atomicAdd((unsigned long long *)&a.counters[CNT_CAND], (unsigned long long)ncand);
}

// Whether an eighth of bucket b has a list that overflowed.
__device__ __forceinline__ bool bucket_ovf(const int32_t *ovf, int64_t b) {
    const int4 o = reinterpret_cast<const int4 *>(ovf)[2 * b], p = reinterpret_cast<const int4 *>(ovf)[2 * b + 1];
    return (o.x | o.y | o.z | o.w | p.x | p.y | p.z | p.w) != 0;
}

// Value of v in lane U of this lane's quad.
template <int U>
__device__ __forceinline__ float quad_from(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), U * 0x55, 0xf, 0xf, true));
}

template <int U>
__device__ __forceinline__ Terms4 quad_from(const Terms4 &t) {
    return {quad_from<U>(t.a), quad_from<U>(t.b), quad_from<U>(t.c), quad_from<U>(t.d)};
}

// Density and EOS over the lists, four lanes a particle and 16 particles a
// wave: a lane evaluates every fourth entry (eight entries a round, their
// gathers of 36 of a record's 80 bytes issued together), and the terms are
// added in list order from the quad's lanes, so that the sums are the walk's.
// Bound: in small runs the chain of the one wave on a SIMD (a VALU instruction
// every eight cycles or so), in large ones the latency and address rate of the
// gathers, for which two loads in flight a lane leave 50 registers and eight
// waves a SIMD.  Against one lane a particle with eight loads in flight (106
// registers, four waves; with the softening sums up to 131,072): 39 -> 18 us at
// 4,096 particles, 88 -> 75 at 65,752, 397 -> 344 at 1,048,576.
template <bool SOFT, bool WALK>
__global__ __launch_bounds__(64) void k_density_quad(Tables t, Soa s, DensArgs a) {
    const int g = xcd_block(blockIdx.x, gridDim.x), b = t.boff + (g >> 2);
    const int lane = threadIdx.x, tl = 16 * (g & 3) + (lane >> 2), u = lane & 3;
    if (bucket_ovf(a.ovf, b)) {
        if (!WALK || (g & 3)) return;
        if (lane == 0 && a.counters) atomicAdd((unsigned long long *)&a.counters[CNT_NBR_OVF], 1ull);
        density_bucket<SOFT>(t, s, a, b);
        return;
    }
    const bool ok = tl < t.b_cnt[b];
    const int i = t.b_beg[b] + tl;
    double xi = 0.0, yi = 0.0, zi = 0.0, hi = 0.0;
    int len = 0;
    if (ok) {
        const PairRec *q = a.rec + i;
        xi = q->x; yi = q->y; zi = q->z; hi = q->h;
        len = q->len;
    }
    const int maxlen = wave_max_i(len);
    const int32_t *lp = a.lst + (int64_t)b * SPHX_NBR_MAX * 64;
    KahanF acc;
    acc.init();
    SoftSum soft;
    soft.init();
    for (int k0 = 0; k0 < maxlen; k0 += 8) {
        float w[2] = {0.0f, 0.0f}, gx[2] = {0.0f, 0.0f}, gy[2] = {0.0f, 0.0f}, gz[2] = {0.0f, 0.0f};
#pragma unroll
        for (int v = 0; v < 2; ++v) {
            const int k = k0 + 4 * v + u;
            if (k < len) {
#pragma clang fp contract(off)
                const PairRec *q = a.rec + lp[nbr_slot(k, tl)];
                const double2 p0 = reinterpret_cast<const double2 *>(q)[0];
                const double2 p1 = reinterpret_cast<const double2 *>(q)[1];
                const float m = q->m;
                const double dx = xi - p0.x, dy = yi - p0.y, dz = zi - p1.x;
                const double r2 = sphx_r2(dx, dy, dz);
                w[v] = density_term(m, dx, dy, dz, r2, hi + p1.y);
                if (SOFT) {
                    const float f = SoftSum::factor(m, r2, hi, p1.y);
                    gx[v] = f * (float)dx;
                    gy[v] = f * (float)dy;
                    gz[v] = f * (float)dz;
                }
            }
        }
#pragma unroll
        for (int v = 0; v < 2; ++v) {
            auto add = [&](int k, float aw, float ax, float ay, float az) {
                if (k < len) {
                    acc.add(aw);
                    if (SOFT) {
                        soft.x.add(ax);
                        soft.y.add(ay);
                        soft.z.add(az);
                    }
                }
            };
            const int k = k0 + 4 * v;
            add(k, quad_from<0>(w[v]), quad_from<0>(gx[v]), quad_from<0>(gy[v]), quad_from<0>(gz[v]));
            add(k + 1, quad_from<1>(w[v]), quad_from<1>(gx[v]), quad_from<1>(gy[v]), quad_from<1>(gz[v]));
            add(k + 2, quad_from<2>(w[v]), quad_from<2>(gx[v]), quad_from<2>(gy[v]), quad_from<2>(gz[v]));
            add(k + 3, quad_from<3>(w[v]), quad_from<3>(gx[v]), quad_from<3>(gy[v]), quad_from<3>(gz[v]));
        }
    }
    if (ok && u == 0) {
        density_store(s, a, i, acc);
        if (SOFT) soft.store(s, i);
    }
}

// Calls f for the wave's bucket if its lists overflowed.  A wave a bucket: runs
// whose lists all overflow (wide h, many neighbours) fill the device.  With 64
// consecutive buckets a wave, density with 500 neighbours took 23 ms at 65,752
// particles, of which these walks take 0.5.
template <class F>
__device__ __forceinline__ void if_overflowed(const Tables &t, const int32_t *ovf, F f) {
    const int b = t.boff + xcd_block(blockIdx.x, gridDim.x);
    if (bucket_ovf(ovf, b)) f(b);
}

// The walk for the buckets whose lists overflowed.
template <bool SOFT>
__global__ __launch_bounds__(64) void k_density_ovf(Tables t, Soa s, DensArgs a) {
    if_overflowed(t, a.ovf, [&](int b) {
        if (threadIdx.x == 0 && a.counters) atomicAdd((unsigned long long *)&a.counters[CNT_NBR_OVF], 1ull);
        density_bucket<SOFT>(t, s, a, b);
    });
}

__device__ __forceinline__ void divcurl_store(const Soa &s, int i, bool ok, const KahanF &kd,
                                              const KahanF &kx, const KahanF &ky,
                                              const KahanF &kz) {
    if (ok) {
        double ir = 1.0 / s.rho[i];
        s.divv[i] = -kd.value() * ir;
        double cx = kx.value() * ir, cy = ky.value() * ir, cz = kz.value() * ir;
        s.curlv[i] = sqrt(cx * cx + cy * cy + cz * cz);
    }
}

// div/curl of the particles of bucket b by the candidate walk.
__device__ __forceinline__ void divcurl_bucket(const Tables &t, const Soa &s, int b) {
    __shared__ double sx[64], sy[64], sz[64], sh[64], svx[64], svy[64], svz[64];
    __shared__ float sm[64];
    int lane = threadIdx.x;
    int cnt = t.b_cnt[b];
    int i = t.b_beg[b] + lane;
    bool ok = lane < cnt;
    double xi = ok ? s.x[i] : 0.0, yi = ok ? s.y[i] : 0.0, zi = ok ? s.z[i] : 0.0;
    double hi = ok ? s.h[i] : 0.0;
    double vxi = ok ? s.vx[i] : 0.0, vyi = ok ? s.vy[i] : 0.0, vzi = ok ? s.vz[i] : 0.0;
    double hI = t.bhmax[b];
    const double ib[6] = {t.bxl[b], t.bxh[b], t.byl[b], t.byh[b], t.bzl[b], t.bzh[b]};
    KahanF kd, kx, ky, kz;
    kd.init(); kx.init(); ky.init(); kz.init();
    const int r = t.b_run[b];
    const uint64_t cuts = bucket_cuts(t, r, i, ok, lane);
    for (int g0 = 0; g0 < cnt;) {
      const int g1 = seg_end(cuts, g0, cnt);
      const bool mine = lane >= g0 && lane < g1;
      double gb[6], hS;
      if (cuts) {
          seg_box(ok && mine, xi, yi, zi, hi, gb, &hS);
      } else {
          for (int k = 0; k < 6; ++k) gb[k] = ib[k];
          hS = hI;
      }
      g0 = g1;
      for_candidates(
        t, r, gb, lane, [&](int S) { return hS + t.shmax[S]; }, [&](int J) { return hS + t.bhmax[J]; },
        [&](int J) {
            int jc = t.b_cnt[J], j0 = t.b_beg[J];
            int j = j0 + lane;
            double xj = 0.0, yj = 0.0, zj = 0.0, hj = 0.0;
            bool keep = false;
            if (lane < jc) {
                xj = s.x[j]; yj = s.y[j]; zj = s.z[j]; hj = s.h[j];
                keep = near_box(gb, xj, yj, zj, hS + hj);
            }
            Kept k = keep_mask(keep, lane);
            if (k.n == 0) return;
            __syncthreads();
            if (keep) {
                int q = k.slot;
                sx[q] = xj; sy[q] = yj; sz[q] = zj; sh[q] = hj;
                svx[q] = s.vx[j]; svy[q] = s.vy[j]; svz[q] = s.vz[j];
                sm[q] = (float)s.m[j];
            }
            __syncthreads();
            // candidates four at a time, their LDS loads issued before the tests
            // (each pair is met in the same order as one at a time)
            auto pair = [&](int q, double dx, double dy, double dz, double r2, double tt) {
                    divcurl_pair(vxi, vyi, vzi, svx[q], svy[q], svz[q], sm[q], dx, dy, dz, r2,
                                 tt, kd, kx, ky, kz);
                };
            int q0 = 0;
            for (; q0 + 4 <= k.n; q0 += 4) {
                double cx[4], cy[4], cz[4], ch[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    cx[u] = sx[q0 + u]; cy[u] = sy[q0 + u]; cz[u] = sz[q0 + u]; ch[u] = sh[q0 + u];
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    double dx = xi - cx[u], dy = yi - cy[u], dz = zi - cz[u];
                    double r2 = sphx_r2(dx, dy, dz);
                    double tt = hi + ch[u];
                    if (mine && r2 <= sphx_sq(tt)) pair(q0 + u, dx, dy, dz, r2, tt);
                }
            }
            for (int q = q0; q < k.n; ++q) {
                double dx = xi - sx[q], dy = yi - sy[q], dz = zi - sz[q];
                double r2 = sphx_r2(dx, dy, dz);
                double tt = hi + sh[q];
                if (mine && r2 <= sphx_sq(tt)) pair(q, dx, dy, dz, r2, tt);
            }
        });
    }
    divcurl_store(s, i, ok, kd, kx, ky, kz);
}

__global__ __launch_bounds__(64) void k_divcurl(Tables t, Soa s) {
    divcurl_bucket(t, s, t.boff + xcd_block(blockIdx.x, gridDim.x));
}

// Hydro acceleration and du/dt of the particles of bucket b by the candidate walk.
__device__ __forceinline__ void hydro_bucket(const Tables &t, const Soa &s, const HydroArgs &a,
                                             int b, bool add_g = false) {
    __shared__ double sx[64], sy[64], sz[64], sh[64], svx[64], svy[64], svz[64];
    __shared__ float sm[64], srho[64], spr[64], sc[64], sf[64];
    int lane = threadIdx.x;
    int cnt = t.b_cnt[b];
    int i = t.b_beg[b] + lane;
    bool ok = lane < cnt;
    double xi = ok ? s.x[i] : 0.0, yi = ok ? s.y[i] : 0.0, zi = ok ? s.z[i] : 0.0;
    double hi = ok ? s.h[i] : 0.0;
    HydroI I;
    I.vx = ok ? s.vx[i] : 0.0;
    I.vy = ok ? s.vy[i] : 0.0;
    I.vz = ok ? s.vz[i] : 0.0;
    I.rho = ok ? (float)s.rho[i] : 1.0f;
    I.pr = ok ? (float)(s.P[i] / (s.rho[i] * s.rho[i])) : 0.0f;
    I.c = ok ? (float)s.c[i] : 0.0f;
    I.f = (ok && a.balsara) ? (float)balsara_f(s.divv[i], s.curlv[i], s.c[i], s.h[i]) : 1.0f;
    double hI = t.bhmax[b];
    const double ib[6] = {t.bxl[b], t.bxh[b], t.byl[b], t.byh[b], t.bzl[b], t.bzh[b]};
    KahanF kx, ky, kz, kdu;
    kx.init(); ky.init(); kz.init(); kdu.init();
    const int r = t.b_run[b];
    const uint64_t cuts = bucket_cuts(t, r, i, ok, lane);
    for (int g0 = 0; g0 < cnt;) {
      const int g1 = seg_end(cuts, g0, cnt);
      const bool mine = lane >= g0 && lane < g1;
      double gb[6], hS;
      if (cuts) {
          seg_box(ok && mine, xi, yi, zi, hi, gb, &hS);
      } else {
          for (int k = 0; k < 6; ++k) gb[k] = ib[k];
          hS = hI;
      }
      g0 = g1;
      for_candidates(
        t, r, gb, lane, [&](int S) { return hS + t.shmax[S]; }, [&](int J) { return hS + t.bhmax[J]; },
        [&](int J) {
            int jc = t.b_cnt[J], j0 = t.b_beg[J];
            int j = j0 + lane;
            double xj = 0.0, yj = 0.0, zj = 0.0, hj = 0.0;
            bool keep = false;
            if (lane < jc) {
                xj = s.x[j]; yj = s.y[j]; zj = s.z[j]; hj = s.h[j];
                keep = near_box(gb, xj, yj, zj, hS + hj);
            }
            Kept k = keep_mask(keep, lane);
            if (k.n == 0) return;
            __syncthreads();
            if (keep) {
                int q = k.slot;
                sx[q] = xj; sy[q] = yj; sz[q] = zj; sh[q] = hj;
                svx[q] = s.vx[j]; svy[q] = s.vy[j]; svz[q] = s.vz[j];
                double rj = s.rho[j];
                sm[q] = (float)s.m[j];
                srho[q] = (float)rj;
                spr[q] = (float)(s.P[j] / (rj * rj));
                sc[q] = (float)s.c[j];
                sf[q] = a.balsara ? (float)balsara_f(s.divv[j], s.curlv[j], s.c[j], s.h[j]) : 1.0f;
            }
            __syncthreads();
            // candidates four at a time, their LDS loads issued before the tests
            // (each pair is met in the same order as one at a time)
            auto pair = [&](int q, double dx, double dy, double dz, double r2, double tt) {
                    hydro_pair(a, I, svx[q], svy[q], svz[q], sm[q], srho[q], spr[q], sc[q],
                               sf[q], dx, dy, dz, r2, tt, kx, ky, kz, kdu);
                };
            int q0 = 0;
            for (; q0 + 4 <= k.n; q0 += 4) {
                double cx[4], cy[4], cz[4], ch[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    cx[u] = sx[q0 + u]; cy[u] = sy[q0 + u]; cz[u] = sz[q0 + u]; ch[u] = sh[q0 + u];
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    double dx = xi - cx[u], dy = yi - cy[u], dz = zi - cz[u];
                    double r2 = sphx_r2(dx, dy, dz);
                    double tt = hi + ch[u];
                    if (mine && r2 <= sphx_sq(tt)) pair(q0 + u, dx, dy, dz, r2, tt);
                }
            }
            for (int q = q0; q < k.n; ++q) {
                double dx = xi - sx[q], dy = yi - sy[q], dz = zi - sz[q];
                double r2 = sphx_r2(dx, dy, dz);
                double tt = hi + sh[q];
                if (mine && r2 <= sphx_sq(tt)) pair(q, dx, dy, dz, r2, tt);
            }
        });
    }
    if (ok) {
        // add_g: the total acceleration, gravity + a_sph, as sphx_combine adds it
        s.ax[i] = add_g ? s.gx[i] + kx.value() : kx.value();
        s.ay[i] = add_g ? s.gy[i] + ky.value() : ky.value();
        s.az[i] = add_g ? s.gz[i] + kz.value() : kz.value();
        s.du[i] = kdu.value();
    }
}

__global__ __launch_bounds__(64) void k_hydro(Tables t, Soa s, HydroArgs a) {
    hydro_bucket(t, s, a, t.boff + xcd_block(blockIdx.x, gridDim.x));
}

// ---------------------------------------------------------------------------
// Neighbour-list passes.  The density walk records, for every particle, the
// indices of the particles it accepted (r_ij^2 <= (h_i + h_j)^2) in the order
// it met them, and a record of the values the pair passes stage for a
// neighbour.  Positions and h do not change between the density pass and the
// hydro pass of a step, and div/curl and hydro accept exactly the pairs density
// accepts, so iterating a particle's list visits the same pairs in the same
// order as the candidate walk: with the shared pair terms the sums are
// bit-identical, without the walk's candidate tests or its wave-wide pair
// evaluations for candidates that only some lanes accept.  Buckets where a list
// overflowed (more than SPHX_NBR_MAX neighbours) are left to the walk.
// ---------------------------------------------------------------------------
struct ListArgs {
    const int32_t *lst;
    const PairRec *rec;
    const int32_t *ovf;
    const float *fbal;   // Balsara factor per particle (hydro with the switch on)
};

__device__ __forceinline__ double rec_dbl(uint32_t lo, uint32_t hi) {
    return __hiloint2double((int)hi, (int)lo);
}

// The position, h, velocity and mass of record j (four 16-byte loads).
struct RecA {
    double x, y, z, h, vx, vy, vz;
    float m, rho;
};
__device__ __forceinline__ RecA load_rec_a(const PairRec *rec, int j) {
    const uint4 *q = reinterpret_cast<const uint4 *>(rec + j);
    uint4 a = q[0], b = q[1], c = q[2], d = q[3];
    RecA o;
    o.x = rec_dbl(a.x, a.y); o.y = rec_dbl(a.z, a.w);
    o.z = rec_dbl(b.x, b.y); o.h = rec_dbl(b.z, b.w);
    o.vx = rec_dbl(c.x, c.y); o.vy = rec_dbl(c.z, c.w);
    o.vz = rec_dbl(d.x, d.y);
    o.m = __uint_as_float(d.z); o.rho = __uint_as_float(d.w);
    return o;
}
// P / rho^2, sound speed and list length of record j (the fifth 16 bytes).
__device__ __forceinline__ uint4 load_rec_b(const PairRec *rec, int j) {
    return reinterpret_cast<const uint4 *>(rec + j)[4];
}

__global__ __launch_bounds__(64) void k_divcurl_list(Tables t, Soa s, ListArgs L) {
    const int b = t.boff + xcd_block(blockIdx.x, gridDim.x);
    if (bucket_ovf(L.ovf, b)) return;  // the walk launch takes this bucket
    const int lane = threadIdx.x;
    const int cnt = t.b_cnt[b];
    const int i = t.b_beg[b] + lane;
    const bool ok = lane < cnt;
    RecA me{};
    int len = 0;
    if (ok) {
        me = load_rec_a(L.rec, i);
        len = (int)load_rec_b(L.rec, i).z;
    }
    const int maxlen = wave_max_i(len);
    const int32_t *lp = L.lst + (int64_t)b * SPHX_NBR_MAX * 64;
    KahanF kd, kx, ky, kz;
    kd.init(); kx.init(); ky.init(); kz.init();
    for_list(lp, lane, len, maxlen, ok ? i : 0, [&](int j) { return load_rec_a(L.rec, j); },
             [&](const RecA &o) {
        double dx = me.x - o.x, dy = me.y - o.y, dz = me.z - o.z;
        double r2 = sphx_r2(dx, dy, dz);
        double tt = me.h + o.h;
        divcurl_pair(me.vx, me.vy, me.vz, o.vx, o.vy, o.vz, o.m, dx, dy, dz, r2, tt, kd, kx, ky,
                     kz);
    });
    divcurl_store(s, i, ok, kd, kx, ky, kz);
}

__global__ __launch_bounds__(64) void k_hydro_list(Tables t, Soa s, HydroArgs a, ListArgs L) {
    const int b = t.boff + xcd_block(blockIdx.x, gridDim.x);
    if (bucket_ovf(L.ovf, b)) return;  // the walk launch takes this bucket
    const int lane = threadIdx.x;
    const int cnt = t.b_cnt[b];
    const int i = t.b_beg[b] + lane;
    const bool ok = lane < cnt;
    RecA me{};
    HydroI I;
    I.vx = I.vy = I.vz = 0.0;
    I.rho = 1.0f; I.pr = 0.0f; I.c = 0.0f; I.f = 1.0f;
    int len = 0;
    if (ok) {
        me = load_rec_a(L.rec, i);
        uint4 e = load_rec_b(L.rec, i);
        I.vx = me.vx; I.vy = me.vy; I.vz = me.vz;
        I.rho = me.rho;
        I.pr = __uint_as_float(e.x);
        I.c = __uint_as_float(e.y);
        if (a.balsara) I.f = L.fbal[i];
        len = (int)e.z;
    }
    const int maxlen = wave_max_i(len);
    const int32_t *lp = L.lst + (int64_t)b * SPHX_NBR_MAX * 64;
    KahanF kx, ky, kz, kdu;
    kx.init(); ky.init(); kz.init(); kdu.init();
    struct Rec {
        RecA o;
        uint4 e;
        float fj;
    };
    for_list(lp, lane, len, maxlen, ok ? i : 0,
             [&](int j) {
                 return Rec{load_rec_a(L.rec, j), load_rec_b(L.rec, j), a.balsara ? L.fbal[j] : 1.0f};
             },
             [&](const Rec &R) {
        const RecA &o = R.o;
        const uint4 &e = R.e;
        const float fj = R.fj;
        double dx = me.x - o.x, dy = me.y - o.y, dz = me.z - o.z;
        double r2 = sphx_r2(dx, dy, dz);
        double tt = me.h + o.h;
        hydro_pair(a, I, o.vx, o.vy, o.vz, o.m, o.rho, __uint_as_float(e.x), __uint_as_float(e.y),
                   fj, dx, dy, dz, r2, tt, kx, ky, kz, kdu);
    });
    if (ok) {
        s.ax[i] = kx.value();
        s.ay[i] = ky.value();
        s.az[i] = kz.value();
        s.du[i] = kdu.value();
    }
}

// div/curl and hydro of bucket b in one list pass, for steps without the
// Balsara switch (hydro then reads nothing div/curl produces): each
// neighbour's record is gathered once for both, and each of the eight sums
// meets its pairs in the list order, as the two separate passes do, so the
// results are the same.  The stored acceleration is the total, gravity +
// a_sph, added as sphx_combine adds it.
__device__ __forceinline__ void dchydro_bucket(const Tables &t, const Soa &s, const HydroArgs &a,
                                               const ListArgs &L, int b) {
    if (bucket_ovf(L.ovf, b)) return;  // the walk launches take this bucket
    const int lane = threadIdx.x;
    const int cnt = t.b_cnt[b];
    const int i = t.b_beg[b] + lane;
    const bool ok = lane < cnt;
    RecA me{};
    HydroI I;
    I.vx = I.vy = I.vz = 0.0;
    I.rho = 1.0f; I.pr = 0.0f; I.c = 0.0f; I.f = 1.0f;
    int len = 0;
    if (ok) {
        me = load_rec_a(L.rec, i);
        uint4 e = load_rec_b(L.rec, i);
        I.vx = me.vx; I.vy = me.vy; I.vz = me.vz;
        I.rho = me.rho;
        I.pr = __uint_as_float(e.x);
        I.c = __uint_as_float(e.y);
        len = (int)e.z;
    }
    const int maxlen = wave_max_i(len);
    const int32_t *lp = L.lst + (int64_t)b * SPHX_NBR_MAX * 64;
    KahanF kd, kx, ky, kz, hx, hy, hz, hdu;
    kd.init(); kx.init(); ky.init(); kz.init();
    hx.init(); hy.init(); hz.init(); hdu.init();
    struct Rec {
        RecA o;
        uint4 e;
    };
    for_list(lp, lane, len, maxlen, ok ? i : 0,
             [&](int j) { return Rec{load_rec_a(L.rec, j), load_rec_b(L.rec, j)}; },
             [&](const Rec &R) {
        const RecA &o = R.o;
        const uint4 &e = R.e;
        double dx = me.x - o.x, dy = me.y - o.y, dz = me.z - o.z;
        double r2 = sphx_r2(dx, dy, dz);
        double tt = me.h + o.h;
        divcurl_pair(me.vx, me.vy, me.vz, o.vx, o.vy, o.vz, o.m, dx, dy, dz, r2, tt, kd, kx, ky,
                     kz);
        hydro_pair(a, I, o.vx, o.vy, o.vz, o.m, o.rho, __uint_as_float(e.x), __uint_as_float(e.y),
                   1.0f, dx, dy, dz, r2, tt, hx, hy, hz, hdu);
    });
    divcurl_store(s, i, ok, kd, kx, ky, kz);
    if (ok) {
        s.ax[i] = s.gx[i] + hx.value();
        s.ay[i] = s.gy[i] + hy.value();
        s.az[i] = s.gz[i] + hz.value();
        s.du[i] = hdu.value();
    }
}

__global__ __launch_bounds__(64) void k_dchydro_list(Tables t, Soa s, HydroArgs a, ListArgs L) {
    dchydro_bucket(t, s, a, L, t.boff + xcd_block(blockIdx.x, gridDim.x));
}

// The same with four lanes a particle (see k_density_quad), the walks of an
// overflowed bucket included.  37.5 -> 23 us at 4,096 particles, and the
// overflow launch (4.5 us) gone.
__global__ __launch_bounds__(64) void k_dchydro_quad(Tables t, Soa s, HydroArgs a, ListArgs L) {
    const int g = xcd_block(blockIdx.x, gridDim.x), b = t.boff + (g >> 2);
    const int lane = threadIdx.x, tl = 16 * (g & 3) + (lane >> 2), u = lane & 3;
    if (bucket_ovf(L.ovf, b)) {
        if (g & 3) return;
        divcurl_bucket(t, s, b);
        hydro_bucket(t, s, a, b, true);
        return;
    }
    const bool ok = tl < t.b_cnt[b];
    const int i = t.b_beg[b] + tl;
    RecA me{};
    HydroI I;
    I.vx = I.vy = I.vz = 0.0;
    I.rho = 1.0f; I.pr = 0.0f; I.c = 0.0f; I.f = 1.0f;
    int len = 0;
    if (ok) {
        me = load_rec_a(L.rec, i);
        uint4 e = load_rec_b(L.rec, i);
        I.vx = me.vx; I.vy = me.vy; I.vz = me.vz;
        I.rho = me.rho;
        I.pr = __uint_as_float(e.x);
        I.c = __uint_as_float(e.y);
        len = (int)e.z;
    }
    const int maxlen = wave_max_i(len);
    const int32_t *lp = L.lst + (int64_t)b * SPHX_NBR_MAX * 64;
    KahanF kd, kx, ky, kz, hx, hy, hz, hdu;
    kd.init(); kx.init(); ky.init(); kz.init();
    hx.init(); hy.init(); hz.init(); hdu.init();
    for (int k0 = 0; k0 < maxlen; k0 += 8) {
        Terms4 d[2] = {}, h[2] = {};
#pragma unroll
        for (int v = 0; v < 2; ++v) {
            const int k = k0 + 4 * v + u;
            if (k < len) {
                const int j = lp[nbr_slot(k, tl)];
                const RecA o = load_rec_a(L.rec, j);
                const uint4 e = load_rec_b(L.rec, j);
                const double dx = me.x - o.x, dy = me.y - o.y, dz = me.z - o.z;
                const double tt = me.h + o.h;
                const PairGeom pg = pair_geom(dx, dy, dz, sphx_r2(dx, dy, dz), tt);
                d[v] = divcurl_terms(me.vx, me.vy, me.vz, o.vx, o.vy, o.vz, o.m, pg);
                h[v] = hydro_terms(a, I, o.vx, o.vy, o.vz, o.m, o.rho, __uint_as_float(e.x),
                                   __uint_as_float(e.y), 1.0f, tt, pg);
            }
        }
#pragma unroll
        for (int v = 0; v < 2; ++v) {
            auto add = [&](int k, const Terms4 &p, const Terms4 &q) {
                if (k < len) {
                    kd.add(p.a); kx.add(p.b); ky.add(p.c); kz.add(p.d);
                    hx.add(q.a); hy.add(q.b); hz.add(q.c); hdu.add(q.d);
                }
            };
            const int k = k0 + 4 * v;
            add(k, quad_from<0>(d[v]), quad_from<0>(h[v]));
            add(k + 1, quad_from<1>(d[v]), quad_from<1>(h[v]));
            add(k + 2, quad_from<2>(d[v]), quad_from<2>(h[v]));
            add(k + 3, quad_from<3>(d[v]), quad_from<3>(h[v]));
        }
    }
    const bool out = ok && u == 0;
    divcurl_store(s, i, out, kd, kx, ky, kz);
    if (out) {
        s.ax[i] = s.gx[i] + hx.value();
        s.ay[i] = s.gy[i] + hy.value();
        s.az[i] = s.gz[i] + hz.value();
        s.du[i] = hdu.value();
    }
}

__global__ __launch_bounds__(64) void k_divcurl_ovf(Tables t, Soa s, const int32_t *ovf) {
    if_overflowed(t, ovf, [&](int b) { divcurl_bucket(t, s, b); });
}

__global__ __launch_bounds__(64) void k_hydro_ovf(Tables t, Soa s, HydroArgs a,
                                                  const int32_t *ovf) {
    if_overflowed(t, ovf, [&](int b) { hydro_bucket(t, s, a, b, false); });
}

// The overflow walks of the fused pass, div/curl and then hydro (which without
// the Balsara switch reads nothing of it), in one launch.
__global__ __launch_bounds__(64) void k_dchydro_ovf(Tables t, Soa s, HydroArgs a,
                                                    const int32_t *ovf) {
    if_overflowed(t, ovf, [&](int b) {
        divcurl_bucket(t, s, b);
        hydro_bucket(t, s, a, b, true);
    });
}

// Balsara factor of every particle of [p0, p1), as the walk computes it.
__global__ void k_fbal(Soa s, int64_t p0, int64_t p1, float *__restrict__ fbal) {
    int64_t i = p0 + (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < p1) fbal[i] = (float)balsara_f(s.divv[i], s.curlv[i], s.c[i], s.h[i]);
}

// The gas half of every particle's record from s.rho, s.P and s.c, as the
// density pass writes it, and with fbal the Balsara factors.
__global__ void k_rec_gas(Soa s, PairRec *__restrict__ rec, int64_t n, float *__restrict__ fbal) {
    int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const double rho = s.rho[i];
    rec[i].rho = (float)rho;
    rec[i].pr = (float)(s.P[i] / (rho * rho));
    rec[i].c = (float)s.c[i];
    if (fbal) fbal[i] = (float)balsara_f(s.divv[i], s.curlv[i], s.c[i], s.h[i]);
}

// kNN smoothing length (do_smoothingX, LIBSX:762-783): h = 0.5 sqrt(v) with v
// the kth smallest r^2 (0-based, self included) from particle i to all
// particles of its run.  Each lane keeps a bracket: lo2 (exclusive, klo
// values <= lo2), up2 (a value with >= kth + 1 values <= it, once known) and
// the probe of the next walk.  A walk counts the values in (lo2, probe] and
// keeps up to KNN_CAP of them in LDS; when the rank falls inside and they
// fit, the value of that rank is selected exactly; otherwise the bracket
// grows (too few) or is bisected in value (too many).  The first probe is the
// radius of a count iteration whose band is [kth + 1, kth + 56], so one walk
// usually suffices.
constexpr int KNN_CAP = 128;

struct KnnArgs {
    int32_t kth;
    int32_t max_walks;
    int64_t *counters;  // lanes left unresolved -> CNT_H_CAPPED
};

__global__ __launch_bounds__(64) void k_knn(Tables t, Soa s, KnnArgs a) {
    __shared__ double sx[64], sy[64], sz[64];
    __shared__ double lst[KNN_CAP * 64];
    int b = t.boff + xcd_block(blockIdx.x, gridDim.x);
    int lane = threadIdx.x;
    int cnt = t.b_cnt[b];
    int i = t.b_beg[b] + lane;
    bool ok = lane < cnt;
    double xi = ok ? s.x[i] : 0.0, yi = ok ? s.y[i] : 0.0, zi = ok ? s.z[i] : 0.0;
    const int r = t.b_run[b];
    const uint64_t cuts = bucket_cuts(t, r, i, ok, lane);
    double lo2 = -1.0, up2 = INFINITY;
    double probe = ok ? sphx_sq(2.0 * s.h[i]) : 0.0;
    int klo = 0;
    bool done = !ok;
    double res = 0.0;
    for (int walk = 0; walk < a.max_walks && __any(!done); ++walk) {
        int cin = 0;
        for (int g0 = 0; g0 < cnt;) {
            const int g1 = seg_end(cuts, g0, cnt);
            const bool mine = lane >= g0 && lane < g1;
            const bool act = mine && !done;
            g0 = g1;
            // a probe of 0 is legitimate (coincident particles): walk whenever
            // a lane of the segment is active; reach 0 still finds the
            // buckets whose box contains the particle
            if (!__any(act)) continue;
            double P = wave_max_d(act ? probe : 0.0);
            double R = sqrt(P);
            double gb[6], hdummy;
            seg_box(ok && mine, xi, yi, zi, 0.0, gb, &hdummy);
            for_candidates(
                t, r, gb, lane, [&](int) { return R; }, [&](int) { return R; },
                [&](int J) {
                    int jc = t.b_cnt[J], j0 = t.b_beg[J];
                    double xj = 0.0, yj = 0.0, zj = 0.0;
                    bool keep = false;
                    if (lane < jc) {
                        xj = s.x[j0 + lane];
                        yj = s.y[j0 + lane];
                        zj = s.z[j0 + lane];
                        keep = near_box(gb, xj, yj, zj, R);
                    }
                    Kept k = keep_mask(keep, lane);
                    if (k.n == 0) return;
                    __syncthreads();
                    if (keep) {
                        sx[k.slot] = xj;
                        sy[k.slot] = yj;
                        sz[k.slot] = zj;
                    }
                    __syncthreads();
                    // candidates four at a time, their LDS loads issued first (the
                    // values are appended in the same order)
                    int q = 0;
                    for (; q + 4 <= k.n; q += 4) {
                        double cx[4], cy[4], cz[4];
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            cx[u] = sx[q + u]; cy[u] = sy[q + u]; cz[u] = sz[q + u];
                        }
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            double v = sphx_r2(cx[u] - xi, cy[u] - yi, cz[u] - zi);
                            if (act && v > lo2 && v <= probe) {
                                if (cin < KNN_CAP) lst[cin * 64 + lane] = v;
                                ++cin;
                            }
                        }
                    }
                    for (; q < k.n; ++q) {
                        double v = sphx_r2(sx[q] - xi, sy[q] - yi, sz[q] - zi);
                        if (act && v > lo2 && v <= probe) {
                            if (cin < KNN_CAP) lst[cin * 64 + lane] = v;
                            ++cin;
                        }
                    }
                });
        }
        if (!done) {
            int have = klo + cin;
            if (have <= a.kth) {
                // too few values up to the probe: move the bracket up
                lo2 = probe;
                klo = have;
                probe = up2 < INFINITY ? up2 : 4.0 * probe;
            } else if (cin <= KNN_CAP) {
                int rk = a.kth - klo;
                for (int c = 0; c < cin; ++c) {
                    double v = lst[c * 64 + lane];
                    int less = 0, leq = 0;
                    for (int d = 0; d < cin; ++d) {
                        double w = lst[d * 64 + lane];
                        less += w < v ? 1 : 0;
                        leq += w <= v ? 1 : 0;
                    }
                    if (less <= rk && rk < leq) res = v;
                }
                done = true;
            } else {
                // too many to keep: bisect the bracket in the ordering of
                // the IEEE bit patterns (monotonic for values >= 0), so ties
                // and tiny values resolve within 64 halvings
                up2 = probe;
                unsigned long long lb = (unsigned long long)__double_as_longlong(lo2 < 0.0 ? 0.0 : lo2);
                unsigned long long pb = (unsigned long long)__double_as_longlong(probe);
                double mid = __longlong_as_double((long long)(lb + (pb - lb) / 2));
                if (mid > lo2 && mid < probe) {
                    probe = mid;
                } else {
                    res = probe;  // every value left in the bracket is the same
                    done = true;
                }
            }
        }
    }
    if (ok) {
        if (!done) atomicAdd((unsigned long long *)&a.counters[CNT_H_CAPPED], 1ull);
        s.h[i] = done ? 0.5 * sqrt(res) : NAN;
    }
}

// Neighbour lists under r_ij^2 <= (h_i + h_j)^2 through the bucket culling.
// counts == nullptr: fill mode, writing the neighbours' caller ids (s.id) at
// offsets[id_i - r0] for targets with r0 <= id_i < r1.
__global__ __launch_bounds__(64) void k_nbr(Tables t, Soa s, int64_t r0, int64_t r1,
                                            int32_t *__restrict__ counts,
                                            const int64_t *__restrict__ offsets,
                                            int32_t *__restrict__ idx) {
    __shared__ double sx[64], sy[64], sz[64], sh[64];
    __shared__ int32_t sid[64];
    int b = t.boff + xcd_block(blockIdx.x, gridDim.x);
    int lane = threadIdx.x;
    int cnt = t.b_cnt[b];
    int i = t.b_beg[b] + lane;
    bool ok = lane < cnt;
    double xi = ok ? s.x[i] : 0.0, yi = ok ? s.y[i] : 0.0, zi = ok ? s.z[i] : 0.0;
    double hi = ok ? s.h[i] : 0.0;
    int32_t myid = ok ? s.id[i] : -1;
    bool want = ok && myid >= r0 && myid < r1;
    int64_t o = (want && !counts) ? offsets[myid - r0] : 0;
    double hI = t.bhmax[b];
    const double ib[6] = {t.bxl[b], t.bxh[b], t.byl[b], t.byh[b], t.bzl[b], t.bzh[b]};
    int c = 0;
    for_candidates(
        t, t.b_run[b], ib, lane, [&](int S) { return hI + t.shmax[S]; },
        [&](int J) { return hI + t.bhmax[J]; },
        [&](int J) {
            int jc = t.b_cnt[J], j0 = t.b_beg[J];
            __syncthreads();
            if (lane < jc) {
                sx[lane] = s.x[j0 + lane];
                sy[lane] = s.y[j0 + lane];
                sz[lane] = s.z[j0 + lane];
                sh[lane] = s.h[j0 + lane];
                sid[lane] = s.id[j0 + lane];
            }
            __syncthreads();
            for (int q = 0; q < jc; ++q) {
                double r2 = sphx_r2(xi - sx[q], yi - sy[q], zi - sz[q]);
                double tt = hi + sh[q];
                if (want && r2 <= sphx_sq(tt)) {
                    if (!counts) idx[o + c] = sid[q];
                    ++c;
                }
            }
        });
    if (want && counts) counts[myid - r0] = c;
}

}  // namespace

int sphx_knn_pass(Engine &E, int kth, hipStream_t st) {
    if (E.n == 0) return SPHX_OK;
    if (E.nb_launch() == 0) return SPHX_OK;
    KnnArgs a{kth, 200, E.counters};
    k_knn<<<E.nb_launch(), 64, 0, st>>>(E.tview(), E.s, a);
    SPHX_HIP(hipGetLastError());
    return SPHX_OK;
}

int sphx_neighbor_pass(Engine &E, int64_t r0, int64_t r1, int32_t *counts, const int64_t *offsets,
                       int32_t *idx, hipStream_t st) {
    if (E.n == 0) return SPHX_OK;
    k_nbr<<<E.t.nb, 64, 0, st>>>(E.t, E.s, r0, r1, counts, offsets, idx);
    SPHX_HIP(hipGetLastError());
    return SPHX_OK;
}

// Small runs walk a half, a quarter or an eighth of a bucket per group: with one
// wave per bucket most SIMDs would hold a single wave or none, and a group's chain of
// loads, tests and LDS round trips sets the time.  Smaller groups gather more
// candidate buckets in all, which costs more once the chip is full.  Measured,
// one / two / four groups a bucket, on a collapsing Evrard sphere (us, boxes
// included, the density pass as it was then): smoothing 77 / 46 / 40 at 4,096 particles, 119 / 77 / 91 at 32,768,
// 159 / 112 / 149 at 65,752, 146 / 165 / 238 at 131,072; lists and density 154
// / 96 / 80 at 4,096, 277 / 164 / 155 at 65,752, 255 / 218 / 224 at 131,072,
// 330 / 363 / 387 at 262,144.  Four / eight groups: lists and density 66 / 57 at
// 4,096, 88 / 81 at 16,384, 108 / 112 at 24,576; smoothing 33 / 28 at 2,048, 36 /
// 36 at 4,096, 51 / 56 at 8,192 (left at four).
int Engine::smooth_parts() const { return nb_launch() <= 384 ? 4 : (nb_launch() <= 1536 ? 2 : 1); }
// Small runs, whose passes are bounded by launches and by the chain of one
// wave a SIMD: the list passes walk an overflowed bucket themselves (that costs
// registers, and the launch it saves 4.5 us), and the div/curl and hydro pass
// gives a particle four lanes.  One pass with four lanes against one with one
// lane and its overflow launch: 24.6 against 41 us at 4,096 particles, 37.6
// against 45 at 32,768, 45 against 44 at 46,341, 56 against 53 at 65,752, 639
// against 521 at 1,048,576, where the gathers bound it.
bool Engine::list_small() const { return nb_launch() <= 512; }
int Engine::list_parts() const {
    const unsigned nb = nb_launch();
    return nb <= 256 ? 8 : nb <= 1536 ? 4 : nb <= 3072 ? 2 : 1;
}

int Engine::smoothing(hipStream_t st, bool predictor) {
    if (n == 0 || nb_launch() == 0) return SPHX_OK;
    SmoothArgs a{p.nngb, p.ndown, p.nup, p.max_iter, (predictor && p.h_predictor) ? 1 : 0,
                 d_run, h_iters, counters, sphx_h_step(p.h_mode), p.h_min, 0, 0, 0, 0};
    const int64_t need = (int64_t)p.nup - p.ndown + 2;
    if (p.ndown >= 1 && need <= HW_CAP - HW_SPARE) {
        a.hwin = 1;
        a.wslack = (int)(HW_CAP - need) / 4;
        a.wlo = std::max(p.ndown - 1 - a.wslack, 0);
        a.whi = (int)std::min<int64_t>((int64_t)p.nup + 1 + a.wslack, INT32_MAX);
    }
    const int parts = smooth_parts();
    auto launch = [&](auto k4, auto k2, auto k1) {
        if (parts == 4) k4<<<nb_launch() * 4, 64, 0, st>>>(tview(), s, a);
        else if (parts == 2) k2<<<nb_launch() * 2, 64, 0, st>>>(tview(), s, a);
        else k1<<<nb_launch(), 64, 0, st>>>(tview(), s, a);
    };
    if (p.h_mode == 5) launch(k_smoothing_steps<5, 4>, k_smoothing_steps<5, 2>, k_smoothing_steps<5, 1>);
    else if (p.h_mode == 4) launch(k_smoothing_steps<4, 4>, k_smoothing_steps<4, 2>, k_smoothing_steps<4, 1>);
    else if (p.h_mode >= 2) launch(k_smoothing_steps<2, 4>, k_smoothing_steps<2, 2>, k_smoothing_steps<2, 1>);
    else launch(k_smoothing<4>, k_smoothing<2>, k_smoothing<1>);
    SPHX_HIP(hipGetLastError());
    return SPHX_OK;
}

bool Engine::lists_ready() const {
    return use_lists && nbr && prec && fbal && nbr_ovf && nbr_bcap >= t.nb && nbr_pcap >= n;
}

// The lists and the geometric half of the records.
int Engine::build_lists(hipStream_t st) {
    if (n == 0 || nb_launch() == 0) return SPHX_OK;
    if (!lists_ready()) {
        sphx_set_error("neighbour lists requested but not allocated");
        return SPHX_ERR_STATE;
    }
    DensArgs a{p.gamma, tmpi, counters, nbr, prec, nbr_ovf};
    const int nb = (int)nb_launch(), parts = list_parts();
    if (parts == 8) k_lists<8><<<nb * 8, 64, 0, st>>>(tview(), s, a);
    else if (parts == 4) k_lists<4><<<nb * 4, 64, 0, st>>>(tview(), s, a);
    else if (parts == 2) k_lists<2><<<nb * 2, 64, 0, st>>>(tview(), s, a);
    else k_lists<1><<<nb, 64, 0, st>>>(tview(), s, a);
    SPHX_HIP(hipGetLastError());
    return SPHX_OK;
}

// The rest of the records, and the Balsara factors, from given rho, P and c
// (and div v, curl v) for a hydro pass that no density pass precedes.
int Engine::fill_records(hipStream_t st) {
    if (n == 0) return SPHX_OK;
    k_rec_gas<<<(unsigned)((n + 255) / 256), 256, 0, st>>>(s, prec, n, p.balsara ? fbal : nullptr);
    SPHX_HIP(hipGetLastError());
    return SPHX_OK;
}

int Engine::density_eos(hipStream_t st, bool lists, bool soft) {
    if (n == 0 || nb_launch() == 0) return SPHX_OK;
    if (!lists) {
        DensArgs a{p.gamma, tmpi, counters, nullptr, nullptr, nullptr};
        if (soft) k_density<true><<<nb_launch(), 64, 0, st>>>(tview(), s, a);
        else k_density<false><<<nb_launch(), 64, 0, st>>>(tview(), s, a);
        SPHX_HIP(hipGetLastError());
        return SPHX_OK;
    }
    SPHX_CHECK(build_lists(st));
    DensArgs a{p.gamma, tmpi, counters, nbr, prec, nbr_ovf};
    const int nb = (int)nb_launch();
    if (list_small()) {
        if (soft) k_density_quad<true, true><<<4 * nb, 64, 0, st>>>(tview(), s, a);
        else k_density_quad<false, true><<<4 * nb, 64, 0, st>>>(tview(), s, a);
    } else {
        if (soft) k_density_quad<true, false><<<4 * nb, 64, 0, st>>>(tview(), s, a);
        else k_density_quad<false, false><<<4 * nb, 64, 0, st>>>(tview(), s, a);
        if (soft) k_density_ovf<true><<<nb, 64, 0, st>>>(tview(), s, a);
        else k_density_ovf<false><<<nb, 64, 0, st>>>(tview(), s, a);
    }
    SPHX_HIP(hipGetLastError());
    return SPHX_OK;
}

int Engine::divcurl(hipStream_t st, bool lists) {
    if (n == 0 || nb_launch() == 0) return SPHX_OK;
    if (lists) {
        ListArgs L{nbr, prec, nbr_ovf, fbal};
        k_divcurl_list<<<nb_launch(), 64, 0, st>>>(tview(), s, L);
        k_divcurl_ovf<<<nb_launch(), 64, 0, st>>>(tview(), s, nbr_ovf);
        if (p.balsara) {
            int64_t p0 = rrun >= 0 ? rp0 : 0, p1 = rrun >= 0 ? rp1 : n;
            if (p1 > p0)
                k_fbal<<<(unsigned)((p1 - p0 + 255) / 256), 256, 0, st>>>(s, p0, p1, fbal);
        }
    } else {
        k_divcurl<<<nb_launch(), 64, 0, st>>>(tview(), s);
    }
    SPHX_HIP(hipGetLastError());
    return SPHX_OK;
}

int Engine::divcurl_hydro_lists(hipStream_t st) {
    if (n == 0 || nb_launch() == 0) return SPHX_OK;
    if (p.balsara || !lists_ready()) {
        sphx_set_error("the fused list pass needs the lists and no Balsara switch");
        return SPHX_ERR_STATE;
    }
    HydroArgs a{(float)p.alpha, (float)p.beta, (float)(p.eta * p.eta), (float)p.av_w_eps,
                p.av_form, p.balsara};
    ListArgs L{nbr, prec, nbr_ovf, fbal};
    const int nb = (int)nb_launch();
    if (list_small()) {
        k_dchydro_quad<<<4 * nb, 64, 0, st>>>(tview(), s, a, L);
        SPHX_HIP(hipGetLastError());
        return SPHX_OK;
    }
    k_dchydro_list<<<nb, 64, 0, st>>>(tview(), s, a, L);
    k_dchydro_ovf<<<nb, 64, 0, st>>>(tview(), s, a, nbr_ovf);
    SPHX_HIP(hipGetLastError());
    return SPHX_OK;
}

int Engine::hydro(hipStream_t st, bool lists) {
    if (n == 0 || nb_launch() == 0) return SPHX_OK;
    HydroArgs a{(float)p.alpha, (float)p.beta, (float)(p.eta * p.eta), (float)p.av_w_eps,
                p.av_form, p.balsara};
    if (lists) {
        ListArgs L{nbr, prec, nbr_ovf, fbal};
        k_hydro_list<<<nb_launch(), 64, 0, st>>>(tview(), s, a, L);
        k_hydro_ovf<<<nb_launch(), 64, 0, st>>>(tview(), s, a, nbr_ovf);
    } else {
        k_hydro<<<nb_launch(), 64, 0, st>>>(tview(), s, a);
    }
    SPHX_HIP(hipGetLastError());
    return SPHX_OK;
}
