// Barnes-Hut gravity: Morton-built octree, monopole moments, group walk.
//
// Replaces the reference's iterative octree (Particles_in_BH_Tree_II/
// Evrard_test/bh_tree_iteration_v2.h: single-block atomic insertion build
// 149-367, per-warp stack walk 454-588, theta = 0.5) with a build that
// follows the sorted 63-bit Morton keys: every octree cell is a contiguous
// key range, and a cell's eight children are found by binary search on the
// next three key bits, one level per pass.  Moments (mass, centre of mass,
// max eps) are summed bottom-up in FP64.  The walk is per group (one
// wavefront): the groups are the largest cells holding at most 64 particles
// (unsplittable leaves of coincident particles are cut into runs of 64), so a
// group's bounding box is always inside one cell's cube -- unlike 64
// consecutive Morton indices, which can straddle a jump of the curve and then
// open most of the tree.  A cell is accepted for the whole group when its
// distance from the group's bounding box exceeds s/theta + |com - centre|
// (cell side s); accepted cells and the particles of opened leaves go to an
// LDS interaction list that is flushed through the FP32 spline-softened pair
// formula with Kahan-compensated sums.
#include <algorithm>

#include "sphx_internal.h"

namespace {

constexpr int BH_LEAF = 8;        // particles per leaf at most
// Cell stack and interaction list capacities per group (one wave).  A deep
// walk (small opening angle) opens many cells per step, and the larger stack
// keeps its batches of popped cells large; at larger angles the smaller
// stack's occupancy wins.  A list of 128 entries
// and four entries evaluated together leave four waves a SIMD, which the pairs'
// FP32 issue fills (five by spilling took as long); a list of 512 and batches
// of eight left two to three (the walk as it was then, 4M-particle Plummer
// sphere, theta 0.3 / 0.5 / 0.7: 60 / 18.1 / 10.1 ms against 45 / 13.8 / 7.5;
// 100 ms at 0.3 with the smaller stack; now 32.5 / 11.2 / 6.3 ms).
constexpr int BH_SCAP = 1024;
constexpr int BH_SCAP_DEEP = 2048;
constexpr double BH_DEEP_THETA = 0.35;  // the larger stack below this angle
constexpr int BH_SLACK = 160;     // > 7 x 21 levels of pure depth-first growth
constexpr int BH_ICAP = 128;
constexpr int BH_BATCH = 4;       // list entries evaluated together
static_assert(BH_ICAP == 128, "the near masks of a full list are two wave ballots");
static_assert(BH_SCAP > BH_SLACK + 7 * 64, "a full batch must fit above the slack");
static_assert(BH_SCAP_DEEP > BH_SCAP, "the deep-walk stack is the larger one");
constexpr int BHT = 256;

// What the walk reads of a cell, packed so that one cell costs two 32-byte
// loads: the monopole (FP64 centre of mass) and the opening/link record.
struct __align__(32) BhMono {
    double cx, cy, cz;
    float mass, emax;
};
struct __align__(32) BhLink {
    float size, delta;
    int32_t child, nchild, beg, cnt, pad0, pad1;
};

struct BhTree {
    int32_t *beg, *cnt, *child, *nchild;
    double *mass, *emax;
    BhMono *mono;
    BhLink *link;
    int32_t *ncell;  // cells of each level, BH_LEVELS of them, zero past the deepest
    int64_t cap;     // cells the arrays hold
};
constexpr int BH_LEVELS = 23;

__device__ __forceinline__ int digit_at(uint64_t key, int shift) { return (int)((key >> shift) & 7ull); }

// Cells of a level: [*beg, *beg + returned), as far as the arrays hold them.
__device__ __forceinline__ int64_t bh_level(const BhTree &T, int level, int64_t *beg) {
    int64_t b = 0;
    for (int l = 0; l < level; ++l) b += T.ncell[l];
    *beg = b;
    return min((int64_t)T.ncell[level], max((int64_t)0, T.cap - b));
}

__global__ void k_bh_root(BhTree T, int32_t n, bool fresh, int32_t *__restrict__ gcount,
                          int64_t *__restrict__ stats) {
    const int t = threadIdx.x;
    if (t < 3) gcount[t] = 0;
    if (t < 4) stats[t] = 0;
    if (!fresh) return;
    if (t < BH_LEVELS) T.ncell[t] = t == 0;
    if (t == 0) {
        T.beg[0] = 0;
        T.cnt[0] = n;
    }
}

// One level of the build: eight lanes a cell find its child boundaries (first
// index of each child digit) side by side, a workgroup takes room for its cells'
// children with one atomic, and the children are written.  The cells' order
// within a level depends on the atomics; no result does, the walk follows links.
// Bound: the chain of dependent key loads of a search (20 at the root).  A search
// by one lane a cell (28 us a level at 1,048,576 particles), three launches of a
// scan, an emitting one and a wait for the level's count -> one launch a level
// and the counts left on the device: build of 1,048,576 particles 800 -> 315 us,
// of 2,000 343 -> 120.
__global__ __launch_bounds__(BHT) void k_bh_split(BhTree T, const uint64_t *__restrict__ keys, int level) {
    __shared__ int32_t wsum[BHT / 64], base;
    const int tid = threadIdx.x, lane = tid & 63, d = tid & 7;
    int64_t f0;
    const int64_t fc = bh_level(T, level, &f0), next = f0 + T.ncell[level];
    const int shift = 3 * (20 - level);
    for (int64_t t0 = (int64_t)blockIdx.x * (BHT / 8); t0 < fc; t0 += (int64_t)gridDim.x * (BHT / 8)) {
        const int64_t t = t0 + (tid >> 3), i = f0 + t;
        int b = 0, c = 0;
        if (t < fc) {
            b = T.beg[i];
            c = T.cnt[i];
        }
        const bool leaf = c <= BH_LEAF || level >= 21;
        int lo = b, hi = leaf || d == 0 ? b : b + c;  // first index with digit >= d
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (digit_at(keys[mid], shift) < d) lo = mid + 1;
            else hi = mid;
        }
        int end = __shfl_down(lo, 1, 8);
        if (d == 7) end = b + c;
        const bool has = !leaf && end > lo;
        const uint64_t m = __ballot(has);
        const int mine = (int)((m >> (lane & 56)) & 0xff);
        if (lane == 0) wsum[tid >> 6] = __popcll(m);
        __syncthreads();
        if (tid == 0) {
            int s = 0;
            for (int w = 0; w < BHT / 64; ++w) {
                const int v = wsum[w];
                wsum[w] = s;
                s += v;
            }
            base = s ? atomicAdd(&T.ncell[level + 1], s) : 0;
        }
        __syncthreads();
        const int64_t first = next + base + wsum[tid >> 6] + __popcll(m & ((1ull << (lane & 56)) - 1));
        if (has) {
            const int64_t o = first + __popc(mine & ((1 << d) - 1));
            if (o < T.cap) {
                T.beg[o] = lo;
                T.cnt[o] = end - lo;
            }
        }
        if (t < fc && d == 0) {
            T.child[i] = leaf ? -1 : (int32_t)first;
            T.nchild[i] = __popc(mine);
        }
        __syncthreads();
    }
}

__device__ __forceinline__ uint32_t compact3(uint64_t v) {
    // gather every third bit of v (bit 3b -> bit b)
    v &= 0x1249249249249249ull;
    v = (v | (v >> 2)) & 0x10c30c30c30c30c3ull;
    v = (v | (v >> 4)) & 0x100f00f00f00f00full;
    v = (v | (v >> 8)) & 0x1f0000ff0000ffull;
    v = (v | (v >> 16)) & 0x1f00000000ffffull;
    v = (v | (v >> 32)) & 0x1fffffull;
    return (uint32_t)v;
}

// Moments of the cells of one level (children are one level deeper and done).
__global__ __launch_bounds__(BHT) void k_bh_moments(BhTree T, int level, const uint64_t *__restrict__ keys,
                                                    const double *__restrict__ x,
                                                    const double *__restrict__ y,
                                                    const double *__restrict__ z,
                                                    const double *__restrict__ m,
                                                    const double *__restrict__ eps,
                                                    const double *__restrict__ rbox) {
    int64_t l0;
    const int64_t nl = bh_level(T, level, &l0);
    const double ext = fmax(rbox[1] - rbox[0], fmax(rbox[3] - rbox[2], rbox[5] - rbox[4]));
    // cell0 = side of a level-21 cell
    const double cell0 = ext > 0.0 ? ext * (1.0 + 0x1p-30) / (double)(1ull << 21) : 1.0;
    const double side = cell0 * (double)(1ull << (21 - level));
    for (int64_t t = (int64_t)blockIdx.x * BHT + threadIdx.x; t < nl; t += (int64_t)gridDim.x * BHT) {
        const int64_t i = l0 + t;
        const int b = T.beg[i], cnt = T.cnt[i], child = T.child[i], nchild = T.nchild[i];
        double M = 0.0, sx = 0.0, sy = 0.0, sz = 0.0, em = 0.0;
        if (child < 0) {
            for (int q = b; q < b + cnt; ++q) {
                double mq = m[q];
                M += mq;
                sx += mq * x[q]; sy += mq * y[q]; sz += mq * z[q];
                em = fmax(em, eps[q]);
            }
        } else if ((int64_t)child + nchild <= T.cap) {
            for (int c = child; c < child + nchild; ++c) {
                double mc = T.mass[c];
                const BhMono mo = T.mono[c];
                M += mc;
                sx += mc * mo.cx; sy += mc * mo.cy; sz += mc * mo.cz;
                em = fmax(em, T.emax[c]);
            }
        }
        double cx = M > 0.0 ? sx / M : 0.0, cy = M > 0.0 ? sy / M : 0.0, cz = M > 0.0 ? sz / M : 0.0;
        uint64_t pre = level > 0 ? keys[b] >> (3 * (21 - level)) : 0ull;
        double gx = rbox[0] + (compact3(pre >> 2) + 0.5) * side;
        double gy = rbox[2] + (compact3(pre >> 1) + 0.5) * side;
        double gz = rbox[4] + (compact3(pre) + 0.5) * side;
        double dl = sqrt((cx - gx) * (cx - gx) + (cy - gy) * (cy - gy) + (cz - gz) * (cz - gz));
        T.mass[i] = M;
        T.emax[i] = em;
        BhMono mo;
        mo.cx = cx; mo.cy = cy; mo.cz = cz;
        mo.mass = (float)M;
        mo.emax = (float)em;
        T.mono[i] = mo;
        BhLink lk;
        // rounded up so that the FP32 opening test is never looser than the FP64 one
        lk.size = __double2float_ru(side);
        lk.delta = __double2float_ru(dl);
        lk.child = child;
        lk.nchild = nchild;
        lk.beg = b;
        lk.cnt = cnt;
        lk.pad0 = lk.pad1 = 0;
        T.link[i] = lk;
    }
}

// Walk groups: the children (cnt <= 64) of a cell with more than 64
// particles, consecutive ones packed while their sum stays <= 64; the root
// when it has at most 64; runs of 64 inside an unsplittable leaf with more.
// Each particle lands in exactly one group; the list order (atomic append)
// does not affect any particle's result.
// A group of a cell with many particles sees most of them as single entries:
// outliers packed over the whole of a large cell, or one small child beside
// full ones.  A wave alone needs some 130 cycles an entry, so such a group in
// one wave outlasts all the others.  It goes to several waves, each of which
// walks the tree and sums its part of the entries: one for every BH_PART
// particles of the cell (of the cells that begin in a range of them) and
// BH_OUT for what lies outside (every BH_OUT-th by the cell's first particle).
// Walk at theta 0.5 over a Plummer sphere, one wave a group -> parts: 3.46 ->
// 0.42 ms for 65,536 particles, 2.12 -> 1.52 for 524,288.  2,048 particles a
// wave took 0.65 ms for 131,072, where 1,024 take 0.55 and 512 take 0.59; four
// waves outside took 1.20 ms for 262,144, eight 0.99 and sixteen 0.86.
constexpr int BH_PART = 1024, BH_PARTS_MAX = 256, BH_OUT = 16;
static_assert(BH_PART > BH_PARTS_MAX, "no part of a cell's range is empty");

// A small run has too few groups to fill the device: all its groups go to
// several waves (every SHARE-th entry by the cell's first particle), at the
// price of a tree walk for each.  Evrard sphere with 1 / 2 / 4 / 8 waves: 194 /
// 126 / 86 / 75 us for 8,192 particles, 287 / 176 / 140 / 208 for 32,768, 338 /
// 222 / 241 / 353 for 65,536, 385 / 379 / 408 / 671 for 131,072.
static int bh_share(int64_t n) { return n <= 8192 ? 8 : n <= 32768 ? 4 : n <= 98304 ? 2 : 1; }

struct BhGroups {
    int32_t *beg, *cnt;  // groups of one wave
    // items of the others, a wave each: {first particle, particles | items of
    // the group << 8 in its first | share << 20 | shares - 1 << 24, lo, hi}; a
    // wave sums the entries of its share in [lo, hi), or outside [hi, lo)
    int4 *part;
    int32_t *count;      // [0] groups of one wave, [1] items of the others, [2] the others
    int share;
};

__device__ __forceinline__ void bh_add_group(const BhGroups &g, int beg, int cnt, int cell, int ccnt) {
    const int parts = min(ccnt / BH_PART, BH_PARTS_MAX);
    if (parts >= 2) {
        // no range is empty: a part has at least BH_PART > BH_PARTS_MAX particles
        const int all = parts + BH_OUT, step = (ccnt + parts - 1) / parts;
        const int k = atomicAdd(&g.count[1], all);
        atomicAdd(&g.count[2], 1);
        for (int p = 0; p < parts; ++p)
            g.part[k + p] = make_int4(beg, cnt | (p ? 0 : all << 8), cell + min(ccnt, p * step),
                                      cell + min(ccnt, (p + 1) * step));
        for (int p = 0; p < BH_OUT; ++p)
            g.part[k + parts + p] = make_int4(beg, cnt | p << 20 | (BH_OUT - 1) << 24, cell + ccnt, cell);
    } else if (g.share > 1) {
        const int k = atomicAdd(&g.count[1], g.share);
        atomicAdd(&g.count[2], 1);
        for (int p = 0; p < g.share; ++p)
            g.part[k + p] = make_int4(beg, cnt | (p ? 0 : g.share << 8) | p << 20 | (g.share - 1) << 24, 0, INT32_MAX);
    } else {
        const int k = atomicAdd(&g.count[0], 1);
        g.beg[k] = beg;
        g.cnt[k] = cnt;
    }
}

__device__ __forceinline__ void bh_cell_groups(const BhTree &T, int64_t i, const BhGroups &G) {
    const int c = T.cnt[i], b = T.beg[i];
    if (i == 0 && c <= 64) bh_add_group(G, b, c, b, c);
    if (c <= 64) return;
    if (T.child[i] >= 0) {
        if ((int64_t)T.child[i] + T.nchild[i] > T.cap) return;  // to be built again
        // consecutive small children are packed into one group of at most 64
        // (their union stays inside this cell's cube)
        int pb = -1, pc = 0;
        for (int q = T.child[i]; q < T.child[i] + T.nchild[i]; ++q) {
            int cq = T.cnt[q];
            if (cq > 64 || pc + cq > 64) {
                if (pc > 0) bh_add_group(G, pb, pc, b, c);
                pb = -1;
                pc = 0;
            }
            if (cq <= 64) {
                if (pc == 0) pb = T.beg[q];
                pc += cq;
            }
        }
        if (pc > 0) bh_add_group(G, pb, pc, b, c);
    } else {
        for (int o = 0; o < c; o += 64) bh_add_group(G, b + o, min(64, c - o), b, 0);
    }
}

// Over the levels 0 to top, those that have been split.
__global__ __launch_bounds__(BHT) void k_bh_groups(BhTree T, int top, BhGroups G) {
    int64_t beg;
    const int64_t n = bh_level(T, top, &beg) + beg;
    for (int64_t i = (int64_t)blockIdx.x * BHT + threadIdx.x; i < min(n, T.cap); i += (int64_t)gridDim.x * BHT)
        bh_cell_groups(T, i, G);
}

// Inclusive prefix sum over the wave, every lane active: within the rows of 16
// lanes, then the rows' totals (row_shr 1, 2, 4, 8, row_bcast 15 and 31).
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t u) {
    int v = (int)u;
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
    return (uint32_t)v;
}
__device__ __forceinline__ uint32_t wave_last(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

struct BhArgs {
    const double *x, *y, *z, *m, *eps;
    const int32_t *gbeg, *gcnt;   // groups of one wave
    const int4 *part;             // items of the others, npart of them: first in the grid
    int32_t npart;
    double4 *psum;                // their sums, 64 an item
    int64_t n;
    double G, theta;
    double *ax, *ay, *az, *pot;
    int64_t *stats;  // [0] interactions, [1] frontier overflow, [2] max list fill
    int64_t *ovf;    // engine counter of overflowing groups (nullable)
};

// One list entry against lane i, its geometry already formed: (dx, dy, dz)
// from i to the entry, r2 = |d|^2 and t = eps_i + eps_j, twice the pair's
// softening e = (eps_i + eps_j) / 2.  Newtonian where r2 >= t^2 (that is
// r >= 2e: (4e) e and t t round the same product), the cubic-spline softened
// kernel inside.
template <bool POT>
__device__ __forceinline__ void bh_eval(float dx, float dy, float dz, float r2, float t, float mj,
                                        float &ax, float &ay, float &az, float &ph) {
    float f, p;
    // r^-1 once for both branches; inside the softening length it also gives
    // r = r^2 r^-1 (a transcendental costs several FP32 instructions' issue
    // time, and a wave whose lanes split between the branches runs both)
    const float ri = __builtin_amdgcn_rsqf(r2);
    if (r2 >= t * t) {
        f = ri * ri * ri;
        p = ri;
    } else {
        float e = 0.5f * t;
        float r = r2 > 0.0f ? r2 * ri : 0.0f;
        float ie = __builtin_amdgcn_rcpf(e);
        float q = r * ie;
        if (q <= 1.0f) {
            float q2 = q * q;
            f = ie * ie * ie * (4.0f / 3.0f - 1.2f * q2 + 0.5f * q2 * q);
            p = (POT && r2 > 0.0f) ? ie * (1.4f - 2.0f * q2 * (1.0f / 3.0f - 0.15f * q2 + 0.05f * q2 * q))
                                   : 0.0f;
        } else {
            float w = 2.0f - q;
            float w2 = w * w;
            f = ri * ri * ri * (1.0f - w2 * w2 * (1.0f - 0.8f * w + w2 * (1.0f / 6.0f)));
            float q2 = q * q;
            p = POT ? -ri * (1.0f / 15.0f) -
                          ie * q2 * (4.0f / 3.0f - q + 0.3f * q2 - q2 * q * (1.0f / 30.0f)) + 1.6f * ie
                    : 0.0f;
        }
    }
    float s = mj * f;
    ax = __builtin_fmaf(s, dx, ax);
    ay = __builtin_fmaf(s, dy, ay);
    az = __builtin_fmaf(s, dz, az);
    if (POT) ph = __builtin_fmaf(mj, p, ph);
}

// The Newtonian branch of bh_eval alone, for entries every lane sees at
// r >= 2e: the same operations, so the same bits.
template <bool POT>
__device__ __forceinline__ void bh_far(float dx, float dy, float dz, float r2, float mj, float &ax,
                                       float &ay, float &az, float &ph) {
    float ri = __builtin_amdgcn_rsqf(r2);
    float f = ri * ri * ri;
    float s = mj * f;
    ax = __builtin_fmaf(s, dx, ax);
    ay = __builtin_fmaf(s, dy, ay);
    az = __builtin_fmaf(s, dz, az);
    if (POT) ph = __builtin_fmaf(mj, ri, ph);
}

// bh_eval without the potential and without a branch: the outer formula with w
// = 2 - q clamped at zero is the Newtonian one from q = 2 on, so one choice
// (q <= 1) is left.
__device__ __forceinline__ void bh_soft(float dx, float dy, float dz, float r2, float t, float mj,
                                        float &ax, float &ay, float &az) {
    const float ri = __builtin_amdgcn_rsqf(fmaxf(r2, 1.17549435e-38f));
    const float ie = 2.0f * __builtin_amdgcn_rcpf(t);
    const float q = r2 * ri * ie, q2 = q * q;
    const float in = ie * ie * ie * __builtin_fmaf(q2, __builtin_fmaf(0.5f, q, -1.2f), 4.0f / 3.0f);
    const float w = fmaxf(2.0f - q, 0.0f), w2 = w * w;
    const float out = ri * ri * ri * __builtin_fmaf(-w2 * w2, __builtin_fmaf(w2, 1.0f / 6.0f, __builtin_fmaf(-0.8f, w, 1.0f)), 1.0f);
    const float s = mj * (q <= 1.0f ? in : out);
    ax = __builtin_fmaf(s, dx, ax);
    ay = __builtin_fmaf(s, dy, ay);
    az = __builtin_fmaf(s, dz, az);
}

template <bool POT>
__device__ __forceinline__ void bh_pair(float xi, float yi, float zi, float ei, float4 j, float ej,
                                        float &ax, float &ay, float &az, float &ph) {
    float dx = j.x - xi, dy = j.y - yi, dz = j.z - zi;
    float r2 = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz));
    bh_eval<POT>(dx, dy, dz, r2, ei + ej, j.w, ax, ay, az, ph);
}

// Bound: FP32 issue of the waves' pairs (0.28-0.30 VALU instructions a SIMD-cycle
// on 1,048,576 particles and more, where a loop of pairs alone reaches 0.33; the
// walk's own instructions are a fifth of it).  So a list's entries are first tested against the group's box, 64 at a
// time, and four that no particle can see softened are taken without a test (13
// instructions an entry for 17); softened ones without a branch (34 for some
// 45); a group of at most 32 or 16 particles gives each two or four lanes; the
// three counts of a batch are scanned in one word, and opened leaves listed 64
// particles at a time.  VALU instructions of the launch, with the groups in
// parts, before -> after: 1.65 -> 1.22 x 10^9 on an Evrard sphere of 1,048,576
// particles with eps = h, theta 0.5 (2.33 -> 1.85 ms), 1.15 -> 0.79 x 10^9 on a
// Plummer sphere of 524,288 (2.68 -> 1.48 ms).
//
// The walk of one group of gn particles, P lanes a particle (P W = 64): lane
// (sub, p) sums every P-th entry of the list for particle p.  Of the accepted
// cells and opened leaves it sums those whose first particle lies in [lo, hi).
template <bool POT, int SCAP, int P>
__device__ __forceinline__ void bh_walk_group(const BhTree &T, const BhArgs &a, int32_t *stk, float4 *il,
                                              float *ie, int64_t g0, int gn, int lo, int hi,
                                              int smask, int sval, double4 *psum) {
    constexpr int W = 64 / P, STEP = BH_BATCH * P;
    const int lane = threadIdx.x, sub = lane / W, pl = lane % W;
    const int64_t i = g0 + pl;
    const bool ok = pl < gn;
    double xd = ok ? a.x[i] : 0.0, yd = ok ? a.y[i] : 0.0, zd = ok ? a.z[i] : 0.0;
    double lx = wave_min_d(ok ? xd : INFINITY), hx = wave_max_d(ok ? xd : -INFINITY);
    double ly = wave_min_d(ok ? yd : INFINITY), hy = wave_max_d(ok ? yd : -INFINITY);
    double lz = wave_min_d(ok ? zd : INFINITY), hz = wave_max_d(ok ? zd : -INFINITY);
    const double ox = 0.5 * (lx + hx), oy = 0.5 * (ly + hy), oz = 0.5 * (lz + hz);
    const float xi = (float)(xd - ox), yi = (float)(yd - oy), zi = (float)(zd - oz);
    const float ei = ok ? (float)a.eps[i] : 1.0f;
    // The group's box and largest softening as the pairs see them: an entry at
    // r >= 2e of the box is at r >= 2e of every particle by the same FP32
    // operations, each of which keeps order under rounding.
    const float bx = (float)(lx - ox), cx = (float)(hx - ox);
    const float by = (float)(ly - oy), cy = (float)(hy - oy);
    const float bz = (float)(lz - oz), cz = (float)(hz - oz);
    const float emax = wave_max_f(ok ? fabsf(ei) : 0.0f);
    float ax = 0.f, ay = 0.f, az = 0.f, ph = 0.f;
    KahanF kx, ky, kz, kp;
    kx.init(); ky.init(); kz.init(); kp.init();
    int icnt = 0;
    int64_t ninter = 0;
    int overflow = 0, maxfill = 0;
    if (lane == 0) stk[0] = 0;
    int sp = 1;
    __syncthreads();

    // Ballot of the entries q0 + lane of the list that some particle may see softened.
    auto near_mask = [&](int q0) -> uint64_t {
        bool near = false;
        if (q0 + lane < icnt) {
            const float4 j = il[q0 + lane];
            const float t = emax + fabsf(ie[q0 + lane]);
            const float dx = fmaxf(0.0f, fmaxf(bx - j.x, j.x - cx));
            const float dy = fmaxf(0.0f, fmaxf(by - j.y, j.y - cy));
            const float dz = fmaxf(0.0f, fmaxf(bz - j.z, j.z - cz));
            const float r2 = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz));
            near = !(r2 >= t * t);
        }
        return __ballot(near);
    };
    auto flush = [&]() {
        __syncthreads();
        // entries STEP at a time, BH_BATCH a lane, their LDS loads issued before the
        // pairs are evaluated
        const int full = icnt - icnt % STEP;
        uint64_t near = near_mask(0);
        const uint64_t near1 = near_mask(64);
        for (int q = 0; q < full; q += STEP) {
            if (q == 64) near = near1;
            float4 j[BH_BATCH];
            float dx[BH_BATCH], dy[BH_BATCH], dz[BH_BATCH], r2[BH_BATCH];
#pragma unroll
            for (int k = 0; k < BH_BATCH; ++k) j[k] = il[q + k * P + sub];
#pragma unroll
            for (int k = 0; k < BH_BATCH; ++k) {
                dx[k] = j[k].x - xi;
                dy[k] = j[k].y - yi;
                dz[k] = j[k].z - zi;
                r2[k] = __builtin_fmaf(dx[k], dx[k], __builtin_fmaf(dy[k], dy[k], dz[k] * dz[k]));
            }
            bool far = true;
            float t[BH_BATCH];
            if (near & ((1ull << STEP) - 1)) {
#pragma unroll
                for (int k = 0; k < BH_BATCH; ++k) {
                    t[k] = ei + ie[q + k * P + sub];
                    far = far && r2[k] >= t[k] * t[k];
                }
                // lanes past the group's end take part in the vote as far
                far = __all(far || !ok);
            }
            near >>= STEP;
            if (far) {
#pragma unroll
                for (int k = 0; k < BH_BATCH; ++k) bh_far<POT>(dx[k], dy[k], dz[k], r2[k], j[k].w, ax, ay, az, ph);
            } else {
#pragma unroll
                for (int k = 0; k < BH_BATCH; ++k) {
                    if (POT) bh_eval<POT>(dx[k], dy[k], dz[k], r2[k], t[k], j[k].w, ax, ay, az, ph);
                    else bh_soft(dx[k], dy[k], dz[k], r2[k], t[k], j[k].w, ax, ay, az);
                }
            }
        }
        for (int q = full + sub; q < icnt; q += P) bh_pair<POT>(xi, yi, zi, ei, il[q], ie[q], ax, ay, az, ph);
        kx.add(ax); ky.add(ay); kz.add(az);
        if (POT) kp.add(ph);
        ax = ay = az = ph = 0.f;
        ninter += icnt;
        maxfill = max(maxfill, icnt);
        icnt = 0;
        __syncthreads();
    };

    // Depth-first in batches: pop up to 64 cells from the top of the stack,
    // classify them, push the children of the opened ones.  A popped cell adds
    // at most 7 net entries, so popping at most (cap - slack - sp) / 7 keeps the
    // stack inside cap - slack; past that the walk is pure depth-first (one
    // cell per batch), whose growth is bounded by 7 x the tree depth (<= 147),
    // inside the slack.  The particles of opened leaves, eight a cell at most,
    // take the place of its children above them while they are listed.
    while (sp > 0) {
        int room = (SCAP - BH_SLACK - sp) / 7;
        int take = room < 1 ? 1 : (room < 64 ? room : 64);
        take = sp < take ? sp : take;
        int base = sp - take;
        int node = lane < take ? stk[base + lane] : -1;
        sp = base;
        __syncthreads();
        // what a lane adds: an accepted cell, leaf particles or children,
        // from lnk on; the three counts are scanned as fields of one word
        uint32_t mine = 0;
        int rem = 0, lnk = 0;
        BhMono mo{};
        BhLink lk{};
        if (node >= 0) {
            mo = T.mono[node];
            lk = T.link[node];
        }
        const int end = lk.beg + lk.cnt;
        if (node >= 0 && (lo < hi ? lk.beg < hi && end > lo : lk.beg < hi || end > lo)) {
            const bool own = (lo < hi ? lk.beg >= lo : lk.beg < hi || lk.beg >= lo) && (lk.beg & smask) == sval;
            double dx = fmax(0.0, fmax(lx - mo.cx, mo.cx - hx));
            double dy = fmax(0.0, fmax(ly - mo.cy, mo.cy - hy));
            double dz = fmax(0.0, fmax(lz - mo.cz, mo.cz - hz));
            // d theta > s + theta delta, both sides >= 0, compared squared
            const double d2 = dx * dx + dy * dy + dz * dz;
            const double rhs = (double)lk.size + a.theta * (double)lk.delta;
            if (d2 * (a.theta * a.theta) > rhs * rhs) {
                mine = own ? 1u : 0u;
            } else if (lk.child < 0) {
                rem = own ? lk.cnt : 0;
                lnk = lk.beg;
                mine = (uint32_t)min(rem, 8) << 8;
            } else {
                lnk = lk.child;
                mine = (uint32_t)lk.nchild << 20;
            }
        }
        uint32_t incl = wave_incl_scan(mine);
        uint32_t tot = wave_last(incl);
        const int nacc = tot & 0xff, nch = tot >> 20;
        int nleaf = (tot >> 8) & 0xfff;
        // accepted cells: at most one entry per lane
        if (icnt + nacc > BH_ICAP) flush();
        if (mine & 1u) {
            const int q = icnt + (int)((incl - mine) & 0xff);
            il[q] = make_float4((float)(mo.cx - ox), (float)(mo.cy - oy),
                                (float)(mo.cz - oz), mo.mass);
            ie[q] = mo.emax;
        }
        icnt += nacc;
        // children onto the stack, the leaf particles' indices above them
        const int top = sp + nch;
        {
            const uint32_t before = incl - mine;
            const int nq = (mine >> 8 & 0xfff) + (int)(mine >> 20);
            const int at = mine >> 20 ? sp + (int)(before >> 20) : top + (int)(before >> 8 & 0xfff);
            if (top + nleaf > SCAP) overflow = 1;
#pragma unroll
            for (int q = 0; q < 8; ++q)
                if (q < nq && at + q < SCAP) stk[at + q] = lnk + q;
        }
        sp = min(top, SCAP);
        while (nleaf > 0) {
            __syncthreads();
            nleaf = min(nleaf, SCAP - top);
            for (int s = 0; s < nleaf;) {
                if (icnt == BH_ICAP) flush();
                const int c = min(min(64, nleaf - s), BH_ICAP - icnt);
                if (lane < c) {
                    const int p = stk[top + s + lane];
                    il[icnt + lane] = make_float4((float)(a.x[p] - ox), (float)(a.y[p] - oy),
                                                  (float)(a.z[p] - oz), (float)a.m[p]);
                    ie[icnt + lane] = (float)a.eps[p];
                }
                icnt += c;
                s += c;
            }
            // an unsplittable leaf (coincident particles) holds more than eight
            rem -= 8;
            lnk += 8;
            nleaf = 0;
            if (__any(rem > 0)) {
                mine = (uint32_t)max(0, min(rem, 8));
                incl = wave_incl_scan(mine);
                nleaf = (int)wave_last(incl);
                __syncthreads();
                const int at = top + (int)(incl - mine);
                if (top + nleaf > SCAP) overflow = 1;
                for (int q = 0; q < (int)mine; ++q)
                    if (at + q < SCAP) stk[at + q] = lnk + q;
            }
        }
        __syncthreads();
    }
    flush();
    double fx = kx.value(), fy = ky.value(), fz = kz.value(), fp = POT ? kp.value() : 0.0;
#pragma unroll
    for (int o = 32; o >= W; o >>= 1) {
        fx += __shfl_xor(fx, o, 64);
        fy += __shfl_xor(fy, o, 64);
        fz += __shfl_xor(fz, o, 64);
        if (POT) fp += __shfl_xor(fp, o, 64);
    }
    if (psum) {
        if (sub == 0) psum[lane] = make_double4(fx, fy, fz, fp);
    } else if (ok && sub == 0) {
        a.ax[i] = a.G * fx;
        a.ay[i] = a.G * fy;
        a.az[i] = a.G * fz;
        if (POT) a.pot[i] = -a.G * fp;
    }
    if (lane == 0) {
        atomicAdd((unsigned long long *)&a.stats[0], (unsigned long long)(ninter * gn));
        if (overflow) {
            atomicAdd((unsigned long long *)&a.stats[1], 1ull);
            if (a.ovf) atomicAdd((unsigned long long *)a.ovf, 1ull);
        }
        atomicMax((unsigned long long *)&a.stats[2], (unsigned long long)maxfill);
    }
}

template <bool POT, int SCAP>
__global__ __launch_bounds__(64) void k_bh_walk(BhTree T, BhArgs a) {
    __shared__ int32_t stk[SCAP];
    __shared__ float4 il[BH_ICAP];
    __shared__ float ie[BH_ICAP];
    int64_t g0;
    int gn, lo = 0, hi = INT32_MAX, smask = 0, sval = 0;
    double4 *psum = nullptr;
    if ((int)blockIdx.x < a.npart) {
        const int4 it = a.part[blockIdx.x];
        g0 = it.x;
        gn = it.y & 0xff;
        sval = it.y >> 20 & 15;
        smask = it.y >> 24 & 15;
        lo = it.z;
        hi = it.w;
        psum = a.psum + 64 * (int64_t)blockIdx.x;
    } else {
        // deep cells last in the list, and first here: theirs are the long walks
        const int g = gridDim.x - 1 - blockIdx.x;
        g0 = a.gbeg[g];
        gn = a.gcnt[g];
    }
    if (gn > 32) bh_walk_group<POT, SCAP, 1>(T, a, stk, il, ie, g0, gn, lo, hi, smask, sval, psum);
    else if (gn > 16) bh_walk_group<POT, SCAP, 2>(T, a, stk, il, ie, g0, gn, lo, hi, smask, sval, psum);
    else bh_walk_group<POT, SCAP, 4>(T, a, stk, il, ie, g0, gn, lo, hi, smask, sval, psum);
}

// The sums of a group in parts, in the order of the parts.
template <bool POT>
__global__ __launch_bounds__(64) void k_bh_join(BhArgs a) {
    const int4 it = a.part[blockIdx.x];
    const int parts = it.y >> 8 & 0xfff, gn = it.y & 0xff, lane = threadIdx.x;
    if (parts == 0 || lane >= gn) return;
    double x = 0.0, y = 0.0, z = 0.0, p = 0.0;
#pragma unroll 8
    for (int k = 0; k < parts; ++k) {
        const double4 v = a.psum[64 * ((int64_t)blockIdx.x + k) + lane];
        x += v.x;
        y += v.y;
        z += v.z;
        p += v.w;
    }
    const int64_t i = it.x + lane;
    a.ax[i] = a.G * x;
    a.ay[i] = a.G * y;
    a.az[i] = a.G * z;
    if (POT) a.pot[i] = -a.G * p;
}

}  // namespace

// Host side: tree storage (owned here, not by the engine) and the build.
struct BhHost {
    BhTree T{};
    int64_t cap = 0;
    BhGroups g{};
    int64_t gcap = 0;
    double4 *psum = nullptr;
    int64_t icap = 0, pcap = 0;
    int64_t *stats = nullptr;
    std::vector<void *> owned;
    ~BhHost() {
        for (void *q : owned) hipFree(q);
    }
    int alloc(void **ptr, size_t bytes) {
        void *q = nullptr;
        if (hipMalloc(&q, bytes ? bytes : 8) != hipSuccess) {
            sphx_set_error("hipMalloc failed for the Barnes-Hut tree");
            return SPHX_ERR_NOMEM;
        }
        owned.push_back(q);
        *ptr = q;
        return SPHX_OK;
    }
};

static int bh_alloc_nodes(BhHost &H, int64_t need) {
    if (need <= H.cap) return SPHX_OK;
    int64_t cap = std::max<int64_t>(need, 2 * H.cap);
    BhTree T{};
    int32_t **ip[] = {&T.beg, &T.cnt, &T.child, &T.nchild};
    double **dp[] = {&T.mass, &T.emax};
    for (int32_t **q : ip) SPHX_CHECK(H.alloc((void **)q, sizeof(int32_t) * cap));
    for (double **q : dp) SPHX_CHECK(H.alloc((void **)q, sizeof(double) * cap));
    SPHX_CHECK(H.alloc((void **)&T.mono, sizeof(BhMono) * cap));
    SPHX_CHECK(H.alloc((void **)&T.link, sizeof(BhLink) * cap));
    SPHX_CHECK(H.alloc((void **)&T.ncell, sizeof(int32_t) * (BH_LEVELS + 3)));
    T.cap = cap;
    H.T = T;
    H.cap = cap;
    return SPHX_OK;
}

// Build the octree and walk it for every particle of the engine (single run,
// Morton-sorted, eps in E.s.eps); accelerations into E.s.gx..gz, potential
// into E.s.pot when with_pot.
int sphx_bh_run(Engine &E, BhHost &H, double theta, bool with_pot, hipStream_t st, BhStats *out) {
    int64_t n = E.n;
    if (n == 0) return SPHX_OK;
    if (E.R != 1 || E.max_runs != 1 || E.rrun >= 0) {
        sphx_set_error("Barnes-Hut gravity needs a single-run engine");
        return SPHX_ERR_STATE;
    }
    const double *eps = E.p.eps_from_h ? E.s.h : E.s.eps;
    hipEvent_t ev[3];
    for (auto &e : ev) SPHX_HIP(hipEventCreate(&e));
    struct EvFree {
        hipEvent_t *e;
        ~EvFree() {
            for (int k = 0; k < 3; ++k) hipEventDestroy(e[k]);
        }
    } evfree{ev};
    SPHX_HIP(hipEventRecord(ev[0], st));
    SPHX_CHECK(bh_alloc_nodes(H, std::max<int64_t>(1024, n / 2)));
    if (!H.stats) SPHX_CHECK(H.alloc((void **)&H.stats, sizeof(int64_t) * 4));
    const double *rbox = E.bbox + 6 * (int64_t)E.t.ns;
    // Levels 0 to top are built, summed and cut into groups without waiting for
    // their counts, seven levels more than a uniform cloud takes (an empty level
    // costs 5 us, a wait 20).  A deeper tree is split on, summed and cut again,
    // and built anew where the arrays do not hold its cells.
    int top = 6, from = 0;
    for (int64_t c = 8; c < n; c *= 8) ++top;
    top = std::min(top, 21);
    int32_t ncell[BH_LEVELS], ng[3] = {0, 0, 0};
    int64_t nodes = 0;
    for (;;) {
        // at most 8^level cells, of the nodes that the arrays hold
        auto blocks = [&](int level, int per) {
            const int64_t c = level < 7 ? (int64_t)1 << (3 * level) : H.cap;
            return (unsigned)std::min<int64_t>((std::min(c, H.cap) + per - 1) / per, 4096);
        };
        const int64_t gneed = H.cap + n / 64 + 1;
        // Items of groups in parts: eight groups at most of a cell of c >= 2 BH_PART
        // particles, at every level, take c / BH_PART + BH_OUT.
        H.g.share = bh_share(n);
        const int64_t pneed = (H.g.share > 1 ? gneed * H.g.share : 1) +
                              8 * (n / BH_PART) * (BH_OUT / 2 + 1) * (top + 1);
        if (gneed > H.gcap) {
            SPHX_CHECK(H.alloc((void **)&H.g.beg, sizeof(int32_t) * gneed));
            SPHX_CHECK(H.alloc((void **)&H.g.cnt, sizeof(int32_t) * gneed));
            H.gcap = gneed;
        }
        if (pneed > H.icap) {
            SPHX_CHECK(H.alloc((void **)&H.g.part, sizeof(int4) * pneed));
            H.icap = pneed;
        }
        H.g.count = H.T.ncell + BH_LEVELS;
        k_bh_root<<<1, 64, 0, st>>>(H.T, (int32_t)n, from == 0, H.g.count, H.stats);
        for (int l = from; l <= top; ++l) k_bh_split<<<blocks(l, BHT / 8), BHT, 0, st>>>(H.T, E.keys, l);
        for (int l = top; l >= 0; --l)
            k_bh_moments<<<blocks(l, BHT), BHT, 0, st>>>(H.T, l, E.keys, E.s.x, E.s.y, E.s.z, E.s.m, eps, rbox);
        k_bh_groups<<<blocks(7, BHT), BHT, 0, st>>>(H.T, top, H.g);
        SPHX_HIP(hipGetLastError());
        int32_t back[BH_LEVELS + 3];
        SPHX_HIP(hipMemcpyAsync(back, H.T.ncell, sizeof(back), hipMemcpyDeviceToHost, st));
        SPHX_HIP(hipStreamSynchronize(st));
        std::copy(back, back + BH_LEVELS, ncell);
        std::copy(back + BH_LEVELS, back + BH_LEVELS + 3, ng);
        nodes = 0;
        for (int32_t c : ncell) nodes += c;
        if (nodes <= H.cap && (top == 21 || ncell[top + 1] == 0)) {
            if (ng[0] < 0 || ng[0] > gneed || ng[1] < 0 || ng[1] > pneed || ng[0] + ng[1] == 0) {
                sphx_set_error("Barnes-Hut group list inconsistent with the tree");
                return SPHX_ERR_STATE;
            }
            break;
        }
        from = top + 1;
        if (nodes > H.cap) {
            SPHX_CHECK(bh_alloc_nodes(H, nodes + nodes / 4));
            from = 0;
        }
        top = std::min(top + 4, 21);
    }
    // levels up to the first empty one
    int depth = 1;
    while (depth < 21 && ncell[depth] > 0) ++depth;
    if (ng[1] > H.pcap) {
        const int64_t c = std::max<int64_t>(ng[1], 2 * H.pcap);
        SPHX_CHECK(H.alloc((void **)&H.psum, sizeof(double4) * 64 * c));
        H.pcap = c;
    }
    SPHX_HIP(hipEventRecord(ev[1], st));
    BhArgs a{E.s.x, E.s.y, E.s.z, E.s.m, eps, H.g.beg, H.g.cnt, H.g.part, ng[1], H.psum, n, E.p.G, theta,
             E.s.gx, E.s.gy, E.s.gz, with_pot ? E.s.pot : nullptr, H.stats,
             E.counters + CNT_BH_OVERFLOW};
    const bool deep = theta < BH_DEEP_THETA;
    const unsigned grid = (unsigned)(ng[0] + ng[1]);
    if (with_pot && deep) k_bh_walk<true, BH_SCAP_DEEP><<<grid, 64, 0, st>>>(H.T, a);
    else if (with_pot) k_bh_walk<true, BH_SCAP><<<grid, 64, 0, st>>>(H.T, a);
    else if (deep) k_bh_walk<false, BH_SCAP_DEEP><<<grid, 64, 0, st>>>(H.T, a);
    else k_bh_walk<false, BH_SCAP><<<grid, 64, 0, st>>>(H.T, a);
    if (ng[1] > 0) {
        if (with_pot) k_bh_join<true><<<(unsigned)ng[1], 64, 0, st>>>(a);
        else k_bh_join<false><<<(unsigned)ng[1], 64, 0, st>>>(a);
    }
    SPHX_HIP(hipGetLastError());
    SPHX_HIP(hipEventRecord(ev[2], st));
    if (out) {
        int64_t sv[4] = {0, 0, 0, 0};
        SPHX_HIP(hipMemcpyAsync(sv, H.stats, sizeof(sv), hipMemcpyDeviceToHost, st));
        SPHX_HIP(hipStreamSynchronize(st));
        out->nodes = nodes;
        out->depth = depth;
        out->interactions = sv[0];
        out->overflow = sv[1];
        out->max_fill = sv[2];
        out->groups = ng[0] + ng[2];
        float b = 0.f, w = 0.f;
        SPHX_HIP(hipEventElapsedTime(&b, ev[0], ev[1]));
        SPHX_HIP(hipEventElapsedTime(&w, ev[1], ev[2]));
        out->build_ms = b;
        out->walk_ms = w;
    }
    return SPHX_OK;
}

BhHost *sphx_bh_host_new() { return new BhHost(); }
void sphx_bh_host_free(BhHost *h) { delete h; }
