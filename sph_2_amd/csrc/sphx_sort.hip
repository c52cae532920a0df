// Morton keys, stable merge sort, permutation gather and bucket boxes.
//
// Replaces the reference's neighbour structures (counting-sort cells of
// Particles_in_BH_Tree_II/Evrard_test/ngb_v3.h:58-117, atomics-filled grid
// cells of Particles_in_Gridcells/final_revision_uniform_grid/
// hfvCLibs_v7_grid_v0.h:680-708) with Morton-ordered 64-particle buckets:
// one wavefront per bucket, bucket and super-bucket AABBs for culling.
#include <utility>

#include "sphx_internal.h"

namespace {

__device__ __forceinline__ uint64_t spread3(uint64_t v) {
    // Spread the low 21 bits of v so bit b lands at bit 3b.
    v &= 0x1fffffull;
    v = (v | (v << 32)) & 0x1f00000000ffffull;
    v = (v | (v << 16)) & 0x1f0000ff0000ffull;
    v = (v | (v << 8)) & 0x100f00f00f00f00full;
    v = (v | (v << 4)) & 0x10c30c30c30c30c3ull;
    v = (v | (v << 2)) & 0x1249249249249249ull;
    return v;
}

// Bounding box of each super-bucket straight from the particles (before the
// sort, in the current order; supers never straddle runs).
__global__ __launch_bounds__(1024) void k_super_box_pos(Tables t, const double *__restrict__ x,
                                                       const double *__restrict__ y,
                                                       const double *__restrict__ z,
                                                       double *__restrict__ out /* 6 per super */) {
    __shared__ double part[16][6];
    const int sidx = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int b0 = t.s_bbeg[sidx], b1 = t.s_bend[sidx];
    const int p0 = t.b_beg[b0];
    const int p1 = t.b_beg[b1 - 1] + t.b_cnt[b1 - 1];
    double v[6] = {INFINITY, -INFINITY, INFINITY, -INFINITY, INFINITY, -INFINITY};
    for (int i = p0 + tid; i < p1; i += 1024) {
        const double a = x[i], b = y[i], c = z[i];
        v[0] = fmin(v[0], a); v[1] = fmax(v[1], a);
        v[2] = fmin(v[2], b); v[3] = fmax(v[3], b);
        v[4] = fmin(v[4], c); v[5] = fmax(v[5], c);
    }
    for (int k = 0; k < 6; k += 2) {
        v[k] = wave_min_d(v[k]);
        v[k + 1] = wave_max_d(v[k + 1]);
    }
    if (lane == 0)
        for (int k = 0; k < 6; ++k) part[w][k] = v[k];
    __syncthreads();
    if (tid < 6) {
        double r = part[0][tid];
        for (int q = 1; q < 16; ++q) r = (tid & 1) ? fmax(r, part[q][tid]) : fmin(r, part[q][tid]);
        out[6 * sidx + tid] = r;
    }
}

// Per-run bounding box from the super boxes; one wavefront per run.
__global__ void k_run_box(Tables t, const double *__restrict__ sbox, double *__restrict__ rbox) {
    int r = blockIdx.x;
    int lane = threadIdx.x;
    double v[6] = {INFINITY, -INFINITY, INFINITY, -INFINITY, INFINITY, -INFINITY};
    for (int s = t.r_sbeg[r] + lane; s < t.r_send[r]; s += 64) {
        for (int a = 0; a < 6; a += 2) {
            v[a] = fmin(v[a], sbox[6 * s + a]);
            v[a + 1] = fmax(v[a + 1], sbox[6 * s + a + 1]);
        }
    }
    for (int a = 0; a < 6; a += 2) {
        v[a] = wave_min_d(v[a]);
        v[a + 1] = wave_max_d(v[a + 1]);
    }
    if (lane == 0)
        for (int a = 0; a < 6; ++a) rbox[6 * r + a] = v[a];
}

// key = run << (3*bits) | interleave(ix, iy, iz); ix = floor((x - lo) * scale)
// clamped to [0, 2^bits - 1], scale = 2^bits / (extent * (1 + 2^-30)) over the
// run's cubic box.  All FP64, separately rounded.
struct MortonIn {
    const double *x, *y, *z;
    const int32_t *run;  // null: one run
    const double *rbox;
    int bits;
};
__device__ __forceinline__ uint64_t morton_key(const MortonIn &in, int64_t i) {
#pragma clang fp contract(off)
    int r = in.run ? in.run[i] : 0;
    const double *b = in.rbox + 6 * r;
    double ex = b[1] - b[0], ey = b[3] - b[2], ez = b[5] - b[4];
    double ext = fmax(ex, fmax(ey, ez));
    double cells = (double)(1ull << in.bits);
    double scale = ext > 0.0 ? cells / (ext * (1.0 + 0x1p-30)) : 0.0;
    uint64_t maxc = (1ull << in.bits) - 1ull;
    double fx = (in.x[i] - b[0]) * scale, fy = (in.y[i] - b[2]) * scale, fz = (in.z[i] - b[4]) * scale;
    uint64_t ix = fx <= 0.0 ? 0ull : (uint64_t)fx;
    uint64_t iy = fy <= 0.0 ? 0ull : (uint64_t)fy;
    uint64_t iz = fz <= 0.0 ? 0ull : (uint64_t)fz;
    ix = ix > maxc ? maxc : ix;
    iy = iy > maxc ? maxc : iy;
    iz = iz > maxc ? maxc : iz;
    uint64_t key = (spread3(ix) << 2) | (spread3(iy) << 1) | spread3(iz);
    return key | ((uint64_t)r) << (3 * in.bits);
}

__global__ void k_morton(MortonIn in, int64_t n, uint64_t *__restrict__ keys) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) keys[i] = morton_key(in, i);
}

// ---------------------------------------------------------------------------
// Stable sort of (key, value) by the 63-bit key: tiles of 4,096 sorted in LDS,
// then merged pairwise.  What bounds the sort of a run is launches and the
// chain of dependent memory trips, not bandwidth (24 bytes a particle and pass),
// so it is a merge sort: one launch for the tiles, which also make the keys
// from the positions, and one per doubling, against the 32 of an eight-pass
// radix sort (histogram, two scans and scatter each).  Half kick, drift, keys,
// sort and gather together: 141 -> 49 us at 4,096 particles, 153 -> 78 at
// 65,752, 162 -> 83 at 131,072, 360 -> 213 at 1,048,576.
// ---------------------------------------------------------------------------
constexpr int ST_TILE = 4096, ST_THREADS = 1024, ST_ITEMS = ST_TILE / ST_THREADS;
constexpr int MG_CHUNK = 1024, MG_THREADS = 256, MG_ITEMS = MG_CHUNK / MG_THREADS;
static_assert(ST_ITEMS == 4 && MG_ITEMS == 4, "four items a thread");
static_assert((2 * ST_TILE) % MG_CHUNK == 0, "a chunk lies inside one pair of runs");

// How many of the first d outputs of the stable merge of A[0, nA) and B[0, nB)
// come from A (equal keys: A first).
__device__ __forceinline__ int merge_split(const uint64_t *A, int nA, const uint64_t *B, int nB, int d) {
    int lo = d > nB ? d - nB : 0, hi = d < nA ? d : nA;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (A[mid] <= B[d - 1 - mid]) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// Four consecutive outputs of the merge from (a, b) on: their indices into
// [A | B], with B at offset offB of the same array.
__device__ __forceinline__ void merge_four(const uint64_t *A, int nA, const uint64_t *B, int nB, int a,
                                           int b, int offB, uint64_t *key, int *at) {
    uint64_t ka = a < nA ? A[a] : ~0ull, kb = b < nB ? B[b] : ~0ull;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const bool ta = b >= nB || (a < nA && ka <= kb);
        key[k] = ta ? ka : kb;
        at[k] = ta ? a : offB + b;
        if (ta) {
            ++a;
            ka = a < nA ? A[a] : ~0ull;
        } else {
            ++b;
            kb = b < nB ? B[b] : ~0ull;
        }
    }
}

// One tile per workgroup, four items a thread: sorted in registers, then merged
// in LDS, doubling from runs of four.  Item i's value is v0 + i; MAKE makes the
// keys from the positions, else they come from kin (which may be kout: a
// workgroup has its tile in LDS before it writes it).
template <bool MAKE>
__global__ __launch_bounds__(ST_THREADS) void k_sort_tiles(MortonIn in, const uint64_t *kin, int64_t n,
                                                           int32_t v0, uint64_t *kout,
                                                           int32_t *__restrict__ vout) {
    __shared__ uint64_t K[ST_TILE];
    __shared__ uint16_t P[ST_TILE];  // position in the tile
    const int tid = threadIdx.x;
    const int64_t base = (int64_t)blockIdx.x * ST_TILE;
    const int cnt = (int)(n - base < ST_TILE ? n - base : ST_TILE);
    uint64_t key[4];
    int at[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int q = 4 * tid + k;
        at[k] = q;
        key[k] = ~0ull;  // past the end: after every key (keys have 63 bits)
        if (q < cnt) key[k] = MAKE ? morton_key(in, base + q) : kin[base + q];
    }
    auto order = [&](int i, int j) {
        const bool sw = key[j] < key[i] || (key[j] == key[i] && at[j] < at[i]);
        const uint64_t ki = sw ? key[j] : key[i], kj = sw ? key[i] : key[j];
        const int pi = sw ? at[j] : at[i], pj = sw ? at[i] : at[j];
        key[i] = ki; key[j] = kj; at[i] = pi; at[j] = pj;
    };
    order(0, 1); order(2, 3); order(0, 2); order(1, 3); order(1, 2);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        K[4 * tid + k] = key[k];
        P[4 * tid + k] = (uint16_t)at[k];
    }
    __syncthreads();
    for (int w = 4; w < cnt; w <<= 1) {
        const int s = (4 * tid) / (2 * w) * (2 * w), d = 4 * tid - s;
        const uint64_t *A = K + s, *B = K + s + w;
        const int a = merge_split(A, w, B, w, d);
        int idx[4];
        merge_four(A, w, B, w, a, d - a, w, key, idx);
#pragma unroll
        for (int k = 0; k < 4; ++k) at[k] = P[s + idx[k]];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            K[4 * tid + k] = key[k];
            P[4 * tid + k] = (uint16_t)at[k];
        }
        __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int q = 4 * tid + k;
        if (q < cnt) {
            kout[base + q] = key[k];
            vout[base + q] = v0 + (int32_t)base + at[k];
        }
    }
}

// merge_split over global memory by one wavefront, 64 probes at a time.
__device__ __forceinline__ int merge_split_wave(const uint64_t *A, int nA, const uint64_t *B, int nB,
                                                int d, int lane) {
    int lo = d > nB ? d - nB : 0, hi = d < nA ? d : nA;
    while (lo < hi) {
        const int step = (hi - lo + 63) / 64;
        const int b = lo + lane * step;                    // this lane's piece of [lo, hi)
        const int e = (b + step < hi ? b + step : hi) - 1;  // its last index
        // pieces whose last element is among A's come first
        const int c = __popcll(__ballot(b < hi && A[b < hi ? e : lo] <= B[d - 1 - (b < hi ? e : lo)]));
        lo += c * step;
        if (lo >= hi) return hi;
        hi = (lo + step < hi ? lo + step : hi) - 1;  // known not to be among A's
    }
    return lo;
}

// One pass: runs of `len` merged pairwise, 1,024 outputs per workgroup.
__global__ __launch_bounds__(MG_THREADS) void k_merge(const uint64_t *__restrict__ kin,
                                                      const int32_t *__restrict__ vin, int64_t n,
                                                      int64_t len, uint64_t *__restrict__ kout,
                                                      int32_t *__restrict__ vout) {
    __shared__ uint64_t K[MG_CHUNK];
    __shared__ int32_t V[MG_CHUNK];
    __shared__ int split[2];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int64_t base = (int64_t)blockIdx.x * MG_CHUNK;
    const int64_t s = base / (2 * len) * (2 * len);
    const int nA = (int)(n - s < len ? n - s : len);
    const int64_t rest = n - s - nA;
    const int nB = (int)(rest < len ? rest : len);
    const uint64_t *A = kin + s, *B = A + nA;
    const int d0 = (int)(base - s), d1 = d0 + MG_CHUNK < nA + nB ? d0 + MG_CHUNK : nA + nB;
    if (w < 2) {
        const int a = merge_split_wave(A, nA, B, nB, w == 0 ? d0 : d1, lane);
        if (lane == 0) split[w] = a;
    }
    __syncthreads();
    const int a0 = split[0], ca = split[1] - a0, b0 = d0 - a0, cb = (d1 - d0) - ca;
    for (int q = tid; q < ca + cb; q += MG_THREADS) {
        const int64_t g = s + (q < ca ? a0 + q : nA + b0 + (q - ca));
        K[q] = kin[g];
        V[q] = vin[g];
    }
    __syncthreads();
    const int d = 4 * tid;
    if (d >= ca + cb) return;
    const int a = merge_split(K, ca, K + ca, cb, d);
    uint64_t key[4];
    int idx[4];
    merge_four(K, ca, K + ca, cb, a, d - a, ca, key, idx);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        if (d + k < ca + cb) {
            kout[base + d + k] = key[k];
            vout[base + d + k] = V[idx[k]];
        }
    }
}

struct GatherList {
    const double *src[16];
    double *dst[16];
    const int32_t *isrc[4];
    int32_t *idst[4];
    int nd, ni;
};

// The gather of the sort, one wave per bucket, with the bucket's box from the
// positions it has in hand (the boxes the smoothing walk reads; a launch less).
__global__ __launch_bounds__(64) void k_gather(GatherList g, const int32_t *__restrict__ perm,
                                               Tables t) {
    const int b = blockIdx.x, lane = threadIdx.x;
    const bool ok = lane < t.b_cnt[b];
    const int i = t.b_beg[b] + lane;
    const int32_t p = ok ? perm[i] : 0;
    double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    if (ok) {
        for (int a = 0; a < 3; ++a) {  // x, y, z
            const double v = g.src[a][p];
            g.dst[a][i] = v;
            lo[a] = hi[a] = v;
        }
        for (int a = 3; a < g.nd; ++a) g.dst[a][i] = g.src[a][p];
        for (int a = 0; a < g.ni; ++a) g.idst[a][i] = g.isrc[a][p];
    }
    for (int a = 0; a < 3; ++a) {
        lo[a] = wave_min_d(lo[a]);
        hi[a] = wave_max_d(hi[a]);
    }
    if (lane == 0) {
        t.bxl[b] = lo[0]; t.bxh[b] = hi[0];
        t.byl[b] = lo[1]; t.byh[b] = hi[1];
        t.bzl[b] = lo[2]; t.bzh[b] = hi[2];
    }
}

// Box and largest h and softening of each 64-particle bucket: one wave each.
__global__ __launch_bounds__(64) void k_bucket_boxes(Tables t, const double *__restrict__ x,
                                                     const double *__restrict__ y,
                                                     const double *__restrict__ z,
                                                     const double *__restrict__ h,
                                                     const double *__restrict__ eps, int with_h) {
    const int b = blockIdx.x, lane = threadIdx.x;
    const int cnt = t.b_cnt[b];
    const int i = t.b_beg[b] + lane;
    const bool ok = lane < cnt;
    double a = ok ? x[i] : INFINITY, bb = ok ? y[i] : INFINITY, c = ok ? z[i] : INFINITY;
    const double xl = wave_min_d(a), yl = wave_min_d(bb), zl = wave_min_d(c);
    a = ok ? x[i] : -INFINITY; bb = ok ? y[i] : -INFINITY; c = ok ? z[i] : -INFINITY;
    const double xh = wave_max_d(a), yh = wave_max_d(bb), zh = wave_max_d(c);
    double hm = 0.0, em = 0.0;
    if (with_h) {
        hm = wave_max_d(ok ? h[i] : 0.0);
        em = wave_max_d(ok ? (eps ? eps[i] : h[i]) : 0.0);
    }
    if (lane == 0) {
        t.bxl[b] = xl; t.bxh[b] = xh; t.byl[b] = yl; t.byh[b] = yh;
        t.bzl[b] = zl; t.bzh[b] = zh;
        if (with_h) { t.bhmax[b] = hm; t.bemax[b] = em; }
    }
}

// Box and largest h of each super (up to SPHX_SUPER consecutive buckets) from
// its buckets' boxes: lane k takes buckets k, k + 64, ... of the super.
__global__ __launch_bounds__(64) void k_super_boxes(Tables t, int with_h) {
    const int sidx = blockIdx.x, lane = threadIdx.x;
    double S[7] = {INFINITY, -INFINITY, INFINITY, -INFINITY, INFINITY, -INFINITY, 0.0};
    for (int b = t.s_bbeg[sidx] + lane; b < t.s_bend[sidx]; b += 64) {
        S[0] = fmin(S[0], t.bxl[b]); S[1] = fmax(S[1], t.bxh[b]);
        S[2] = fmin(S[2], t.byl[b]); S[3] = fmax(S[3], t.byh[b]);
        S[4] = fmin(S[4], t.bzl[b]); S[5] = fmax(S[5], t.bzh[b]);
        if (with_h) S[6] = fmax(S[6], t.bhmax[b]);
    }
    const double xl = wave_min_d(S[0]), xh = wave_max_d(S[1]), yl = wave_min_d(S[2]),
                 yh = wave_max_d(S[3]), zl = wave_min_d(S[4]), zh = wave_max_d(S[5]);
    const double hm = with_h ? wave_max_d(S[6]) : 0.0;
    if (lane == 0) {
        t.sxl[sidx] = xl; t.sxh[sidx] = xh; t.syl[sidx] = yl; t.syh[sidx] = yh;
        t.szl[sidx] = zl; t.szh[sidx] = zh;
        if (with_h) t.shmax[sidx] = hm;
    }
}

__global__ void k_aos_to_soa(const double *__restrict__ a, int64_t n, double *__restrict__ x,
                             double *__restrict__ y, double *__restrict__ z) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    x[i] = a[3 * i];
    y[i] = a[3 * i + 1];
    z[i] = a[3 * i + 2];
}

__global__ void k_soa_to_aos(const double *__restrict__ x, const double *__restrict__ y,
                             const double *__restrict__ z, int64_t n, double *__restrict__ a) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    a[3 * i] = x[i];
    a[3 * i + 1] = y[i];
    a[3 * i + 2] = z[i];
}

inline unsigned grid_for(int64_t n, int threads) { return (unsigned)((n + threads - 1) / threads); }

}  // namespace

int sphx_aos_to_soa(const double *aos, int64_t n, double *x, double *y, double *z,
                    hipStream_t st) {
    if (n <= 0) return SPHX_OK;
    k_aos_to_soa<<<grid_for(n, 256), 256, 0, st>>>(aos, n, x, y, z);
    SPHX_HIP(hipGetLastError());
    return SPHX_OK;
}

int sphx_soa_to_aos(const double *x, const double *y, const double *z, int64_t n, double *aos,
                    hipStream_t st) {
    if (n <= 0) return SPHX_OK;
    k_soa_to_aos<<<grid_for(n, 256), 256, 0, st>>>(x, y, z, n, aos);
    SPHX_HIP(hipGetLastError());
    return SPHX_OK;
}

// Passes of pairwise merges over n items.
static int merge_passes(int64_t n) {
    int m = 0;
    while (((int64_t)ST_TILE << m) < n) ++m;
    return m;
}

// Merge the sorted tiles in (ka, va) until one run is left; it ends in ka / va
// after an even number of passes, else in kb / vb.
static int merge_tiles(uint64_t *ka, int32_t *va, uint64_t *kb, int32_t *vb, int64_t n, hipStream_t st) {
    const unsigned grid = grid_for(n, MG_CHUNK);
    for (int64_t len = ST_TILE; len < n; len <<= 1) {
        k_merge<<<grid, MG_THREADS, 0, st>>>(ka, va, n, len, kb, vb);
        std::swap(ka, kb);
        std::swap(va, vb);
    }
    SPHX_HIP(hipGetLastError());
    return SPHX_OK;
}

// Sort n keys in place with their indices, counted from v0, in vals; the other
// two arrays are scratch.
int sphx_sort_keys(uint64_t *keys, int32_t *vals, uint64_t *keys_tmp, int32_t *vals_tmp, int64_t n,
                   int32_t v0, hipStream_t st) {
    if (n <= 0) return SPHX_OK;
    const bool odd = merge_passes(n) & 1;
    uint64_t *ka = odd ? keys_tmp : keys, *kb = odd ? keys : keys_tmp;
    int32_t *va = odd ? vals_tmp : vals, *vb = odd ? vals : vals_tmp;
    k_sort_tiles<false><<<grid_for(n, ST_TILE), ST_THREADS, 0, st>>>(MortonIn{}, keys, n, v0, ka, va);
    SPHX_HIP(hipGetLastError());
    return merge_tiles(ka, va, kb, vb, n, st);
}

static int run_bits(int max_runs) {
    int rb = 0;
    while ((1 << rb) < max_runs) ++rb;
    return rb;
}

// Bits per axis: 21 for a lone run; fewer when run ids share the 63-bit key.
// Depends on the engine's run capacity only, so a run sorts the same way
// whether it is alone or packed with others.
int sphx_morton_bits(int max_runs) {
    int b = (63 - run_bits(max_runs)) / 3;
    return b > 21 ? 21 : b;
}

// Boxes of the runs (E.bbox), and where their keys come from.
static int morton_in(Engine &E, MortonIn *in, hipStream_t st) {
    Tables &t = E.t;
    double *sbox = E.bbox;                 // 6 per super
    double *rbox = E.bbox + 6 * (int64_t)t.ns;  // 6 per run
    k_super_box_pos<<<t.ns, 1024, 0, st>>>(t, E.s.x, E.s.y, E.s.z, sbox);
    k_run_box<<<t.R, 64, 0, st>>>(t, sbox, rbox);
    SPHX_HIP(hipGetLastError());
    *in = MortonIn{E.s.x, E.s.y, E.s.z, E.max_runs > 1 ? E.s.run : nullptr, rbox,
                   sphx_morton_bits(E.max_runs)};
    return SPHX_OK;
}

// Unsorted keys of every particle.
int sphx_launch_morton(Engine &E, hipStream_t st) {
    MortonIn in;
    SPHX_CHECK(morton_in(E, &in, st));
    k_morton<<<grid_for(E.n, 256), 256, 0, st>>>(in, E.n, E.keys);
    SPHX_HIP(hipGetLastError());
    return SPHX_OK;
}

// Persistent arrays gathered by the sort, and the derived arrays that serve
// as their destinations (recomputed after every sort).  After the gather the
// roles swap; applying the swap twice restores the original assignment.
static void sort_roles(Engine &E, double **dst[12], double **spare[12], int32_t **idst[4],
                       int32_t **ispare[4]) {
    Soa &s = E.s;
    double **d[12] = {&s.x, &s.y, &s.z, &s.vx, &s.vy, &s.vz, &s.u, &s.m,
                      &s.h, &s.eps, &s.ut_prev, &s.divv};
    double **sp[12] = {&s.gx, &s.gy, &s.gz, &s.rho, &s.P, &s.c, &s.curlv, &s.du,
                       &s.pot, &s.ax, &s.ay, &s.az};
    int32_t **id[4] = {&s.k, &s.id, &s.run, &s.bin};
    int32_t **isp[4] = {&E.tmpi, &E.perm2, &E.h_iters, &E.bin_spare};
    for (int a = 0; a < 12; ++a) { dst[a] = d[a]; spare[a] = sp[a]; }
    for (int a = 0; a < 4; ++a) { idst[a] = id[a]; ispare[a] = isp[a]; }
}

void Engine::swap_sorted() {
    double **d[12], **sp[12];
    int32_t **id[4], **isp[4];
    sort_roles(*this, d, sp, id, isp);
    for (int a = 0; a < 12; ++a) std::swap(*d[a], *sp[a]);
    for (int a = 0; a < 4; ++a) std::swap(*id[a], *isp[a]);
    gpar ^= 1;
}

int Engine::sort_and_permute(hipStream_t st, bool gather_state) {
    if (n == 0) return SPHX_OK;
    MortonIn in;
    SPHX_CHECK(morton_in(*this, &in, st));
    const bool odd = merge_passes(n) & 1;
    uint64_t *ka = odd ? keys2 : keys, *kb = odd ? keys : keys2;
    int32_t *va = odd ? perm2 : perm, *vb = odd ? perm : perm2;
    k_sort_tiles<true><<<grid_for(n, ST_TILE), ST_THREADS, 0, st>>>(in, nullptr, n, 0, ka, va);
    SPHX_HIP(hipGetLastError());
    SPHX_CHECK(merge_tiles(ka, va, kb, vb, n, st));
    if (!gather_state) return SPHX_OK;
    double **d[12], **sp[12];
    int32_t **id[4], **isp[4];
    sort_roles(*this, d, sp, id, isp);
    GatherList g{};
    g.nd = 12;
    g.ni = 4;
    for (int a = 0; a < 12; ++a) {
        g.src[a] = *d[a];
        g.dst[a] = *sp[a];
    }
    for (int a = 0; a < 4; ++a) {
        g.isrc[a] = *id[a];
        g.idst[a] = *isp[a];
    }
    k_gather<<<t.nb, 64, 0, st>>>(g, perm, t);
    SPHX_HIP(hipGetLastError());
    swap_sorted();
    sorted_boxes = true;
    return SPHX_OK;
}

int Engine::build_boxes(hipStream_t st, bool with_h) {
    if (n == 0) return SPHX_OK;
    const double *e = p.eps_from_h ? nullptr : s.eps;
    // right after a sort the gather has left the buckets' boxes
    if (with_h || !sorted_boxes)
        k_bucket_boxes<<<t.nb, 64, 0, st>>>(t, s.x, s.y, s.z, s.h, e, with_h ? 1 : 0);
    sorted_boxes = false;
    k_super_boxes<<<t.ns, 64, 0, st>>>(t, with_h ? 1 : 0);
    SPHX_HIP(hipGetLastError());
    return SPHX_OK;
}
