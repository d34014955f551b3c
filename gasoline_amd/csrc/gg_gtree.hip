// Gravity tree build on the device: the tree of gasoline's pkdBuildBinary
// (pkd.c:2627-2723), node for node.
//
// Cells split in three stages: those of more than 4096 particles level by
// level over the whole chip, then each cell of at most 4096 in one workgroup
// down to 512, then each of at most 512 in another, which also makes that
// subtree's records.  Every cell is split at the midpoint of the longest axis
// of its particles' bounding box (pkd.c:2493-2505) unless it holds nBucket
// particles or fewer or has no extent (pkd.c:2489).  The partition reproduces
// pkdUpperPart's Hoare scan (pkd.c:1109-1157): a Hoare scan swaps the k-th
// particle of the lower part that belongs above with the k-th particle,
// counted from the top, of the upper part that belongs below, so each
// particle's destination follows from prefix counts.  pkdActiveTypeOrder's
// partitions (pkd.c:1304-1355) run the same way over each system.  Cells get
// their preorder ids from subtree sizes, which climb from the buckets with
// the records.  Mass, softening and centre of mass are summed as the
// reference sums them (buckets over their particles in storage order, cells
// from their children, lower then upper), and bounds, Bmax and fOpen2 are
// exact, so every quantity the walk decides on is the reference's to the
// bit.  The multipole moments (pkdCalcCell, pkd.c:2018-2135) are sums over a
// bucket's particles and, above, the children's moved to the cell's centre;
// they enter only the force arithmetic, which they change by 1e-16 of itself
// against sums over every cell's particles.
//
// Several independent systems build at once: each is a root of its own.
#include "gg_internal.h"

#include <algorithm>
#include <cfloat>
#include <climits>
#include <cmath>
#include <type_traits>
#include <vector>

namespace gg {
namespace {

int nblk(int64_t n, int b) { return (int)((n + b - 1) / b); }

constexpr int LMAX = 512;        // cells of at most LMAX particles finish in one workgroup
constexpr int LSML = 128;        // systems of at most LSML particles finish in one wavefront
constexpr int MID = 4096;        // cells of at most MID particles reach LMAX in one workgroup
constexpr int DMAX = 2048;       // levels above MID a tree may have

// A cell, in a slot of its own: the cells above LMAX from slot 0 up, the
// subtrees of k_gt_sub from the last slot down, each in its preorder.
struct GNode {
    int lo, hi, par, root;       // particle range, parent and root slots
    int ch0, ch1, dim, s;        // children (-1), split axis (-1: bucket), split position
    int size, nab;               // cells and buckets with active particles of the subtree
    int pre, bpre;               // preorder id and bucket rank (within the subtree of
                                 // k_gt_sub; absolute for the cells of the level loop)
    int sizeLo, nabLo;           // the lower child's, above LMAX
    double split;
};

// Numeric record of a cell: mass, softening, centre of mass, the largest
// squared distance of a particle from it, and the raw moments about it of
// second (6: xx yy zz xy xz yz), third (10) and fourth (15) order.
constexpr int GM_B = 5, GM_Q = 6, GM_T = 12, GM_F = 22;
constexpr int gm_stride(int order) { return order >= 4 ? 37 : (order == 3 ? 22 : 12); }

// ------------------------------------------------------------ levels
// Cells of more than MID particles split level by level over tiles of ts
// particles; each tile lies in one cell of the level.  A level takes four
// launches: k_gt_ctl (one workgroup: split decisions, child ids, the tile
// list), k_gt_count (each tile's lower-part flags as bits, and their number),
// k_gt_rank (the upper part's misplaced particles by rank) and k_gt_swap (the
// Hoare swaps, and the children's bounds as the particles pass through
// registers).  Only particles of cells that still split are read.  Cells of
// at most MID particles are left to k_gt_mid.
struct GLevel {
    int a, b;            // cells of the level: ids a..b-1
    int ntile;           // tiles of its splitting cells
    int nunit;           // cells left to k_gt_mid so far
    int next;            // slots taken from the first one up
    int nloc;            // slots taken from the last one down
    int nsub;            // cells left to k_gt_sub
    int err;             // 1: a split left one side empty, 2: out of slots
    int need;            // a particle lacks the type bit of the orders
    int maxb;            // largest bucket
    int lv[DMAX + 1];    // first cell of each level
};

// Doubles as unsigned integers of the same order, for atomic min and max.
__device__ __forceinline__ unsigned long long ord_key(double v)
{
    const long long b = __double_as_longlong(v);
    return (unsigned long long)(b < 0 ? ~b : (b | (long long)0x8000000000000000ull));
}

__device__ __forceinline__ double ord_val(unsigned long long k)
{
    const long long b = (long long)k;
    return __longlong_as_double(b < 0 ? (b & 0x7fffffffffffffffll) : ~b);
}

// A cell's bounds while its particles are still being scanned: six keys, each
// in a 128-byte line of its own.  Every tile of a cell adds to its six, and
// atomics on one line are served one after another: side by side they made
// k_gt_swap take 53 us on the root of 2^21 particles, 35 in lines of their own.
constexpr int BOX_S = 16, BOX_N = 6 * BOX_S;
__device__ __forceinline__ void box_init(unsigned long long *b)
{
    for (int d = 0; d < 3; ++d) {
        b[BOX_S * d] = ~0ull;
        b[BOX_S * (3 + d)] = 0ull;
    }
}

// The last of nr ascending first positions (or tiles) that is <= i.
__device__ __forceinline__ int root_of(int i, int nr, const int *__restrict__ rlo)
{
    int lo = 0, hi = nr - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (rlo[mid] <= i) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// The systems by size, so that a forest of very many small ones costs what
// its particles cost: those of more than MID particles are the cells of the
// first level (with bounds), those of more than LMAX go to k_gt_mid, those
// of more than nBucket to k_gt_sub (those of at most LSML first), and the
// rest are buckets (k_gt_tiny).  The host gives every 256 systems their first
// entries of the lists.  A single system is the whole store and has none of
// these arrays.
struct Roots {
    int n, nr, nBucket;
    int nbig, nunit, nsub[2], maxTiny;   // systems of each list, the largest bucket
    const int *lo, *hi;                  // particle ranges
    const int *bslot, *blo, *bhi;        // those of more than MID particles
    const int *base[3];                  // per 256 systems: nsub[0], nsub[1], nunit
    const int *tslot, *toff;             // those of more than LMAX: slot, first tile of the
    int ntroot;                          // type orders
};

// Root cells, their lists, the empty bounds and the level state.
__global__ __launch_bounds__(256) void k_gt_roots(Roots R, GNode *__restrict__ nd,
                                                  unsigned long long *__restrict__ box,
                                                  int *__restrict__ unit, int *__restrict__ sub,
                                                  GLevel *__restrict__ L)
{
    __shared__ int ws[4][3];
    const int k = blockIdx.x * 256 + threadIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (k == 0) {
        L->a = 0;
        L->b = L->next = R.nr;
        L->nunit = R.nunit;
        L->nsub = R.nsub[0] + R.nsub[1];
        L->maxb = R.maxTiny;
        L->ntile = L->nloc = L->err = L->need = 0;
    }
    if (k < R.nbig) box_init(box + BOX_N * (size_t)k);
    int cnt = 0;
    if (k < R.nr) {
        GNode &g = nd[k];
        g.lo = R.nr > 1 ? R.lo[k] : 0;
        g.hi = R.nr > 1 ? R.hi[k] : R.n - 1;
        g.par = -1;
        g.root = k;
        g.ch0 = g.ch1 = -1;
        g.dim = -1;
        g.split = 0.0;
        cnt = g.hi - g.lo + 1;
    }
    const int cls = cnt <= R.nBucket ? -1 : cnt <= LSML ? 0 : cnt <= LMAX ? 1 : cnt <= MID ? 2 : -1;
    unsigned long long m[3];
    for (int q = 0; q < 3; ++q) {
        m[q] = __ballot(cls == q);
        if (lane == 0) ws[w][q] = __popcll(m[q]);
    }
    __syncthreads();
    for (int q = 0; q < 3; ++q) {
        if (cls != q) continue;
        int at = (R.nr > 1 ? R.base[q][blockIdx.x] : 0) + __popcll(m[q] & ((1ull << lane) - 1));
        for (int v = 0; v < w; ++v) at += ws[v][q];
        if (q == 2) unit[at] = k;
        else sub[q ? R.nsub[0] + at : at] = k;
    }
}

// Min/max of a wavefront's lo/hi.  Lanes 0, 8, 16 return the lower bounds x,
// y, z, lanes 32, 40, 48 the upper ones.  The lanes share the six values out
// as the reduction goes (three, two, one each), so it takes 9 exchanges of a
// double; one butterfly per value takes 36, and k_gt_mid spent a quarter of
// its time in the LDS pipe on them.
__device__ __forceinline__ bool box_lane(int lane) { return !(lane & 7) && (lane & 24) != 24; }
__device__ __forceinline__ double wave_box(const double *lo, const double *hi, int lane)
{
    const bool h = lane & 32, r = lane & 16, e = lane & 8;
    double a[3];                             // minima of lo, or of -hi
    for (int d = 0; d < 3; ++d) {
        const double t = __shfl_xor(h ? lo[d] : -hi[d], 32);
        a[d] = h ? -hi[d] : lo[d];
        a[d] = t < a[d] ? t : a[d];
    }
    const double t0 = __shfl_xor(r ? a[0] : a[2], 16), t1 = __shfl_xor(a[1], 16);
    double k0 = r ? a[2] : a[0], k1 = a[1];
    k0 = t0 < k0 ? t0 : k0;
    k1 = t1 < k1 ? t1 : k1;
    double v = r || !e ? k0 : k1;
    const double t2 = __shfl_xor(r || e ? k0 : k1, 8);
    v = t2 < v ? t2 : v;
    for (int o = 4; o > 0; o >>= 1) {
        const double t = __shfl_xor(v, o);
        v = t < v ? t : v;
    }
    return h ? -v : v;
}

// Min/max of a workgroup's lo/hi (256 threads), left to threads 0..5 as
// order keys: thread d < 3 the lower bound d, 3 + d the upper.
__device__ __forceinline__ unsigned long long block_box(double *lo, double *hi, double (*sm)[6])
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const double x = wave_box(lo, hi, lane);
    if (box_lane(lane)) sm[w][(lane >> 5) * 3 + ((lane >> 3) & 3)] = x;
    __syncthreads();
    if (threadIdx.x >= 6) return 0;
    double v = sm[0][threadIdx.x];
    for (int k = 1; k < 4; ++k) {
        const double t = sm[k][threadIdx.x];
        v = threadIdx.x < 3 ? (t < v ? t : v) : (t > v ? t : v);
    }
    return ord_key(v);
}

constexpr int INIT_E = 8;        // particles per thread of k_gt_init

// Positions into storage order, the bounds of the systems of more than MID
// particles, and whether a particle lacks the type bit of msrBuildTree's
// second order (L->need, master.c:4262).
__global__ __launch_bounds__(256) void k_gt_init(Roots R, const double *__restrict__ r,
                                                 const uint32_t *__restrict__ bits,
                                                 double *__restrict__ x, double *__restrict__ y,
                                                 double *__restrict__ z, int *__restrict__ src,
                                                 unsigned long long *__restrict__ box,
                                                 GLevel *__restrict__ L)
{
    __shared__ double sm[4][6];
    const int first = blockIdx.x * (256 * INIT_E), last = min(R.n, first + 256 * INIT_E) - 1;
    const int lane = threadIdx.x & 63;
    // the system of a position among the large ones (-1: of none), and its end
    auto big = [&](int i, int &end) {
        if (R.nr == 1) {
            end = R.n - 1;
            return R.nbig - 1;
        }
        if (R.nbig == 0 || i < R.blo[0]) return -1;
        const int q = root_of(i, R.nbig, R.blo);
        end = R.bhi[q];
        return i <= end ? q : -1;
    };
    int e0 = 0, e1 = 0;
    const int r0 = big(first, e0), r1 = big(last, e1);
    // all of the block in one large system, or none of it in any (a large
    // system is longer than a block)
    static_assert(MID >= 256 * INIT_E, "a large system within a block holds one of its ends");
    const bool one = r0 == r1;
    double lo[3] = {DBL_MAX, DBL_MAX, DBL_MAX}, hi[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
    bool lack = false;
    for (int e = 0; e < INIT_E; ++e) {
        const int i = first + e * 256 + threadIdx.x, i0 = i - lane;   // i0: the wavefront's first
        if (i0 > last) break;
        const bool in = i <= last;
        double v[3] = {0.0, 0.0, 0.0};
        if (in) {
            for (int d = 0; d < 3; ++d) v[d] = r[3 * (size_t)i + d];
            x[i] = v[0];
            y[i] = v[1];
            z[i] = v[2];
            src[i] = i;
            lack |= !(bits[i] & GG_TYPE_TREEACTIVE);
        }
        if (!one) {
            // a block over several systems: 64 particles of one share their
            // atomics (one per particle made a forest of 48 systems of 1024 to
            // 16384 particles take 150 us here, 27 this way)
            int end = 0;
            const int q0 = big(i0, end);
            if (q0 >= 0 && min(i0 + 63, last) <= end) {
                double l[3], h[3];
                for (int d = 0; d < 3; ++d) {
                    const bool ok = in && v[d] == v[d];
                    l[d] = ok ? v[d] : DBL_MAX;
                    h[d] = ok ? v[d] : -DBL_MAX;
                }
                const double k = wave_box(l, h, lane);
                if (box_lane(lane)) {
                    unsigned long long *b = box + BOX_N * (size_t)q0 +
                                            BOX_S * ((lane >> 5) * 3 + ((lane >> 3) & 3));
                    if (lane < 32) atomicMin(b, ord_key(k));
                    else atomicMax(b, ord_key(k));
                }
                continue;
            }
        }
        if (!in) continue;
        if (one) {
            if (r0 < 0) continue;
            for (int d = 0; d < 3; ++d) {
                lo[d] = v[d] < lo[d] ? v[d] : lo[d];
                hi[d] = v[d] > hi[d] ? v[d] : hi[d];
            }
        } else {
            int end = 0;
            const int q = big(i, end);
            if (q < 0) continue;
            unsigned long long *b = box + BOX_N * (size_t)q;
            for (int d = 0; d < 3; ++d) {
                if (v[d] != v[d]) continue;
                atomicMin(b + BOX_S * d, ord_key(v[d]));
                atomicMax(b + BOX_S * (3 + d), ord_key(v[d]));
            }
        }
    }
    if (__ballot(lack) && lane == 0) atomicOr(&L->need, 1);
    if (!one || r0 < 0) return;
    const unsigned long long k = block_box(lo, hi, sm);
    unsigned long long *b = box + BOX_N * (size_t)r0 + BOX_S * threadIdx.x;
    if (threadIdx.x < 3) atomicMin(b, k);
    else if (threadIdx.x < 6) atomicMax(b, k);
}

// The host's copy of a device word (pinned memory, -1 until written).
__device__ __forceinline__ void tell_host(int *p, int v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

__global__ void k_gt_tell(const int *__restrict__ v, int *__restrict__ host)
{
    tell_host(host, *v);
}

// One workgroup decides the level's cells (pkd.c:2489-2505): cells of more
// than MID particles with any extent split at the middle of their longest axis
// and get two child ids; the others join the unit list.  Then the tiles of the
// splitting cells.  The first level's cells are the systems of more than MID
// particles (list, if they are not the only ones).  The tile count goes to
// *host.  One workgroup because a level has at most 2 n / MID cells and every
// later launch waits for it: 4-6 us a level, against the three scans, the
// decision and id kernels and the host's wait it replaces.
constexpr int CTL_T = 1024;
__global__ __launch_bounds__(CTL_T) void k_gt_ctl(int ts, int depth, int cap, int nlist,
                                                  const int *__restrict__ list, GLevel *L,
                                                  GNode *__restrict__ nd,
                                                  const unsigned long long *__restrict__ box,
                                                  unsigned long long *__restrict__ kbox,
                                                  int4 *__restrict__ tiles,
                                                  int *__restrict__ unit, int *host)
{
#pragma clang fp contract(off)
    __shared__ int soff[CTL_T + 1], scell[CTL_T], sfirst[CTL_T];
    __shared__ int ws[CTL_T / 64][3];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int a = L->a, b = L->b, nunit0 = L->nunit;
    const bool bad = L->err != 0;
    __syncthreads();                     // (read before any wavefront below sets it)
    const int nc = list ? nlist : b - a;
    int nsp = 0, ntl = 0, nun = 0;       // splits, tiles and units so far
    for (int base = 0; base < nc && !bad; base += CTL_T) {
        const int i = base + tid, c = i >= nc ? 0 : list ? list[i] : a + i;
        int split = 0, nt = 0, un = 0, lo = 0;
        if (i < nc) {
            GNode &g = nd[c];
            lo = g.lo;
            const int cnt = g.hi - lo + 1;
            if (cnt <= MID) {
                un = 1;
            } else {
                const unsigned long long *k = box + BOX_N * (size_t)i;
                double bmin[3], bmax[3];
                for (int d = 0; d < 3; ++d) {
                    bmin[d] = ord_val(k[BOX_S * d]);
                    bmax[d] = ord_val(k[BOX_S * (3 + d)]);
                }
                bool extent = false;
                for (int d = 0; d < 3; ++d) extent |= bmax[d] > bmin[d];
                if (extent && b + 2 * i + 2 > cap) {   // (a bound on its children's slots)
                    atomicOr(&L->err, 2);
                } else if (extent) {
                    int d = 0;
                    for (int q = 1; q < 3; ++q)
                        if (bmax[q] - bmin[q] > bmax[d] - bmin[d]) d = q;
                    g.dim = d;
                    g.split = 0.5 * (bmin[d] + bmax[d]);
                    split = 1;
                    nt = (cnt + ts - 1) / ts;
                } else {
                    un = 1;              // coincident particles: a bucket (dim -1)
                }
            }
        }
        int is = split, it = nt, iu = un;
        for (int o = 1; o < 64; o <<= 1) {
            const int us = __shfl_up(is, o), ut = __shfl_up(it, o), uu = __shfl_up(iu, o);
            if (lane >= o) {
                is += us;
                it += ut;
                iu += uu;
            }
        }
        if (lane == 63) {
            ws[w][0] = is;
            ws[w][1] = it;
            ws[w][2] = iu;
        }
        __syncthreads();
        int ts0 = 0, tt0 = 0, tu0 = 0, ps = 0, pt = 0, pu = 0;
        for (int k = 0; k < CTL_T / 64; ++k) {
            if (k < w) {
                ps += ws[k][0];
                pt += ws[k][1];
                pu += ws[k][2];
            }
            ts0 += ws[k][0];
            tt0 += ws[k][1];
            tu0 += ws[k][2];
        }
        const int t0 = pt + it - nt;     // this cell's first tile in the chunk
        soff[tid] = t0;
        scell[tid] = c;
        sfirst[tid] = lo;
        if (tid == 0) soff[CTL_T] = tt0;
        if (split) {
            const int kid = 2 * (nsp + ps + is - 1);
            GNode &g = nd[c];
            g.ch0 = b + kid;
            g.ch1 = b + kid + 1;
            for (int q = 0; q < 2; ++q) {
                GNode &h = nd[b + kid + q];
                h.par = c;
                h.root = g.root;
                h.ch0 = h.ch1 = -1;
                h.dim = -1;
                h.split = 0.0;
                box_init(kbox + BOX_N * (size_t)(kid + q));
            }
        }
        if (un) unit[nunit0 + nun + pu + iu - 1] = c;
        __syncthreads();
        for (int t = tid; t < tt0; t += CTL_T) {   // the last cell whose first tile is <= t
            int l = 0, h = CTL_T - 1;
            while (l < h) {
                const int mid = (l + h + 1) >> 1;
                if (soff[mid] <= t) l = mid;
                else h = mid - 1;
            }
            tiles[ntl + t] = make_int4(scell[l], sfirst[l] + (t - soff[l]) * ts, ntl + soff[l],
                                       ntl + soff[l + 1]);
        }
        nsp += ts0;
        ntl += tt0;
        nun += tu0;
        __syncthreads();
    }
    if (tid == 0) {
        L->ntile = ntl;
        L->lv[depth] = a;
        L->a = b;
        L->b = L->next = b + 2 * nsp;
        L->nunit = nunit0 + nun;
        tell_host(host + 1, nunit0 + nun);
        tell_host(host, ntl);
    }
}

struct TileArgs {
    int ts;                              // particles per tile (a multiple of 256)
    uint32_t mask;                       // type orders: the bits of the lower part
    const GLevel *L;
    const int4 *tiles;                   // cell, first particle, the cell's tiles
    GNode *nd;
    double *x, *y, *z;
    int *src;
    const uint32_t *bits;                // caller order
    unsigned long long *flag;            // lower-part flags, ts / 64 words per tile
    int *tcnt, *tpre;                    // per tile: lower-part particles, those before it
    int *posR;
    int *err;
};

// The tiles of the type orders: every system of more than LMAX particles is
// partitioned, none split.
__global__ __launch_bounds__(256) void k_gt_type_tiles(Roots R, int ts, int ntile,
                                                       const GNode *__restrict__ nd,
                                                       int4 *__restrict__ tiles,
                                                       GLevel *__restrict__ L)
{
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t == 0) L->ntile = ntile;
    if (t >= ntile) return;
    int c = 0, t0 = 0, t1 = ntile;
    if (R.nr > 1) {
        const int q = root_of(t, R.ntroot, R.toff);
        c = R.tslot[q];
        t0 = R.toff[q];
        t1 = q + 1 < R.ntroot ? R.toff[q + 1] : ntile;
    }
    tiles[t] = make_int4(c, nd[c].lo + (t - t0) * ts, t0, t1);
}

// Both type orders of the systems of at most LMAX particles, a wavefront each:
// the Hoare swaps on the particles' indices in LDS, then the particles in
// that order.  (As tiles, systems of 4 particles would take six launches of a
// workgroup each.)
constexpr int TY_W = 4;
__global__ __launch_bounds__(64 * TY_W) void k_gt_type_small(Roots R, const double *__restrict__ r,
                                                             const uint32_t *__restrict__ bits,
                                                             double *__restrict__ x,
                                                             double *__restrict__ y,
                                                             double *__restrict__ z,
                                                             int *__restrict__ src)
{
    __shared__ short idx_[TY_W][LMAX], posR_[TY_W][LMAX];
    __shared__ unsigned char bit_[TY_W][LMAX];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    short *idx = idx_[w], *posR = posR_[w];
    unsigned char *bit = bit_[w];
    const unsigned long long below = (1ull << lane) - 1;
    auto wave_fence = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    for (int k = blockIdx.x * TY_W + w; k < R.nr; k += gridDim.x * TY_W) {
        const int lo = R.nr > 1 ? R.lo[k] : 0, cnt = (R.nr > 1 ? R.hi[k] : R.n - 1) - lo + 1;
        if (cnt < 2 || cnt > LMAX) continue;
        for (int i = lane; i < cnt; i += 64) {
            const uint32_t t = bits[lo + i];
            idx[i] = (short)i;
            bit[i] = (t & GG_TYPE_TREEACTIVE ? 2 : 0) |
                     (t & (GG_TYPE_ACTIVE | GG_TYPE_TREEACTIVE) ? 1 : 0);
        }
        wave_fence();
        for (int mask = 1; mask <= 2; ++mask) {
            int nl = 0;
            for (int c0 = 0; c0 < cnt; c0 += 64)
                nl += __popcll(__ballot(c0 + lane < cnt && (bit[idx[c0 + lane]] & mask)));
            int run = 0;
            for (int c0 = 0; c0 < cnt; c0 += 64) {   // upper positions holding a lower one
                const int i = c0 + lane;
                const bool f = i < cnt && (bit[idx[i]] & mask);
                const unsigned long long m = __ballot(f);
                const int ex = run + __popcll(m & below);
                if (f && i >= nl) posR[nl - 1 - ex] = (short)i;
                run += __popcll(m);
            }
            wave_fence();
            run = 0;
            for (int c0 = 0; c0 < nl; c0 += 64) {    // lower positions holding an upper one
                const int i = c0 + lane;
                const bool in = i < nl, f = in && (bit[idx[i]] & mask);
                const unsigned long long m = __ballot(f);
                const int ex = run + __popcll(m & below);
                if (in && !f) {
                    const int j = posR[i - ex];
                    const short u = idx[i];
                    idx[i] = idx[j];
                    idx[j] = u;
                }
                run += __popcll(m);
            }
            wave_fence();
        }
        for (int i = lane; i < cnt; i += 64) {
            const int s = idx[i];
            if (s == i) continue;
            src[lo + i] = lo + s;
            x[lo + i] = r[3 * (size_t)(lo + s)];
            y[lo + i] = r[3 * (size_t)(lo + s) + 1];
            z[lo + i] = r[3 * (size_t)(lo + s) + 2];
        }
        wave_fence();
    }
}

// mode 0: the coordinate below the cell's split; mode 1: a type bit of mask.
template <int MODE>
__device__ __forceinline__ bool lower_flag(const TileArgs &A, const double *v, double split, int i)
{
    if (MODE == 1) return (A.bits[A.src[i]] & A.mask) != 0;
    return v[i] < split;
}

__device__ __forceinline__ const double *split_axis(const TileArgs &A, int dim)
{
    return dim == 0 ? A.x : (dim == 1 ? A.y : A.z);
}

template <int MODE> __global__ __launch_bounds__(256) void k_gt_count(TileArgs A)
{
    __shared__ int wc[4];
    const int t = blockIdx.x;
    if (t >= A.L->ntile) return;
    const int4 T = A.tiles[t];
    const int hi = A.nd[T.x].hi, last = min(hi, T.y + A.ts - 1);
    const double split = A.nd[T.x].split;
    const double *v = split_axis(A, A.nd[T.x].dim);
    unsigned long long *fw = A.flag + (size_t)t * (A.ts / 64);
    int c = 0;
    for (int j = threadIdx.x; j < A.ts; j += 256) {
        const int i = T.y + j;
        const bool f = i <= last && lower_flag<MODE>(A, v, split, i);
        const unsigned long long m = __ballot(f);
        if ((threadIdx.x & 63) == 0) fw[j >> 6] = m;
        c += __popcll(m);
    }
    if ((threadIdx.x & 63) == 0) wc[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) A.tcnt[t] = wc[0] + wc[1] + wc[2] + wc[3];
}

constexpr int TW = 64;                   // flag words of a tile, at most (one wavefront scans them)

// The tile's flag words and, before each, the number of flags of its cell
// (pre: those of the cell's earlier tiles).
__device__ __forceinline__ void tile_flags(const TileArgs &A, int t, int pre,
                                           unsigned long long *fw, int *fp)
{
    if (threadIdx.x < 64) {
        const int l = threadIdx.x;
        const unsigned long long m = l < A.ts / 64 ? A.flag[(size_t)t * (A.ts / 64) + l] : 0;
        const int c = __popcll(m);
        int inc = c;
        for (int o = 1; o < 64; o <<= 1) {
            const int u = __shfl_up(inc, o);
            if (l >= o) inc += u;
        }
        fw[l] = m;
        fp[l] = pre + inc - c;
    }
    __syncthreads();
}

// Split position s = lo + number of lower-part particles (the first tile of
// a cell writes it and the children's ranges); a split that leaves one side
// empty (the reference asserts against it, pkd.c:2512-2516) sets *err.  Then
// the upper part's positions that hold a lower particle, by rank counted
// down from hi: posR[lo + k].
template <int MODE> __global__ __launch_bounds__(256) void k_gt_rank(TileArgs A)
{
    __shared__ unsigned long long fw[TW];
    __shared__ int fp[TW], red[2][4];
    const int t = blockIdx.x;
    if (t >= A.L->ntile) return;
    const int4 T = A.tiles[t];
    int pre = 0, tot = 0;
    for (int k = T.z + threadIdx.x; k < T.w; k += 256) {
        const int c = A.tcnt[k];
        tot += c;
        if (k < t) pre += c;
    }
    for (int o = 32; o > 0; o >>= 1) {
        pre += __shfl_xor(pre, o);
        tot += __shfl_xor(tot, o);
    }
    if ((threadIdx.x & 63) == 0) {
        red[0][threadIdx.x >> 6] = pre;
        red[1][threadIdx.x >> 6] = tot;
    }
    __syncthreads();
    pre = red[0][0] + red[0][1] + red[0][2] + red[0][3];
    const int nl = red[1][0] + red[1][1] + red[1][2] + red[1][3];
    tile_flags(A, t, pre, fw, fp);
    GNode &g = A.nd[T.x];
    const int lo = g.lo, hi = g.hi, s = lo + nl;
    if (threadIdx.x == 0) {
        A.tpre[t] = pre;
        if (t == T.z) {
            g.s = s;
            if (MODE == 0) {
                if (s == lo || s > hi) atomicOr(A.err, 1);
                GNode &l = A.nd[g.ch0], &u = A.nd[g.ch1];
                l.lo = lo;
                l.hi = s - 1;
                u.lo = s;
                u.hi = hi;
            }
        }
    }
    const int last = min(hi, T.y + A.ts - 1);
    for (int i = T.y + threadIdx.x; i <= last; i += 256) {
        if (i < s) continue;
        const int j = i - T.y;
        const unsigned long long m = fw[j >> 6], bit = 1ull << (j & 63);
        if (!(m & bit)) continue;
        A.posR[lo + nl - 1 - (fp[j >> 6] + __popcll(m & (bit - 1)))] = i;
    }
}

// The swaps of the Hoare scan: the lower-part position holding the k-th
// upper particle (counted up from lo) <-> posR[lo + k], each pair swapped
// by its lower member.  Every particle passes through registers once, so
// the children's bounds are taken on the way (mode 0).  It moves 24-28 bytes
// a particle and 56 a swapped one.  Measured per level: 23 us on a 2^21
// Plummer sphere (count 6.0, rank 4.6, control 6.0) and 10.3 us on 3 10^5
// particles (4.1, 3.8, 5.1), where the chain of loads and the bounds'
// reduction bound it rather than the bytes.
template <int MODE>
__global__ __launch_bounds__(256) void k_gt_swap(TileArgs A, unsigned long long *__restrict__ kbox)
{
    __shared__ unsigned long long fw[TW];
    __shared__ int fp[TW];
    __shared__ double sm[2][4][6];
    const int t = blockIdx.x;
    if (t >= A.L->ntile) return;
    const int4 T = A.tiles[t];
    tile_flags(A, t, A.tpre[t], fw, fp);
    const GNode &g = A.nd[T.x];
    const int lo = g.lo, hi = g.hi, s = g.s, ch0 = g.ch0;
    // a child that goes to k_gt_mid takes its bounds there
    const bool need[2] = {MODE == 0 && s - lo > MID, MODE == 0 && hi - s + 1 > MID};
    const int last = min(hi, T.y + A.ts - 1);
    double bl[2][3], bh[2][3];
    for (int q = 0; q < 2; ++q)
        for (int d = 0; d < 3; ++d) {
            bl[q][d] = DBL_MAX;
            bh[q][d] = -DBL_MAX;
        }
    auto grow = [&](int q, const double *v) {
        for (int d = 0; d < 3; ++d) {
            bl[q][d] = v[d] < bl[q][d] ? v[d] : bl[q][d];
            bh[q][d] = v[d] > bh[q][d] ? v[d] : bh[q][d];
        }
    };
    for (int i = T.y + threadIdx.x; i <= last; i += 256) {
        const int j = i - T.y;
        const unsigned long long m = fw[j >> 6], bit = 1ull << (j & 63);
        const bool f = m & bit, low = i < s;
        if (!low && f) continue;         // its partner's thread takes it
        if (MODE == 1 && (!low || f)) continue;
        const double v[3] = {A.x[i], A.y[i], A.z[i]};
        if (low && !f) {
            const int p = A.posR[i - (fp[j >> 6] + __popcll(m & (bit - 1)))];
            const double u[3] = {A.x[p], A.y[p], A.z[p]};
            const int si = A.src[i], sp = A.src[p];
            A.x[i] = u[0];
            A.y[i] = u[1];
            A.z[i] = u[2];
            A.src[i] = sp;
            A.x[p] = v[0];
            A.y[p] = v[1];
            A.z[p] = v[2];
            A.src[p] = si;
            if (MODE == 0) {
                grow(0, u);
                grow(1, v);
            }
        } else if (MODE == 0) {
            if (low) grow(0, v);
            else grow(1, v);
        }
    }
    if (!need[0] && !need[1]) return;
    const int kid = ch0 - A.L->a;        // the children's level starts at L->a now
    for (int q = 0; q < 2; ++q) {
        if (!need[q]) continue;
        const unsigned long long k = block_box(bl[q], bh[q], sm[q]);
        unsigned long long *b = kbox + BOX_N * (size_t)(kid + q) + BOX_S * threadIdx.x;
        if (threadIdx.x < 3) atomicMin(b, k);
        else if (threadIdx.x < 6) atomicMax(b, k);
    }
}

// The cells of the unit list, each by one workgroup: a cell of LMAX..MID
// particles is split in LDS, level by level with the rules above, until its
// parts hold at most LMAX (listed for k_gt_sub).  The cells it closes (split,
// or coincident and left buckets) are listed in seg from the cell's first
// particle on, level by level, with the levels' ends in segl and their
// numbers in useg (that of the levels negative if buckets are among the
// cells), for the upward pass.
// At most MID / LMAX parts are open at a time, so a level is a handful of
// wavefront passes over the particles between barriers instead of four
// launches.  Its barriers and LDS round trips bound it: 88 us for a cell of 4096
// Plummer particles (160 with a butterfly per bound, the flags' prefix left to
// one wavefront and the slots' atomics waited for in every level).  Flags are
// bits, 64 particles a word, and ranks come from a prefix over the 64 words.
// MID is what the LDS holds: 140 KB, one workgroup per CU.
constexpr int MID_T = 1024, MID_O = MID / LMAX, MID_W = MID / 64;
static_assert(6 * MID_O <= 64, "one lane per bound of an open part");
static_assert(MID_W == 64, "one wavefront scans the flag words");
__global__ __launch_bounds__(MID_T) void k_gt_mid(const int *__restrict__ unit, int cap,
                                                  GLevel *L, GNode *__restrict__ nd,
                                                  double *__restrict__ px, double *__restrict__ py,
                                                  double *__restrict__ pz, int *__restrict__ perm,
                                                  int *__restrict__ sub, int *__restrict__ seg,
                                                  int *__restrict__ segl, int2 *__restrict__ useg)
{
#pragma clang fp contract(off)
    __shared__ double lx[MID], ly[MID], lz[MID];
    __shared__ int ls[MID];
    __shared__ unsigned short posR[MID];
    __shared__ unsigned long long fbits[MID_W];
    __shared__ int subl[MID], sub0_sh, nsub_sh;
    __shared__ int olo[2][MID_O], ohi[2][MID_O], onode[2][MID_O];
    __shared__ unsigned long long cb[MID_O][6];
    __shared__ double csplit[MID_O];
    __shared__ int cdim[MID_O], nopen[2], full;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int rootId = unit[blockIdx.x];
    const int glo = nd[rootId].lo, cnt = nd[rootId].hi - glo + 1;
    const int troot = nd[rootId].root;
    if (cnt > MID || cnt <= LMAX) {
        if (tid == 0) {
            useg[blockIdx.x] = make_int2(cnt > MID, -(cnt > MID));
            if (cnt > MID) {             // coincident particles: a bucket
                seg[glo] = rootId;
                segl[glo] = 1;
            } else {
                sub[atomicAdd(&L->nsub, 1)] = rootId;
            }
        }
        return;
    }
    for (int i = tid; i < cnt; i += MID_T) {
        lx[i] = px[glo + i];
        ly[i] = py[glo + i];
        lz[i] = pz[glo + i];
        ls[i] = perm[glo + i];
    }
    if (tid == 0) {
        olo[0][0] = 0;
        ohi[0][0] = cnt - 1;
        onode[0][0] = rootId;
        nopen[0] = 1;
        full = 0;
    }
    if (tid < 6 * MID_O) cb[tid / 6][tid % 6] = tid % 6 < 3 ? ~0ull : 0ull;
    __syncthreads();
    const int w0 = w * (MID / (MID_T / 64));             // this wavefront's particles
    constexpr int WN = MID / MID_T;                      // its words
    int cur = 0, depth = 0, nseg = 0, nsubl = 0;        // (the counts: wavefront 0)
    bool leaves = false;
    for (; nopen[cur] > 0; ++depth) {
        const int no = nopen[cur];
        for (int q = 0; q < no; ++q) {                   // bounds
            const int lo = olo[cur][q], hi = ohi[cur][q];
            if (hi < w0 || lo >= w0 + 64 * WN) continue;
            double bl[3] = {DBL_MAX, DBL_MAX, DBL_MAX}, bh[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
            for (int k = 0; k < WN; ++k) {
                const int i = w0 + 64 * k + lane;
                if (i < lo || i > hi) continue;
                const double v[3] = {lx[i], ly[i], lz[i]};
                for (int d = 0; d < 3; ++d) {
                    bl[d] = v[d] < bl[d] ? v[d] : bl[d];
                    bh[d] = v[d] > bh[d] ? v[d] : bh[d];
                }
            }
            const double v = wave_box(bl, bh, lane);
            if (box_lane(lane)) {
                unsigned long long *k = &cb[q][(lane >> 5) * 3 + ((lane >> 3) & 3)];
                if (lane < 32) atomicMin(k, ord_key(v));
                else atomicMax(k, ord_key(v));
            }
        }
        __syncthreads();
        int got = 0;                                     // the level's first slot (lane 0)
        if (w == 0) {                                    // split decisions
            bool extent = false;
            if (lane < no) {
                double bmin[3], bmax[3];
                for (int d = 0; d < 3; ++d) {
                    bmin[d] = ord_val(cb[lane][d]);
                    bmax[d] = ord_val(cb[lane][3 + d]);
                    extent |= bmax[d] > bmin[d];
                }
                int d = 0;
                for (int k = 1; k < 3; ++k)
                    if (bmax[k] - bmin[k] > bmax[d] - bmin[d]) d = k;
                cdim[lane] = extent ? d : -1;            // -1: coincident, a bucket
                csplit[lane] = 0.5 * (bmin[d] + bmax[d]);
            }
            const unsigned long long me = __ballot(extent);
            if (lane == 0) {
                nopen[cur ^ 1] = 0;
                if (me) got = atomicAdd(&L->next, 2 * __popcll(me));   // waited for below
            }
        }
        __syncthreads();
        bool f[WN];                                      // lower-part flags
        for (int k = 0; k < WN; ++k) f[k] = false;
        for (int q = 0; q < no; ++q) {
            const int lo = olo[cur][q], hi = ohi[cur][q], dim = cdim[q];
            if (hi < w0 || lo >= w0 + 64 * WN || dim < 0) continue;
            const double *v = dim == 0 ? lx : (dim == 1 ? ly : lz), split = csplit[q];
            for (int k = 0; k < WN; ++k) {
                const int i = w0 + 64 * k + lane;
                if (i >= lo && i <= hi) f[k] = v[i] < split;
            }
        }
        unsigned long long fm[WN];
        for (int k = 0; k < WN; ++k) {
            fm[k] = __ballot(f[k]);
            if (lane == 0) fbits[(w0 >> 6) + k] = fm[k];
        }
        __syncthreads();
        // every wavefront: lane l holds word l of the flags and those before it
        const unsigned long long word = fbits[lane];
        int inc = __popcll(word);
        for (int o = 1; o < 64; o <<= 1) {
            const int u = __shfl_up(inc, o);
            if (lane >= o) inc += u;
        }
        const int pre = inc - __popcll(word), all = __builtin_amdgcn_readlane(inc, 63);
        auto F = [&](int i) {                            // flags of positions below i
            const int l = min(i >> 6, MID_W - 1);
            const int n = __shfl(pre, l) + __popcll(__shfl(word, l) & ((1ull << (i & 63)) - 1));
            return i >= MID ? all : n;
        };
        int part[WN], Fi[WN];                            // swap partner's rank slot, -1: none
        for (int k = 0; k < WN; ++k) {
            part[k] = -1;
            Fi[k] = __builtin_amdgcn_readlane(pre, (w0 >> 6) + k) +
                    __popcll(fm[k] & ((1ull << lane) - 1));
        }
        for (int q = 0; q < no; ++q) {
            const int lo = olo[cur][q], hi = ohi[cur][q];
            if (hi < w0 || lo >= w0 + 64 * WN || cdim[q] < 0) continue;
            const int F0 = F(lo), nl = F(hi + 1) - F0;
            for (int k = 0; k < WN; ++k) {
                const int i = w0 + 64 * k + lane;
                if (i < lo || i > hi) continue;
                if (i >= lo + nl && f[k])
                    posR[lo + nl - 1 - (Fi[k] - F0)] = (unsigned short)i;
                if (i < lo + nl && !f[k]) part[k] = i - (Fi[k] - F0);
            }
        }
        __syncthreads();
        if (w == 0) {                                    // nodes of the two parts
            const bool in = lane < no;
            int lo = 0, hi = -1, s = 0;
            bool sp = false;
            if (in) {
                lo = olo[cur][lane];
                hi = ohi[cur][lane];
            }
            const int nl = F(hi + 1) - F(lo);
            if (in) {
                s = lo;
                if (cdim[lane] >= 0) {
                    s = lo + nl;
                    sp = s > lo && s <= hi;
                    if (!sp) atomicOr(&L->err, 1);       // one side empty: reported
                }
            }
            const bool sub0 = sp && s - lo <= LMAX, sub1 = sp && hi - s + 1 <= LMAX;
            const unsigned long long ms = __ballot(sp), u0 = __ballot(sub0), u1 = __ballot(sub1);
            const unsigned long long below = (1ull << lane) - 1;
            const int id0 = __shfl(got, 0) + 2 * __popcll(ms & below);
            const int su0 = nsubl + __popcll(u0 & below) + __popcll(u1 & below);
            nsubl += __popcll(u0) + __popcll(u1);        // at most one per particle
            if (lane < 6 * MID_O) cb[lane / 6][lane % 6] = lane % 6 < 3 ? ~0ull : 0ull;
            if (__shfl(got, 0) + 2 * __popcll(ms) > cap) {   // out of slots: built again
                sp = false;
                if (lane == 0) {
                    atomicOr(&L->err, 2);
                    full = 1;
                }
            }
            if (sp && sub0) subl[su0] = id0;
            if (sp && sub1) subl[su0 + sub0] = id0 + 1;
            const int me = in ? onode[cur][lane] : 0;
            if (in) seg[glo + nseg + lane] = me;
            leaves |= __ballot(in && !sp) != 0;
            nseg += no;
            if (lane == 0) segl[glo + depth] = nseg;
            if (sp) {
                GNode &g = nd[me];
                g.dim = cdim[lane];
                g.split = csplit[lane];
                g.s = glo + s;
                g.ch0 = id0;
                g.ch1 = id0 + 1;
            }
            for (int q = 0; q < 2; ++q) {
                const int a0 = q ? s : lo, a1 = q ? hi : s - 1;
                const bool open = sp && a1 - a0 + 1 > LMAX;
                const unsigned long long mo = __ballot(open);
                if (sp) {
                    GNode &h = nd[id0 + q];
                    h.lo = glo + a0;
                    h.hi = glo + a1;
                    h.par = me;
                    h.root = troot;
                    h.ch0 = h.ch1 = -1;
                    h.split = 0.0;
                    h.dim = -1;
                }
                const int at = nopen[cur ^ 1] + __popcll(mo & ((1ull << lane) - 1));
                if (open) {
                    olo[cur ^ 1][at] = a0;
                    ohi[cur ^ 1][at] = a1;
                    onode[cur ^ 1][at] = id0 + q;
                }
                if (lane == 0) nopen[cur ^ 1] += __popcll(mo);
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            }
        }
        for (int k = 0; k < WN; ++k) {                   // the swaps
            if (part[k] < 0) continue;
            const int i = w0 + 64 * k + lane, j = posR[part[k]];
            double d = lx[i]; lx[i] = lx[j]; lx[j] = d;
            d = ly[i]; ly[i] = ly[j]; ly[j] = d;
            d = lz[i]; lz[i] = lz[j]; lz[j] = d;
            const int u = ls[i]; ls[i] = ls[j]; ls[j] = u;
        }
        cur ^= 1;
        __syncthreads();
        if (full) return;
    }
    if (tid == 0) {
        useg[blockIdx.x] = make_int2(nseg, leaves ? -depth : depth);
        sub0_sh = nsubl ? atomicAdd(&L->nsub, nsubl) : 0;
        nsub_sh = nsubl;
    }
    __syncthreads();
    for (int k = tid; k < nsub_sh; k += MID_T) sub[sub0_sh + k] = subl[k];
    for (int i = tid; i < cnt; i += MID_T) {
        px[glo + i] = lx[i];
        py[glo + i] = ly[i];
        pz[glo + i] = lz[i];
        perm[glo + i] = ls[i];
    }
}

// ------------------------------------------------------ numeric records
// Positions of the raw moments: third order xxx xyy xxy yyy xxz yyz xyz xzz
// yzz zzz, fourth xxxx xyyy xxxy yyyy xxxz yyyz xxyy xxyz xyyz xxzz xyzz
// xzzz yyzz yzzz zzzz.
__device__ constexpr int T_IX[10][3] = {{0, 0, 0}, {0, 1, 1}, {0, 0, 1}, {1, 1, 1}, {0, 0, 2},
                                        {1, 1, 2}, {0, 1, 2}, {0, 2, 2}, {1, 2, 2}, {2, 2, 2}};
__device__ constexpr int F_IX[15][4] = {{0, 0, 0, 0}, {0, 1, 1, 1}, {0, 0, 0, 1}, {1, 1, 1, 1},
                                        {0, 0, 0, 2}, {1, 1, 1, 2}, {0, 0, 1, 1}, {0, 0, 1, 2},
                                        {0, 1, 1, 2}, {0, 0, 2, 2}, {0, 1, 2, 2}, {0, 2, 2, 2},
                                        {1, 1, 2, 2}, {1, 2, 2, 2}, {2, 2, 2, 2}};
__device__ constexpr int q_at(int a, int b)   // xx yy zz xy xz yz
{
    return a == b ? a : a + b + 2;
}
__device__ constexpr int t_at(int a, int b, int c)   // any order of indices
{
    const int n[3] = {(a == 0) + (b == 0) + (c == 0), (a == 1) + (b == 1) + (c == 1),
                      (a == 2) + (b == 2) + (c == 2)};
    for (int k = 0; k < 10; ++k) {
        int m[3] = {0, 0, 0};
        for (int j = 0; j < 3; ++j) ++m[T_IX[k][j]];
        if (m[0] == n[0] && m[1] == n[1] && m[2] == n[2]) return k;
    }
    return -1;
}

// The raw moments of a particle of mass m at d from the expansion centre,
// added to g.
template <int ORDER>
__device__ __forceinline__ void mom_particle(double m, const double *d, double *g)
{
    double q[6];
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int b = a; b < 3; ++b) {
            q[q_at(a, b)] = m * d[a] * d[b];
            g[GM_Q + q_at(a, b)] += q[q_at(a, b)];
        }
    if constexpr (ORDER >= 3) {
        double t[10];
#pragma unroll
        for (int k = 0; k < 10; ++k) {
            t[k] = q[q_at(T_IX[k][0], T_IX[k][1])] * d[T_IX[k][2]];
            g[GM_T + k] += t[k];
        }
        if constexpr (ORDER >= 4) {
#pragma unroll
            for (int k = 0; k < 15; ++k)
                g[GM_F + k] += t[t_at(F_IX[k][0], F_IX[k][1], F_IX[k][2])] * d[F_IX[k][3]];
        }
    }
}

// A child's raw moments c moved from its centre of mass to the parent's,
// which lies -d from it, and added to g.  The child's first moment about
// its own centre vanishes.
template <int ORDER>
__device__ __forceinline__ void mom_shift(const double *c, const double *d, double *g)
{
    const double m = c[0];
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int b = a; b < 3; ++b)
            g[GM_Q + q_at(a, b)] += c[GM_Q + q_at(a, b)] + m * d[a] * d[b];
    if constexpr (ORDER >= 3) {
#pragma unroll
        for (int k = 0; k < 10; ++k) {
            constexpr auto &X = T_IX;
            const int i = X[k][0], j = X[k][1], l = X[k][2];
            g[GM_T + k] += c[GM_T + k] + c[GM_Q + q_at(i, j)] * d[l]
                           + c[GM_Q + (i <= l ? q_at(i, l) : q_at(l, i))] * d[j]
                           + c[GM_Q + (j <= l ? q_at(j, l) : q_at(l, j))] * d[i]
                           + m * d[i] * d[j] * d[l];
        }
    }
    if constexpr (ORDER >= 4) {
#pragma unroll
        for (int k = 0; k < 15; ++k) {
            const int i = F_IX[k][0], j = F_IX[k][1], l = F_IX[k][2], o = F_IX[k][3];
            // i <= j <= l <= o throughout F_IX
            g[GM_F + k] += c[GM_F + k] + c[GM_T + t_at(i, j, l)] * d[o]
                           + c[GM_T + t_at(i, j, o)] * d[l] + c[GM_T + t_at(i, l, o)] * d[j]
                           + c[GM_T + t_at(j, l, o)] * d[i]
                           + c[GM_Q + q_at(i, j)] * d[l] * d[o] + c[GM_Q + q_at(i, l)] * d[j] * d[o]
                           + c[GM_Q + q_at(i, o)] * d[j] * d[l] + c[GM_Q + q_at(j, l)] * d[i] * d[o]
                           + c[GM_Q + q_at(j, o)] * d[i] * d[l] + c[GM_Q + q_at(l, o)] * d[i] * d[j]
                           + m * d[i] * d[j] * d[l] * d[o];
        }
    }
}

// Mass, mass-weighted softening and centre of mass of a cell from its
// children's, lower then upper (pkd.c:2510-2576).
__device__ __forceinline__ void mass_children(const double *c0, const double *c1, double *g)
{
#pragma clang fp contract(off)
    double M = 0.0, S = 0.0, R[3] = {0.0, 0.0, 0.0};
    for (int k = 0; k < 2; ++k) {
        const double *q = k ? c1 : c0;
        const double fm = q[0];
        M += fm;
        S += fm * q[1];
        for (int d = 0; d < 3; ++d) R[d] += fm * q[2 + d];
    }
    if (M > 0) {
        S /= M;
        for (int d = 0; d < 3; ++d) R[d] /= M;
    }
    g[0] = M;
    g[1] = S;
    for (int d = 0; d < 3; ++d) g[2 + d] = R[d];
}

// Squared distance as Bmax takes it (pkd.c:2018-2135), before its root.
__device__ __forceinline__ double cm_d2(double x, double y, double z, const double *cm)
{
#pragma clang fp contract(off)
    const double dx = x - cm[0], dy = y - cm[1], dz = z - cm[2];
    return dx * dx + dy * dy + dz * dz;
}

// A bucket's record by one thread: mass, softening and centre of mass over
// its particles in storage order, then the moments, and bb: the active
// particles' bounds, the largest softening and their number (pkd.c:2916-2937,
// walk.c:319-324).  get(i, p, m, h) loads particle i; returns whether active.
template <int ORDER, typename Get>
__device__ __forceinline__ int bucket_record(int lo, int hi, Get get, double *g, double *bb)
{
#pragma clang fp contract(off)
    double M = 0.0, S = 0.0, R[3] = {0.0, 0.0, 0.0};
    double bl[3] = {DBL_MAX, DBL_MAX, DBL_MAX}, bh[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
    double fsm = 0.0;
    int na = 0;
    for (int i = lo; i <= hi; ++i) {
        double p[3], m, h;
        const bool act = get(i, p, m, h);
        M += m;
        S += m * h;
        for (int d = 0; d < 3; ++d) R[d] += m * p[d];
        if (h > fsm) fsm = h;
        if (!act) continue;
        ++na;
        for (int d = 0; d < 3; ++d) {
            if (p[d] < bl[d]) bl[d] = p[d];
            if (p[d] > bh[d]) bh[d] = p[d];
        }
    }
    if (M > 0) {
        S /= M;
        for (int d = 0; d < 3; ++d) R[d] /= M;
    }
    g[0] = M;
    g[1] = S;
    for (int d = 0; d < 3; ++d) g[2 + d] = R[d];
    double b2 = 0.0;
    for (int i = lo; i <= hi; ++i) {
        double p[3], m, h;
        get(i, p, m, h);
        const double d2 = cm_d2(p[0], p[1], p[2], R);
        if (d2 > b2) b2 = d2;
        const double d[3] = {p[0] - R[0], p[1] - R[1], p[2] - R[2]};
        mom_particle<ORDER>(m, d, g);
    }
    g[GM_B] = b2;
    for (int d = 0; d < 3; ++d) {
        bb[d] = bl[d];
        bb[3 + d] = bh[d];
    }
    bb[6] = fsm;
    bb[7] = (double)na;
    return na;
}

struct TreeArgs {
    int nBucket, cap;                    // slots
    GLevel *L;
    GNode *nd;
    double *gm, *bb8;                    // numeric record and bucket bounds per slot
    double *px, *py, *pz, *pm, *ph;      // storage order
    uint32_t *pact;
    int *perm;
    const double *m, *h;                 // caller order
    const uint32_t *bits;
    const int *sub;                      // cells left to k_gt_sub
    int2 *subn;                          // their first slot and cells below them
    const int *unit, *seg, *segl;        // cells left to k_gt_mid and what it closed
    const int2 *useg;
};

// The subtree of one cell of at most LMAX particles, by one workgroup in LDS:
// the splits with the rules above, then the preorder of its cells, their
// slots, and their records from the particles that are still in LDS.  A level
// of splits takes one barrier: a part of more than 32 particles is split by
// one wavefront, two smaller ones by its halves, and each reserves its
// children with LDS atomics.  Sizes and records climb from the buckets, the
// second child to arrive computing the parent, so a level needs no barrier
// there.  Moments come from the children's by shifting (31 values, ~400
// operations a cell) instead of from every particle of every cell.
// Two forms: LM = LMAX particles by T = 256 threads (57 KB of LDS, two
// workgroups a CU) for the parts of larger cells, and LM = LSML by one
// wavefront (14 KB, eleven a CU) for small systems, of which a forest may have
// very many and each takes its latency whatever its size.  A workgroup takes
// entries t0 to t1 of the list (t1 < 0: all) in turn, and slots for several
// small subtrees by one atomic (chunk, where there is room to lose part of
// one): the atomics on the level's line, 10 ns each, bound a forest of small
// systems whatever the occupancy.  200000 systems of 20 particles, a build:
// 14.0 ms with the first form alone, 11.1 with the second, 2.5 with both.
template <int ORDER, int LM, int T>
__global__ __launch_bounds__(T) void k_gt_sub(TreeArgs A, int t0, int t1, int chunk)
{
#pragma clang fp contract(off)
    constexpr int GS = gm_stride(ORDER), SN = 2 * LM;
    __shared__ double lx[LM], ly[LM], lz[LM], nsp[SN];
    __shared__ double lm[LM], lh[LM];
    __shared__ int ls[LM], arr[SN];
    __shared__ short posR[LM];
    __shared__ short nlo[SN], nhi[SN], npar[SN], nch[SN], nsz[SN], nac[SN], npre[SN], nbp[SN];
    __shared__ signed char ndm[SN];
    __shared__ unsigned char lact[LM];
    __shared__ short qa[3][2][LM / 2];  // open cells of a level: larger, smaller than 33
    __shared__ int qn[3][2], nloc_sh, slot_sh, maxb_sh;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, half = lane >> 5, l32 = lane & 31;
    // No early exit when slots have run out: other workgroups of this launch
    // set that bit while this one starts, so its wavefronts could read it
    // differently and part of them leave the rest to LDS they never filled.
    // Every listed subtree is valid whatever the bit; room, one value for the
    // workgroup, guards the writes past the slots.
    const int nsub = t1 < 0 ? A.L->nsub : t1, next = A.L->next;
    int slot = 0, left = 0;              // slots in hand (thread 0)
    if (tid == 0) maxb_sh = 0;
    for (int t = t0 + blockIdx.x; t < nsub; t += gridDim.x) {
        const int root = A.sub[t];
        const int glo = A.nd[root].lo, cnt = A.nd[root].hi - glo + 1, troot = A.nd[root].root;
        for (int i = tid; i < cnt; i += T) {
            lx[i] = A.px[glo + i];
            ly[i] = A.py[glo + i];
            lz[i] = A.pz[glo + i];
            ls[i] = A.perm[glo + i];
        }
        if (tid == 0) {
            nlo[0] = 0;
            nhi[0] = (short)(cnt - 1);
            npar[0] = nch[0] = -1;
            ndm[0] = -1;
            nsp[0] = 0.0;
            nloc_sh = 1;
            for (int k = 0; k < 3; ++k) qn[k][0] = qn[k][1] = 0;
            if (cnt > A.nBucket) {
                const int big = cnt > 32 ? 0 : 1;
                qa[0][big][0] = 0;
                qn[0][big] = 1;
            }
        }
        __syncthreads();
        // the split cell k (range lo..hi, lower part lo..s-1): its children,
        // queued for the next level if they may split
        auto children = [&](int k, int lo, int hi, int s, int dim, double split, int nxt) {
            const int c = atomicAdd(&nloc_sh, 2);
            ndm[k] = (signed char)dim;
            nsp[k] = split;
            nch[k] = (short)c;
            for (int q = 0; q < 2; ++q) {
                const int a0 = q ? s : lo, a1 = q ? hi : s - 1, m = a1 - a0 + 1;
                nlo[c + q] = (short)a0;
                nhi[c + q] = (short)a1;
                npar[c + q] = (short)k;
                nch[c + q] = -1;
                ndm[c + q] = -1;
                nsp[c + q] = 0.0;
                if (m > A.nBucket) {
                    const int b = m > 32 ? 0 : 1;
                    qa[nxt][b][atomicAdd(&qn[nxt][b], 1)] = (short)(c + q);
                }
            }
        };
        for (int cur = 0; qn[cur][0] + qn[cur][1] > 0;) {
            const int nxt = cur == 2 ? 0 : cur + 1, nn2 = nxt == 2 ? 0 : nxt + 1;
            const int nbig = qn[cur][0], nsml = qn[cur][1];
            if (tid == 0) qn[nn2][0] = qn[nn2][1] = 0;   // the queue after the next
            for (int b = w; b < nbig; b += T / 64) {
                const int k = qa[cur][0][b];
                const int lo = nlo[k], hi = nhi[k];
                double bmin[3] = {DBL_MAX, DBL_MAX, DBL_MAX};
                double bmax[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
                for (int i = lo + lane; i <= hi; i += 64) {
                    const double v[3] = {lx[i], ly[i], lz[i]};
                    for (int d = 0; d < 3; ++d) {
                        bmin[d] = v[d] < bmin[d] ? v[d] : bmin[d];
                        bmax[d] = v[d] > bmax[d] ? v[d] : bmax[d];
                    }
                }
                const double bx = wave_box(bmin, bmax, lane);
                for (int d = 0; d < 3; ++d) {
                    bmin[d] = __shfl(bx, 8 * d);
                    bmax[d] = __shfl(bx, 32 + 8 * d);
                }
                int dim = 0;
                for (int q = 1; q < 3; ++q)
                    if (bmax[q] - bmin[q] > bmax[dim] - bmin[dim]) dim = q;
                if (!(bmax[0] > bmin[0]) && !(bmax[1] > bmin[1]) && !(bmax[2] > bmin[2])) continue;
                const double split = 0.5 * (bmin[dim] + bmax[dim]);
                const double *cc = dim == 0 ? lx : (dim == 1 ? ly : lz);
                int nl = 0;
                for (int c0 = lo; c0 <= hi; c0 += 64) {
                    const int i = c0 + lane;
                    nl += __popcll(__ballot(i <= hi && cc[i] < split));
                }
                const int s = lo + nl;
                if (s == lo || s > hi) {   // one side empty: reported, left a bucket
                    if (lane == 0) atomicOr(&A.L->err, 1);
                    continue;
                }
                int run = 0;
                for (int c0 = lo; c0 <= hi; c0 += 64) {   // upper positions holding a lower one
                    const int i = c0 + lane;
                    const bool f = i <= hi && cc[i] < split;
                    const unsigned long long m = __ballot(f);
                    const int ex = run + __popcll(m & ((1ull << lane) - 1));
                    if (f && i >= s) posR[lo + (nl - 1 - ex)] = (short)i;
                    run += __popcll(m);
                }
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                run = 0;
                for (int c0 = lo; c0 < s; c0 += 64) {     // lower positions holding an upper one
                    const int i = c0 + lane;
                    const bool in = i < s, f = in && cc[i] < split;
                    const unsigned long long m = __ballot(f);
                    const int ex = run + __popcll(m & ((1ull << lane) - 1));
                    if (in && !f) {
                        const int j = posR[lo + (i - lo) - ex];
                        double d = lx[i]; lx[i] = lx[j]; lx[j] = d;
                        d = ly[i]; ly[i] = ly[j]; ly[j] = d;
                        d = lz[i]; lz[i] = lz[j]; lz[j] = d;
                        const int u = ls[i]; ls[i] = ls[j]; ls[j] = u;
                    }
                    run += __popcll(m);
                }
                if (lane == 0) children(k, lo, hi, s, dim, split, nxt);
            }
            for (int b = 2 * w; b < nsml; b += T / 32) {   // at most 32 particles: half a
                const bool have = b + half < nsml;             // wavefront each
                const int k = have ? qa[cur][1][b + half] : 0;
                const int lo = have ? nlo[k] : 0, hi = have ? nhi[k] : -1;
                const int i = lo + l32;
                const bool in = i <= hi;
                double bmin[3] = {DBL_MAX, DBL_MAX, DBL_MAX};
                double bmax[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
                if (in) {
                    const double v[3] = {lx[i], ly[i], lz[i]};
                    for (int d = 0; d < 3; ++d) {       // comparisons, as in the larger cells
                        bmin[d] = v[d] < bmin[d] ? v[d] : bmin[d];
                        bmax[d] = v[d] > bmax[d] ? v[d] : bmax[d];
                    }
                }
                for (int o = 16; o > 0; o >>= 1)
                    for (int d = 0; d < 3; ++d) {
                        const double l = __shfl_xor(bmin[d], o), h = __shfl_xor(bmax[d], o);
                        bmin[d] = l < bmin[d] ? l : bmin[d];
                        bmax[d] = h > bmax[d] ? h : bmax[d];
                    }
                int dim = 0;
                for (int q = 1; q < 3; ++q)
                    if (bmax[q] - bmin[q] > bmax[dim] - bmin[dim]) dim = q;
                const bool ext = have && (bmax[0] > bmin[0] || bmax[1] > bmin[1] ||
                                          bmax[2] > bmin[2]);
                const double split = 0.5 * (bmin[dim] + bmax[dim]);
                const double *cc = dim == 0 ? lx : (dim == 1 ? ly : lz);
                const bool f = ext && in && cc[i] < split;
                const unsigned long long mm = __ballot(f);
                const uint32_t m = (uint32_t)(mm >> (32 * half));
                const int nl = __popc(m), s = lo + nl, ex = __popc(m & ((1u << l32) - 1));
                const bool ok = ext && s > lo && s <= hi;
                if (ext && !ok && l32 == 0) atomicOr(&A.L->err, 1);
                if (ok && f && i >= s) posR[lo + (nl - 1 - ex)] = (short)i;
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                if (ok && i < s && !f) {
                    const int j = posR[i - ex];
                    double d = lx[i]; lx[i] = lx[j]; lx[j] = d;
                    d = ly[i]; ly[i] = ly[j]; ly[j] = d;
                    d = lz[i]; lz[i] = lz[j]; lz[j] = d;
                    const int u = ls[i]; ls[i] = ls[j]; ls[j] = u;
                }
                if (ok && l32 == 0) children(k, lo, hi, s, dim, split, nxt);
            }
            cur = nxt;
            __syncthreads();
        }
        // storage-order particles; the cells' slots
        const int nloc = nloc_sh;
        if (tid == 0) {
            const int need = nloc - 1;
            if (need == 0) {
                slot_sh = 0;
            } else if (4 * need > chunk) {
                slot_sh = atomicAdd(&A.L->nloc, need);
            } else {
                if (need > left) {
                    slot = atomicAdd(&A.L->nloc, chunk);
                    left = chunk;
                }
                slot_sh = slot;
                slot += need;
                left -= need;
            }
        }
        for (int i = tid; i < cnt; i += T) {
            const int s = ls[i];
            const double mm = A.m[s], hh = A.h[s];
            const uint32_t bt = A.bits[s];
            lm[i] = mm;
            lh[i] = hh;
            lact[i] = bt & 1u;
            A.px[glo + i] = lx[i];
            A.py[glo + i] = ly[i];
            A.pz[glo + i] = lz[i];
            A.perm[glo + i] = s;
            A.pm[glo + i] = mm;
            A.ph[glo + i] = hh;
            A.pact[glo + i] = bt;
        }
        for (int k = tid; k < nloc; k += T) arr[k] = 0;
        __syncthreads();
        const int used = slot_sh + nloc - 1;             // from the last slot down
        const bool room = next + used <= A.cap;
        if (!room && tid == 0) atomicOr(&A.L->err, 2);
        // sizes and active buckets, climbing from the buckets
        for (int k = tid; k < nloc; k += T) {
            if (nch[k] >= 0) continue;
            int na = 0;
            for (int i = nlo[k]; i <= nhi[k]; ++i) na |= lact[i];
            atomicMax(&maxb_sh, nhi[k] - nlo[k] + 1);
            nsz[k] = 1;
            nac[k] = (short)na;
            for (int c = npar[k]; c >= 0; c = npar[c]) {
                if (__hip_atomic_fetch_add(&arr[c], 1, __ATOMIC_ACQ_REL,
                                           __HIP_MEMORY_SCOPE_WORKGROUP) == 0)
                    break;
                const int c0 = nch[c];
                nsz[c] = (short)(1 + nsz[c0] + nsz[c0 + 1]);
                nac[c] = (short)(nac[c0] + nac[c0 + 1]);
            }
        }
        __syncthreads();
        for (int k = tid; k < nloc; k += T) {        // preorder ids and bucket ranks
            int p = 0, bp = 0;
            for (int c = k; npar[c] >= 0; c = npar[c]) {
                const int c0 = nch[npar[c]];
                ++p;
                if (c != c0) {
                    p += nsz[c0];
                    bp += nac[c0];
                }
            }
            npre[k] = (short)p;
            nbp[k] = (short)bp;
            arr[k] = 0;
        }
        __syncthreads();
        if (room) {
            const int s1 = A.cap - used;                 // slot of preorder id 1
            auto slot = [&](int k) { return k == 0 ? root : s1 + npre[k] - 1; };
            auto get = [&](int i, double *p, double &mm, double &hh) {
                p[0] = lx[i];
                p[1] = ly[i];
                p[2] = lz[i];
                mm = lm[i];
                hh = lh[i];
                return lact[i] != 0;
            };
            for (int k = tid; k < nloc; k += T) {    // records, climbing likewise
                if (nch[k] >= 0) continue;
                double g[GS];
                for (int q = 0; q < GS; ++q) g[q] = 0.0;
                const int sk = slot(k);
                bucket_record<ORDER>(nlo[k], nhi[k], get, g, A.bb8 + 8 * (size_t)sk);
                double *o = A.gm + (size_t)GS * sk;
                for (int q = 0; q < GS; ++q) o[q] = g[q];
                for (int c = npar[k]; c >= 0; c = npar[c]) {
                    if (__hip_atomic_fetch_add(&arr[c], 1, __ATOMIC_ACQ_REL,
                                               __HIP_MEMORY_SCOPE_WORKGROUP) == 0)
                        break;
                    const double *c0 = A.gm + (size_t)GS * slot(nch[c]);
                    const double *c1 = A.gm + (size_t)GS * slot(nch[c] + 1);
                    for (int q = 0; q < GS; ++q) g[q] = 0.0;
                    mass_children(c0, c1, g);
                    for (int q = 0; q < 2; ++q) {
                        const double *cq = q ? c1 : c0;
                        const double d[3] = {cq[2] - g[2], cq[3] - g[3], cq[4] - g[4]};
                        mom_shift<ORDER>(cq, d, g);
                    }
                    o = A.gm + (size_t)GS * slot(c);
                    for (int q = 0; q < GS; ++q) o[q] = g[q];
                }
            }
            __syncthreads();
            for (int k = tid >> 4; k < nloc; k += T / 16) {   // Bmax, 16 lanes per cell
                if (nch[k] < 0) continue;                // buckets have theirs
                double *o = A.gm + (size_t)GS * slot(k);
                const double cm[3] = {o[2], o[3], o[4]};
                double b2 = 0.0;
                for (int i = nlo[k] + (tid & 15); i <= nhi[k]; i += 16) {
                    const double d2 = cm_d2(lx[i], ly[i], lz[i], cm);
                    b2 = d2 > b2 ? d2 : b2;
                }
                for (int q = 8; q > 0; q >>= 1) {
                    const double u = __shfl_xor(b2, q);
                    b2 = u > b2 ? u : b2;
                }
                if ((tid & 15) == 0) o[GM_B] = b2;
            }
            for (int k = tid; k < nloc; k += T) {
                GNode &g = A.nd[slot(k)];
                const int c = nch[k];
                if (k > 0) {
                    g.lo = glo + nlo[k];
                    g.hi = glo + nhi[k];
                    g.root = troot;
                    g.pre = npre[k];
                    g.bpre = nbp[k];
                }
                g.dim = ndm[k];
                g.split = nsp[k];
                g.size = nsz[k];
                g.nab = nac[k];
                g.ch0 = c < 0 ? -1 : slot(c);
                g.ch1 = c < 0 ? -1 : slot(c + 1);
            }
            if (tid == 0) A.subn[t] = make_int2(s1, nloc - 1);
        }
        __syncthreads();
    }
    if (tid == 0 && maxb_sh > 0) atomicMax(&A.L->maxb, maxb_sh);
}

// The systems of at most nBucket particles, a bucket each, by one thread.
template <int ORDER> __global__ __launch_bounds__(256) void k_gt_tiny(int nr, TreeArgs A)
{
    constexpr int GS = gm_stride(ORDER);
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= nr) return;
    GNode &g = A.nd[c];
    if (g.hi - g.lo >= A.nBucket) return;
    for (int i = g.lo; i <= g.hi; ++i) {
        const int s = A.perm[i];
        A.pm[i] = A.m[s];
        A.ph[i] = A.h[s];
        A.pact[i] = A.bits[s];
    }
    double v[GS];
    for (int k = 0; k < GS; ++k) v[k] = 0.0;
    const int na = bucket_record<ORDER>(
        g.lo, g.hi,
        [&](int i, double *p, double &m, double &h) {
            p[0] = A.px[i];
            p[1] = A.py[i];
            p[2] = A.pz[i];
            m = A.pm[i];
            h = A.ph[i];
            return (A.pact[i] & 1u) != 0;
        },
        v, A.bb8 + 8 * (size_t)c);
    double *o = A.gm + (size_t)GS * c;
    for (int k = 0; k < GS; ++k) o[k] = v[k];
    g.size = 1;
    g.nab = na > 0;
}

// The record of a bucket of more than LMAX coincident particles, by one
// wavefront: 64 particles at a time into registers, the sums that follow the
// storage order (mass, softening, centre) taken from them lane by lane, all
// else by lane and reduced.  By one lane each particle cost two chains of
// loads: a build with 10^5 of them took 69 ms, 9.9 this way.
__device__ __forceinline__ double lane_d(double v, int l)
{
    const long long b = __double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)b, l);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}

template <int ORDER> __device__ void large_bucket(const TreeArgs &A, int c, int lane)
{
#pragma clang fp contract(off)
    constexpr int GS = gm_stride(ORDER);
    GNode &g = A.nd[c];
    const int lo = g.lo, hi = g.hi;
    double M = 0.0, S = 0.0, R[3] = {0.0, 0.0, 0.0};
    double bl[3] = {DBL_MAX, DBL_MAX, DBL_MAX}, bh[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
    double fsm = 0.0;
    int na = 0;
    for (int b = lo; b <= hi; b += 64) {
        const int i = b + lane;
        double m = 0.0, mh = 0.0, mp[3] = {0.0, 0.0, 0.0};
        bool act = false;
        if (i <= hi) {
            const int s = A.perm[i];
            const double p[3] = {A.px[i], A.py[i], A.pz[i]}, h = A.h[s];
            const uint32_t t = A.bits[s];
            m = A.m[s];
            A.pm[i] = m;
            A.ph[i] = h;
            A.pact[i] = t;
            act = t & 1u;
            mh = m * h;
            if (h > fsm) fsm = h;
            for (int d = 0; d < 3; ++d) {
                mp[d] = m * p[d];
                if (act && p[d] < bl[d]) bl[d] = p[d];
                if (act && p[d] > bh[d]) bh[d] = p[d];
            }
        }
        na += __popcll(__ballot(act));
        const int n = min(64, hi - b + 1);
        for (int l = 0; l < n; ++l) {
            M += lane_d(m, l);
            S += lane_d(mh, l);
            for (int d = 0; d < 3; ++d) R[d] += lane_d(mp[d], l);
        }
    }
    if (M > 0) {
        S /= M;
        for (int d = 0; d < 3; ++d) R[d] /= M;
    }
    double v[GS], b2 = 0.0;
    for (int k = 0; k < GS; ++k) v[k] = 0.0;
    for (int i = lo + lane; i <= hi; i += 64) {
        const double d2 = cm_d2(A.px[i], A.py[i], A.pz[i], R);
        if (d2 > b2) b2 = d2;
        const double d[3] = {A.px[i] - R[0], A.py[i] - R[1], A.pz[i] - R[2]};
        mom_particle<ORDER>(A.pm[i], d, v);
    }
    for (int o = 32; o > 0; o >>= 1) {
        double t = __shfl_xor(b2, o);
        b2 = t > b2 ? t : b2;
        t = __shfl_xor(fsm, o);
        fsm = t > fsm ? t : fsm;
        for (int d = 0; d < 3; ++d) {
            t = __shfl_xor(bl[d], o);
            bl[d] = t < bl[d] ? t : bl[d];
            t = __shfl_xor(bh[d], o);
            bh[d] = t > bh[d] ? t : bh[d];
        }
        for (int k = GM_Q; k < GS; ++k) v[k] += __shfl_xor(v[k], o);
    }
    if (lane) return;
    v[0] = M;
    v[1] = S;
    for (int d = 0; d < 3; ++d) v[2 + d] = R[d];
    v[GM_B] = b2;
    double *o = A.gm + (size_t)GS * c, *bb = A.bb8 + 8 * (size_t)c;
    for (int k = 0; k < GS; ++k) o[k] = v[k];
    for (int d = 0; d < 3; ++d) {
        bb[d] = bl[d];
        bb[3 + d] = bh[d];
    }
    bb[6] = fsm;
    bb[7] = (double)na;
    g.size = 1;
    g.nab = na > 0;
    atomicMax(&A.L->maxb, hi - lo + 1);
}

// A split cell above LMAX, by a pair of lanes (q 0, 1): its record and its
// subtree's counts from its children's.
template <int ORDER> __device__ __forceinline__ void upper_record(const TreeArgs &A, int c, int q)
{
#pragma clang fp contract(off)
    constexpr int GS = gm_stride(ORDER);
    GNode &g = A.nd[c];
    double v[GS];
    for (int k = 0; k < GS; ++k) v[k] = 0.0;
    const int i0 = g.ch0, i1 = g.ch1;
    const double *c0 = A.gm + (size_t)GS * i0, *c1 = A.gm + (size_t)GS * i1;
    mass_children(c0, c1, v);
    const double *cq = q ? c1 : c0;
    const double d[3] = {cq[2] - v[2], cq[3] - v[3], cq[4] - v[4]};
    mom_shift<ORDER>(cq, d, v);
    for (int k = GM_Q; k < GS; ++k) v[k] += __shfl_xor(v[k], 1);
    if (q) return;
    v[GM_B] = 0.0;
    double *o = A.gm + (size_t)GS * c;
    for (int k = 0; k < GS; ++k) o[k] = v[k];
    const int s0 = A.nd[i0].size, a0 = A.nd[i0].nab;
    g.sizeLo = s0;
    g.nabLo = a0;
    g.size = 1 + s0 + A.nd[i1].size;
    g.nab = a0 + A.nd[i1].nab;
}

// What k_gt_mid closed in one unit: buckets, then the split cells, deepest
// level first (one wavefront).
template <int ORDER> __global__ __launch_bounds__(64) void k_gt_up_unit(TreeArgs A)
{
    const int lane = threadIdx.x;
    if (A.L->err & 2) return;
    const int2 u = A.useg[blockIdx.x];
    if (u.y == 0) return;
    const int base = A.nd[A.unit[blockIdx.x]].lo;
    const bool leaves = u.y < 0;
    if (leaves) {
        for (int e = 0; e < u.x; e += 64) {
            const int c = e + lane < u.x ? A.seg[base + e + lane] : -1;
            for (unsigned long long m = __ballot(c >= 0 && A.nd[c].dim < 0); m; m &= m - 1)
                large_bucket<ORDER>(A, __shfl(c, __ffsll((long long)m) - 1), lane);
        }
        __syncthreads();
    }
    for (int l = abs(u.y) - 1; l >= 0; --l) {
        const int e0 = l ? A.segl[base + l - 1] : 0, e1 = A.segl[base + l];
        for (int e = e0 + (lane >> 1); e < e1; e += 32) {
            const int c = A.seg[base + e];
            if (!(leaves && A.nd[c].dim < 0)) upper_record<ORDER>(A, c, lane & 1);
        }
        __syncthreads();
    }
}

// One workgroup: the splitting cells of the levels above MID from the deepest
// up, then the roots' preorder ids and first bucket ranks, then those of the
// level's children downwards; to the host the cells, active buckets, largest
// bucket and error word.  A level holds at most 2 n / MID cells, usually a
// few, so what it costs is one record's chain of loads: about 2 us between
// barriers against 4.7 us for a launch of its own (18 of them on a galaxy of
// 50k particles, 26 on 2^21).
constexpr int TOP_T = 512, TOP_R = 8;                    // TOP_R: roots per thread
template <int ORDER>
__global__ __launch_bounds__(TOP_T) void k_gt_up_top(int nr, int nlist,
                                                     const int *__restrict__ list, int nlev,
                                                     TreeArgs A, int *host)
{
    __shared__ int2 ws[TOP_T / 64];
    int2 run = make_int2(0, 0);
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    // A build that failed has cells without a record: the host gets zeros for
    // its totals (a word of -1 would read as not yet written).
    const int err = A.L->err, lev = err ? 0 : nlev;
    if (err) nr = 0;
    auto splits = [&](int c) {                           // (the others are units)
        const GNode &g = A.nd[c];
        return g.hi - g.lo >= MID && g.dim >= 0;
    };
    // a level's cells (the first one's may be a list)
    auto cells = [&](int d, int first, int step, auto f) {
        const int *ls = d ? nullptr : list;
        const int a = A.L->lv[d], nc = ls ? nlist : A.L->lv[d + 1] - a;
        for (int i = first; i < nc; i += step) {
            const int c = ls ? ls[i] : a + i;
            if (splits(c)) f(c);
        }
        __syncthreads();
    };
    for (int d = lev - 1; d >= 0; --d)
        cells(d, tid >> 1, TOP_T / 2, [&](int c) { upper_record<ORDER>(A, c, tid & 1); });
    for (int b = 0; b < nr; b += TOP_T * TOP_R) {
        const int k0 = b + tid * TOP_R;
        int sz[TOP_R], na[TOP_R], ts = 0, ta = 0;
        for (int q = 0; q < TOP_R; ++q) {
            sz[q] = k0 + q < nr ? A.nd[k0 + q].size : 0;
            na[q] = k0 + q < nr ? A.nd[k0 + q].nab : 0;
        }
        for (int q = 0; q < TOP_R; ++q) {
            ts += sz[q];
            ta += na[q];
        }
        int is = ts, ia = ta;
        for (int o = 1; o < 64; o <<= 1) {
            const int us = __shfl_up(is, o), ua = __shfl_up(ia, o);
            if (lane >= o) {
                is += us;
                ia += ua;
            }
        }
        if (lane == 63) ws[w] = make_int2(is, ia);
        __syncthreads();
        int ps = run.x + is - ts, pa = run.y + ia - ta;
        for (int q = 0; q < TOP_T / 64; ++q) {
            if (q < w) {
                ps += ws[q].x;
                pa += ws[q].y;
            }
            run.x += ws[q].x;
            run.y += ws[q].y;
        }
        for (int q = 0; q < TOP_R; ++q) {
            if (k0 + q >= nr) break;
            A.nd[k0 + q].pre = ps;
            A.nd[k0 + q].bpre = pa;
            ps += sz[q];
            pa += na[q];
        }
        __syncthreads();
    }
    if (tid == 0) {
        tell_host(host + 1, run.x);
        tell_host(host + 2, run.y);
        tell_host(host + 3, A.L->maxb);
        tell_host(host + 4, A.L->next);
        tell_host(host + 5, A.L->nsub);
        tell_host(host, err);
    }
    for (int d = 0; d < lev; ++d)
        cells(d, tid, TOP_T, [&](int c) {
            const GNode &g = A.nd[c];
            GNode &l = A.nd[g.ch0], &u = A.nd[g.ch1];
            l.pre = g.pre + 1;
            l.bpre = g.bpre;
            u.pre = g.pre + 1 + g.sizeLo;
            u.bpre = g.bpre + g.nabLo;
        });
}

// Largest squared distances of the cells above LMAX: per unit, those of the
// cells k_gt_mid closed, and the unit's particles against every cell above
// it, by one atomic a cell.  The workgroup holds the unit's particles in
// registers, four a thread, 256 in a row to a wavefront, and takes the cells
// from a list in LDS; a wavefront passes over cells it has no particle of.
// With a wavefront to each closed cell its latest loads were waited for one
// after another: 43 us for 4096 particles, 66 us with 18 cells above a unit;
// 18 and 28 us this way.
constexpr int BM_T = 1024, BM_E = 4, BM_A = 256;         // BM_A: cells of the list
template <int ORDER> __global__ __launch_bounds__(BM_T) void k_gt_up_bmax(TreeArgs A)
{
    constexpr int GS = gm_stride(ORDER);
    __shared__ unsigned long long bm[BM_A];
    __shared__ double cx[BM_A], cy[BM_A], cz[BM_A];
    __shared__ int cell[BM_A], first[BM_A], last[BM_A];
    __shared__ int na_sh, up_sh;
    if (A.L->err & 2) return;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int root = A.unit[blockIdx.x];
    const int lo = A.nd[root].lo, hi = A.nd[root].hi;
    const int nclosed = A.useg[blockIdx.x].x;
    int up = A.nd[root].par;
    for (int done = 0; done < nclosed || up >= 0;) {
        const int nc = min(BM_A, nclosed - done);
        if (tid < nc) {                                  // closed cells
            const int c = A.seg[lo + done + tid];
            const bool leaf = A.nd[c].dim < 0;           // buckets have theirs
            cell[tid] = c;
            first[tid] = leaf ? 1 : A.nd[c].lo;
            last[tid] = leaf ? 0 : A.nd[c].hi;
        }
        if (tid == BM_T - 64) {                          // cells above
            int k = nc;
            for (; up >= 0 && k < BM_A; up = A.nd[up].par) {
                cell[k] = up;
                first[k] = lo;
                last[k++] = hi;
            }
            na_sh = k;
            up_sh = up;
        }
        __syncthreads();
        const int na = na_sh;
        up = up_sh;
        if (tid < na) {
            const double *o = A.gm + (size_t)GS * cell[tid];
            cx[tid] = o[2];
            cy[tid] = o[3];
            cz[tid] = o[4];
            bm[tid] = 0;
        }
        __syncthreads();
        for (int b = lo; b <= hi; b += BM_T * BM_E) {
            const int wlo = b + w * 64 * BM_E, whi = min(hi, wlo + 64 * BM_E - 1);
            if (wlo > hi) continue;
            double x[BM_E], y[BM_E], z[BM_E];
            for (int q = 0; q < BM_E; ++q) {
                const int i = min(hi, wlo + 64 * q + lane);
                x[q] = A.px[i];
                y[q] = A.py[i];
                z[q] = A.pz[i];
            }
            for (int k = 0; k < na; ++k) {
                const int c0 = first[k], c1 = last[k];
                if (c0 > whi || c1 < wlo) continue;
                const double cm[3] = {cx[k], cy[k], cz[k]};
                double b2 = 0.0;
                for (int q = 0; q < BM_E; ++q) {
                    const int i = wlo + 64 * q + lane;
                    const double d2 = cm_d2(x[q], y[q], z[q], cm);
                    b2 = i >= c0 && i <= c1 && d2 > b2 ? d2 : b2;
                }
                for (int q = 32; q > 0; q >>= 1) {
                    const double v = __shfl_xor(b2, q);
                    b2 = v > b2 ? v : b2;
                }
                if (lane == 0) atomicMax(&bm[k], (unsigned long long)__double_as_longlong(b2));
            }
        }
        __syncthreads();
        if (tid < na) {
            double *o = A.gm + (size_t)GS * cell[tid] + GM_B;
            if (tid >= nc) atomicMax(reinterpret_cast<unsigned long long *>(o), bm[tid]);
            else if (first[tid] <= last[tid]) *o = __longlong_as_double((long long)bm[tid]);
        }
        done += nc;
        __syncthreads();
    }
}

// What the walk and the parity tools read, in preorder.
struct EmitArgs {
    int iOpenType;
    double dCrit;
    int *tint;
    double *tdbl;
    WalkNode *wn;
    double *cell, *momOH;
    int *bucket, *broot;
    double *bbox;
};

// Preorder id and first bucket rank of a cell above LMAX or of a subtree of
// k_gt_sub, up the parents to a cell of the levels above MID (those before
// ntop), which has its own.
__device__ __forceinline__ int2 climb(const GNode *__restrict__ nd, int ntop, int c)
{
    int p = 0, b = 0;
    while (c >= ntop) {
        const int up = nd[c].par;
        const GNode &g = nd[up];
        ++p;
        if (g.ch1 == c) {
            p += g.sizeLo;
            b += g.nabLo;
        }
        c = up;
    }
    return make_int2(p + nd[c].pre, b + nd[c].bpre);
}

// Per cell at preorder id c: the parity record (iDim, pLower, pUpper, iLower,
// iNext, 0; mass, softening, c.o.m., fOpen2, Bmax, fSplit), the walk record,
// the cell record (traceless Q as the walk stores it, walk.c:41-48) and the
// reduced O/H; fOpen2 by pkdCalcOpen (pkd.c:2228-2264).  Of a bucket with
// active particles also its entry of the bucket list (rank bk).
template <int ORDER>
__device__ __forceinline__ void emit_cell(const TreeArgs &A, const EmitArgs &E, int slot, int c,
                                          int bk)
{
#pragma clang fp contract(off)
    constexpr int GS = gm_stride(ORDER);
    const GNode &g = A.nd[slot];
    const double *M = A.gm + (size_t)GS * slot;
    const double Bmax = sqrt(M[GM_B]);
    double dOpen;
    if (E.iOpenType == 1) {
        dOpen = 2 / sqrt(3.0) * Bmax / E.dCrit;
        if (dOpen < Bmax) dOpen = Bmax;
    } else {
        dOpen = Bmax;
    }
    const double fOpen2 = dOpen * dOpen;
    const GNode &rt = A.nd[g.root];
    const int next = c + g.size < rt.pre + rt.size ? c + g.size : -1;
    const int second = g.ch1 >= 0 ? c + 1 + A.nd[g.ch0].size : -1;
    int *ti = E.tint + 6 * (size_t)c;   // iLower: the first child is c + 1 in preorder
    ti[0] = g.dim;
    ti[1] = g.lo;
    ti[2] = g.hi;
    ti[3] = g.dim >= 0 ? c + 1 : -1;
    ti[4] = next;
    ti[5] = 0;
    double *td = E.tdbl + 8 * (size_t)c;
    for (int k = 0; k < 5; ++k) td[k] = M[k];
    td[5] = fOpen2;
    td[6] = Bmax;
    td[7] = g.split;
    WalkNode w;
    w.cx = M[2];
    w.cy = M[3];
    w.cz = M[4];
    w.fOpen2 = fOpen2;
    w.fSoft = M[1];
    w.pLower = g.lo;
    w.pUpper = g.hi;
    w.iLower = g.dim >= 0 ? c + 1 : -1;
    w.iNext = next;
    w.iUpper = second;
    w.pad1 = 0;
    E.wn[c] = w;
    double *r = E.cell + (size_t)CR_N * c;
    r[CR_M] = M[0];
    for (int d = 0; d < 3; ++d) r[CR_X + d] = M[2 + d];
    r[CR_H] = M[1];
    const double *Q = M + GM_Q;
    for (int k = 0; k < 6; ++k) r[CR_QR + k] = Q[k];
    const double tr = Q[0] + Q[1] + Q[2];
    for (int k = 0; k < 3; ++k) r[CR_QT + k] = Q[k] - tr / 3.0;
    for (int k = 3; k < 6; ++k) r[CR_QT + k] = Q[k];
    if constexpr (ORDER >= 3) {
        double *o = E.momOH + (size_t)OH_N * c;
        const double *T = M + GM_T;
        const double tx = T[0] + T[1] + T[7], ty = T[2] + T[3] + T[8], tz = T[4] + T[5] + T[9];
        o[0] = T[0] - 0.6 * tx;
        o[1] = T[1] - 0.2 * tx;
        o[2] = T[2] - 0.2 * ty;
        o[3] = T[3] - 0.6 * ty;
        o[4] = T[4] - 0.2 * tz;
        o[5] = T[5] - 0.2 * tz;
        o[6] = T[6];
        o[7] = T[7] - 0.2 * tx;
        o[8] = T[8] - 0.2 * ty;
        o[9] = T[9] - 0.6 * tz;
        if constexpr (ORDER >= 4) {
            const double *F = M + GM_F;
            const double sxx = F[0] + F[6] + F[9], syy = F[6] + F[3] + F[12];
            const double szz = F[9] + F[12] + F[14], sxy = F[2] + F[1] + F[10];
            const double sxz = F[4] + F[8] + F[11], syz = F[7] + F[5] + F[13];
            const double s4 = sxx + syy + szz;
            o[10] = F[0] - 6.0 / 7.0 * (sxx - 0.1 * s4);
            o[11] = F[1] - 3.0 / 7.0 * sxy;
            o[12] = F[2] - 3.0 / 7.0 * sxy;
            o[13] = F[3] - 6.0 / 7.0 * (syy - 0.1 * s4);
            o[14] = F[4] - 3.0 / 7.0 * sxz;
            o[15] = F[5] - 3.0 / 7.0 * syz;
            o[16] = F[6] - 1.0 / 7.0 * (sxx + syy - 0.2 * s4);
            o[17] = F[7] - 1.0 / 7.0 * syz;
            o[18] = F[8] - 1.0 / 7.0 * sxz;
            o[19] = F[9] - 1.0 / 7.0 * (sxx + szz - 0.2 * s4);
            o[20] = F[10] - 1.0 / 7.0 * sxy;
            o[21] = F[11] - 3.0 / 7.0 * sxz;
            o[22] = F[12] - 1.0 / 7.0 * (syy + szz - 0.2 * s4);
            o[23] = F[13] - 3.0 / 7.0 * syz;
            o[24] = F[14] - 6.0 / 7.0 * (szz - 0.1 * s4);
        }
    }
    if (g.dim < 0 && g.nab) {
        E.bucket[bk] = c;
        E.broot[bk] = rt.pre;
        for (int d = 0; d < 8; ++d) E.bbox[8 * (size_t)bk + d] = A.bb8[8 * (size_t)slot + d];
    }
}

// Blocks below nub: a thread per slot above LMAX and per system that is a
// bucket.  The others: a wavefront per subtree of k_gt_sub, its cells in
// preorder (consecutive slots and ids).
template <int ORDER>
__global__ __launch_bounds__(256) void k_gt_emit(int nub, int nup, int nsub, int nr, TreeArgs A,
                                                 EmitArgs E)
{
    if ((int)blockIdx.x < nub) {
        const int c = blockIdx.x * 256 + threadIdx.x;
        if (c >= nup) return;
        const GNode &g = A.nd[c];
        if (g.hi - g.lo < LMAX && !(c < nr && g.hi - g.lo < A.nBucket)) return;   // with its subtree
        const int2 p = climb(A.nd, A.L->b, c);
        emit_cell<ORDER>(A, E, c, p.x, p.y);
        return;
    }
    const int t = (blockIdx.x - nub) * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (t >= nsub) return;
    const int root = A.sub[t];
    const int2 s = A.subn[t], p = climb(A.nd, A.L->b, root);
    for (int k = lane; k <= s.y; k += 64) {
        const int slot = k ? s.x + k - 1 : root;
        emit_cell<ORDER>(A, E, slot, p.x + k, p.y + (k ? A.nd[slot].bpre : 0));
    }
}

}  // namespace

// The stream running dry without the word is an error, so the wait always ends.
int host_word(hipStream_t st, const int *p, int *v)
{
    for (unsigned it = 0;; ++it) {
        *v = __atomic_load_n(p, __ATOMIC_ACQUIRE);
        if (*v != -1) return GG_OK;
        if ((it & 1023u) != 1023u) continue;
        const hipError_t e = hipStreamQuery(st);
        if (e == hipErrorNotReady) continue;
        GG_HIP(e);
        *v = __atomic_load_n(p, __ATOMIC_ACQUIRE);
        GG_CHECK(*v != -1, GG_EHIP, "a device word never reached the host");
        return GG_OK;
    }
}

// Particles per tile: enough tiles to fill the chip on a small store, fewer
// of them (each block adds up its cell's tile counts) on a large one.  Builds
// of Plummer spheres with 1024 / 2048 / 4096, us: 5000 particles 392 / 400 / 416,
// 30011 718 / 773 / 890, 3 10^5 1026 / 1125 / 1339, 2^20 1789 / 1857 / 2088,
// 2^21 2930 / 2933 / 3114, 2^22 5133 / 5020 / 5140, 2^24 19822 / 18933 / 19131;
// uniform boxes the same way.
static int tile_size(int n) { return n < (1 << 21) ? 1024 : 2048; }

// One partition pass over the tiles k_gt_ctl listed.
template <int MODE>
static int gt_partition(hipStream_t st, const TileArgs &A, int grid, unsigned long long *kbox)
{
    hipLaunchKernelGGL(k_gt_count<MODE>, dim3(grid), dim3(256), 0, st, A);
    hipLaunchKernelGGL(k_gt_rank<MODE>, dim3(grid), dim3(256), 0, st, A);
    hipLaunchKernelGGL(k_gt_swap<MODE>, dim3(grid), dim3(256), 0, st, A, kbox);
    GG_HIP(hipGetLastError());
    return GG_OK;
}

// One build with slots for cap cells; *room tells whether they were enough.
static int gtree_try(GGPKD pkd, int nSys, const int *sysOff, int nBucket, int iOpenType,
                     double dCrit, int iOrder, int cap, bool *room)
{
    GravDev &G = pkd->grav;
    hipStream_t st = pkd->stream;
    const int n = pkd->nLocal;
    // roots: the non-empty systems, their ranges and what each size's stage
    // reads (Roots), in one array for the device
    const int ts = tile_size(n);
    std::vector<int> up;
    int nr = 0;
    for (int s = 0; s < nSys; ++s) nr += sysOff[s + 1] > sysOff[s];
    Roots R{};
    R.n = n;
    R.nr = nr;
    R.nBucket = nBucket;
    size_t oBig = 0, oBase[3] = {0, 0, 0}, oT = 0;
    int nttile = 0;                  // tiles of the type orders
    if (nr == 1) {                   // the whole store
        R.nbig = n > MID;
        R.nunit = n > LMAX && n <= MID;
        R.nsub[n > LSML] = n > nBucket && n <= LMAX;
        R.maxTiny = n <= nBucket ? n : 0;
        if (n > LMAX) nttile = nblk(n, ts);
    } else {
        std::vector<int> big, mid, base[3];              // (roots above MID and LMAX)
        up.resize(2 * (size_t)nr);
        for (int s = 0, k = 0; s < nSys; ++s) {
            const int cnt = sysOff[s + 1] - sysOff[s];
            if (cnt <= 0) continue;
            if ((k & 255) == 0) {
                base[0].push_back(R.nsub[0]);
                base[1].push_back(R.nsub[1]);
                base[2].push_back(R.nunit);
            }
            up[k] = sysOff[s];
            up[nr + k] = sysOff[s + 1] - 1;
            if (cnt > MID) big.push_back(k);
            else if (cnt > LMAX) ++R.nunit;
            else if (cnt > nBucket) ++R.nsub[cnt > LSML];
            else R.maxTiny = std::max(R.maxTiny, cnt);
            if (cnt > LMAX) mid.push_back(k);
            ++k;
        }
        R.nbig = (int)big.size();
        R.ntroot = (int)mid.size();
        auto add = [&](const std::vector<int> &v) {
            const size_t at = up.size();
            up.insert(up.end(), v.begin(), v.end());
            return at;
        };
        oBig = add(big);
        for (int k : big) up.push_back(up[k]);
        for (int k : big) up.push_back(up[nr + k]);
        for (int q = 0; q < 3; ++q) oBase[q] = add(base[q]);
        oT = add(mid);
        for (int k : mid) {
            up.push_back(nttile);
            nttile += nblk(up[nr + k] - up[k] + 1, ts);
        }
    }
    const size_t n1 = (size_t)n;
    // tiles of a level, or of the type orders, and a level's cells, at most
    const size_t mtile = std::max<size_t>(n1 / ts + n1 / MID + 1, nttile);
    const size_t mbox = 2 * (n1 / MID) + 2;
    const int order = iOrder >= 4 ? 4 : (iOrder == 3 ? 3 : 2);
    GG_TRY(G.px.reserve(sizeof(double) * n1));
    GG_TRY(G.py.reserve(sizeof(double) * n1));
    GG_TRY(G.pz.reserve(sizeof(double) * n1));
    GG_TRY(G.pm.reserve(sizeof(double) * n1));
    GG_TRY(G.ph.reserve(sizeof(double) * n1));
    GG_TRY(G.pact.reserve(sizeof(uint32_t) * n1));
    GG_TRY(G.perm.reserve(sizeof(int) * n1));
    GG_TRY(G.acc.reserve(sizeof(double) * 5 * n1));
    GG_TRY(G.gposR.reserve(sizeof(int) * n1));
    GG_TRY(G.gnode.reserve(sizeof(GNode) * (size_t)cap));
    GG_TRY(G.gm.reserve(sizeof(double) * gm_stride(order) * (size_t)cap));
    GG_TRY(G.gbb8.reserve(sizeof(double) * 8 * (size_t)cap));
    GG_TRY(G.gbox.reserve(sizeof(unsigned long long) * 2 * BOX_N * mbox));
    GG_TRY(G.gtile.reserve(sizeof(int4) * mtile));
    GG_TRY(G.gflag.reserve(sizeof(unsigned long long) * mtile * (ts / 64)));
    GG_TRY(G.gtcnt.reserve(sizeof(int) * 2 * mtile));
    GG_TRY(G.gunit.reserve((sizeof(int) + sizeof(int2)) * (size_t)n));
    GG_TRY(G.gsub.reserve((sizeof(int) + sizeof(int2)) * (size_t)n));
    GG_TRY(G.gseg.reserve(sizeof(int) * 2 * n1));
    GG_TRY(G.glev.reserve(sizeof(GLevel)));
    GG_TRY(G.groot.reserve(sizeof(int) * std::max<size_t>(up.size(), 1)));
    if (!G.hst)
        GG_HIP(hipHostMalloc((void **)&G.hst, sizeof(int) * GravDev::NHST, hipHostMallocDefault));
    GLevel *L = G.glev.as<GLevel>();
    TreeArgs T;
    T.nBucket = nBucket;
    T.cap = cap;
    T.L = L;
    T.nd = G.gnode.as<GNode>();
    T.gm = G.gm.as<double>();
    T.bb8 = G.gbb8.as<double>();
    T.px = G.px.as<double>();
    T.py = G.py.as<double>();
    T.pz = G.pz.as<double>();
    T.pm = G.pm.as<double>();
    T.ph = G.ph.as<double>();
    T.pact = G.pact.as<uint32_t>();
    T.perm = G.perm.as<int>();
    T.m = pkd->f[GG_MASS].as<double>();
    T.h = pkd->f[GG_SOFT].as<double>();
    T.bits = pkd->f[GG_IACTIVE].as<uint32_t>();
    // a unit, or a cell left to k_gt_sub, holds a particle: at most n of each
    int2 *subn = G.gsub.as<int2>(), *useg = G.gunit.as<int2>();
    int *sub = reinterpret_cast<int *>(subn + n), *unit = reinterpret_cast<int *>(useg + n);
    int *seg = G.gseg.as<int>(), *segl = seg + n;
    T.sub = sub;
    T.subn = subn;
    T.unit = unit;
    T.useg = useg;
    T.seg = seg;
    T.segl = segl;
    const int *rl = G.groot.as<int>();
    R.lo = rl;
    R.hi = rl + nr;
    R.bslot = rl + oBig;
    R.blo = R.bslot + R.nbig;
    R.bhi = R.blo + R.nbig;
    for (int q = 0; q < 3; ++q) R.base[q] = rl + oBase[q];
    R.tslot = rl + oT;
    R.toff = R.tslot + R.ntroot;
    const int *list = nr > 1 ? R.bslot : nullptr;        // the first level's cells
    unsigned long long *box[2];
    box[0] = G.gbox.as<unsigned long long>();
    box[1] = box[0] + BOX_N * mbox;
    volatile int *hv = G.hst;
    for (int k = 0; k < 16; ++k) hv[k] = -1;
    if (nr > 1)
        GG_HIP(hipMemcpyAsync(G.groot.p, up.data(), sizeof(int) * up.size(), hipMemcpyHostToDevice,
                              st));
    hipLaunchKernelGGL(k_gt_roots, dim3(nblk(nr, 256)), dim3(256), 0, st, R, T.nd, box[0], unit,
                       sub, L);
    hipLaunchKernelGGL(k_gt_init, dim3(nblk(n, 256 * INIT_E)), dim3(256), 0, st, R,
                       pkd->f[GG_R].as<double>(), T.bits, T.px, T.py, T.pz, T.perm, box[0], L);
    hipLaunchKernelGGL(k_gt_tell, dim3(1), dim3(1), 0, st, &L->need, G.hst);
    GG_HIP(hipGetLastError());
    TileArgs A;
    A.ts = ts;
    A.mask = 0;
    A.L = L;
    A.tiles = G.gtile.as<int4>();
    A.nd = T.nd;
    A.x = T.px;
    A.y = T.py;
    A.z = T.pz;
    A.src = T.perm;
    A.bits = T.bits;
    A.flag = G.gflag.as<unsigned long long>();
    A.tcnt = G.gtcnt.as<int>();
    A.tpre = A.tcnt + mtile;
    A.posR = G.gposR.as<int>();
    A.err = &L->err;
    // msrBuildTree's active-type orders (master.c:4262).  A particle with
    // the second order's bit has one of the first's, so where all have it
    // both orders leave everything in place.
    int lack = 0;
    GG_TRY(host_word(st, G.hst, &lack));
    if (lack && nttile > 0) {
        hipLaunchKernelGGL(k_gt_type_tiles, dim3(nblk(nttile, 256)), dim3(256), 0, st, R, ts,
                           nttile, T.nd, G.gtile.as<int4>(), L);
        A.mask = GG_TYPE_ACTIVE | GG_TYPE_TREEACTIVE;
        GG_TRY(gt_partition<1>(st, A, nttile, nullptr));
        A.mask = GG_TYPE_TREEACTIVE;
        GG_TRY(gt_partition<1>(st, A, nttile, nullptr));
    }
    const int ntroot = nr > 1 ? R.ntroot : n > LMAX;
    if (lack && ntroot < nr)
        hipLaunchKernelGGL(k_gt_type_small, dim3(std::min(nblk(nr, TY_W), 8192)), dim3(64 * TY_W),
                           0, st, R, pkd->f[GG_R].as<double>(), T.bits, T.px, T.py, T.pz, T.perm);
    int nunit = R.nunit, nlev = 0;
    if (R.nbig > 0) {
        const int grid = (int)(n1 / ts + n1 / MID + 1);  // tiles of a level
        // The levels.  The host learns a level's tile count while its
        // partition runs, in time to queue the next level behind it.
        for (int depth = 0;; ++depth) {
            GG_CHECK(depth < DMAX, GG_EUNSUP, "tree deeper than %d levels", DMAX);
            int *h = G.hst + 16 + 4 * (depth & 3);
            for (int k = 0; k < 2; ++k) ((volatile int *)h)[k] = -1;
            hipLaunchKernelGGL(k_gt_ctl, dim3(1), dim3(CTL_T), 0, st, ts, depth, cap, R.nbig,
                               depth ? nullptr : list, L, T.nd, box[depth & 1],
                               box[(depth & 1) ^ 1], G.gtile.as<int4>(), unit, h);
            GG_TRY(gt_partition<0>(st, A, grid, box[(depth & 1) ^ 1]));
            int nt = 0;
            GG_TRY(host_word(st, h, &nt));
            if (nt == 0) {
                GG_TRY(host_word(st, h + 1, &nunit));
                nlev = depth;            // levels with a splitting cell
                break;
            }
        }
    }
    // the units and the subtrees below them, then the records upwards
    int *ht = G.hst + 4;
    if (nunit > 0)
        hipLaunchKernelGGL(k_gt_mid, dim3(nunit), dim3(MID_T), 0, st, unit, cap, L, T.nd, T.px,
                           T.py, T.pz, T.perm, sub, seg, segl, useg);
    auto by_order = [&](auto f) {
        if (order == 4) f(std::integral_constant<int, 4>{});
        else if (order == 3) f(std::integral_constant<int, 3>{});
        else f(std::integral_constant<int, 2>{});
    };
    by_order([&](auto o) {
        constexpr int O = decltype(o)::value;
        if (R.nsub[0] > 0) {
            const int grid = std::min(R.nsub[0], 2560);
            hipLaunchKernelGGL((k_gt_sub<O, LSML, 64>), dim3(grid), dim3(64), 0, st, T, 0,
                               R.nsub[0], cap < 2 * n + 2 ? R.nsub[0] / grid : 0);
        }
        if (R.nsub[1] + nunit > 0)
            hipLaunchKernelGGL((k_gt_sub<O, LMAX, 256>), dim3(std::min(std::max(n / 64, 1), 2048)),
                               dim3(256), 0, st, T, R.nsub[0], -1, 0);
        if (R.maxTiny > 0)
            hipLaunchKernelGGL(k_gt_tiny<O>, dim3(nblk(nr, 256)), dim3(256), 0, st, nr, T);
        if (nunit > 0) hipLaunchKernelGGL(k_gt_up_unit<O>, dim3(nunit), dim3(64), 0, st, T);
        hipLaunchKernelGGL(k_gt_up_top<O>, dim3(1), dim3(TOP_T), 0, st, nr, R.nbig, list, nlev, T,
                           ht);
        if (nunit > 0) hipLaunchKernelGGL(k_gt_up_bmax<O>, dim3(nunit), dim3(BM_T), 0, st, T);
    });
    GG_HIP(hipGetLastError());
    int tot[6];   // error word, cells, active buckets, largest bucket, slots above LMAX, subtrees
    for (int k = 0; k < 6; ++k) GG_TRY(host_word(st, ht + k, tot + k));
    const int err = tot[0], nn = tot[1], nb = tot[2], nup = tot[4], nsub = tot[5];
    GG_CHECK(!(err & 1), GG_EUNSUP,
             "a cell split leaves one side empty (positions differ in the last bit only)");
    *room = !(err & 2);
    if (!*room) return GG_OK;
    G.maxBucket = tot[3];     // > 64 only for cells of coincident particles (pkd.c:2489)
    GG_TRY(G.wnode.reserve(sizeof(WalkNode) * (size_t)nn));
    GG_TRY(G.cell.reserve(sizeof(double) * CR_N * (size_t)nn));
    GG_TRY(G.momOH.reserve(sizeof(double) * OH_N * (size_t)(iOrder >= 3 ? nn : 1)));
    GG_TRY(G.tint.reserve(sizeof(int) * 6 * (size_t)nn));
    GG_TRY(G.tdbl.reserve(sizeof(double) * 8 * (size_t)nn));
    GG_TRY(G.bucket.reserve(sizeof(int) * std::max(nb, 1)));
    GG_TRY(G.broot.reserve(sizeof(int) * std::max(nb, 1)));
    GG_TRY(G.bbox.reserve(sizeof(double) * 8 * (size_t)std::max(nb, 1)));
    EmitArgs E;
    E.iOpenType = iOpenType;
    E.dCrit = dCrit;
    E.tint = G.tint.as<int>();
    E.tdbl = G.tdbl.as<double>();
    E.wn = G.wnode.as<WalkNode>();
    E.cell = G.cell.as<double>();
    E.momOH = G.momOH.as<double>();
    E.bucket = G.bucket.as<int>();
    E.broot = G.broot.as<int>();
    E.bbox = G.bbox.as<double>();
    const int nub = nblk(nup, 256);
    by_order([&](auto o) {
        hipLaunchKernelGGL(k_gt_emit<decltype(o)::value>, dim3(nub + nblk(nsub, 4)), dim3(256), 0,
                           st, nub, nup, nsub, nr, T, E);
    });
    GG_HIP(hipGetLastError());
    G.nNodes = nn;
    G.nb = nb;
    return GG_OK;
}

int gtree_build(GGPKD pkd, int nSys, const int *sysOff, int nBucket, int iOpenType, double dCrit,
                int iOrder)
{
    GravDev &G = pkd->grav;
    hipStream_t st = pkd->stream;
    const int n = pkd->nLocal;
    G.built = 0;
    if (n == 0) {   // an empty store: one empty bucket (pkd.c:2684-2712)
        const int ti[6] = {-1, 0, -1, -1, -1, 0};
        const double td[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        WalkNode w{};
        w.pLower = 0;
        w.pUpper = -1;
        w.iLower = w.iNext = w.iUpper = -1;
        GG_TRY(G.wnode.reserve(sizeof w));
        GG_TRY(G.tint.reserve(sizeof ti));
        GG_TRY(G.tdbl.reserve(sizeof td));
        GG_HIP(hipMemcpyAsync(G.tint.p, ti, sizeof ti, hipMemcpyHostToDevice, st));
        GG_HIP(hipMemcpyAsync(G.tdbl.p, td, sizeof td, hipMemcpyHostToDevice, st));
        GG_HIP(hipMemcpyAsync(G.wnode.p, &w, sizeof w, hipMemcpyHostToDevice, st));
        GG_HIP(hipStreamSynchronize(st));
        G.nNodes = 1;
        G.nb = G.maxBucket = 0;
    } else {
        // Slots: buckets of nBucket hold about 0.65 nBucket particles, so
        // 3 n / nBucket cells; twice that fits all but odd distributions,
        // which build again with the most a tree can have.
        const int64_t most = 2 * (int64_t)n + 2;
        const int64_t guess = 6 * (int64_t)n / nBucket + 2 * (int64_t)nSys + 4096;
        GG_CHECK(most <= INT_MAX, GG_EINVAL, "%d particles: too many for one tree", n);
        bool room = false;
        GG_TRY(gtree_try(pkd, nSys, sysOff, nBucket, iOpenType, dCrit, iOrder,
                         (int)std::min(most, guess), &room));
        if (!room)
            GG_TRY(gtree_try(pkd, nSys, sysOff, nBucket, iOpenType, dCrit, iOrder, (int)most,
                             &room));
        GG_CHECK(room, GG_EHIP, "tree cell capacity exceeded");
    }
    const int nb = G.nb;
    GG_TRY(G.cnt.reserve(sizeof(int) * 3 * std::max(nb, 1)));
    GG_TRY(G.off.reserve(sizeof(int64_t) * (3 * (size_t)std::max(nb, 1) + 1)));
    G.n = n;
    G.iRoot = 0;
    G.nSys = nSys;
    G.iOrder = iOrder;
    G.nBucket = nBucket;
    G.built = 1;
    G.listsCurrent = 0;
    ++G.treeId;
    return GG_OK;
}

}  // namespace gg
