// Gravity tree build on the device: the tree of gasoline's pkdBuildBinary
// (pkd.c:2627-2723), node for node.
//
// Large cells level by level over the whole chip, then each cell of at most
// 4096 particles in one workgroup, then each of at most 512 in another:
// every cell is split at the midpoint of the
// longest axis of its particles' bounding box (pkd.c:2493-2505) unless it
// holds nBucket particles or fewer or has no extent (pkd.c:2489).  The
// partition reproduces pkdUpperPart's Hoare scan (pkd.c:1109-1157): a Hoare
// scan swaps the k-th particle of the lower part that belongs above with the
// k-th particle, counted from the top, of the upper part that belongs below,
// so each particle's destination follows from prefix counts and the cells
// of a level partition in parallel.  pkdActiveTypeOrder's partitions
// (pkd.c:1304-1355) run the same way over each system.  Cells are numbered
// in preorder afterwards, from subtree sizes.  Mass, softening and centre of
// mass are summed as the reference sums them (buckets over their particles
// in storage order, cells from their children, lower then upper), and
// bounds, Bmax and fOpen2 are exact, so every quantity the walk decides on
// is the reference's to the bit.  The multipole moments (pkdCalcCell,
// pkd.c:2018-2135) are direct sums over each cell's particles in a fixed
// but different order; they enter only the force arithmetic.
//
// Several independent systems build at once: each is a root of its own.
#include "gg_internal.h"
#include "gg_scan.h"

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <vector>

namespace gg {
namespace {

int nblk(int64_t n, int b) { return (int)((n + b - 1) / b); }

constexpr int MOM_CH = 2048;     // particles per moment work item
constexpr int NM = 32;           // per item: raw Q (6), O (10), H (15), Bmax
constexpr int MOM_SMALL = 64;    // cells of at most this many particles: a thread each
constexpr int LMAX = 512;        // cells of at most LMAX particles finish in one workgroup
constexpr int MID = 4096;        // cells of at most MID particles reach LMAX in one workgroup

constexpr int DMAX = 2048;       // depths a tree may have

// Per cell in creation order.
struct GNode {
    int lo, hi, par, side;       // particle range, parent, 0 lower / 1 upper
    int ch0, ch1, dim, root;     // children (-1), split axis (-1: bucket), root cell
    int s, size, pre, depth;     // split position, subtree size, preorder id, level
    double split;
};

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
    int next;            // first free node id once the levels are done
    int err;             // 1: a split left one side empty
    int need[2];         // particles lacking a type bit of each order
    int maxb;            // largest bucket
    int maxdep;          // deepest cell k_gt_mid made
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

__device__ __forceinline__ void box_init(unsigned long long *b)
{
    for (int d = 0; d < 3; ++d) {
        b[d] = ~0ull;
        b[3 + d] = 0ull;
    }
}

// The last root whose first position is <= i.
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

// Root cells, their empty bounds and the level state.
__global__ void k_gt_roots(int nr, const int *__restrict__ rlo, const int *__restrict__ rhi,
                           GNode *__restrict__ nd, unsigned long long *__restrict__ box,
                           int *__restrict__ unit, GLevel *__restrict__ L)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k == 0) {
        L->a = 0;
        L->b = L->next = nr;
        L->ntile = L->nunit = L->err = L->need[0] = L->need[1] = L->maxb = L->maxdep = 0;
    }
    if (k >= nr) return;
    GNode &g = nd[k];
    g.lo = rlo[k];
    g.hi = rhi[k];
    g.par = -1;
    g.side = -1;
    g.root = k;
    g.ch0 = g.ch1 = -1;
    g.dim = -1;
    g.split = 0.0;
    g.depth = 0;
    box_init(box + 6 * (size_t)k);
    unit[k] = k;
}

// Min/max of a workgroup's lo/hi (256 threads), left to threads 0..5 as
// order keys: thread d < 3 the lower bound d, 3 + d the upper.
__device__ __forceinline__ unsigned long long block_box(double *lo, double *hi, double (*sm)[6])
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int o = 32; o > 0; o >>= 1)
        for (int d = 0; d < 3; ++d) {
            const double l = __shfl_xor(lo[d], o), h = __shfl_xor(hi[d], o);
            lo[d] = l < lo[d] ? l : lo[d];
            hi[d] = h > hi[d] ? h : hi[d];
        }
    if (lane == 0)
        for (int d = 0; d < 3; ++d) {
            sm[w][d] = lo[d];
            sm[w][3 + d] = hi[d];
        }
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

// Positions into storage order, the roots' bounds, and whether a particle
// lacks the type bits of msrBuildTree's orders (*need, master.c:4262).
__global__ __launch_bounds__(256) void k_gt_init(int n, int nr, const int *__restrict__ rlo,
                                                 const double *__restrict__ r,
                                                 const uint32_t *__restrict__ bits,
                                                 double *__restrict__ x, double *__restrict__ y,
                                                 double *__restrict__ z, int *__restrict__ src,
                                                 unsigned long long *__restrict__ box,
                                                 GLevel *__restrict__ L)
{
    __shared__ double sm[4][6];
    const int first = blockIdx.x * (256 * INIT_E), last = min(n, first + 256 * INIT_E) - 1;
    const int r0 = root_of(first, nr, rlo), r1 = root_of(last, nr, rlo);
    double lo[3] = {DBL_MAX, DBL_MAX, DBL_MAX}, hi[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
    bool lack0 = false, lack1 = false;
    for (int e = 0; e < INIT_E; ++e) {
        const int i = first + e * 256 + threadIdx.x;
        if (i > last) break;
        const double v[3] = {r[3 * (size_t)i], r[3 * (size_t)i + 1], r[3 * (size_t)i + 2]};
        x[i] = v[0];
        y[i] = v[1];
        z[i] = v[2];
        src[i] = i;
        const uint32_t t = bits[i];
        lack0 |= !(t & (GG_TYPE_ACTIVE | GG_TYPE_TREEACTIVE));
        lack1 |= !(t & GG_TYPE_TREEACTIVE);
        if (r0 == r1) {
            for (int d = 0; d < 3; ++d) {
                lo[d] = v[d] < lo[d] ? v[d] : lo[d];
                hi[d] = v[d] > hi[d] ? v[d] : hi[d];
            }
        } else {
            unsigned long long *b = box + 6 * (size_t)root_of(i, nr, rlo);
            for (int d = 0; d < 3; ++d) {
                if (v[d] != v[d]) continue;
                atomicMin(b + d, ord_key(v[d]));
                atomicMax(b + 3 + d, ord_key(v[d]));
            }
        }
    }
    const unsigned long long m0 = __ballot(lack0), m1 = __ballot(lack1);
    if ((threadIdx.x & 63) == 0) {
        if (m0) atomicOr(&L->need[0], 1);
        if (m1) atomicOr(&L->need[1], 1);
    }
    if (r0 != r1) return;
    const unsigned long long k = block_box(lo, hi, sm);
    unsigned long long *b = box + 6 * (size_t)r0;
    if (threadIdx.x < 3) atomicMin(b + threadIdx.x, k);
    else if (threadIdx.x < 6) atomicMax(b + threadIdx.x, k);
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

// One workgroup decides the level's cells (mode 0, pkd.c:2489-2505): cells of
// more than MID particles with any extent split at the middle of their
// longest axis and get two child ids; the others join the unit list.  Then
// the tiles of the splitting cells.  mode 1 (the type orders): every cell
// is partitioned, none split.  The tile count goes to *host.  One workgroup
// because a level has at most 2 n / MID cells and every later launch waits
// for it: 4-6 us a level, against the three scans, the decision and id
// kernels and the host's wait it replaces.
constexpr int CTL_T = 1024;
__global__ __launch_bounds__(CTL_T) void k_gt_ctl(int mode, int ts, int depth, GLevel *L,
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
    int nsp = 0, ntl = 0, nun = 0;       // splits, tiles and units so far
    for (int base = a; base < b && !bad; base += CTL_T) {
        const int c = base + tid;
        int split = 0, nt = 0, un = 0, lo = 0;
        if (c < b) {
            GNode &g = nd[c];
            lo = g.lo;
            const int cnt = g.hi - lo + 1;
            if (mode == 1) {
                nt = (cnt + ts - 1) / ts;
            } else if (cnt <= MID) {
                un = 1;
            } else {
                const unsigned long long *k = box + 6 * (size_t)(c - a);
                double bmin[3], bmax[3];
                for (int d = 0; d < 3; ++d) {
                    bmin[d] = ord_val(k[d]);
                    bmax[d] = ord_val(k[3 + d]);
                }
                bool extent = false;
                for (int d = 0; d < 3; ++d) extent |= bmax[d] > bmin[d];
                if (extent) {
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
                h.side = q;
                h.root = g.root;
                h.ch0 = h.ch1 = -1;
                h.dim = -1;
                h.split = 0.0;
                h.depth = depth + 1;
                box_init(kbox + 6 * (size_t)(kid + q));
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
        if (mode == 0) {
            L->a = b;
            L->b = L->next = b + 2 * nsp;
            L->nunit = nunit0 + nun;
            tell_host(host + 1, nunit0 + nun);
            tell_host(host + 2, b + 2 * nsp);
        }
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

constexpr int TW = 64;                   // flag words of the largest tile

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
// a particle and 56 a swapped one.  Measured per level: 31 us on a 2^21
// Plummer sphere (count 6.3, rank 4.6, control 5.9) and 14 us on 3 10^5
// particles (4.3, 3.9, 5.4), where the chain of loads and the bounds'
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
    const int hi = g.hi, s = g.s, ch0 = g.ch0;
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
    if (MODE == 1) return;
    const int kid = ch0 - A.L->a;        // the children's level starts at L->a now
    for (int q = 0; q < 2; ++q) {
        const unsigned long long k = block_box(bl[q], bh[q], sm[q]);
        unsigned long long *b = kbox + 6 * (size_t)(kid + q);
        if (threadIdx.x < 3) atomicMin(b + threadIdx.x, k);
        else if (threadIdx.x < 6) atomicMax(b + threadIdx.x, k);
    }
}

// The cells of the unit list, each by one workgroup: a cell of LMAX..MID
// particles is split in LDS, level by level with the rules above, until its
// parts hold at most LMAX (marked for k_gt_local, dim -2, or left buckets).
// At most MID / LMAX parts are open at a time, so a level is a handful of
// wavefront passes over the particles between barriers (7 us measured on one
// full cell) instead of four launches.  Flags are bits, 64 particles a word, and ranks come
// from a prefix over the 64 words.  MID is what the LDS holds: 124 KB, one
// workgroup per CU.
constexpr int MID_T = 1024, MID_O = MID / LMAX, MID_W = MID / 64;
static_assert(MID_W == 64, "one wavefront scans the flag words");
__global__ __launch_bounds__(MID_T) void k_gt_mid(const int *__restrict__ unit, GLevel *L,
                                                  int nBucket, GNode *__restrict__ nd,
                                                  double *__restrict__ px, double *__restrict__ py,
                                                  double *__restrict__ pz, int *__restrict__ perm,
                                                  int *__restrict__ err)
{
#pragma clang fp contract(off)
    __shared__ double lx[MID], ly[MID], lz[MID];
    __shared__ int ls[MID];
    __shared__ unsigned short posR[MID];
    __shared__ unsigned long long fbits[MID_W + 1];
    __shared__ int wpre[MID_W + 1];
    __shared__ int olo[2][MID_O], ohi[2][MID_O], onode[2][MID_O];
    __shared__ unsigned long long cb[MID_O][6];
    __shared__ double csplit[MID_O];
    __shared__ int cdim[MID_O], nopen[2];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int rootId = unit[blockIdx.x];
    const int glo = nd[rootId].lo, cnt = nd[rootId].hi - glo + 1;
    const int troot = nd[rootId].root, rdepth = nd[rootId].depth;
    if (cnt > MID) return;               // coincident particles: a bucket
    if (cnt <= LMAX) {
        if (tid == 0 && cnt > nBucket) nd[rootId].dim = -2;
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
        fbits[MID_W] = 0;
    }
    __syncthreads();
    // flags of positions below i
    auto F = [&](int i) {
        return wpre[i >> 6] + __popcll(fbits[i >> 6] & ((1ull << (i & 63)) - 1));
    };
    const int w0 = w * (MID / (MID_T / 64));             // this wavefront's particles
    constexpr int WN = MID / MID_T;                      // its words
    int cur = 0, depth = 0;
    for (; nopen[cur] > 0; ++depth) {
        const int no = nopen[cur];
        if (tid < 6 * no) cb[tid / 6][tid % 6] = tid % 6 < 3 ? ~0ull : 0ull;
        if (tid == 0) nopen[cur ^ 1] = 0;
        __syncthreads();
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
            for (int o = 32; o > 0; o >>= 1)
                for (int d = 0; d < 3; ++d) {
                    const double l = __shfl_xor(bl[d], o), h = __shfl_xor(bh[d], o);
                    bl[d] = l < bl[d] ? l : bl[d];
                    bh[d] = h > bh[d] ? h : bh[d];
                }
            if (lane == 0)
                for (int d = 0; d < 3; ++d) {
                    atomicMin(&cb[q][d], ord_key(bl[d]));
                    atomicMax(&cb[q][3 + d], ord_key(bh[d]));
                }
        }
        __syncthreads();
        if (tid < no) {                                  // split decisions
            double bmin[3], bmax[3];
            bool extent = false;
            for (int d = 0; d < 3; ++d) {
                bmin[d] = ord_val(cb[tid][d]);
                bmax[d] = ord_val(cb[tid][3 + d]);
                extent |= bmax[d] > bmin[d];
            }
            int d = 0;
            for (int k = 1; k < 3; ++k)
                if (bmax[k] - bmin[k] > bmax[d] - bmin[d]) d = k;
            cdim[tid] = extent ? d : -1;                 // -1: coincident, a bucket
            csplit[tid] = 0.5 * (bmin[d] + bmax[d]);
        }
        __syncthreads();
        for (int k = 0; k < WN; ++k) {                   // lower-part flags
            const int i = w0 + 64 * k + lane;
            bool f = false;
            for (int q = 0; q < no; ++q)
                if (i >= olo[cur][q] && i <= ohi[cur][q] && cdim[q] >= 0)
                    f = (cdim[q] == 0 ? lx[i] : (cdim[q] == 1 ? ly[i] : lz[i])) < csplit[q];
            const unsigned long long m = __ballot(f);
            if (lane == 0) fbits[(w0 >> 6) + k] = m;
        }
        __syncthreads();
        if (w == 0) {
            const int c = __popcll(fbits[lane]);
            int inc = c;
            for (int o = 1; o < 64; o <<= 1) {
                const int u = __shfl_up(inc, o);
                if (lane >= o) inc += u;
            }
            wpre[lane] = inc - c;
            if (lane == 63) wpre[MID_W] = inc;
        }
        __syncthreads();
        int part[WN];                                    // swap partner's rank slot, -1: none
        for (int k = 0; k < WN; ++k) {
            const int i = w0 + 64 * k + lane;
            part[k] = -1;
            for (int q = 0; q < no; ++q) {
                const int lo = olo[cur][q], hi = ohi[cur][q];
                if (i < lo || i > hi || cdim[q] < 0) continue;
                const int F0 = F(lo), nl = F(hi + 1) - F0, Fi = F(i) - F0;
                const bool f = (fbits[i >> 6] >> (i & 63)) & 1;
                if (i >= lo + nl && f) posR[lo + nl - 1 - Fi] = (unsigned short)i;
                if (i < lo + nl && !f) part[k] = i - Fi;
            }
        }
        if (w == 0) {                                    // nodes of the two parts
            const bool in = lane < no;
            int lo = 0, hi = -1, s = 0;
            bool sp = false;
            if (in) {
                lo = olo[cur][lane];
                hi = ohi[cur][lane];
                s = lo;
                if (cdim[lane] >= 0) {
                    s = lo + F(hi + 1) - F(lo);
                    sp = s > lo && s <= hi;
                    if (!sp) atomicOr(err, 1);           // one side empty: reported
                }
            }
            const unsigned long long ms = __ballot(sp);
            int id0 = 0;
            if (lane == 0 && ms) id0 = atomicAdd(&L->next, 2 * __popcll(ms));
            id0 = __shfl(id0, 0) + 2 * __popcll(ms & ((1ull << lane) - 1));
            const int me = in ? onode[cur][lane] : 0;
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
                    h.side = q;
                    h.root = troot;
                    h.ch0 = h.ch1 = -1;
                    h.split = 0.0;
                    h.depth = rdepth + depth + 1;
                    h.dim = !open && a1 - a0 + 1 > nBucket ? -2 : -1;
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
        __syncthreads();
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
    }
    if (tid == 0) atomicMax(&L->maxdep, rdepth + depth);
    for (int i = tid; i < cnt; i += MID_T) {
        px[glo + i] = lx[i];
        py[glo + i] = ly[i];
        pz[glo + i] = lz[i];
        perm[glo + i] = ls[i];
    }
}

// Work items of the cells [a, b): ceil(count / ch) each for cells of more
// than minc particles, none for the others.
__global__ void k_gt_items(int a, int b, int ch, int minc, const GNode *__restrict__ nd,
                           int *__restrict__ nit)
{
    const int c = a + blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= b) return;
    const int cnt = nd[c].hi - nd[c].lo + 1;
    nit[c - a] = cnt > minc ? (cnt + ch - 1) / ch : 0;
}

// Subtree sizes and preorder ids, over the nodes of one depth (list).
__global__ void k_gt_size(int m, const int *__restrict__ list, GNode *__restrict__ nd)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= m) return;
    GNode &g = nd[list[k]];
    g.size = 1 + (g.ch0 >= 0 ? nd[g.ch0].size : 0) + (g.ch1 >= 0 ? nd[g.ch1].size : 0);
}

__global__ void k_gt_pre(int m, const int *__restrict__ list, GNode *__restrict__ nd)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= m) return;
    const GNode &g = nd[list[k]];
    if (g.ch0 >= 0) nd[g.ch0].pre = g.pre + 1;
    if (g.ch1 >= 0) nd[g.ch1].pre = g.pre + 1 + (g.ch0 >= 0 ? nd[g.ch0].size : 0);
}

// Nodes by depth: a count per depth, then each node to its depth's list.
// Each workgroup counts in LDS
// first, so the global counters see one atomic per workgroup and depth.

__global__ __launch_bounds__(256) void k_gt_depth_count(int nn, int ndep,
                                                        const GNode *__restrict__ nd,
                                                        int *__restrict__ cnt)
{
    __shared__ int h[DMAX];
    for (int d = threadIdx.x; d < ndep; d += 256) h[d] = 0;
    __syncthreads();
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c < nn) atomicAdd(&h[nd[c].depth], 1);
    __syncthreads();
    for (int d = threadIdx.x; d < ndep; d += 256)
        if (h[d]) atomicAdd(&cnt[d], h[d]);
}

__global__ __launch_bounds__(256) void k_gt_depth_list(int nn, int ndep,
                                                       const GNode *__restrict__ nd,
                                                       int *__restrict__ cur,
                                                       int *__restrict__ list)
{
    __shared__ int h[DMAX], b0[DMAX];
    for (int d = threadIdx.x; d < ndep; d += 256) h[d] = 0;
    __syncthreads();
    const int c = blockIdx.x * 256 + threadIdx.x;
    const bool ok = c < nn;
    const int dep = ok ? nd[c].depth : 0;
    const int r = ok ? atomicAdd(&h[dep], 1) : 0;
    __syncthreads();
    for (int d = threadIdx.x; d < ndep; d += 256)
        if (h[d]) b0[d] = atomicAdd(&cur[d], h[d]);
    __syncthreads();
    if (ok) list[b0[dep] + r] = c;
}

// Cells marked for the local build, and the scratch node slots each
// reserves for its descendants (2 count - 2 at most).
__global__ void k_gt_lmark(int nn, const GNode *__restrict__ nd, int *__restrict__ flag,
                           int *__restrict__ res)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nn) return;
    const bool l = nd[c].dim == -2;
    flag[c] = l;
    res[c] = l ? 2 * (nd[c].hi - nd[c].lo + 1) - 2 : 0;
}

__global__ void k_gt_lcompact(int nn, const int *__restrict__ flag, const int64_t *__restrict__ pos,
                              int *__restrict__ list)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c < nn && flag[c]) list[pos[c]] = c;
}

// The subtree of one marked cell (at most LMAX particles), built in LDS by
// one workgroup with the rules of the level loop: per level, each cell's
// bounds and split decision (a wavefront per cell), child ids in order,
// then each split cell's partition by the Hoare pairing of the k-th
// misplaced particles from either end (a wavefront per cell).  The cell is
// local node 0; descendant k >= 1 (in creation order) goes to scratch slot
// lres[root] + k - 1 with its links as local ids, and *used receives the
// node count; k_gt_lcopy then moves them into place.  The particles are
// written back in their new order.
__global__ __launch_bounds__(256) void k_gt_local(const int *__restrict__ lroot,
                                                  const int64_t *__restrict__ lres, int nBucket,
                                                  GNode *__restrict__ nd, GNode *__restrict__ scr,
                                                  int *__restrict__ used,
                                                  double *__restrict__ px, double *__restrict__ py,
                                                  double *__restrict__ pz, int *__restrict__ perm,
                                                  int *__restrict__ err)
{
#pragma clang fp contract(off)
    __shared__ double lx[LMAX], ly[LMAX], lz[LMAX];
    __shared__ int ls[LMAX];
    __shared__ short posR[LMAX];
    __shared__ short qa[2][LMAX];              // cells of the current / next level
    __shared__ short nlo[2 * LMAX], nhi[2 * LMAX];   // cell ranges (local positions)
    __shared__ short coff[LMAX], cs[LMAX];     // child offset (-1: none), split position
    __shared__ signed char cdim[LMAX];
    __shared__ double csplit[LMAX];
    __shared__ int wsum[4];
    __shared__ int nsplit_sh;
    const int rootId = lroot[blockIdx.x];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int glo = nd[rootId].lo, cnt = nd[rootId].hi - glo + 1;
    const int troot = nd[rootId].root, rdepth = nd[rootId].depth;
    GNode *const sb = scr + lres[rootId] - 1;   // local node k >= 1 at sb[k]
    for (int i = threadIdx.x; i < cnt; i += 256) {
        lx[i] = px[glo + i];
        ly[i] = py[glo + i];
        lz[i] = pz[glo + i];
        ls[i] = perm[glo + i];
    }
    if (threadIdx.x == 0) {
        nlo[0] = 0;
        nhi[0] = (short)(cnt - 1);
        qa[0][0] = 0;
    }
    __syncthreads();
    int nq = 1, cur = 0, nloc = 1, depth = 0;
    while (nq > 0) {
        // bounds, decision and lower-part count, a wavefront per cell
        for (int t = w; t < nq; t += 4) {
            const int k = qa[cur][t];
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
            for (int o = 32; o > 0; o >>= 1)
                for (int d = 0; d < 3; ++d) {
                    const double l = __shfl_xor(bmin[d], o), h = __shfl_xor(bmax[d], o);
                    bmin[d] = l < bmin[d] ? l : bmin[d];
                    bmax[d] = h > bmax[d] ? h : bmax[d];
                }
            bool extent = false;
            for (int d = 0; d < 3; ++d) extent |= bmax[d] > bmin[d];
            int dim = -1;
            double split = 0.0;
            if (hi - lo + 1 > nBucket && extent) {
                int d = 0;
                for (int q = 1; q < 3; ++q)
                    if (bmax[q] - bmin[q] > bmax[d] - bmin[d]) d = q;
                dim = d;
                split = 0.5 * (bmin[d] + bmax[d]);
            }
            int s = lo;
            if (dim >= 0) {
                const double *cc = dim == 0 ? lx : (dim == 1 ? ly : lz);
                int nl = 0;
                for (int c0 = lo; c0 <= hi; c0 += 64) {
                    const int i = c0 + lane;
                    nl += __popcll(__ballot(i <= hi && cc[i] < split));
                }
                s = lo + nl;
                if (s == lo || s > hi) {   // one side empty: reported, left a bucket
                    if (lane == 0) atomicOr(err, 1);
                    dim = -1;
                    s = lo;
                }
            }
            if (lane == 0) {
                GNode &g = k == 0 ? nd[rootId] : sb[k];
                g.lo = glo + lo;
                g.hi = glo + hi;
                g.dim = dim;
                g.split = dim >= 0 ? split : 0.0;
                g.ch0 = g.ch1 = -1;
                g.s = glo + s;
                g.root = troot;
                g.depth = rdepth + depth;
                coff[t] = dim >= 0 ? 1 : 0;
                cdim[t] = (signed char)dim;
                csplit[t] = split;
                cs[t] = (short)s;
            }
        }
        __syncthreads();
        {   // child offsets: exclusive sum of the split flags
            int v[4], sum = 0;
            for (int q = 0; q < 4; ++q) {
                const int t = threadIdx.x * 4 + q;
                v[q] = t < nq ? coff[t] : 0;
                sum += v[q];
            }
            int inc = sum;
            for (int o = 1; o < 64; o <<= 1) {
                const int u = __shfl_up(inc, o);
                if (lane >= o) inc += u;
            }
            if (lane == 63) wsum[w] = inc;
            __syncthreads();
            int ex = inc - sum, tot = 0;
            for (int q = 0; q < 4; ++q) {
                if (q < w) ex += wsum[q];
                tot += wsum[q];
            }
            for (int q = 0; q < 4; ++q) {
                const int t = threadIdx.x * 4 + q;
                if (t < nq) coff[t] = v[q] ? (short)ex : (short)-1;
                ex += v[q];
            }
            if (threadIdx.x == 0) nsplit_sh = tot;
        }
        __syncthreads();
        const int nsplit = nsplit_sh;
        // partitions and children, a wavefront per split cell
        for (int t = w; t < nq; t += 4) {
            const int co = coff[t];
            if (co < 0) continue;
            const int k = qa[cur][t];
            const int lo = nlo[k], hi = nhi[k], s = cs[t];
            const double split = csplit[t];
            const double *cc = cdim[t] == 0 ? lx : (cdim[t] == 1 ? ly : lz);
            const int nl = s - lo;
            int run = 0;
            for (int c0 = lo; c0 <= hi; c0 += 64) {   // upper positions holding a lower particle
                const int i = c0 + lane;
                const bool f = i <= hi && cc[i] < split;
                const unsigned long long m = __ballot(f);
                const int incl = run + __popcll(m & (lane == 63 ? ~0ull : ((1ull << (lane + 1)) - 1)));
                if (f && i >= s) posR[lo + (nl - incl)] = (short)i;
                run += __popcll(m);
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            run = 0;
            for (int c0 = lo; c0 < s; c0 += 64) {     // lower positions holding an upper one
                const int i = c0 + lane;
                const bool in = i < s;
                const bool f = in && cc[i] < split;
                const unsigned long long m = __ballot(f);
                const int excl = run + __popcll(m & ((1ull << lane) - 1));
                if (in && !f) {
                    const int j = posR[lo + (i - lo) - excl];
                    double d = lx[i]; lx[i] = lx[j]; lx[j] = d;
                    d = ly[i]; ly[i] = ly[j]; ly[j] = d;
                    d = lz[i]; lz[i] = lz[j]; lz[j] = d;
                    const int u = ls[i]; ls[i] = ls[j]; ls[j] = u;
                }
                run += __popcll(m);
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            if (lane == 0) {
                const int a0 = nloc + 2 * co, a1 = a0 + 1;
                nlo[a0] = (short)lo;
                nhi[a0] = (short)(s - 1);
                nlo[a1] = (short)s;
                nhi[a1] = (short)hi;
                qa[cur ^ 1][2 * co] = (short)a0;
                qa[cur ^ 1][2 * co + 1] = (short)a1;
                GNode &g = k == 0 ? nd[rootId] : sb[k];
                g.ch0 = a0;
                g.ch1 = a1;
                sb[a0].par = k;
                sb[a0].side = 0;
                sb[a1].par = k;
                sb[a1].side = 1;
            }
        }
        __syncthreads();
        nloc += 2 * nsplit;
        nq = 2 * nsplit;
        cur ^= 1;
        ++depth;
    }
    for (int i = threadIdx.x; i < cnt; i += 256) {
        px[glo + i] = lx[i];
        py[glo + i] = ly[i];
        pz[glo + i] = lz[i];
        perm[glo + i] = ls[i];
    }
    if (threadIdx.x == 0) used[blockIdx.x] = nloc - 1;
}

// The descendants of local build r from scratch to nodes nng + dbase[r] ...,
// links turned from local ids (0: the marked cell) to node ids.
__global__ __launch_bounds__(256) void k_gt_lcopy(const int *__restrict__ lroot,
                                                  const int64_t *__restrict__ lres,
                                                  const int *__restrict__ used,
                                                  const int64_t *__restrict__ dbase, int nng,
                                                  GNode *__restrict__ nd,
                                                  const GNode *__restrict__ scr)
{
    const int r = blockIdx.x, rootId = lroot[r], u = used[r];
    const int db = nng + (int)dbase[r];
    const GNode *const sb = scr + lres[rootId] - 1;
    auto fin = [&](int k) { return k < 0 ? -1 : (k == 0 ? rootId : db + k - 1); };
    for (int k = 1 + threadIdx.x; k <= u; k += 256) {
        GNode g = sb[k];
        g.ch0 = fin(g.ch0);
        g.ch1 = fin(g.ch1);
        g.par = fin(g.par);
        nd[db + k - 1] = g;
    }
    if (threadIdx.x == 0) {
        GNode &g = nd[rootId];
        g.ch0 = fin(g.ch0);
        g.ch1 = fin(g.ch1);
    }
}

// Storage-order particle fields: masses, softenings, type bits by source.
__global__ void k_gt_gather(int n, const int *__restrict__ src, const double *__restrict__ m,
                            const double *__restrict__ h, const uint32_t *__restrict__ bits,
                            double *__restrict__ pm, double *__restrict__ ph,
                            uint32_t *__restrict__ pact)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int s = src[i];
    pm[i] = m[s];
    ph[i] = h[s];
    pact[i] = bits[s];
}

// Mass, mass-weighted softening and centre of mass (pkd.c:2510-2576):
// buckets over their particles in storage order, cells from their
// children, lower then upper.  Deepest level first, one depth per launch.
__global__ void k_gt_mass(int m, const int *__restrict__ list, const GNode *__restrict__ nd,
                          const double *__restrict__ x, const double *__restrict__ y,
                          const double *__restrict__ z, const double *__restrict__ pm,
                          const double *__restrict__ ph, double *__restrict__ cm)
{
#pragma clang fp contract(off)
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= m) return;
    const int c = list[k];
    const GNode &g = nd[c];
    double fm, M = 0.0, S = 0.0, R[3] = {0.0, 0.0, 0.0};
    if (g.dim >= 0) {
        for (int k = 0; k < 2; ++k) {
            const int ch = k ? g.ch1 : g.ch0;
            if (ch == -1) continue;
            const double *q = cm + 5 * (size_t)ch;
            fm = q[0];
            M += fm;
            S += fm * q[1];
            for (int d = 0; d < 3; ++d) R[d] += fm * q[2 + d];
        }
    } else {
        for (int i = g.lo; i <= g.hi; ++i) {
            fm = pm[i];
            M += fm;
            S += fm * ph[i];
            R[0] += fm * x[i];
            R[1] += fm * y[i];
            R[2] += fm * z[i];
        }
    }
    if (M > 0) {
        S /= M;
        for (int d = 0; d < 3; ++d) R[d] /= M;
    }
    double *o = cm + 5 * (size_t)c;
    o[0] = M;
    o[1] = S;
    for (int d = 0; d < 3; ++d) o[2 + d] = R[d];
}

// Cell of each moment item (a thread per cell writes its items).
__global__ void k_gt_itemcell(int nn, const int64_t *__restrict__ ioff, int *__restrict__ icell)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nn) return;
    for (int64_t k = ioff[c]; k < ioff[c + 1]; ++k) icell[k] = c;
}

// One particle's terms of the moments about (cx, cy, cz): raw Q (6),
// reduced O (10) and H (15), and its distance for Bmax.
template <int ORDER>
__device__ __forceinline__ void mom_accum(double mm, double dx, double dy, double dz, double *Q,
                                          double *O, double *H, double &Bmax)
{
#pragma clang fp contract(off)
    constexpr bool wantO = ORDER >= 3, wantH = ORDER >= 4;
    const double d2 = dx * dx + dy * dy + dz * dz;
    const double d1 = sqrt(d2);
    if (d1 > Bmax) Bmax = d1;
    if (wantH) {
        H[0] += mm * (dx * dx * dx * dx - 6.0 / 7.0 * d2 * (dx * dx - 0.1 * d2));
        H[1] += mm * (dx * dy * dy * dy - 3.0 / 7.0 * d2 * dx * dy);
        H[2] += mm * (dx * dx * dx * dy - 3.0 / 7.0 * d2 * dx * dy);
        H[3] += mm * (dy * dy * dy * dy - 6.0 / 7.0 * d2 * (dy * dy - 0.1 * d2));
        H[4] += mm * (dx * dx * dx * dz - 3.0 / 7.0 * d2 * dx * dz);
        H[5] += mm * (dy * dy * dy * dz - 3.0 / 7.0 * d2 * dy * dz);
        H[6] += mm * (dx * dx * dy * dy - 1.0 / 7.0 * d2 * (dx * dx + dy * dy - 0.2 * d2));
        H[7] += mm * (dx * dx * dy * dz - 1.0 / 7.0 * d2 * dy * dz);
        H[8] += mm * (dx * dy * dy * dz - 1.0 / 7.0 * d2 * dx * dz);
        H[9] += mm * (dx * dx * dz * dz - 1.0 / 7.0 * d2 * (dx * dx + dz * dz - 0.2 * d2));
        H[10] += mm * (dx * dy * dz * dz - 1.0 / 7.0 * d2 * dx * dy);
        H[11] += mm * (dx * dz * dz * dz - 3.0 / 7.0 * d2 * dx * dz);
        H[12] += mm * (dy * dy * dz * dz - 1.0 / 7.0 * d2 * (dy * dy + dz * dz - 0.2 * d2));
        H[13] += mm * (dy * dz * dz * dz - 3.0 / 7.0 * d2 * dy * dz);
        H[14] += mm * (dz * dz * dz * dz - 6.0 / 7.0 * d2 * (dz * dz - 0.1 * d2));
    }
    if (wantO) {
        O[0] += mm * (dx * dx * dx - 0.6 * d2 * dx);
        O[1] += mm * (dx * dy * dy - 0.2 * d2 * dx);
        O[2] += mm * (dx * dx * dy - 0.2 * d2 * dy);
        O[3] += mm * (dy * dy * dy - 0.6 * d2 * dy);
        O[4] += mm * (dx * dx * dz - 0.2 * d2 * dz);
        O[5] += mm * (dy * dy * dz - 0.2 * d2 * dz);
        O[6] += mm * dx * dy * dz;
        O[7] += mm * (dx * dz * dz - 0.2 * d2 * dx);
        O[8] += mm * (dy * dz * dz - 0.2 * d2 * dy);
        O[9] += mm * (dz * dz * dz - 0.6 * d2 * dz);
    }
    Q[0] += mm * dx * dx;
    Q[1] += mm * dy * dy;
    Q[2] += mm * dz * dz;
    Q[3] += mm * dx * dy;
    Q[4] += mm * dx * dz;
    Q[5] += mm * dy * dz;
}

// Partial moments of one item (one wavefront): raw Q (6), reduced O (10)
// and H (15) about the cell's centre of mass, and the largest distance.
// Per-lane sums, then a fixed butterfly: the result does not depend on
// scheduling.
template <int ORDER>
__global__ __launch_bounds__(256) void k_gt_moments(int nitem, const int *__restrict__ icell,
                                                    const int64_t *__restrict__ ioff,
                                                    const GNode *__restrict__ nd,
                                                    const double *__restrict__ cm,
                                                    const double *__restrict__ x,
                                                    const double *__restrict__ y,
                                                    const double *__restrict__ z,
                                                    const double *__restrict__ pm,
                                                    double *__restrict__ part)
{
#pragma clang fp contract(off)
    const int it = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (it >= nitem) return;
    const int c = icell[it];
    const GNode &g = nd[c];
    if (g.hi - g.lo + 1 <= MOM_SMALL) return;   // k_gt_moments_small's
    const int first = g.lo + (int)(it - ioff[c]) * MOM_CH;
    const int last = min(g.hi, first + MOM_CH - 1);
    const double cx = cm[5 * (size_t)c + 2], cy = cm[5 * (size_t)c + 3], cz = cm[5 * (size_t)c + 4];
    constexpr bool wantO = ORDER >= 3, wantH = ORDER >= 4;
    double Q[6] = {0, 0, 0, 0, 0, 0}, O[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    double H[15] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    double Bmax = 0.0;
    for (int i = first + lane; i <= last; i += 64) {
        const double mm = pm[i];
        const double dx = x[i] - cx, dy = y[i] - cy, dz = z[i] - cz;
        mom_accum<ORDER>(mm, dx, dy, dz, Q, O, H, Bmax);
    }
    for (int o = 32; o > 0; o >>= 1) {
        for (int k = 0; k < 6; ++k) Q[k] += __shfl_xor(Q[k], o);
        if (wantO)
            for (int k = 0; k < 10; ++k) O[k] += __shfl_xor(O[k], o);
        if (wantH)
            for (int k = 0; k < 15; ++k) H[k] += __shfl_xor(H[k], o);
        Bmax = fmax(Bmax, __shfl_xor(Bmax, o));
    }
    if (lane == 0) {
        double *p = part + (size_t)NM * it;
        for (int k = 0; k < 6; ++k) p[k] = Q[k];
        for (int k = 0; k < 10; ++k) p[6 + k] = O[k];
        for (int k = 0; k < 15; ++k) p[16 + k] = H[k];
        p[31] = Bmax;
    }
}

// Cells of at most MOM_SMALL particles (most cells: the buckets and the
// levels just above them): one thread each sums its cell's particles in
// order, with no cross-lane reduction.  Each such cell is one item.
template <int ORDER>
__global__ __launch_bounds__(256) void k_gt_moments_small(int nitem, const int *__restrict__ icell,
                                                          const GNode *__restrict__ nd,
                                                          const double *__restrict__ cm,
                                                          const double *__restrict__ x,
                                                          const double *__restrict__ y,
                                                          const double *__restrict__ z,
                                                          const double *__restrict__ pm,
                                                          double *__restrict__ part)
{
#pragma clang fp contract(off)
    const int it = blockIdx.x * blockDim.x + threadIdx.x;
    if (it >= nitem) return;
    const int c = icell[it];
    const GNode &g = nd[c];
    if (g.hi - g.lo + 1 > MOM_SMALL) return;
    const double cx = cm[5 * (size_t)c + 2], cy = cm[5 * (size_t)c + 3], cz = cm[5 * (size_t)c + 4];
    double Q[6] = {0, 0, 0, 0, 0, 0}, O[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    double H[15] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    double Bmax = 0.0;
    for (int i = g.lo; i <= g.hi; ++i) {
        const double mm = pm[i];
        const double dx = x[i] - cx, dy = y[i] - cy, dz = z[i] - cz;
        mom_accum<ORDER>(mm, dx, dy, dz, Q, O, H, Bmax);
    }
    double *p = part + (size_t)NM * it;
    for (int k = 0; k < 6; ++k) p[k] = Q[k];
    for (int k = 0; k < 10; ++k) p[6 + k] = O[k];
    for (int k = 0; k < 15; ++k) p[16 + k] = H[k];
    p[31] = Bmax;
}

// Per cell in preorder: the parity record (iDim, pLower, pUpper, iLower,
// iNext, 0; mass, softening, c.o.m., fOpen2, Bmax, fSplit), the walk record,
// the cell record and O/H: moments summed over the cell's items in order,
// traceless Q as the walk stores it (walk.c:41-48), fOpen2 by pkdCalcOpen
// (pkd.c:2228-2264).
// Cells of more than one moment item (one wavefront per cell): lane j sums
// the items j, j + 64, ..., a fixed butterfly combines the lanes, and the
// total replaces the cell's first item.
__global__ __launch_bounds__(256) void k_gt_combine(int nn, int nv,
                                                    const int64_t *__restrict__ ioff,
                                                    double *__restrict__ part)
{
    const int b = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (b >= nn) return;
    const int64_t i0 = ioff[b], i1 = ioff[b + 1];
    if (i1 - i0 < 2) return;
    double M[31];
    for (int k = 0; k < 31; ++k) M[k] = 0.0;
    double Bmax = 0.0;
    for (int64_t it = i0 + lane; it < i1; it += 64) {
        const double *p = part + (size_t)NM * it;
        for (int k = 0; k < nv; ++k) M[k] += p[k];
        Bmax = fmax(Bmax, p[31]);
    }
    for (int o = 32; o > 0; o >>= 1) {
        for (int k = 0; k < nv; ++k) M[k] += __shfl_xor(M[k], o);
        Bmax = fmax(Bmax, __shfl_xor(Bmax, o));
    }
    if (lane) return;
    double *p = part + (size_t)NM * i0;
    for (int k = 0; k < nv; ++k) p[k] = M[k];
    p[31] = Bmax;
}

__global__ void k_gt_emit(int nn, int iOrder, int iOpenType, double dCrit,
                          const GNode *__restrict__ nd, const double *__restrict__ cm,
                          const int64_t *__restrict__ ioff, const double *__restrict__ part,
                          int *__restrict__ tint, double *__restrict__ tdbl,
                          WalkNode *__restrict__ wn, double *__restrict__ cell,
                          double *__restrict__ momOH)
{
#pragma clang fp contract(off)
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nn) return;
    const GNode &g = nd[b];
    const int c = g.pre;
    const double *q = cm + 5 * (size_t)b;
    const double *M = part + (size_t)NM * ioff[b];
    const double Bmax = M[31];
    double dOpen;
    if (iOpenType == 1) {
        dOpen = 2 / sqrt(3.0) * Bmax / dCrit;
        if (dOpen < Bmax) dOpen = Bmax;
    } else {
        dOpen = Bmax;
    }
    const double fOpen2 = g.hi >= g.lo ? dOpen * dOpen : 0.0;
    const GNode &rt = nd[g.root];
    const int end = rt.pre + rt.size;
    const int first = g.ch0 >= 0 ? nd[g.ch0].pre : -1;
    const int second = g.ch1 >= 0 ? nd[g.ch1].pre : -1;
    const int next = c + g.size < end ? c + g.size : -1;
    int *ti = tint + 6 * (size_t)c;   // iLower: the first child is c + 1 in preorder
    ti[0] = g.dim;
    ti[1] = g.lo;
    ti[2] = g.hi;
    ti[3] = g.dim >= 0 ? c + 1 : -1;
    ti[4] = next;
    ti[5] = 0;
    double *td = tdbl + 8 * (size_t)c;
    for (int k = 0; k < 5; ++k) td[k] = q[k];
    td[5] = fOpen2;
    td[6] = Bmax;
    td[7] = g.split;
    WalkNode w;
    w.cx = q[2];
    w.cy = q[3];
    w.cz = q[4];
    w.fOpen2 = fOpen2;
    w.fSoft = q[1];
    w.pLower = g.lo;
    w.pUpper = g.hi;
    w.iLower = first;
    w.iNext = next;
    w.iUpper = second;
    w.pad1 = 0;
    wn[c] = w;
    double *r = cell + (size_t)CR_N * c;
    r[CR_M] = q[0];
    for (int d = 0; d < 3; ++d) r[CR_X + d] = q[2 + d];
    r[CR_H] = q[1];
    for (int k = 0; k < 6; ++k) r[CR_QR + k] = M[k];
    const double tr = M[0] + M[1] + M[2];
    r[CR_QT] = M[0] - tr / 3.0;
    r[CR_QT + 1] = M[1] - tr / 3.0;
    r[CR_QT + 2] = M[2] - tr / 3.0;
    r[CR_QT + 3] = M[3];
    r[CR_QT + 4] = M[4];
    r[CR_QT + 5] = M[5];
    if (iOrder >= 3)
        for (int k = 0; k < 25; ++k) momOH[(size_t)OH_N * c + k] = M[6 + k];
}

// Buckets with an active particle: flag by preorder id; bounds of the
// active particles, largest softening, active count (pkd.c:2916-2937,
// walk.c:319-324); the largest bucket, active or not (the fused walk maps a
// bucket's targets, and an opened bucket's particles, onto one wavefront).
__global__ void k_gt_bucket(int nn, const GNode *__restrict__ nd, const double *__restrict__ x,
                            const double *__restrict__ y, const double *__restrict__ z,
                            const double *__restrict__ ph, const uint32_t *__restrict__ pact,
                            int *__restrict__ flag, double *__restrict__ bb8,
                            int *__restrict__ maxb)
{
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nn) return;
    const GNode &g = nd[b];
    const int c = g.pre;
    if (g.dim >= 0 || g.lo > g.hi) {
        flag[c] = 0;
        return;
    }
    double lo[3] = {DBL_MAX, DBL_MAX, DBL_MAX}, hi[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
    int na = 0;
    double fsm = 0.0;
    for (int i = g.lo; i <= g.hi; ++i) {
        if (ph[i] > fsm) fsm = ph[i];
        if (!(pact[i] & 1u)) continue;
        ++na;
        const double r[3] = {x[i], y[i], z[i]};
        for (int d = 0; d < 3; ++d) {
            if (r[d] < lo[d]) lo[d] = r[d];
            if (r[d] > hi[d]) hi[d] = r[d];
        }
    }
    flag[c] = na > 0;
    atomicMax(maxb, g.hi - g.lo + 1);
    double *o = bb8 + 8 * (size_t)c;
    for (int d = 0; d < 3; ++d) {
        o[d] = lo[d];
        o[3 + d] = hi[d];
    }
    o[6] = fsm;
    o[7] = (double)na;
}

__global__ void k_gt_bucket_list(int nn, const int *__restrict__ flag,
                                 const int64_t *__restrict__ pos, const double *__restrict__ bb8,
                                 const int *__restrict__ rootOf, int *__restrict__ bucket,
                                 double *__restrict__ bbox, int *__restrict__ broot)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nn || !flag[c]) return;
    const int k = (int)pos[c];
    bucket[k] = c;
    for (int d = 0; d < 8; ++d) bbox[8 * (size_t)k + d] = bb8[8 * (size_t)c + d];
    broot[k] = rootOf[c];
}

__global__ void k_gt_rootof(int nn, const GNode *__restrict__ nd, int *__restrict__ rootOf)
{
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nn) return;
    rootOf[nd[b].pre] = nd[nd[b].root].pre;
}

}  // namespace

// Waits until the kernels queued on the stream have written *p (pinned,
// tell_host; -1 before).  The stream running dry without it is an error, so
// the wait always ends.
static int host_word(hipStream_t st, const int *p, int *v)
{
    for (unsigned it = 0;; ++it) {
        *v = __atomic_load_n(p, __ATOMIC_ACQUIRE);
        if (*v != -1) return GG_OK;
        if ((it & 1023u) != 1023u) continue;
        const hipError_t e = hipStreamQuery(st);
        if (e == hipErrorNotReady) continue;
        GG_HIP(e);
        *v = __atomic_load_n(p, __ATOMIC_ACQUIRE);
        GG_CHECK(*v != -1, GG_EHIP, "the tree build's device state never arrived");
        return GG_OK;
    }
}

// Particles per tile: enough tiles to fill the chip on a small store, fewer
// of them (each block adds up its cell's tile counts) on a large one.
static int tile_size(int n) { return n < (1 << 19) ? 1024 : (n < (1 << 22) ? 2048 : 4096); }

// One partition pass over the tiles k_gt_ctl listed.
template <int MODE>
static int gt_partition(GravDev &G, hipStream_t st, const TileArgs &A, int grid,
                        unsigned long long *kbox)
{
    hipLaunchKernelGGL(k_gt_count<MODE>, dim3(grid), dim3(256), 0, st, A);
    hipLaunchKernelGGL(k_gt_rank<MODE>, dim3(grid), dim3(256), 0, st, A);
    hipLaunchKernelGGL(k_gt_swap<MODE>, dim3(grid), dim3(256), 0, st, A, kbox);
    GG_HIP(hipGetLastError());
    return GG_OK;
}

int gtree_build(GGPKD pkd, int nSys, const int *sysOff, int nBucket, int iOpenType, double dCrit,
                int iOrder)
{
    GravDev &G = pkd->grav;
    hipStream_t st = pkd->stream;
    const int n = pkd->nLocal;
    G.built = 0;
    // roots: the non-empty systems
    std::vector<int> rlo;
    int maxRoot = 0;
    for (int s = 0; s < nSys; ++s)
        if (sysOff[s + 1] > sysOff[s]) {
            rlo.push_back(sysOff[s]);
            maxRoot = std::max(maxRoot, sysOff[s + 1] - sysOff[s]);
        }
    const int nr = (int)rlo.size();
    for (int k = 0; k < nr; ++k) rlo.push_back(k + 1 < nr ? rlo[k + 1] - 1 : n - 1);
    const size_t n1 = (size_t)std::max(n, 1);
    const size_t cap = 2 * n1 + 2;   // cells at most: every split has two children
    const int ts = tile_size(n);
    const size_t mtile = n1 / ts + n1 / MID + std::max(nr, 1) + 1;   // tiles of a level, at most
    const size_t mbox = std::max<size_t>(2 * (n1 / MID) + 2, nr);    // its cells
    GG_TRY(G.px.reserve(sizeof(double) * n1));
    GG_TRY(G.py.reserve(sizeof(double) * n1));
    GG_TRY(G.pz.reserve(sizeof(double) * n1));
    GG_TRY(G.pm.reserve(sizeof(double) * n1));
    GG_TRY(G.ph.reserve(sizeof(double) * n1));
    GG_TRY(G.pact.reserve(sizeof(uint32_t) * n1));
    GG_TRY(G.perm.reserve(sizeof(int) * n1));
    GG_TRY(G.acc.reserve(sizeof(double) * 5 * n1));
    GG_TRY(G.gposR.reserve(sizeof(int) * n1));
    GG_TRY(G.gnode.reserve(sizeof(GNode) * cap));
    GG_TRY(G.gbox.reserve(sizeof(unsigned long long) * 12 * mbox));
    GG_TRY(G.gtile.reserve(sizeof(int4) * mtile));
    GG_TRY(G.gflag.reserve(sizeof(unsigned long long) * mtile * (ts / 64)));
    GG_TRY(G.gtcnt.reserve(sizeof(int) * 2 * mtile));
    GG_TRY(G.gunit.reserve(sizeof(int) * cap));
    GG_TRY(G.glev.reserve(sizeof(GLevel)));
    GG_TRY(G.gnit.reserve(sizeof(int) * cap));
    GG_TRY(G.gioff.reserve(sizeof(int64_t) * (cap + 1)));
    GG_TRY(G.gchoff.reserve(sizeof(int64_t) * (cap + 1)));
    GG_TRY(G.groot.reserve(sizeof(int) * 2 * std::max(nr, 1)));
    if (!G.hst)
        GG_HIP(hipHostMalloc((void **)&G.hst, sizeof(int) * GravDev::NHST, hipHostMallocDefault));
    GLevel *L = G.glev.as<GLevel>();
    GNode *nd = G.gnode.as<GNode>();
    int nn = 0;
    std::vector<std::pair<int, int>> depths;
    if (nr > 0) {
        const int *rl = G.groot.as<int>(), *rh = rl + nr;
        unsigned long long *box[2];
        box[0] = G.gbox.as<unsigned long long>();
        box[1] = box[0] + 6 * mbox;
        volatile int *hv = G.hst;
        for (int k = 0; k < 8; ++k) hv[k] = -1;
        GG_HIP(hipMemcpyAsync(G.groot.p, rlo.data(), sizeof(int) * 2 * nr, hipMemcpyHostToDevice,
                              st));
        hipLaunchKernelGGL(k_gt_roots, dim3(nblk(nr, 256)), dim3(256), 0, st, nr, rl, rh, nd,
                           box[0], G.gunit.as<int>(), L);
        hipLaunchKernelGGL(k_gt_init, dim3(nblk(n, 256 * INIT_E)), dim3(256), 0, st, n, nr, rl,
                           pkd->f[GG_R].as<double>(), pkd->f[GG_IACTIVE].as<uint32_t>(),
                           G.px.as<double>(), G.py.as<double>(), G.pz.as<double>(),
                           G.perm.as<int>(), box[0], L);
        hipLaunchKernelGGL(k_gt_tell, dim3(1), dim3(1), 0, st, &L->need[1], G.hst + 3);
        GG_HIP(hipGetLastError());
        TileArgs A;
        A.ts = ts;
        A.mask = 0;
        A.L = L;
        A.tiles = G.gtile.as<int4>();
        A.nd = nd;
        A.x = G.px.as<double>();
        A.y = G.py.as<double>();
        A.z = G.pz.as<double>();
        A.src = G.perm.as<int>();
        A.bits = pkd->f[GG_IACTIVE].as<uint32_t>();
        A.flag = G.gflag.as<unsigned long long>();
        A.tcnt = G.gtcnt.as<int>();
        A.tpre = A.tcnt + mtile;
        A.posR = G.gposR.as<int>();
        A.err = &L->err;
        const int grid = (int)mtile;
        auto ctl = [&](int mode, int depth, int *host) {
            hipLaunchKernelGGL(k_gt_ctl, dim3(1), dim3(CTL_T), 0, st, mode, ts, depth, L, nd,
                               box[depth & 1], box[(depth & 1) ^ 1], G.gtile.as<int4>(),
                               G.gunit.as<int>(), host);
        };
        // msrBuildTree's active-type orders (master.c:4262).  A particle with
        // the second order's bit has one of the first's, so where all have it
        // both orders leave everything in place.
        int lack = 0;
        GG_TRY(host_word(st, G.hst + 3, &lack));
        if (lack) {
            ctl(1, 0, G.hst + 4);
            A.mask = GG_TYPE_ACTIVE | GG_TYPE_TREEACTIVE;
            GG_TRY(gt_partition<1>(G, st, A, grid, nullptr));
            A.mask = GG_TYPE_TREEACTIVE;
            GG_TRY(gt_partition<1>(G, st, A, grid, nullptr));
        }
        int nunit = nr, nng = nr, nlev = 1;
        if (maxRoot > MID) {
            // The levels.  The host learns a level's tile count while its
            // partition runs, in time to queue the next level behind it.
            for (int depth = 0;; ++depth) {
                GG_CHECK(depth < DMAX, GG_EUNSUP, "tree deeper than %d levels", DMAX);
                int *h = G.hst + 8 + 4 * (depth & 3);
                for (int k = 0; k < 3; ++k) ((volatile int *)h)[k] = -1;
                ctl(0, depth, h);
                GG_TRY(gt_partition<0>(G, st, A, grid, box[(depth & 1) ^ 1]));
                int nt = 0;
                GG_TRY(host_word(st, h, &nt));
                if (nt == 0) {
                    GG_TRY(host_word(st, h + 1, &nunit));
                    GG_TRY(host_word(st, h + 2, &nng));
                    nlev = depth + 1;
                    break;
                }
            }
        }
        if (nunit > 0)
            hipLaunchKernelGGL(k_gt_mid, dim3(nunit), dim3(MID_T), 0, st, G.gunit.as<int>(), L,
                               nBucket, nd, G.px.as<double>(), G.py.as<double>(),
                               G.pz.as<double>(), G.perm.as<int>(), &L->err);
        GG_HIP(hipGetLastError());
        GLevel hl;
        GG_HIP(hipMemcpyAsync(&hl, L, sizeof hl, hipMemcpyDeviceToHost, st));
        GG_HIP(hipStreamSynchronize(st));
        GG_CHECK(!hl.err, GG_EUNSUP,
                 "a cell split leaves one side empty (positions differ in the last bit only)");
        nng = hl.next;
        // cells of at most LMAX particles: their subtrees in one launch, each
        // in node slots reserved after the cells above them
        GG_TRY(G.gbflag.reserve(sizeof(int) * (size_t)nng));
        hipLaunchKernelGGL(k_gt_lmark, dim3(nblk(nng, 256)), dim3(256), 0, st, nng, nd,
                           G.gbflag.as<int>(), G.gnit.as<int>());
        int64_t nloc = 0, nres = 0;
        GG_TRY(exclusive_scan_i64(st, G.gbflag.as<int>(), G.gchoff.as<int64_t>(), nng, G.scan,
                                  &nloc));
        GG_TRY(exclusive_scan_i64(st, G.gnit.as<int>(), G.gioff.as<int64_t>(), nng, G.scan, &nres));
        GG_CHECK((size_t)nng + (size_t)nres <= cap, GG_EHIP, "tree cell capacity exceeded");
        nn = nng;
        if (nloc > 0) {
            GG_TRY(G.glroot.reserve(sizeof(int) * (size_t)nloc));
            GG_TRY(G.glused.reserve(sizeof(int) * (size_t)nloc));
            GG_TRY(G.glbase.reserve(sizeof(int64_t) * ((size_t)nloc + 1)));
            GG_TRY(G.gscr.reserve(sizeof(GNode) * (size_t)std::max<int64_t>(nres, 1)));
            hipLaunchKernelGGL(k_gt_lcompact, dim3(nblk(nng, 256)), dim3(256), 0, st, nng,
                               G.gbflag.as<int>(), G.gchoff.as<int64_t>(), G.glroot.as<int>());
            hipLaunchKernelGGL(k_gt_local, dim3((unsigned)nloc), dim3(256), 0, st,
                               G.glroot.as<int>(), G.gioff.as<int64_t>(), nBucket, nd,
                               G.gscr.as<GNode>(), G.glused.as<int>(), G.px.as<double>(),
                               G.py.as<double>(), G.pz.as<double>(), G.perm.as<int>(),
                               &L->err);
            GG_HIP(hipGetLastError());
            int64_t nused = 0;
            GG_TRY(exclusive_scan_i64(st, G.glused.as<int>(), G.glbase.as<int64_t>(), (int)nloc,
                                      G.scan, &nused));
            int err = 0;
            GG_HIP(hipMemcpyAsync(&err, &L->err, sizeof(int), hipMemcpyDeviceToHost, st));
            GG_HIP(hipStreamSynchronize(st));
            GG_CHECK(!err, GG_EUNSUP,
                     "a cell split leaves one side empty (positions differ in the last bit only)");
            nn = nng + (int)nused;
            hipLaunchKernelGGL(k_gt_lcopy, dim3((unsigned)nloc), dim3(256), 0, st,
                               G.glroot.as<int>(), G.gioff.as<int64_t>(), G.glused.as<int>(),
                               G.glbase.as<int64_t>(), nng, nd, G.gscr.as<GNode>());
            GG_HIP(hipGetLastError());
        }
        // nodes by depth
        const int ndep = std::max(nlev, hl.maxdep + 1) + LMAX + 1;
        GG_CHECK(ndep <= DMAX, GG_EUNSUP, "tree deeper than %d levels", DMAX);
        GG_TRY(G.gdcnt.reserve(sizeof(int) * 2 * (size_t)ndep));
        GG_TRY(G.gdlist.reserve(sizeof(int) * (size_t)nn));
        GG_HIP(hipMemsetAsync(G.gdcnt.p, 0, sizeof(int) * ndep, st));
        hipLaunchKernelGGL(k_gt_depth_count, dim3(nblk(nn, 256)), dim3(256), 0, st, nn, ndep, nd,
                           G.gdcnt.as<int>());
        std::vector<int> dcnt((size_t)ndep), doff((size_t)ndep + 1, 0);
        GG_HIP(hipMemcpyAsync(dcnt.data(), G.gdcnt.p, sizeof(int) * ndep, hipMemcpyDeviceToHost,
                              st));
        GG_HIP(hipStreamSynchronize(st));
        int nd_used = 0;
        for (int d = 0; d < ndep; ++d) {
            doff[d + 1] = doff[d] + dcnt[d];
            if (dcnt[d]) nd_used = d + 1;
        }
        GG_HIP(hipMemcpyAsync(G.gdcnt.as<int>() + ndep, doff.data(), sizeof(int) * ndep,
                              hipMemcpyHostToDevice, st));
        hipLaunchKernelGGL(k_gt_depth_list, dim3(nblk(nn, 256)), dim3(256), 0, st, nn, ndep, nd,
                           G.gdcnt.as<int>() + ndep, G.gdlist.as<int>());
        depths.clear();
        for (int d = 0; d < nd_used; ++d) depths.push_back({doff[d], dcnt[d]});
        const int *dl = G.gdlist.as<int>();
        // preorder numbering from subtree sizes
        for (int d = (int)depths.size() - 1; d >= 0; --d)
            if (depths[d].second)
                hipLaunchKernelGGL(k_gt_size, dim3(nblk(depths[d].second, 256)), dim3(256), 0, st,
                                   depths[d].second, dl + depths[d].first, nd);
        std::vector<GNode> roots((size_t)nr);
        GG_HIP(hipMemcpyAsync(roots.data(), nd, sizeof(GNode) * nr, hipMemcpyDeviceToHost, st));
        GG_HIP(hipStreamSynchronize(st));
        int pre = 0;
        for (int k = 0; k < nr; ++k) {
            roots[k].pre = pre;
            pre += roots[k].size;
        }
        GG_HIP(hipMemcpyAsync(nd, roots.data(), sizeof(GNode) * nr, hipMemcpyHostToDevice, st));
        for (size_t d = 0; d < depths.size(); ++d)
            if (depths[d].second)
                hipLaunchKernelGGL(k_gt_pre, dim3(nblk(depths[d].second, 256)), dim3(256), 0, st,
                                   depths[d].second, dl + depths[d].first, nd);
        GG_HIP(hipGetLastError());
        GG_HIP(hipStreamSynchronize(st));
    }
    const bool empty = nn == 0;
    const int nNodes = empty ? 1 : nn;
    // storage-order particle fields
    if (n > 0)
        hipLaunchKernelGGL(k_gt_gather, dim3(nblk(n, 256)), dim3(256), 0, st, n,
                           G.perm.as<int>(), pkd->f[GG_MASS].as<double>(),
                           pkd->f[GG_SOFT].as<double>(), pkd->f[GG_IACTIVE].as<uint32_t>(),
                           G.pm.as<double>(), G.ph.as<double>(), G.pact.as<uint32_t>());
    GG_TRY(G.wnode.reserve(sizeof(WalkNode) * nNodes));
    GG_TRY(G.cell.reserve(sizeof(double) * CR_N * nNodes));
    GG_TRY(G.momOH.reserve(sizeof(double) * OH_N * (iOrder >= 3 ? nNodes : 1)));
    GG_TRY(G.tint.reserve(sizeof(int) * 6 * nNodes));
    GG_TRY(G.tdbl.reserve(sizeof(double) * 8 * nNodes));
    GG_TRY(G.gcm.reserve(sizeof(double) * 5 * nNodes));
    int nb = 0;
    if (empty) {   // an empty store: one empty bucket (pkd.c:2684-2712)
        const int ti[6] = {-1, 0, -1, -1, -1, 0};
        const double td[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        WalkNode w{};
        w.pLower = 0;
        w.pUpper = -1;
        w.iLower = w.iNext = w.iUpper = -1;
        GG_HIP(hipMemcpyAsync(G.tint.p, ti, sizeof ti, hipMemcpyHostToDevice, st));
        GG_HIP(hipMemcpyAsync(G.tdbl.p, td, sizeof td, hipMemcpyHostToDevice, st));
        GG_HIP(hipMemcpyAsync(G.wnode.p, &w, sizeof w, hipMemcpyHostToDevice, st));
        GG_HIP(hipStreamSynchronize(st));
    } else {
        // mass, softening, c.o.m.: deepest level first
        for (int d = (int)depths.size() - 1; d >= 0; --d)
            if (depths[d].second)
                hipLaunchKernelGGL(k_gt_mass, dim3(nblk(depths[d].second, 256)), dim3(256), 0, st,
                                   depths[d].second, G.gdlist.as<int>() + depths[d].first, nd,
                                   G.px.as<double>(), G.py.as<double>(), G.pz.as<double>(),
                                   G.pm.as<double>(), G.ph.as<double>(), G.gcm.as<double>());
        // moments: work items of MOM_CH particles per cell
        hipLaunchKernelGGL(k_gt_items, dim3(nblk(nn, 256)), dim3(256), 0, st, 0, nn, MOM_CH, 0,
                           nd, G.gnit.as<int>());
        int64_t nitem = 0;
        GG_TRY(exclusive_scan_i64(st, G.gnit.as<int>(), G.gioff.as<int64_t>(), nn, G.scan, &nitem));
        GG_TRY(G.gpart.reserve(sizeof(double) * NM * std::max<int64_t>(nitem, 1)));
        GG_TRY(G.gicell.reserve(sizeof(int) * std::max<int64_t>(nitem, 1)));
        hipLaunchKernelGGL(k_gt_itemcell, dim3(nblk(nn, 256)), dim3(256), 0, st, nn,
                           G.gioff.as<int64_t>(), G.gicell.as<int>());
        if (nitem > 0) {
            auto mom = iOrder >= 4 ? k_gt_moments<4> : (iOrder >= 3 ? k_gt_moments<3>
                                                                      : k_gt_moments<2>);
            hipLaunchKernelGGL(mom, dim3(nblk(nitem, 4)), dim3(256), 0, st, (int)nitem,
                               G.gicell.as<int>(), G.gioff.as<int64_t>(), nd, G.gcm.as<double>(),
                               G.px.as<double>(), G.py.as<double>(), G.pz.as<double>(),
                               G.pm.as<double>(), G.gpart.as<double>());
            auto small = iOrder >= 4 ? k_gt_moments_small<4>
                                     : (iOrder >= 3 ? k_gt_moments_small<3> : k_gt_moments_small<2>);
            hipLaunchKernelGGL(small, dim3(nblk(nitem, 256)), dim3(256), 0, st, (int)nitem,
                               G.gicell.as<int>(), nd, G.gcm.as<double>(), G.px.as<double>(),
                               G.py.as<double>(), G.pz.as<double>(), G.pm.as<double>(),
                               G.gpart.as<double>());
        }
        const int nv = iOrder >= 4 ? 31 : (iOrder >= 3 ? 16 : 6);
        hipLaunchKernelGGL(k_gt_combine, dim3(nblk(nn, 4)), dim3(256), 0, st, nn, nv,
                           G.gioff.as<int64_t>(), G.gpart.as<double>());
        hipLaunchKernelGGL(k_gt_emit, dim3(nblk(nn, 256)), dim3(256), 0, st, nn, iOrder,
                           iOpenType, dCrit, nd, G.gcm.as<double>(), G.gioff.as<int64_t>(),
                           G.gpart.as<double>(), G.tint.as<int>(), G.tdbl.as<double>(),
                           G.wnode.as<WalkNode>(), G.cell.as<double>(), G.momOH.as<double>());
        // active buckets in preorder
        GG_TRY(G.gbflag.reserve(sizeof(int) * nn));
        GG_TRY(G.gbb8.reserve(sizeof(double) * 8 * nn));
        GG_TRY(G.grootof.reserve(sizeof(int) * nn));
        hipLaunchKernelGGL(k_gt_bucket, dim3(nblk(nn, 256)), dim3(256), 0, st, nn, nd,
                           G.px.as<double>(), G.py.as<double>(), G.pz.as<double>(),
                           G.ph.as<double>(), G.pact.as<uint32_t>(), G.gbflag.as<int>(),
                           G.gbb8.as<double>(), &L->maxb);
        hipLaunchKernelGGL(k_gt_rootof, dim3(nblk(nn, 256)), dim3(256), 0, st, nn, nd,
                           G.grootof.as<int>());
        int64_t nb64 = 0;
        GG_TRY(exclusive_scan_i64(st, G.gbflag.as<int>(), G.gchoff.as<int64_t>(), nn, G.scan,
                                  &nb64));
        nb = (int)nb64;
        int maxb = 0;
        GG_HIP(hipMemcpyAsync(&maxb, &L->maxb, sizeof(int), hipMemcpyDeviceToHost,
                              st));
        GG_HIP(hipStreamSynchronize(st));
        G.maxBucket = maxb;     // > 64 only for cells of coincident particles (pkd.c:2489)
        GG_TRY(G.bucket.reserve(sizeof(int) * std::max(nb, 1)));
        GG_TRY(G.broot.reserve(sizeof(int) * std::max(nb, 1)));
        GG_TRY(G.bbox.reserve(sizeof(double) * 8 * std::max(nb, 1)));
        hipLaunchKernelGGL(k_gt_bucket_list, dim3(nblk(nn, 256)), dim3(256), 0, st, nn,
                           G.gbflag.as<int>(), G.gchoff.as<int64_t>(), G.gbb8.as<double>(),
                           G.grootof.as<int>(), G.bucket.as<int>(), G.bbox.as<double>(),
                           G.broot.as<int>());
        GG_HIP(hipGetLastError());
    }
    GG_TRY(G.cnt.reserve(sizeof(int) * 3 * std::max(nb, 1)));
    GG_TRY(G.off.reserve(sizeof(int64_t) * (3 * (size_t)std::max(nb, 1) + 1)));
    GG_HIP(hipStreamSynchronize(st));
    G.nb = nb;
    G.n = n;
    G.nNodes = nNodes;
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
