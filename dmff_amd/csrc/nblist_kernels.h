// Neighbour lists.
//
// Semantics (dmff/common/nblist.py:27-55): the pair set {i < j : minimum-image
// distance < rc}, minimum image by fractional rounding (spatial.py:13-32).
// Internally every site keeps a FULL list (both directions) in a padded row of
// `cap` words, word = j | nbond << 28, so the pair kernels gather without atomics.
//
// Bit-exactness: the squared distance is formed with unfused, single-rounded
// operations in a fixed order (see d2_exact) so the pair set equals the FP64
// brute force of the oracle bit for bit.
#pragma once
#include "admp_common.h"

namespace admp {

// box rows and inverse held in registers by the neighbour search
struct BoxMat {
    double B[9], Binv[9];
};

// d2_exact for a box with zero off-diagonal entries (B and Binv): the terms
// d_k * 0 of the general form add exact zeros, so the value is the same bit for
// bit (a zero's sign aside, which the square removes)
template <class BX>
__device__ __forceinline__ double d2_ortho(const BX& b, double dx, double dy, double dz) {
#pragma clang fp contract(off)
    const double t0 = dx * b.Binv[0], t1 = dy * b.Binv[4], t2 = dz * b.Binv[8];
    const double s0 = t0 - floor(t0 + 0.5), s1 = t1 - floor(t1 + 0.5), s2 = t2 - floor(t2 + 0.5);
    const double d0 = s0 * b.B[0], d1 = s1 * b.B[4], d2 = s2 * b.B[8];
    double r = d0 * d0;
    r = r + d1 * d1;
    r = r + d2 * d2;
    return r;
}

template <class BX>
__device__ __forceinline__ double d2_exact(const BX& b, double dx, double dy, double dz) {
#pragma clang fp contract(off)
    double s[3], d[3];
    for (int c = 0; c < 3; ++c) {
        double t = dx * b.Binv[0 * 3 + c];
        t = t + dy * b.Binv[1 * 3 + c];
        t = t + dz * b.Binv[2 * 3 + c];
        s[c] = t - floor(t + 0.5);
    }
    for (int c = 0; c < 3; ++c) {
        double t = s[0] * b.B[0 * 3 + c];
        t = t + s[1] * b.B[1 * 3 + c];
        t = t + s[2] * b.B[2 * 3 + c];
        d[c] = t;
    }
    double r = d[0] * d[0];
    r = r + d[1] * d[1];
    r = r + d[2] * d[2];
    return r;
}

struct CellGrid {
    int nc[3];
    int ncell;
};

// Validity of a cell grid taken over from an earlier build: every frame's cell
// slabs must stay at least rc wide (nc[d] <= floor(width_d / rc), width_d =
// 1 / |column d of Binv|, the rule the host applies when it sizes the grid).
// flag[f] = 1 where frame f's box needs another grid.
__global__ void k_cell_grid_check(int F, const BoxInfo* __restrict__ boxes, double rc, CellGrid cg,
                                  int* __restrict__ flag) {
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= F) return;
    const double* Bi = boxes[f].Binv;
    int bad = 0;
    for (int d = 0; d < 3; ++d) {
        const double n2 = Bi[d] * Bi[d] + Bi[3 + d] * Bi[3 + d] + Bi[6 + d] * Bi[6 + d];
        const double width = 1.0 / sqrt(n2);
        const double n = floor(width / rc);
        if (!(n >= (double)cg.nc[d])) bad = 1;
    }
    flag[f] = bad;
}

// atomicAdd(&ctr[key], 1) for every active lane of the wavefront with one atomic
// per distinct key (consecutive atoms mostly share a cell, so same-address
// atomics would serialise); returns the lane's old value: the key's base plus
// its rank among the lanes with that key.  Blocks are whole wavefronts.
__device__ __forceinline__ int wave_agg_inc(int* ctr, int key) {
    const int lane = threadIdx.x & 63;
    unsigned long long todo = __ballot(1);
    int res = 0;
    while (todo) {
        const int leader = __ffsll((long long)todo) - 1;
        const int lkey = __shfl(key, leader);
        const unsigned long long same = __ballot(key == lkey) & todo;
        int base = 0;
        if (lane == leader) base = atomicAdd(&ctr[lkey], __popcll(same));
        base = __shfl(base, leader);
        if ((same >> lane) & 1ull) res = base + __popcll(same & ((1ull << lane) - 1ull));
        todo &= ~same;
    }
    return res;
}

__global__ void k_cell_assign(int N, const double4* __restrict__ pos, const BoxInfo* __restrict__ boxes, CellGrid cg,
                              int* __restrict__ cell, int* __restrict__ ccount) {
    const int f = blockIdx.y;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const BoxInfo& b = boxes[f];
    const double4 p = pos[(size_t)f * N + i];
    int c[3];
    for (int d = 0; d < 3; ++d) {
        double s = p.x * b.Binv[0 * 3 + d] + p.y * b.Binv[1 * 3 + d] + p.z * b.Binv[2 * 3 + d];
        s -= floor(s);
        int k = (int)(s * cg.nc[d]);
        if (k >= cg.nc[d]) k = cg.nc[d] - 1;
        if (k < 0) k = 0;
        c[d] = k;
    }
    const int id = (c[0] * cg.nc[1] + c[1]) * cg.nc[2] + c[2];
    cell[(size_t)f * N + i] = id;
    wave_agg_inc(ccount + (size_t)f * cg.ncell, id);
}

// exclusive scan of ncell counts per frame (single block per frame)
// ---------------------------------------------------------------------------
// Exclusive scan of F rows of n ints: out row f has n + 1 entries, the last one
// the row total.  Three launches: 1024-element tiles scanned in registers and
// LDS (k_scan_tiles), the tile totals scanned per row (k_scan_top), tile offsets
// added back (k_scan_add).
// ---------------------------------------------------------------------------
constexpr int SCAN_TILE = 1024;

__device__ __forceinline__ int wave_incl_scan(int v) {
    const int lane = threadIdx.x & 63;
    for (int d = 1; d < 64; d <<= 1) {
        const int t = __shfl_up(v, d, 64);
        if (lane >= d) v += t;
    }
    return v;
}

// block of 256 threads; returns the exclusive prefix of v within the block, total in *tot
__device__ __forceinline__ int block_excl_scan256(int v, int* ws, int* tot) {
    const int incl = wave_incl_scan(v);
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 63) ws[w] = incl;
    __syncthreads();
    int woff = 0;
    for (int k = 0; k < w; ++k) woff += ws[k];
    *tot = ws[0] + ws[1] + ws[2] + ws[3];
    __syncthreads();
    return woff + incl - v;
}

__global__ void __launch_bounds__(256) k_scan_tiles(int n, const int* __restrict__ in, int* __restrict__ out,
                                                    int* __restrict__ tsum, int ntile) {
    __shared__ int ws[4];
    const int f = blockIdx.y, t = blockIdx.x;
    const int* a = in + (size_t)f * n;
    int* o = out + (size_t)f * (n + 1);
    const int base = t * SCAN_TILE + threadIdx.x * 4;
    int v[4], s = 0;
    for (int k = 0; k < 4; ++k) {
        v[k] = base + k < n ? a[base + k] : 0;
        s += v[k];
    }
    int tot;
    int ex = block_excl_scan256(s, ws, &tot);
    for (int k = 0; k < 4; ++k) {
        if (base + k < n) o[base + k] = ex;
        ex += v[k];
    }
    if (threadIdx.x == 0) tsum[(size_t)f * ntile + t] = tot;
}

// one block of 256 per row: exclusive scan of the tile totals in place, row total to out[n]
__global__ void __launch_bounds__(256) k_scan_top(int n, int ntile, int* __restrict__ tsum, int* __restrict__ out) {
    __shared__ int ws[4];
    const int f = blockIdx.x;
    int* ts = tsum + (size_t)f * ntile;
    int carry = 0;
    for (int b = 0; b < ntile; b += 256) {
        const int k = b + threadIdx.x;
        const int v = k < ntile ? ts[k] : 0;
        int tot;
        const int ex = block_excl_scan256(v, ws, &tot);
        if (k < ntile) ts[k] = carry + ex;
        carry += tot;
    }
    if (threadIdx.x == 0) out[(size_t)f * (n + 1) + n] = carry;
}

__global__ void __launch_bounds__(256) k_scan_add(int n, const int* __restrict__ tsum, int* __restrict__ out,
                                                  int ntile) {
    const int f = blockIdx.y, t = blockIdx.x;
    if (t == 0) return;
    const int off = tsum[(size_t)f * ntile + t];
    int* o = out + (size_t)f * (n + 1);
    for (int k = threadIdx.x; k < SCAN_TILE; k += 256) {
        const int idx = t * SCAN_TILE + k;
        if (idx < n) o[idx] += off;
    }
}

// one block of 1024 per row for short rows (one launch instead of the three
// above): tiles of 4096 scanned in turn with a running carry
__global__ void __launch_bounds__(1024) k_scan_small(int n, const int* __restrict__ in, int* __restrict__ out) {
    __shared__ int ws[16];
    const int f = blockIdx.x;
    const int* a = in + (size_t)f * n;
    int* o = out + (size_t)f * (n + 1);
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    int carry = 0;
    for (int base0 = 0; base0 < n; base0 += 4 * 1024) {
        const int base = base0 + threadIdx.x * 4;
        int v[4], sum = 0;
        for (int k = 0; k < 4; ++k) {
            v[k] = base + k < n ? a[base + k] : 0;
            sum += v[k];
        }
        const int incl = wave_incl_scan(sum);
        if (lane == 63) ws[w] = incl;
        __syncthreads();
        int woff = 0, tot = 0;
        for (int k = 0; k < 16; ++k) {
            if (k < w) woff += ws[k];
            tot += ws[k];
        }
        __syncthreads();
        int ex = carry + woff + incl - sum;
        for (int k = 0; k < 4; ++k) {
            if (base + k < n) o[base + k] = ex;
            ex += v[k];
        }
        carry += tot;
    }
    if (threadIdx.x == 0) o[n] = carry;
}

// agg: one atomic per distinct cell per wavefront (for cells holding many
// consecutive atoms); 0: one per atom (many cells, few atoms each)
__global__ void k_cell_fill(int N, int ncell, const int* __restrict__ cell, const int* __restrict__ cstart,
                            int* __restrict__ cfill, int* __restrict__ catoms, int agg) {
    const int f = blockIdx.y;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const int id = cell[(size_t)f * N + i];
    const int slot = agg ? wave_agg_inc(cfill + (size_t)f * ncell, id) : atomicAdd(&cfill[(size_t)f * ncell + id], 1);
    catoms[(size_t)f * N + cstart[(size_t)f * (ncell + 1) + id] + slot] = i;
}

// deterministic order inside each cell: ascending atom index
__global__ void k_cell_sort(int ncell, int N, const int* __restrict__ cstart, int* __restrict__ catoms) {
    const int f = blockIdx.y;
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= ncell) return;
    int* a = catoms + (size_t)f * N;
    const int lo = cstart[(size_t)f * (ncell + 1) + c], hi = cstart[(size_t)f * (ncell + 1) + c + 1];
    for (int k = lo + 1; k < hi; ++k) {
        int v = a[k], m = k - 1;
        while (m >= lo && a[m] > v) { a[m + 1] = a[m]; --m; }
        a[m + 1] = v;
    }
}

// one block of 256 per cell: rank sort of the cell's (distinct) atom indices in LDS.
// Cells larger than the LDS buffer fall back to an insertion sort by one thread.
constexpr int CELL_SORT_CAP = 2048;

__global__ void __launch_bounds__(256) k_cell_sort_block(int ncell, int N, const int* __restrict__ cstart,
                                                         int* __restrict__ catoms) {
    __shared__ int buf[CELL_SORT_CAP];
    const int f = blockIdx.y, c = blockIdx.x;
    int* a = catoms + (size_t)f * N;
    const int lo = cstart[(size_t)f * (ncell + 1) + c], hi = cstart[(size_t)f * (ncell + 1) + c + 1];
    const int cnt = hi - lo;
    if (cnt <= 1) return;
    if (cnt > CELL_SORT_CAP) {
        if (threadIdx.x == 0)
            for (int k = lo + 1; k < hi; ++k) {
                int v = a[k], m = k - 1;
                while (m >= lo && a[m] > v) { a[m + 1] = a[m]; --m; }
                a[m + 1] = v;
            }
        return;
    }
    for (int k = threadIdx.x; k < cnt; k += 256) buf[k] = a[lo + k];
    __syncthreads();
    for (int k = threadIdx.x; k < cnt; k += 256) {
        const int v = buf[k];
        int r = 0;
        for (int m = 0; m < cnt; ++m) r += buf[m] < v;
        a[lo + r] = v;
    }
}

__device__ __forceinline__ int lookup_nbond(int i, int j, const int* __restrict__ xoff, const int* __restrict__ xent) {
    for (int e = xoff[i]; e < xoff[i + 1]; ++e) {
        const int w = xent[e];
        if ((w & NB_MASK) == j) return w >> NB_SHIFT;
    }
    return 0;
}

// positions in cell order, the atom index in .w (exact as a double), so that a
// candidate of the neighbour search is one load
__global__ void k_cell_pos(int N, const double4* __restrict__ pos, const int* __restrict__ catoms,
                           double4* __restrict__ spos) {
    const int f = blockIdx.y;
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= N) return;
    const size_t fo = (size_t)f * N;
    const int j = catoms[fo + k];
    double4 p = pos[fo + j];
    p.w = (double)j;
    spos[fo + k] = p;
}

// one wavefront (64 lanes) per site; blockDim = 256 -> 4 sites per block.  The
// ranges of the (up to 27) neighbour cells are loaded once, one per lane, and
// broadcast; candidates come from the cell-ordered positions.
__global__ void __launch_bounds__(256)
k_nbr_build(int N, int cap, const double4* __restrict__ pos, const BoxInfo* __restrict__ boxes, CellGrid cg,
            double rc2, const int* __restrict__ cell, const int* __restrict__ cstart,
            const double4* __restrict__ spos, const int* __restrict__ xoff, const int* __restrict__ xent,
            int* __restrict__ nbr, int* __restrict__ ncnt, int* __restrict__ nhalf, int* __restrict__ maxcnt) {
    const int f = blockIdx.y;
    const int lane = threadIdx.x & 63;
    const int i = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (i >= N) return;
    const BoxInfo& b = boxes[f];
    const size_t fo = (size_t)f * N;
    const double4 pi_ = pos[fo + i];
    const int ci = cell[fo + i];
    int cc[3];
    cc[2] = ci % cg.nc[2];
    cc[1] = (ci / cg.nc[2]) % cg.nc[1];
    cc[0] = ci / (cg.nc[1] * cg.nc[2]);
    // distinct neighbour cell coordinates per dimension
    int lst[3][3], nl[3];
    for (int d = 0; d < 3; ++d) {
        const int n = cg.nc[d];
        if (n >= 3) {
            lst[d][0] = (cc[d] + n - 1) % n; lst[d][1] = cc[d]; lst[d][2] = (cc[d] + 1) % n; nl[d] = 3;
        } else {
            for (int k = 0; k < n; ++k) lst[d][k] = k;
            nl[d] = n;
        }
    }
    int count = 0, half = 0;
    int* row = nbr + (fo + i) * (size_t)cap;
    const int* cs = cstart + (size_t)f * (cg.ncell + 1);
    const double4* sp = spos + fo;
    BoxMat bm;
#pragma unroll
    for (int q = 0; q < 9; ++q) { bm.B[q] = b.B[q]; bm.Binv[q] = b.Binv[q]; }
    bool ortho = true;
#pragma unroll
    for (int q = 0; q < 9; ++q)
        if (q % 4 != 0) ortho = ortho && bm.B[q] == 0.0 && bm.Binv[q] == 0.0;
    // atom i's exclusion words (the same for the whole wavefront): lane e holds entry e
    const int x0 = xoff[i], nx = xoff[i + 1] - x0;
    const int myx = lane < nx ? xent[x0 + lane] : 0;
    // lane l < ncand holds the range of neighbour cell l (a0-major, a2 fastest)
    const int ncand = nl[0] * nl[1] * nl[2];
    int mylo = 0, myhi = 0;
    if (lane < ncand) {
        const int a2 = lane % nl[2], a1 = (lane / nl[2]) % nl[1], a0 = lane / (nl[2] * nl[1]);
        const int cid = (lst[0][a0] * cg.nc[1] + lst[1][a1]) * cg.nc[2] + lst[2][a2];
        // A cell further than rc from the site has no neighbours: 17 of 27 cells remain on
        // average where cells are little wider than rc (98,304 sites at rc 10: 840 -> 662 us; 64
        // frames of 12,288 at rc 8: 3.49 -> 3.11 ms; one such frame, latency bound: 67 -> 65 us).
        // The distance to the cell's slab along each axis is a lower bound; in an orthogonal
        // box the three add up.  (The far side of a cell, reached the other way round, is at
        // least a cell's width off.)  1e-6 A covers the rounding of cell membership.
        const int at[3] = {lst[0][a0], lst[1][a1], lst[2][a2]};
        double sum = 0, most = 0;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const double* Bi = bm.Binv + d;
            double sd = pi_.x * Bi[0] + pi_.y * Bi[3] + pi_.z * Bi[6];
            sd = (sd - floor(sd)) * cg.nc[d] - cc[d];                       // place in the own cell, 0..1
            // (k_cell_assign's rounding may have found a site on the periodic face on the other side)
            if (sd > 1.5) sd -= cg.nc[d];
            if (sd < -0.5) sd += cg.nc[d];
            const int n = cg.nc[d], off = (at[d] - cc[d] + n) % n;
            const double up = off == 1 ? 1.0 - sd : 1e30, down = off == n - 1 ? sd : 1e30;
            const double w = 1.0 / (n * sqrt(Bi[0] * Bi[0] + Bi[3] * Bi[3] + Bi[6] * Bi[6]));   // slab width
            const double g = off == 0 ? 0.0 : fmax(0.0, fmin(up, down) * w - 1e-6);
            sum += g * g;
            most = fmax(most, g * g);
        }
        if ((ortho ? sum : most) < rc2) {
            mylo = cs[cid];
            myhi = cs[cid + 1];
        }
    }
    for (int q = 0; q < ncand; ++q) {
        const int lo = __shfl(mylo, q, 64), hi = __shfl(myhi, q, 64);
        for (int base = lo; base < hi; base += 64) {
            const int k = base + lane;
            int j = -1;
            bool hit = false;
            if (k < hi) {
                const double4 pj = sp[k];
                j = (int)pj.w;
                const double d2 = ortho ? d2_ortho(bm, pi_.x - pj.x, pi_.y - pj.y, pi_.z - pj.z)
                                        : d2_exact(bm, pi_.x - pj.x, pi_.y - pj.y, pi_.z - pj.z);
                hit = j != i && d2 < rc2;
            }
            const unsigned long long m = __ballot(hit);
            // nbond of (i, j) from i's exclusion words, read lane by lane by the
            // whole wavefront (nx is the same in every lane)
            int nbd = 0;
            if (nx <= 64) {
                bool found = false;
                for (int e = 0; e < nx; ++e) {
                    const int w = __builtin_amdgcn_readlane(myx, e);
                    if (!found && (w & NB_MASK) == j) { nbd = w >> NB_SHIFT; found = true; }
                }
            } else if (hit) {
                nbd = lookup_nbond(i, j, xoff, xent);
            }
            if (hit) {
                const int pre = __popcll(m & ((1ull << lane) - 1ull));
                const int slot = count + pre;
                if (slot < cap) row[slot] = j | (nbd << NB_SHIFT);
            }
            const unsigned long long mh = __ballot(hit && j > i);
            count += __popcll(m);
            half += __popcll(mh);
        }
    }
    if (lane == 0) {
        ncnt[fo + i] = count < cap ? count : cap;
        nhalf[fo + i] = half;
        // only overflowing rows report (the host needs the longest row only to
        // grow the capacity): no same-address atomic per site in the common case
        if (count > cap) atomicMax(maxcnt, count);
    }
}

// reference-format output: rows (i, j, nbond) for j > i, row offsets from an
// exclusive scan of nhalf (one wavefront per site: one thread per site walked a row in
// dependent steps and wrote single words: 65 us for 29,000 pairs of 648 sites against 3.6)
__global__ void __launch_bounds__(256)
k_pairs_out(int N, int cap, int f, const int* __restrict__ nbr, const int* __restrict__ ncnt,
            const int* __restrict__ off, int* __restrict__ out) {
    const int i = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (i >= N) return;
    const size_t fo = (size_t)f * N;
    const int* row = nbr + (fo + i) * (size_t)cap;
    const int n = ncnt[fo + i];
    int o = off[i];
    for (int k0 = 0; k0 < n; k0 += 64) {
        const int w = k0 + lane < n ? row[k0 + lane] : 0;
        const int j = w & NB_MASK;
        const bool keep = k0 + lane < n && j > i;
        const unsigned long long m = __ballot(keep);
        if (keep) {
            int* q = out + (size_t)(o + __popcll(m & ((1ull << lane) - 1ull))) * 3;
            q[0] = i;
            q[1] = j;
            q[2] = w >> NB_SHIFT;
        }
        o += __popcll(m);
    }
}

// user pairs (reference format) -> full lists.  A list sorted by its first site gives a
// wavefront long runs of one i, whose same-address atomics bound these kernels; a run adds
// once, by its first lane, and its lanes take consecutive places (an unsorted list has runs
// of one).  Count and fill, 29,000 pairs of 648 sites: 67 and 67 us with an atomic per row,
// 14 and 14 with one per run.
__device__ __forceinline__ int run_inc(int* ctr, int i, bool live) {
    const int lane = threadIdx.x & 63;
    const int key = live ? i : -1;
    const int prev = __shfl_up(key, 1, 64);
    const unsigned long long heads = __ballot(lane == 0 || prev != key);
    const unsigned long long below = heads & (~0ull >> (63 - lane));         // heads up to this lane
    const int head = 63 - __clzll((long long)below);
    const unsigned long long above = head == 63 ? 0 : heads >> (head + 1);   // the next run's head
    const int len = above ? __ffsll((long long)above) : 64 - head;
    int base = 0;
    if (live && lane == head) base = atomicAdd(ctr + i, len);
    return __shfl(base, head, 64) + (lane - head);
}

template <class I>
__global__ void __launch_bounds__(256)
k_upairs_count(int64_t np, int N, const I* __restrict__ pairs, int* __restrict__ cnt, int* __restrict__ bad) {
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t i = 0, j = 0;
    if (r < np) { i = (int64_t)pairs[r * 3]; j = (int64_t)pairs[r * 3 + 1]; }
    bool live = i < j;  // padding / i >= j rows vanish (dmff/utils.py:65-84)
    if (live && (i < 0 || j >= N)) { atomicExch(bad, 1); live = false; }
    run_inc(cnt, (int)i, live);
    if (live) atomicAdd(&cnt[j], 1);
}

template <class I>
__global__ void __launch_bounds__(256)
k_upairs_fill(int64_t np, int N, int cap, const I* __restrict__ pairs, int* __restrict__ fill,
              int* __restrict__ nbr) {
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t i = 0, j = 0;
    if (r < np) { i = (int64_t)pairs[r * 3]; j = (int64_t)pairs[r * 3 + 1]; }
    const bool live = i < j && i >= 0 && j < N;
    // (on its way before the run's place is waited for: shuffled lists of 332,000 and 1,361,000
    // pairs 230 and 439 us per call with the two in turn, 221 and 421 so; an atomic per row 208
    // and 424, but 320 and 710 for sorted lists, 122 and 213 here)
    const int sj = live ? atomicAdd(&fill[j], 1) : 0;
    const int si = run_inc(fill, (int)i, live);
    if (!live) return;
    int nb = (int)pairs[r * 3 + 2];
    if (nb < 0) nb = 0;
    if (nb > 7) nb = 7;
    if (si < cap) nbr[(size_t)i * cap + si] = (int)j | (nb << NB_SHIFT);
    if (sj < cap) nbr[(size_t)j * cap + sj] = (int)i | (nb << NB_SHIFT);
}

// per-site bitonic sort of the row (unsigned word order) for a deterministic
// summation order; one block per site, row padded to a power of two in LDS
__global__ void k_row_sort(int N, int cap, int* __restrict__ nbr, const int* __restrict__ ncnt) {
    extern __shared__ unsigned int srt[];
    const int i = blockIdx.x;
    const int n = ncnt[i];
    int P = 1;
    while (P < n) P <<= 1;
    unsigned int* row = reinterpret_cast<unsigned int*>(nbr + (size_t)i * cap);
    for (int k = threadIdx.x; k < P; k += blockDim.x) srt[k] = k < n ? row[k] : 0xFFFFFFFFu;
    __syncthreads();
    for (int size = 2; size <= P; size <<= 1)
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int k = threadIdx.x; k < P; k += blockDim.x) {
                const int l = k ^ stride;
                if (l > k) {
                    const bool up = (k & size) == 0;
                    const unsigned int a = srt[k], c = srt[l];
                    if ((a > c) == up) { srt[k] = c; srt[l] = a; }
                }
            }
            __syncthreads();
        }
    for (int k = threadIdx.x; k < n; k += blockDim.x) row[k] = srt[k];
}

}  // namespace admp
