// Reciprocal space of the FP64 products on the matrix cores: the 1-D discrete
// Fourier transforms are dense matrix products (v_mfma_f64_16x16x4), the spread
// is a matrix product over sites, and the passes are fused so that a product takes
// three launches: spread + z transform, (x, y) plane, inverse z transform + gather.
//
// Dense transforms.  A line of K points is folded into its even and odd parts,
// e_n = x_n + x_{K-n} and o_n = x_n - x_{K-n} (n <= K / 2), so that
//   C_k = sum_n e_n cos(2 pi k n / K),   S_k = sum_n o_n sin(2 pi k n / K)
// give frequencies k and K - k at once: H = K / 2 + 1 rows and columns, a quarter of
// the products of the full matrix.  Up to about 64 points this costs less than the LDS
// passes, barriers and index arithmetic of a mixed-radix transform, up to about 90 as
// much, and it does not depend on the factors of K: the radix passes of
// recip2_kernels.h fall back to a direct sum by one thread per line where K is prime.
// Large grids of small factors stay there (radix_faster in admp_api.hip), and so do the
// FP32 passes of the mixed path.
//
// Measured per product, radix passes -> these: 12,288 sites on 50 x 50 x 50 (15 of them per
// solve): spread 14.6 + r2c 7.5 -> 15.6, plane 18.0 -> 21.6, c2r 6.5 + gather 8.1 -> 12.0 us;
// 1,536 sites on 25 x 25 x 25: 15.6 -> 9.4, 13.9 -> 10.4, 9.9 -> 7.7 us; 64 frames of 12,288
// sites: level (1.85 ms).  On axes that are prime or hold a prime factor above 13 the radix
// passes sum directly: for 2,970 sites r2c 74, plane 112 and c2r 70 us of each of eleven
// sweeps, and the evaluation falls from 4.7 to 1.8 ms (with the sweeps' test on the host).
//
// Fragments of v_mfma_f64_16x16x4 (lane l of the wavefront): A holds row l % 16,
// column l / 16 of a 16 x 4 block, B row l / 16, column l % 16 of a 4 x 16 block, and
// register r of the result holds row 4 r + l / 16, column l % 16.
#pragma once
#include "admp_common.h"
#include "recip_kernels.h"
#include "recip2_kernels.h"

namespace admp {

typedef double d4 __attribute__((vector_size(32)));

__device__ __forceinline__ d4 mma4(double a, double b, d4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// LDS written by some lanes of a wavefront and read by others of the same one: the
// unit keeps a wavefront's accesses in order, so only the compiler has to
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// A launch of few workgroups issues its first loads before it looks at its frame's
// converged flag, which saves a load's latency; in one of several rounds of workgroups the
// others cover that, and a converged frame's workgroups leave before they load anything
// (64 converged frames of 169 tiles: 170 us against 7 for the gather).
__device__ __forceinline__ bool early_exit() { return gridDim.x * gridDim.y > 4 * N_CU; }

// largest axis of the dense transforms: the products grow as K^2 per line
constexpr int MM_KMAX = 128;
// largest (x, y) plane held in LDS by the plane pass (one workgroup per CU)
constexpr size_t MM_PLANE_LDS = 152 * 1024;
// row tiles of the transforms' template instances
constexpr int MM_NT = (MM_KMAX / 2 + 1 + 15) / 16;

__host__ __device__ inline int mm_tiles(int K) { return (K / 2 + 1 + 15) / 16; }
__host__ __device__ inline int mm_steps(int K) { return (K / 2 + 1 + 3) / 4; }

// One lane's walk along a row of the transform matrix, four columns a step: entry
// (row, col) is w^(row col) of the axis's K twiddles w^t = (cos, -sin)(2 pi t / K),
// staged in LDS; the byte offset of the exponent is kept reduced modulo K.
struct TwWalk {
    unsigned off, step, lim;
    const unsigned char* tw;
    __device__ __forceinline__ void start(const Cplx<double>* t, int K, int row, int col) {
        tw = reinterpret_cast<const unsigned char*>(t);
        const float inv = 1.0f / (float)K;
        const int a = row * col, b = 4 * row;
        off = 16u * (unsigned)(a - qdiv(a, K, inv) * K);
        step = 16u * (unsigned)(b - qdiv(b, K, inv) * K);
        lim = 16u * (unsigned)K;
    }
    __device__ __forceinline__ Cplx<double> next() {
        const Cplx<double> v = *reinterpret_cast<const Cplx<double>*>(tw + off);
        off += step;
        off = min(off, off - lim);   // unsigned: the difference wraps round when it is negative
        return v;
    }
};

// a double at a byte offset
__device__ __forceinline__ double at8(const void* p, int byte) {
    return *reinterpret_cast<const double*>(reinterpret_cast<const unsigned char*>(p) + byte);
}
__device__ __forceinline__ int clamp56(int v) { return min(max(v, 0), 56); }
// a value moved between lanes by a DPP control (every lane has a source)
template <int CTRL> __device__ __forceinline__ double dpp_move(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xF, 0xF, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// the neighbouring lane's value (lanes 2 i and 2 i + 1 exchange)
__device__ __forceinline__ double swap_pair(double v) { return dpp_move<0xB1>(v); }

// ---------------------------------------------------------------------------
// Spread + real-to-complex z transform.
//
// One workgroup holds the 16 (x, y) columns of a 4 x 4 tile over all z.  A
// z segment of up to 16 points is one 16 x 16 result block: column factors of the
// candidate sites (16 x k) times their z factors (k x 16), k running over (site,
// term).  With the 1-D spline tables v (value), a, b (derivatives) the terms are
//   C0 vz + C1 az + C2 bz,
//   C0 = (q vx + mx ax + Txx bx) vy + vx (my ay + Tyy by) + ax (2 Txy ay),
//   C1 = (mz vx + 2 Txz ax) vy + vx (2 Tyz ay),  C2 = Tzz vx vy;
// charges have one term (four sites per product), dipoles two (C0, C1: two sites),
// quadrupoles three (one site).  A wavefront stages the tables of its next sites in
// its own part of LDS, each with a zero before and after so that points outside a
// support read a zero instead of testing for it.  `wpt` wavefronts share a segment's
// candidates; their partial blocks are added in a fixed order by the transform that
// reads them, so results are bitwise reproducible.
// ---------------------------------------------------------------------------
constexpr int MM_TX = 4, MM_TY = 4;    // columns of a tile
constexpr int MM_TZ = 16;              // most z points of a segment
constexpr int MM_TILE_COPIES = 48;     // most (tile, segment) lists a site appears in: 4 x 4 x 3
__host__ __device__ inline int mm_nseg(int K2) { return (K2 + MM_TZ - 1) / MM_TZ; }
__host__ __device__ inline int mm_seglen(int K2) { return (K2 + mm_nseg(K2) - 1) / mm_nseg(K2); }

template <int LM> struct SpreadShape {
    static constexpr int SPM = LM == 0 ? 4 : LM == 1 ? 2 : 1;     // sites per matrix product
    static constexpr int NST = LM == 2 ? 12 : 20;                 // sites staged per round
    static constexpr int U = LM == 2 ? 4 : 5;                     // products per batch of LDS reads
    // Tables of 8 doubles (6 and the zero ends); one axis of a site holds 1, 2 or 4 of
    // them in an odd number of doubles, so that the lanes that write them, one per (site,
    // axis), fall on different LDS banks (with 16 doubles per axis all lanes met on one
    // bank: 23.1 us per launch at 12,288 sites against 16.0)
    static constexpr int AS = (LM == 0 ? 1 : LM == 1 ? 2 : 4) * 8 + 1;
    static constexpr int TS = 3 * AS;                             // doubles per staged site
    static constexpr int WLDS = NST * TS + 2 * NST;               // doubles per wavefront (tables, offsets)
};
// row stride of the tile's real grid in LDS (odd: columns fall on different banks)
__host__ __device__ inline int mm_zstride(int K2) { return K2 | 1; }
template <int LM> __host__ inline size_t spread_mm_lds(int K2, int wpt) {
    return (2 * (size_t)K2 + (size_t)SpreadShape<LM>::WLDS * mm_nseg(K2) * wpt + (size_t)wpt * 16 * mm_zstride(K2)) *
           sizeof(double);
}

// WRAP: one segment spans the axis (up to 16 points), so a support may wrap round into it
template <int LM, bool WRAP>
__global__ void __launch_bounds__(1024)
k_spread_z(int N, int K0, int K1, int K2, int wpt, const Cplx<double>* __restrict__ twz, const double* __restrict__ wfrac,
           const double* __restrict__ fq, const int* __restrict__ tstart, const int2* __restrict__ tlist, long cap,
           Cplx<double>* __restrict__ hgrid, const PcgState* __restrict__ skip, CgCheck chk) {
    using S = SpreadShape<LM>;
    extern __shared__ unsigned char smem_raw[];
    const int f = blockIdx.y;
    const int nty = (K1 + MM_TY - 1) / MM_TY, ntx = (K0 + MM_TX - 1) / MM_TX;
    const int nseg = mm_nseg(K2), len = mm_seglen(K2), nlist = ntx * nty * nseg;
    const int tile = xcd_item(blockIdx.x, ntx * nty);
    if (tile >= ntx * nty) return;
    const int lane = threadIdx.x & 63, nwave = blockDim.x >> 6;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int part = qdiv(wave, nseg, 1.0f / (float)nseg), seg = wave - part * nseg;
    const int Z0 = seg * len;
    Cplx<double>* tw = reinterpret_cast<Cplx<double>*>(smem_raw);
    double* tab = reinterpret_cast<double*>(tw + K2) + wave * S::WLDS;
    int4* se = reinterpret_cast<int4*>(tab + S::NST * S::TS);
    const int zs = mm_zstride(K2);
    double* G = reinterpret_cast<double*>(tw + K2) + nwave * S::WLDS;
    // The launch finds nothing of its predecessor in its caches, so a chain of loads
    // costs about a microsecond each: everything that does not depend on another load
    // is issued here (the flags are tested once the first sites are on their way).
    // This wavefront's share of the segment's candidates:
    const int li = tile * nseg + seg;
    const int l0 = tstart[(size_t)f * (nlist + 1) + li];
    const int l1 = tstart[(size_t)f * (nlist + 1) + li + 1];
    const int done = skip ? skip[f].done : 0;
    if (early_exit() && done) return;   // frame already converged
    double mxr = 0.0;
    if (chk.on) {
        // every wavefront reduces the same partials in the same order: one decision
        const double* mxp = chk.parts.mx(f, chk.cur);
        for (int k = lane; k < chk.parts.nb; k += 64) mxr = fmax(mxr, mxp[k]);
    }
    for (int t = threadIdx.x; t < K2; t += blockDim.x) tw[t] = twz[t];
    const int ltot = (int)min((long)l1, cap) - l0;
    const int wsh = wpt == 4 ? 2 : wpt - 1;      // wpt is 1, 2 or 4
    const int lo = l0 + ((ltot * part) >> wsh), hi = l0 + ((ltot * (part + 1)) >> wsh);
    // staging: lane = (site of the round, axis)
    const int ss = (lane * 43) >> 7, ax = lane - 3 * ss;
    // (a round's list entries are fetched two rounds ahead, its sites' data one)
    int2 ne = make_int2(0, 0), nl = make_int2(0, 0);
    double nw = 0, nq[6] = {0, 0, 0, 0, 0, 0};
    auto fetch_list = [&](int c) {
        if (ss < min(S::NST, hi - c)) nl = tlist[(size_t)f * cap + c + ss];
    };
    auto fetch = [&](int c) {
        if (ss < min(S::NST, hi - c)) {
            ne = nl;
            const size_t a = (size_t)f * N + ne.x;
            nw = wfrac[a * 3 + ax];
            const double* q = fq + a * 10;
            if (ax == 0) nq[0] = q[0];
            if (LM >= 1) {
                nq[1] = q[1 + ax];                 // mu along this axis
                if (LM == 1 && ax == 0) nq[2] = 0;
            }
            if (LM >= 2) {
                nq[2] = q[4 + ax];                 // Theta along this axis
                if (ax == 0) { nq[3] = q[3]; nq[4] = q[8]; }        // mz, Txz
                if (ax == 1) { nq[3] = q[7]; nq[4] = q[9]; }        // Txy, Tyz
            }
        }
    };
    if (lo < hi) {
        fetch_list(lo);
        fetch(lo);
        fetch_list(lo + S::NST);
    }
    if (done) return;   // frame already converged
    if (chk.on) {
        for (int o = 32; o > 0; o >>= 1) mxr = fmax(mxr, __shfl_xor(mxr, o, 64));
        if (mxr < chk.tol) {
            if (blockIdx.x == 0 && threadIdx.x == 0) {
                chk.st[f].res = mxr;
                chk.st[f].done = 1;
            }
            return;
        }
    }
    // zero ends of this lane's tables
    if (ss < S::NST)
#pragma unroll
        for (int t = 0; t < (LM == 0 ? 1 : LM == 1 ? 2 : 4); ++t) {
            double* T = tab + (ss * 3 + ax) * S::AS + t * 8;
            T[0] = 0.0;
            T[7] = 0.0;
        }
    const int c16 = lane & 15, k4 = lane >> 4;
    const int lx = c16 >> 2, ly = c16 & 3;
    d4 acc = {0, 0, 0, 0};
    for (int c = lo; c < hi; c += S::NST) {
        const int n = min(S::NST, hi - c);
        const int npad = (n + S::SPM * S::U - 1) / (S::SPM * S::U) * (S::SPM * S::U);   // empty sites fill the last batch
        wave_lds_fence();
        if (ss < npad) {
            const bool live = ss < n;
            // byte offsets of the support's start in the tables
            if (ax == 0) {
                const int e = live ? ne.y : 0;
                se[ss] = make_int4((e & 15) * 8, ((e >> 4) & 15) * 8, (e >> 8) * 8, 0);
            }
            double* T = tab + (ss * 3 + ax) * S::AS + 1;
#pragma unroll
            for (int k = 0; k < 6; ++k) {
                double v, d1, d2;
                bs_piece<double>(k, nw, v, d1, d2);
                if (!live) v = d1 = d2 = 0.0;
                if constexpr (LM == 0) {
                    T[k] = ax == 0 ? nq[0] * v : v;                     // q vx; vy; vz
                } else if constexpr (LM == 1) {
                    // q vx + mx ax, vx; vy, my ay; vz, mz az
                    T[k] = ax == 0 ? nq[0] * v + nq[1] * d1 : v;
                    T[8 + k] = ax == 0 ? v : nq[1] * d1;
                } else {
                    // x: q v + mx a + Txx b, mz v + 2 Txz a, v, a;  y: v, my a + Tyy b, 2 Tyz a, 2 Txy a;
                    // z: v, a, Tzz b  (mz belongs to the x factor of the az term)
                    if (ax == 0) {
                        T[k] = nq[0] * v + nq[1] * d1 + nq[2] * d2;
                        T[8 + k] = nq[3] * v + 2.0 * nq[4] * d1;
                        T[16 + k] = v;
                        T[24 + k] = d1;
                    } else if (ax == 1) {
                        T[k] = v;
                        T[8 + k] = nq[1] * d1 + nq[2] * d2;
                        T[16 + k] = 2.0 * nq[4] * d1;
                        T[24 + k] = 2.0 * nq[3] * d1;
                    } else {
                        T[k] = v;
                        T[8 + k] = d1;
                        T[16 + k] = nq[2] * d2;
                    }
                }
            }
        }
        wave_lds_fence();
        if (c + S::NST < hi) {
            fetch(c + S::NST);
            fetch_list(c + 2 * S::NST);
        }
        const int sub = LM == 0 ? k4 : LM == 1 ? k4 >> 1 : 0;     // this lane's site of the product
        const int term = LM == 0 ? 0 : LM == 1 ? (k4 & 1) : k4;
        const int x8 = 8 * lx + 48, y8 = 8 * ly + 48, z8 = 8 * c16 + 48;
        // LDS byte offsets kept per lane (not as a wavefront's base plus a lane's part,
        // which costs an addition per read)
        constexpr int Y = S::AS * 8, Z = 2 * S::AS * 8;
        const int wb = K2 * 16 + (int)(threadIdx.x >> 6) * (S::WLDS * 8);
        int b0 = wb + sub * (S::TS * 8);                                   // the site's tables
        int bx = b0 + (LM == 0 ? 0 : LM == 1 ? 64 * term : 64 * min(term, 2));   // this term's x, z tables
        int be = wb + S::NST * (S::TS * 8) + sub * 16;
        for (int s0 = 0; s0 < npad; s0 += S::SPM * S::U) {
            // a batch reads LDS twice (offsets, then tables) before its products
            int4 e[S::U];
            double A[S::U], B[S::U];
#pragma unroll
            for (int u = 0; u < S::U; ++u) e[u] = *reinterpret_cast<const int4*>(smem_raw + be + u * S::SPM * 16);
#pragma unroll
            for (int u = 0; u < S::U; ++u) {
                const unsigned char* T = smem_raw + u * S::SPM * S::TS * 8;
                const int ix = clamp56(x8 - e[u].x), iy = clamp56(y8 - e[u].y);
                int iz = z8 - e[u].z;
                if (WRAP) iz += iz < 8 ? 8 * K2 : iz >= 8 * K2 + 8 ? -8 * K2 : 0;
                iz = clamp56(iz);
                if constexpr (LM == 0) {
                    A[u] = at8(T, b0 + ix) * at8(T + Y, b0 + iy);
                    B[u] = at8(T + Z, b0 + iz);
                } else if constexpr (LM == 1) {
                    const double y1 = at8(T + Y + 64, b0 + (term ? 0 : iy));     // a zero end for the second term
                    A[u] = at8(T, bx + ix) * at8(T + Y, b0 + iy) + at8(T + 64, b0 + ix) * y1;
                    B[u] = at8(T + Z, bx + iz);
                } else {
                    // terms 0, 1, 2 and an empty fourth
                    A[u] = at8(T, bx + ix) * at8(T + Y, b0 + iy);
                    A[u] += at8(T + 128, b0 + ix) * at8(T + Y, b0 + (term == 0 ? 64 + iy : term == 1 ? 128 + iy : 0));
                    A[u] += at8(T + 192, b0 + ix) * at8(T + Y + 192, b0 + (term == 0 ? iy : 0));
                    B[u] = at8(T + Z, bx + (term < 3 ? iz : 0));
                }
            }
            b0 += S::SPM * S::U * S::TS * 8;
            bx += S::SPM * S::U * S::TS * 8;
            be += S::SPM * S::U * 16;
#pragma unroll
            for (int u = 0; u < S::U; ++u) acc = mma4(A[u], B[u], acc);
        }
    }
    {
        double* g = G + (size_t)part * 16 * zs;
        if (c16 < len && Z0 + c16 < K2)
#pragma unroll
            for (int r = 0; r < 4; ++r) g[(4 * r + k4) * zs + Z0 + c16] = acc[r];
    }
    __syncthreads();
    // z transform of the 16 columns: wavefront = (row tile, cos or sin)
    const int H = K2 / 2 + 1, nt = mm_tiles(K2), ns = mm_steps(K2);
    const int bx = tile / nty, by = tile - bx * nty;
    const int px = bx * MM_TX + lx, py = by * MM_TY + ly;
    // the partial blocks of a segment are added first (wpt > 1)
    if (wpt > 1) {
        for (int t = threadIdx.x; t < 16 * zs; t += blockDim.x) {
            double v = G[t];
            for (int p = 1; p < wpt; ++p) v += G[p * 16 * zs + t];
            G[t] = v;
        }
        __syncthreads();
    }
    for (int w = wave; w < 2 * nt; w += nwave) {
        const int mt = w >> 1, odd = w & 1;
        TwWalk walk;
        walk.start(tw, K2, mt * 16 + c16, k4);
        const double* g = G + c16 * zs;
        // n = 0 (and K / 2) is its own mirror image: it is counted twice in the even sums
        // and taken off once
        const double dbl = odd ? 0.0 : -(g[0] + (K2 & 1 ? 0.0 : (k4 & 1 ? -1.0 : 1.0) * g[K2 >> 1]));
        d4 o = {dbl, dbl, dbl, dbl};
        const double sg = odd ? -1.0 : 1.0;
        int na = k4, nb = k4 ? K2 - k4 : 0;
        for (int ks = 0; ks < ns; ++ks) {
            const Cplx<double> t = walk.next();
            double x = na < H ? g[na] + sg * g[nb] : 0.0;
            o = mma4(odd ? t.y : t.x, x, o);
            na += 4;
            nb = K2 - na;
        }
        if (px < K0 && py < K1) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int k = mt * 16 + 4 * r + k4;
                if (k < H) {
                    double* h = reinterpret_cast<double*>(hgrid + (((size_t)f * H + k) * K0 + px) * K1 + py);
                    h[odd] = o[r];   // (C, -S)
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Dense transform of the complex lines of an LDS array, in place: element e of line
// l at P[l * ls + e * es].  A wavefront takes 8 lines (16 columns: their real and
// imaginary parts) and all NT row tiles of them, so that an operand read from LDS
// serves 2 NT products; results stay in registers until every wavefront has read its
// inputs.  Every 8 lines need a wavefront.  hook.pre(line, k) is read early for every
// output (line, frequency k) and handed to hook.out(v, pre, line, k), whose value is
// written.
// ---------------------------------------------------------------------------
struct NoHook {
    static constexpr bool PRE = false;
    __device__ double pre(int, int) const { return 0.0; }
    __device__ double out(double v, double, int, int) { return v; }
};
template <int NT, class Hook>
__device__ __forceinline__ void mm_lines(Cplx<double>* P, int K, int nl, int ls, int es, const Cplx<double>* tw, int inverse,
                                         Hook& hook) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c16 = lane & 15, k4 = lane >> 4, comp = c16 & 1;
    const int H = K / 2 + 1, ns = mm_steps(K);
    const int line = wave * 8 + (c16 >> 1);
    d4 C[NT], S[NT];
    double pk[NT][4], pm[NT][4];
    double* D = reinterpret_cast<double*>(P);
    if (wave * 8 < nl) {
        const int lc = min(line, nl - 1);
        const unsigned char* col = reinterpret_cast<const unsigned char*>(D + 2 * lc * ls + comp);
        const int e16 = 16 * es;
        if (Hook::PRE && NT <= 3) {   // (more row tiles have no registers for it)
#pragma unroll
            for (int m = 0; m < NT; ++m)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int k = min(m * 16 + 4 * r + k4, H - 1);
                    pk[m][r] = hook.pre(lc, k);
                    pm[m][r] = hook.pre(lc, k > 0 ? K - k : 0);
                }
        }
        // element 0 (and K / 2) is its own mirror image: it is counted twice in the even
        // sums and taken off once
        const double dbl = -(at8(col, 0) + (K & 1 ? 0.0 : (k4 & 1 ? -1.0 : 1.0) * at8(col, (K >> 1) * e16)));
        TwWalk walk[NT];
#pragma unroll
        for (int m = 0; m < NT; ++m) {
            C[m] = d4{dbl, dbl, dbl, dbl};
            S[m] = d4{0, 0, 0, 0};
            walk[m].start(tw, K, m * 16 + c16, k4);
        }
        int oa = k4 * e16, ob = k4 ? (K - k4) * e16 : 0;
        double a = at8(col, oa), b = at8(col, ob);
#pragma unroll 1
        for (int ks = 0; ks < ns; ++ks) {
            const double e = a + b, o = a - b;
            // the next step's operands (past the last step: any element, with no products)
            oa += 4 * e16;
            ob = K * e16 - oa;
            const bool in = ks * 4 + 4 + k4 < H;
            a = at8(col, in ? oa : 0);
            b = at8(col, in ? ob : 0);
            if (!in) a = b = 0.0;
#pragma unroll
            for (int m = 0; m < NT; ++m) {
                const Cplx<double> t = walk[m].next();
                C[m] = mma4(t.x, e, C[m]);
                S[m] = mma4(t.y, o, S[m]);
            }
        }
    }
    __syncthreads();
    // frequency k of the real part: C(re) + sin sum(im) forward (- for the inverse), of
    // the imaginary part C(im) - sin sum(re); frequency K - k with the other sign; S
    // holds minus the sine sums
    const double sg = (comp != 0) != (inverse != 0) ? 1.0 : -1.0;
    if (wave * 8 < nl) {
        double* d = D + 2 * line * ls + comp;
        const bool live = line < nl;
#pragma unroll
        for (int m = 0; m < NT; ++m) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const double s = sg * swap_pair(S[m][r]), c = C[m][r];
                const int k = m * 16 + 4 * r + k4;
                if (live && k < H) {
                    if (Hook::PRE && NT > 3) {
                        pk[m][r] = hook.pre(line, k);
                        pm[m][r] = hook.pre(line, k > 0 ? K - k : 0);
                    }
                    d[2 * k * es] = hook.out(c + s, pk[m][r], line, k);
                    if (k > 0 && 2 * k < K) d[2 * (K - k) * es] = hook.out(c - s, pm[m][r], line, K - k);
                }
            }
        }
    }
    __syncthreads();
}

__device__ __forceinline__ void block_partials7(const double* vals, double* sh, double* out) {
#pragma unroll
    for (int k = 0; k < 7; ++k) {
        const double t = block_sum(vals[k], sh);
        if (threadIdx.x == 0) out[k] = t;
    }
}

struct InflArgs {
    const BoxInfo* boxes;
    const double *bmod0, *bmod1, *bmod2;
    double kappa;
    int kind;
    double pref;
    const double* tab;    // tabulated 2 pref C_k / theta_k^2, plane-major
    const double* tabd;   // pref (dC / d(k^2)) / theta_k^2 (IN_TABLE2_ACC)
    double* part;         // energy and box partials, 7 per block (IN_TABLE_ACC, IN_TABLE2_ACC)
};
// influence function applied to one component of a spectrum.  IN_TABLE: the tabulated
// electrostatic function (solver products).  IN_TABLE_ACC: the same with the energy
// and box-derivative sums, which follow from the table: C = tab theta^2 / (2 pref) and
// dC / d(k^2) = -C (1 / k^2 + 1 / (4 kappa^2)).  IN_TABLE2_ACC: the sums with the derivative
// from a table of its own (the dispersion kinds; k_infl_table2).
enum { IN_TABLE = 0, IN_TABLE2_ACC = 1, IN_TABLE_ACC = 2 };

// Both tables of a dispersion kind.  Their exp and erfc are formed here by every CU at once:
// in the plane pass, on the one CU a plane has, they took 21 of its 49 us (8,580 sites); the
// table takes 3.4 us and the pass 28.
__global__ void __launch_bounds__(256)
k_infl_table2(int K0, int K1, int K2, const BoxInfo* __restrict__ boxes, const double* __restrict__ bmod0,
              const double* __restrict__ bmod1, const double* __restrict__ bmod2, double kappa, int kind, double pref,
              double* __restrict__ tab, double* __restrict__ tabd) {
    const int f = blockIdx.y, H = K2 / 2 + 1, P = K0 * K1;
    const int idx = blockIdx.x * 256 + threadIdx.x;
    if (idx >= P * H) return;
    const int i2 = idx / P, r = idx - i2 * P, i0 = r / K1, i1 = r - i0 * K1;
    const InflPt q = infl_point(boxes[f], K0, K1, K2, i0, i1, i2, kappa, kind);
    const double th = bmod0[i0] * bmod1[i1] * bmod2[i2];
    const double ith2 = 1.0 / (th * th);
    tab[(size_t)f * P * H + idx] = 2.0 * pref * q.C * ith2;
    tabd[(size_t)f * P * H + idx] = pref * q.dC * ith2;
}

template <int KIND> struct InflHook {
    const InflArgs& q;
    const BoxInfo& b;
    const double* tp;     // the plane of the table
    const double* td;     // and of its derivative's
    int K0, K1, K2, y0, i2;
    bool on;              // off: values pass unchanged
    double sum[KIND == IN_TABLE ? 1 : 7];
    static constexpr bool PRE = true;
    __device__ __forceinline__ double pre(int line, int i0) const { return on ? tp[i0 * K1 + y0 + line] : 1.0; }
    __device__ __forceinline__ double out(double v, double t, int line, int i0) {
        if (KIND != IN_TABLE && on) {
            const int i1 = y0 + line;
            const int m0 = i0 < (K0 + 1) / 2 ? i0 : i0 - K0, m1 = i1 < (K1 + 1) / 2 ? i1 : i1 - K1;
            const int m2 = i2 < (K2 + 1) / 2 ? i2 : i2 - K2;
            const double kx = b.kb[0] * m0 + b.kb[1] * m1 + b.kb[2] * m2;
            const double ky = b.kb[3] * m0 + b.kb[4] * m1 + b.kb[5] * m2;
            const double kz = b.kb[6] * m0 + b.kb[7] * m1 + b.kb[8] * m2;
            const double v2 = v * v * ((i2 == 0 || 2 * i2 == K2) ? 1.0 : 2.0), e = 0.5 * t * v2;
            double wd;
            if constexpr (KIND == IN_TABLE2_ACC) {
                wd = -td[i0 * K1 + i1] * v2;
            } else {
                const double ksq = kx * kx + ky * ky + kz * kz;
                wd = ksq > 0.0 ? e * (1.0 / ksq + 1.0 / (4.0 * q.kappa * q.kappa)) : 0.0;
            }
            sum[0] += e;
            sum[1] += wd * kx * kx; sum[2] += wd * ky * ky; sum[3] += wd * kz * kz;
            sum[4] += wd * kx * ky; sum[5] += wd * kx * kz; sum[6] += wd * ky * kz;
        }
        return v * t;
    }
};

// row stride of the plane in LDS (odd: lines fall on different banks)
__host__ __device__ inline int mm_ystride(int K1) { return K1 | 1; }
__host__ inline size_t plane_mm_lds(int K0, int K1) {
    return ((size_t)K0 * mm_ystride(K1) + K0 + K1) * sizeof(Cplx<double>);
}
// a wavefront per 8 lines of either direction: at most MM_PT(NT) threads for NT row tiles
constexpr int MM_PT(int nt) { return nt <= 3 ? 256 * nt : 1024; }
__host__ inline int plane_mm_threads(int K0, int K1) { return 64 * (((K0 > K1 ? K0 : K1) + 7) / 8); }

// Plane pass: one workgroup per (kz, frame) holds the K0 x K1 plane in LDS and does
// the forward y and x transforms, the influence function (on the way out of the x
// transform), and the inverse x and y transforms.  It is bound by the matrix products
// of the one CU a plane has (a 50^2 plane: 784 products, 5.2 us at one per 16 cycles
// and CU), the rest by LDS latency between the four barriers.
template <int NT, int KIND>
__device__ __forceinline__ void plane_mm_body(int f, int i2, int nplane, int K0, int K1, int K2,
                                              const Cplx<double>* __restrict__ twx, const Cplx<double>* __restrict__ twy,
                                              Cplx<double>* __restrict__ hgrid, const InflArgs& q,
                                              const PcgState* __restrict__ skip) {
    extern __shared__ unsigned char smem_raw[];
    const int H = K2 / 2 + 1, P = K0 * K1, ys = mm_ystride(K1);
    Cplx<double>* b0 = reinterpret_cast<Cplx<double>*>(smem_raw);
    Cplx<double>* tx = b0 + K0 * ys;
    Cplx<double>* ty = tx + K0;
    Cplx<double>* pl = hgrid + ((size_t)f * H + i2) * P;
    const float inv = 1.0f / (float)K1;
    const int done = skip ? skip[f].done : 0;
    for (int i = threadIdx.x; i < K0 + K1; i += blockDim.x) tx[i] = i < K0 ? twx[i] : twy[i - K0];
    for (int i0 = threadIdx.x; i0 < P; i0 += 6 * blockDim.x) {
        Cplx<double> v[6];
#pragma unroll
        for (int u = 0; u < 6; ++u) v[u] = pl[min(i0 + u * (int)blockDim.x, P - 1)];
#pragma unroll
        for (int u = 0; u < 6; ++u) {
            const int i = i0 + u * (int)blockDim.x;
            const int x = qdiv(i, K1, inv);
            if (i < P) b0[x * ys + (i - x * K1)] = v[u];
        }
    }
    if (done) return;   // frame already converged
    __syncthreads();
    // forward y, forward x with the influence function, inverse x, inverse y: one copy
    // of the code
    const size_t to = ((size_t)f * H + i2) * P;
    InflHook<KIND> infl{q, q.boxes[f], q.tab + to, KIND == IN_TABLE2_ACC ? q.tabd + to : nullptr, K0, K1, K2, 0, i2, false, {}};
#pragma unroll 1
    for (int t = 0; t < 4; ++t) {
        const bool x = t == 1 || t == 2;
        infl.on = t == 1;
        mm_lines<NT>(b0, x ? K0 : K1, x ? K1 : K0, x ? 1 : ys, x ? ys : 1, x ? tx : ty, t >> 1, infl);
    }
    for (int i = threadIdx.x; i < P; i += blockDim.x) {
        const int x = qdiv(i, K1, inv);
        pl[i] = b0[x * ys + (i - x * K1)];
    }
    if constexpr (KIND != IN_TABLE) {
        __shared__ double sh[16];
        block_partials7(infl.sum, sh, q.part + ((size_t)f * nplane + i2) * 7);
    }
}

template <int NT, int KIND>
__global__ void __launch_bounds__(MM_PT(NT))
k_plane_mm(int K0, int K1, int K2, const Cplx<double>* __restrict__ twx, const Cplx<double>* __restrict__ twy,
           Cplx<double>* __restrict__ hgrid, InflArgs q, const PcgState* __restrict__ skip) {
    plane_mm_body<NT, KIND>(blockIdx.y, blockIdx.x, gridDim.x, K0, K1, K2, twx, twy, hgrid, q, skip);
}

// the plane pass and the real-space product of a solver product in one launch (see
// k_plane_matvec)
template <int NT>
__global__ void __launch_bounds__(MM_PT(NT))
k_plane_mm_matvec(int K0, int K1, int K2, const Cplx<double>* __restrict__ twx, const Cplx<double>* __restrict__ twy,
                  Cplx<double>* __restrict__ hgrid, InflArgs q, int F, int nplane_blocks, int N, int nbf, int cap,
                  const int* __restrict__ nbr, const int* __restrict__ ncnt,
                  const double* __restrict__ pcoef, MatvecRecords src, double* __restrict__ out,
                  const PcgState* __restrict__ skip) {
    const int H = K2 / 2 + 1;
    const int b = blockIdx.x;
    if (b < nplane_blocks) {
        if (b >= H * F) return;
        const int f = b / H, i2 = b - f * H;
        plane_mm_body<NT, IN_TABLE>(f, i2, H, K0, K1, K2, twx, twy, hgrid, q, skip);
        return;
    }
    const int item = xcd_item(b - nplane_blocks, nbf * F);
    if (item >= nbf * F) return;
    real_matvec_body<double, double>(blockDim.x, item, N, nbf, cap, q.boxes, nbr, ncnt, pcoef, src, out, skip);
}

// Planes too large for LDS: y lines and x lines in passes of their own, 32 lines per
// workgroup of 4 wavefronts, on the same plane-major half spectrum.
constexpr int MM_LINE_THREADS = 256;
constexpr int MM_LINES = MM_LINE_THREADS / 64 * 8;
__host__ inline size_t line_mm_lds(int K) { return ((size_t)MM_LINES * (K | 1) + K) * sizeof(Cplx<double>); }

template <int NT>
__global__ void __launch_bounds__(MM_LINE_THREADS)
k_y_mm(int K0, int K1, int H, const Cplx<double>* __restrict__ twy, Cplx<double>* __restrict__ hgrid, int inverse,
       const PcgState* __restrict__ skip) {
    if (skip && skip[blockIdx.y].done) return;  // frame already converged
    extern __shared__ unsigned char smem_raw[];
    Cplx<double>* b0 = reinterpret_cast<Cplx<double>*>(smem_raw);
    const int f = blockIdx.y, ys = K1 | 1;
    Cplx<double>* ty = b0 + MM_LINES * ys;
    for (int i = threadIdx.x; i < K1; i += blockDim.x) ty[i] = twy[i];
    const int nlines = H * K0, l0 = blockIdx.x * MM_LINES, nl = min(MM_LINES, nlines - l0);   // lines (kz, x)
    Cplx<double>* hg = hgrid + ((size_t)f * nlines + l0) * K1;
    const float inv = 1.0f / (float)K1;
    for (int i = threadIdx.x; i < nl * K1; i += blockDim.x) {
        const int l = qdiv(i, K1, inv);
        b0[l * ys + (i - l * K1)] = hg[i];
    }
    __syncthreads();
    NoHook plain;
    mm_lines<NT>(b0, K1, nl, ys, 1, ty, inverse, plain);
    for (int i = threadIdx.x; i < nl * K1; i += blockDim.x) {
        const int l = qdiv(i, K1, inv);
        hg[i] = b0[l * ys + (i - l * K1)];
    }
}

// consecutive y of one kz
template <int NT, int KIND>
__global__ void __launch_bounds__(MM_LINE_THREADS)
k_x_mm(int K0, int K1, int K2, const Cplx<double>* __restrict__ twx, Cplx<double>* __restrict__ hgrid, InflArgs q,
       const PcgState* __restrict__ skip) {
    if (skip && skip[blockIdx.y].done) return;  // frame already converged
    extern __shared__ unsigned char smem_raw[];
    Cplx<double>* b0 = reinterpret_cast<Cplx<double>*>(smem_raw);   // [x][MM_LINES + 1]
    constexpr int es = MM_LINES + 1;
    Cplx<double>* tx = b0 + es * K0;
    for (int i = threadIdx.x; i < K0; i += blockDim.x) tx[i] = twx[i];
    const int f = blockIdx.y, H = K2 / 2 + 1, nyb = (K1 + MM_LINES - 1) / MM_LINES;
    const int i2 = blockIdx.x / nyb, y0 = (blockIdx.x - i2 * nyb) * MM_LINES, nl = min(MM_LINES, K1 - y0);
    Cplx<double>* hg = hgrid + ((size_t)f * H + i2) * K0 * K1 + y0;
    for (int i = threadIdx.x; i < MM_LINES * K0; i += blockDim.x) {
        const int x = i / MM_LINES, y = i % MM_LINES;
        if (y < nl) b0[x * es + y] = hg[(size_t)x * K1 + y];
    }
    __syncthreads();
    const size_t to = ((size_t)f * H + i2) * K0 * K1;
    InflHook<KIND> infl{q, q.boxes[f], q.tab + to, KIND == IN_TABLE2_ACC ? q.tabd + to : nullptr, K0, K1, K2, y0, i2, false, {}};
#pragma unroll 1
    for (int t = 0; t < 2; ++t) {
        infl.on = t == 0;
        mm_lines<NT>(b0, K0, nl, 1, es, tx, t, infl);
    }
    for (int i = threadIdx.x; i < MM_LINES * K0; i += blockDim.x) {
        const int x = i / MM_LINES, y = i % MM_LINES;
        if (y < nl) hg[(size_t)x * K1 + y] = b0[x * es + y];
    }
    if constexpr (KIND != IN_TABLE) {
        __shared__ double sh[16];
        block_partials7(infl.sum, sh, q.part + ((size_t)f * gridDim.x + blockIdx.x) * 7);
    }
}
__host__ inline size_t xline_mm_lds(int K) { return ((size_t)(MM_LINES + 1) * K + K) * sizeof(Cplx<double>); }

// ---------------------------------------------------------------------------
// Complex-to-real z transform + gather.  One workgroup serves the sites whose base
// grid point lies in a 4 x 4 column tile: it transforms the 9 x 9 columns their
// supports touch into LDS (five times the tile's own columns, which still costs less
// than writing the real grid and reading it back in a launch of its own) and gathers
// from there, eight lanes per site (six of them own one x row of the support each),
// in cell-sorted order.  A site's spline tables are formed once, one axis by each of
// three lanes, and shared through LDS.
// ---------------------------------------------------------------------------
constexpr int GZ_COLS = (MM_TX + 5) * (MM_TY + 5);   // 81 columns
constexpr int GZ_CT = (GZ_COLS + 15) / 16;           // column tiles
constexpr int GZ_THREADS = 64 * GZ_CT * 2;           // 12 wavefronts, 96 sites per round
// Threads by the number of tiles.  Up to a tile per CU, a tile's own time is all there is:
// 12 wavefronts.  Past that, smaller workgroups of which two, then four, share a CU, so that
// one tile's loads run beside another's products.  With 12 / 8 / 4 wavefronts: 44 / 40 / 49 us
// for 400 tiles (98304 sites, 80 x 80 x 80), 436 / 309 / 293 us for 10816 (64 frames of 12288
// sites, 50 x 50 x 50), and 3470 / 1156 / 700 us for the latter's final pass beside the pair kernel.
__host__ inline int gather_z_threads(int items) { return items <= N_CU ? GZ_THREADS : items <= 4 * N_CU ? 512 : 256; }
// doubles of a site's tables: ND orders x 6 points x 3 axes, made odd
template <int MODE> struct GatherShape {
    static constexpr int ND = MODE == 0 ? 4 : 2;     // derivative orders needed
    static constexpr int AS = 6 * ND + (MODE == 0 ? 1 : 0);
    static constexpr int TS = 3 * AS + (MODE == 0 ? 0 : 1);
};
template <int MODE> __host__ inline size_t gather_z_lds(int K2, int threads) {
    return (2 * (size_t)K2 + (size_t)GZ_COLS * mm_zstride(K2) + (threads / 8) * GatherShape<MODE>::TS) * sizeof(double);
}
// sum over the eight lanes of a site, in every lane
__device__ __forceinline__ double sum8(double v) {
    v += dpp_move<0xB1>(v);    // lanes 2 i, 2 i + 1
    v += dpp_move<0x4E>(v);    // pairs of a quad
    v += dpp_move<0x141>(v);   // quads (mirrored; a quad's lanes agree)
    return v;
}

template <int MODE>
__global__ void __launch_bounds__(GZ_THREADS)
k_gather_z(int N, int K0, int K1, int K2, const Cplx<double>* __restrict__ twz, const double4* __restrict__ pos,
           const BoxInfo* __restrict__ boxes, int use_dA, const int4* __restrict__ mbase,
           const double* __restrict__ wfrac, const double* __restrict__ fq, const double* __restrict__ Qc,
           const double* __restrict__ U, int qmode, const Cplx<double>* __restrict__ hgrid, double* __restrict__ out3,
           double* __restrict__ g_q, double* __restrict__ g_pos, double* __restrict__ vir_atom,
           const int* __restrict__ cstart, const int* __restrict__ order, const PcgState* __restrict__ skip, CgEpi epi) {
    using GS = GatherShape<MODE>;
    extern __shared__ unsigned char smem_raw[];
    constexpr int ND = GS::ND;
    const int f = blockIdx.y;
    const int nty = (K1 + MM_TY - 1) / MM_TY, ntx = (K0 + MM_TX - 1) / MM_TX;
    const int tile = xcd_item(blockIdx.x, ntx * nty);
    if (tile >= ntx * nty) return;
    const int X0 = tile / nty * MM_TX, Y0 = (tile % nty) * MM_TY;
    Cplx<double>* tw = reinterpret_cast<Cplx<double>*>(smem_raw);
    double* G = reinterpret_cast<double*>(tw + K2);
    const int zs = mm_zstride(K2);
    const int lane = threadIdx.x & 63, nwave = blockDim.x >> 6;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int done = skip ? skip[f].done : 0;
    if (early_exit() && done) return;   // frame already converged
    for (int t = threadIdx.x; t < K2; t += blockDim.x) tw[t] = twz[t];
    // the tile's sites: one run of the cell-sorted order per x row
    const int* cs = cstart + (size_t)f * ((size_t)K0 * K1 * K2 + 1);
    int row0[MM_TX], rown[MM_TX], nsite = 0;
#pragma unroll
    for (int r = 0; r < MM_TX; ++r) {
        const int x = min(X0 + r, K0 - 1);
        const size_t b = ((size_t)x * K1 + Y0) * K2;
        row0[r] = cs[b];
        rown[r] = cs[b + (size_t)min(MM_TY, K1 - Y0) * K2] - row0[r];
        if (X0 + r >= K0) rown[r] = 0;
        nsite += rown[r];
    }
    // a site's inputs, which do not depend on the grid: those of the first round are on
    // their way while the columns are transformed.  Lanes 0..2 of a site own an axis
    // (or component) each.
    const int sl = threadIdx.x >> 3, l8 = threadIdx.x & 7;
    double* M = G + GZ_COLS * zs + sl * GS::TS;
    int si = 0, slx = 0;
    int4 sm = {0, 0, 0, 0};
    double e_pol = 0, e_real = 0, e_z = 0;
    auto load_site = [&](int k) {
        int base = row0[0];
        slx = 0;
#pragma unroll
        for (int r = 0; r < MM_TX; ++r)
            if (slx == r) {
                base = row0[r] + k;
                if (k >= rown[r] && r + 1 < MM_TX) { k -= rown[r]; ++slx; }
            }
        si = order[(size_t)f * N + base];
        const size_t a = (size_t)f * N + si;
        sm = mbase[a];
        if (l8 < 3) {
            if constexpr (MODE == 2) {
                e_pol = epi.pol[si];
                e_real = epi.real[a * 3 + l8];
                e_z = U[a * 3 + l8];
            }
            double m[4][6];
            bspline6<double>(wfrac[a * 3 + l8], m[0], m[1], m[2], m[3]);
#pragma unroll
            for (int o = 0; o < ND; ++o)
#pragma unroll
                for (int k2 = 0; k2 < 6; ++k2) M[l8 * GS::AS + o * 6 + k2] = m[o][k2];
        }
    };
    if (sl < nsite) load_site(sl);
    {
        const int H = K2 / 2 + 1, nt = mm_tiles(K2), ns = mm_steps(K2);
        const int c16 = lane & 15, k4 = lane >> 4;
        const int P = K0 * K1;
        for (int w = wave; w < GZ_CT * nt; w += nwave) {
            const int ct = w % GZ_CT, mt = w / GZ_CT, col = ct * 16 + c16;
            const int cx = (col * 57) >> 9, cy = col - cx * (MM_TY + 5);      // col / 9 below 96
            const bool live = col < GZ_COLS;
            int gx = X0 + cx - 3, gy = Y0 + cy - 3;
            gx = gx < 0 ? gx + K0 : gx >= K0 ? gx - K0 : gx;
            gy = gy < 0 ? gy + K1 : gy >= K1 ? gy - K1 : gy;
            const Cplx<double>* h = hgrid + (size_t)f * H * P + (live ? gx * K1 + gy : 0);
            // x_n = 2 sum_k (Re_k cos - Im_k sin), with k = 0 (and K / 2) counted once
            double once = h[0].x;
            if (!(K2 & 1)) once += (k4 & 1 ? -1.0 : 1.0) * h[(size_t)(H - 1) * P].x;
            once *= -0.5;
            d4 E = {once, once, once, once}, O = {0, 0, 0, 0};
            const Cplx<double>* hk = h + (size_t)k4 * P;
            TwWalk walk;
            walk.start(tw, K2, mt * 16 + c16, k4);
#pragma unroll 1
            for (int k0 = 0; k0 < ns; k0 += 4) {
                Cplx<double> v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    v[u] = Cplx<double>{0, 0};
                    if ((k0 + u) * 4 + k4 < H) v[u] = hk[(size_t)(4 * u) * P];
                }
                hk += (size_t)16 * P;
                if (w == wave && k0 == 0) __syncthreads();   // the twiddles are in LDS
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (k0 + u < ns) {
                        const Cplx<double> t = walk.next();
                        E = mma4(t.x, v[u].x, E);
                        O = mma4(t.y, v[u].y, O);
                    }
            }
            if (live) {
                double* g = G + col * zs;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int n = mt * 16 + 4 * r + k4;
                    if (n < H) {
                        g[n] = 2.0 * (E[r] + O[r]);     // O holds minus the sine sum
                        if (n > 0 && 2 * n < K2) g[K2 - n] = 2.0 * (E[r] - O[r]);
                    }
                }
            }
        }
        if (wave >= GZ_CT * nt) __syncthreads();   // wavefronts without a column tile meet the barrier here
    }
    if (done) return;   // frame already converged
    __syncthreads();
    const BoxInfo& b = boxes[f];
    const double* A = use_dA ? b.dA : b.A;
    double zw = 0;
    for (int k0s = 0; k0s < nsite; k0s += blockDim.x >> 3) {
        const bool active = k0s + sl < nsite;
        if (k0s > 0) {
            wave_lds_fence();     // the tables of the round before have been read
            if (active) load_site(k0s + sl);
            wave_lds_fence();
        }
        const size_t a = (size_t)f * N + si;
        // fp[c][aa][bb]: d^(c,aa,bb) of the fractional potential, c + aa + bb < ND
        double fp[ND][ND][ND];
#pragma unroll
        for (int c = 0; c < ND; ++c)
#pragma unroll
            for (int aa = 0; aa < ND; ++aa)
#pragma unroll
                for (int bb = 0; bb < ND; ++bb) fp[c][aa][bb] = 0.0;
        if (active && l8 < 6) {
            const double *Mx = M, *My = M + GS::AS, *Mz = M + 2 * GS::AS;
            const int my = wrapi(sm.y, K1) - Y0, mz = wrapi(sm.z, K2);
            double mzt[ND][6];
            int gz[6];
#pragma unroll
            for (int k2 = 0; k2 < 6; ++k2) {
                const int z = mz + k2 - 3;
                gz[k2] = z < 0 ? z + K2 : z >= K2 ? z - K2 : z;
#pragma unroll
                for (int o = 0; o < ND; ++o) mzt[o][k2] = Mz[o * 6 + k2];
            }
            double u[ND][ND];
#pragma unroll
            for (int aa = 0; aa < ND; ++aa)
#pragma unroll
                for (int bb = 0; bb < ND; ++bb) u[aa][bb] = 0;
            const double* row = G + ((slx + l8) * (MM_TY + 5) + my) * zs;
#pragma unroll 2
            for (int k1 = 0; k1 < 6; ++k1, row += zs) {
                double ph[6];
#pragma unroll
                for (int k2 = 0; k2 < 6; ++k2) ph[k2] = row[gz[k2]];
                double sz[ND];
#pragma unroll
                for (int o = 0; o < ND; ++o) {
                    sz[o] = 0;
#pragma unroll
                    for (int k2 = 0; k2 < 6; ++k2) sz[o] += ph[k2] * mzt[o][k2];
                }
#pragma unroll
                for (int aa = 0; aa < ND; ++aa) {
                    const double m1 = My[aa * 6 + k1];
#pragma unroll
                    for (int bb = 0; bb < ND; ++bb)
                        if (aa + bb < ND) u[aa][bb] += m1 * sz[bb];
                }
            }
#pragma unroll
            for (int c = 0; c < ND; ++c) {
                const double m0 = Mx[c * 6 + l8];
#pragma unroll
                for (int aa = 0; aa < ND; ++aa)
#pragma unroll
                    for (int bb = 0; bb < ND; ++bb)
                        if (c + aa + bb < ND) fp[c][aa][bb] = m0 * u[aa][bb];
            }
        }
#pragma unroll
        for (int c = 0; c < ND; ++c)
#pragma unroll
            for (int aa = 0; aa < ND; ++aa)
#pragma unroll
                for (int bb = 0; bb < ND; ++bb)
                    if (c + aa + bb < ND && (MODE == 0 || c + aa + bb == 1)) fp[c][aa][bb] = sum8(fp[c][aa][bb]);
        if constexpr (MODE == 0) {
            if (active && l8 == 0)
                gather_site_out<double, 0>(a, A, fp, pos, fq, Qc, U, qmode, out3, g_q, g_pos, vir_atom, 0.0, nullptr,
                                           nullptr, 0.0, zw);
        } else if (active && l8 < 3) {
            // component l8 of dE/dmu, and of the CG product
            const double dm = A[l8 * 3 + 0] * fp[1][0][0] + A[l8 * 3 + 1] * fp[0][1][0] + A[l8 * 3 + 2] * fp[0][0][1];
            if constexpr (MODE == 1) {
                out3[a * 3 + l8] = dm;
            } else {
                const double ap = e_pol < 1e-8 ? 1e-8 : e_pol;
                const double d = DIELECTRIC / ap - 2.0 * DIELECTRIC * epi.f1;
                const double wv = e_real + dm + d * e_z;
                out3[a * 3 + l8] = wv;
                zw += e_z * wv;
            }
        }
    }
    if constexpr (MODE == 2) {
        __shared__ double shz[GZ_THREADS / 64];
        zw = group_sum(zw, 64);
        if (lane == 0) shz[wave] = zw;
        __syncthreads();
        if (threadIdx.x == 0) {
            double t = shz[0];
            for (int w = 1; w < nwave; ++w) t += shz[w];
            epi.parts.zw(f)[tile] = t;
        }
    }
}

}  // namespace admp
