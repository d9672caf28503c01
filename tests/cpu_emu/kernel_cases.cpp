// Single kernels on chosen blocks, for what a whole run on the CPU cannot show: a value in
// memory that another block changes between two wavefronts of one block.  One case per run; the
// exit status is the number of wrong values.
#include "hip/hip_runtime.h"
#include "admp_common.h"
#include "nblist_kernels.h"
#include "pair_kernels.h"
#include "recip_kernels.h"
#include "recip2_kernels.h"
#include "site_kernels.h"
#include <string>
#include <vector>
using namespace admp;

// runs block bx of a launch of g blocks
template <class... KA, class... A> void one_block(void (*k)(KA...), dim3 g, dim3 b, unsigned bx, A... a) {
    using Tup = std::tuple<typename std::decay<KA>::type...>;
    struct Pack { void (*k)(KA...); Tup args; } pk{k, Tup(a...)};
    emu::begin_kernel("one_block", g, b, 0);
    emu::run_block([](void* p) { auto* q = static_cast<Pack*>(p); std::apply(q->k, q->args); }, &pk, bx, 0, 0);
    emu::end_kernel();
}

// The frame's flag, set by block 0 (to the value that it leaves alone) while another block of the
// launch runs, whose wavefronts then read it different.  run(block, residual) runs one block of an
// update; a residual below tol (1) updates nothing, whenever the flag becomes visible.
static PcgState g_st;
static int g_mark;
template <class Run> static int flag_case(Run run, std::vector<double>& out) {
    int bad = 0;
    auto unchanged = [&] { for (double& v : out) { bad += v != 0.0; v = 0.0; } };
    g_st = PcgState{};
    run(0, 0.1);
    g_mark = g_st.done;
    bad += !g_mark;
    unchanged();
    g_st = PcgState{};
    run(1, 1e3);            // leaves large values in LDS
    std::fill(out.begin(), out.end(), 0.0);
    g_st = PcgState{};
    emu::g_after_wave = [] { g_st.done = g_mark; };
    run(1, 0.1);
    emu::g_after_wave = nullptr;
    unchanged();
    return bad;
}

static int jacobi_flag() {
    const int nb = 256, N = nb * 256;
    std::vector<double> pol(N, 1.0), g(3 * N, 1.0), part(nb), U(3 * N, 0.0);
    return flag_case([&](unsigned bx, double res) {
        std::fill(part.begin(), part.end(), res);
        one_block(k_jacobi, dim3(nb), dim3(256), bx, N, 3, 1.0, pol.data(), g.data(), part.data(), U.data(), &g_st);
    }, U);
}

static int cg_flag() {
    const int nb = 4, N = nb * PCG_BLOCK, n3 = 3 * N;
    std::vector<double> pol(N, 1.0), x(n3, 0.0), r(2 * n3, 1e4), z(n3, 1.0), p(n3, 1.0), s(2 * n3, 1.0), w(n3, 1.0),
        rec(N * MREC, 0.0), parts(nb + 4 * nb, 1.0);
    const CgParts cp{parts.data(), nb, nb};
    BoxInfo box{};
    auto run = [&](int cur, unsigned bx) {
        one_block(k_cg_update<double>, dim3(nb), dim3(PCG_BLOCK), bx, N, nb, cur, 1.0, (const BoxInfo*)&box, pol.data(),
                  x.data(), r.data(), z.data(), p.data(), s.data(), w.data(), rec.data(), (double*)nullptr,
                  (const int*)nullptr, (const double*)nullptr, cp, &g_st);
    };
    int bad = flag_case([&](unsigned bx, double res) {
        std::fill(cp.mx(0, 0), cp.mx(0, 0) + nb, res);
        run(0, bx);
    }, x);
    // the updates after it leave the frame alone, though parity 1 holds an older residual
    std::fill(cp.mx(0, 1), cp.mx(0, 1) + nb, 1e3);
    g_st = PcgState{};
    run(0, 0);
    for (int n = 1; n < 4; ++n)
        for (unsigned bx = 0; bx < nb; ++bx) run(n & 1, bx);
    for (double v : x) bad += v != 0.0;
    return bad;
}

// k_nbr_build with a site on the periodic face whose stored cell and recomputed place lie on
// opposite sides of it, as two kernels' roundings may have it: its neighbours on either side stay.
// (lo: the site at 0+, stored in the last cell; else at the box's end, stored in the first.)
static int nbr_face(bool lo, int nc) {
    const double rc = 4.0, L = nc * rc * 1.004;
    const int N = 3, cap = 8;
    const double x0 = lo ? 1e-17 : L * (1.0 - 1e-16);
    // neighbours 0.5 beyond either side of the face, in the last and the first cell
    const double4 pos[N] = {make_double4(x0, 1, 1, 0), make_double4(L - 0.5, 1, 1, 0), make_double4(0.5, 1, 1, 0)};
    BoxInfo box{};
    for (int d = 0; d < 3; ++d) { box.B[4 * d] = L; box.Binv[4 * d] = 1.0 / L; }
    const CellGrid cg{{nc, 1, 1}, nc};
    const int cell[N] = {lo ? nc - 1 : 0, nc - 1, 0};
    std::vector<int> start(nc + 1, 0);
    for (int c : cell) ++start[c + 1];
    for (int c = 0; c < nc; ++c) start[c + 1] += start[c];
    std::vector<int> fill(start);
    double4 spos[N];
    for (int i = 0; i < N; ++i) { spos[fill[cell[i]]] = pos[i]; spos[fill[cell[i]]++].w = i; }
    const int xoff[N + 1] = {0, 0, 0, 0}, xent[1] = {0};
    int nbr[N * cap], ncnt[N], nhalf[N], maxcnt = 0;
    one_block(k_nbr_build, dim3(1), dim3(256), 0, N, cap, pos, (const BoxInfo*)&box, cg, rc * rc, cell, (const int*)start.data(),
              (const double4*)spos, xoff, xent, nbr, ncnt, nhalf, &maxcnt);
    return (ncnt[0] != 2) + (ncnt[1] != 2) + (ncnt[2] != 2);
}
static int nbr_faces() {
    int bad = 0;
    for (int nc : {2, 3, 4, 7}) bad += nbr_face(true, nc) + nbr_face(false, nc);
    return bad;
}

int main(int argc, char** argv) {
    const std::string c = argc > 1 ? argv[1] : "";
    const int bad = c == "jacobi_flag" ? jacobi_flag() : c == "cg_flag" ? cg_flag() : c == "nbr_faces" ? nbr_faces() : -1;
    printf("%s: %d wrong values\n", c.c_str(), bad);
    return bad != 0;
}
