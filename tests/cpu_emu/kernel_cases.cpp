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

// the frame's flag, set by block 0 while another block of the launch runs
static PcgState g_st;
static void set_done() { g_st.done = 1; }

// k_jacobi, block 1 of 256: the residual is below tol, so nothing is updated, whenever block 0's
// flag becomes visible.  (The launch before it leaves large maxima in LDS.)
static int jacobi_flag() {
    const int nb = 256, N = nb * 256;
    std::vector<double> pol(N, 1.0), g(3 * N, 1.0), part(nb, 1e3), U(3 * N, 0.0);
    int bad = 0;
    for (int pass = 0; pass < 2; ++pass) {
        g_st = PcgState{};
        one_block(k_jacobi, dim3(nb), dim3(256), 1, N, 3, 1.0, pol.data(), g.data(), part.data(), U.data(), &g_st);
        if (pass) for (double u : U) bad += u != 0.0;
        std::fill(part.begin(), part.end(), 0.1);
        std::fill(U.begin(), U.end(), 0.0);
        emu::g_after_wave = set_done;
    }
    return bad;
}

// k_cg_update, block 1 of 4, the same: the residual of parity 0 is below tol
static int cg_flag() {
    const int nb = 4, N = nb * PCG_BLOCK, n3 = 3 * N;
    std::vector<double> pol(N, 1.0), x(n3, 0.0), r(2 * n3, 1e4), z(n3, 1.0), p(n3, 1.0), s(2 * n3, 1.0), w(n3, 1.0),
        rec(N * MREC, 0.0), parts(nb + 4 * nb, 1.0);
    const CgParts cp{parts.data(), nb, nb};
    BoxInfo box{};
    std::fill(cp.mx(0, 0), cp.mx(0, 0) + nb, 1e3);
    int bad = 0;
    for (int pass = 0; pass < 2; ++pass) {
        g_st = PcgState{};
        one_block(k_cg_update<double>, dim3(nb), dim3(PCG_BLOCK), 1, N, nb, 0, 1.0, (const BoxInfo*)&box, pol.data(), x.data(),
                  r.data(), z.data(), p.data(), s.data(), w.data(), rec.data(), (double*)nullptr, (const int*)nullptr,
                  (const double*)nullptr, cp, &g_st);
        if (pass) for (double v : x) bad += v != 0.0;
        std::fill(cp.mx(0, 0), cp.mx(0, 0) + nb, 0.1);
        std::fill(x.begin(), x.end(), 0.0);
        emu::g_after_wave = set_done;
    }
    return bad;
}

int main(int argc, char** argv) {
    const std::string c = argc > 1 ? argv[1] : "";
    const int bad = c == "jacobi_flag" ? jacobi_flag() : c == "cg_flag" ? cg_flag() : -1;
    printf("%s: %d wrong values\n", c.c_str(), bad);
    return bad != 0;
}
