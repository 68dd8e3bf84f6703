// First mixed solves on new handles whose FP32 vectors start out with what another
// program left in the memory: this program's hipMalloc fills allocations of a
// vector's size (argv[1] = 1) before it hands them out; for
// test_gpu_alloc_failure.py.  One cell, so that nearly all face rows are padding.
#include <dlfcn.h>

#include <cstdio>
#include <cstdlib>
#include <vector>

#include "mimetic_hybrid.h"

static const size_t kRows = 1024, kRhs = 4;   // padded face rows of one cell, right-hand sides
static bool g_fill = false;

extern "C" int hipMalloc(void **p, size_t n) {
    static auto real = reinterpret_cast<int (*)(void **, size_t)>(dlsym(RTLD_NEXT, "hipMalloc"));
    static auto fill = reinterpret_cast<int (*)(void *, int, size_t)>(dlsym(RTLD_NEXT, "hipMemset"));
    const int e = real(p, n);
    // only the FP32 vectors have this size: no index is ever filled
    if (e == 0 && g_fill && n == kRows * kRhs * sizeof(float)) return fill(*p, 0x4b, n);   // 1.3e7 each
    return e;
}

int main(int, char **argv) {
    g_fill = std::atoi(argv[1]) != 0;
    const int fp[2] = {0, 6}, nb[6] = {-1, -1, -1, -1, -1, -1}, ijk[3] = {0, 0, 0}, cells[2] = {0, 1};
    const int bt[6] = {MHS_BC_DIRICHLET, MHS_BC_DIRICHLET, 0, 0, 0, 0};
    const double vol = 1.0, cc[3] = {0.5, 0.5, 0.5}, g[3] = {0.0, 0.0, -9.81};
    const double perm[9] = {2.0, 0.3, 0.1, 0.3, 1.0, 0.2, 0.1, 0.2, 0.5}, one = 1.0, half = 0.5;
    double area[6], fc[18], fn[18];
    std::vector<double> bv(6 * kRhs, 0.0), src(kRhs, 0.0);
    for (int f = 0; f < 6; ++f) {
        area[f] = 1.0;
        for (int d = 0; d < 3; ++d) {
            fc[3 * f + d] = d == f / 2 ? f % 2 : 0.5;
            fn[3 * f + d] = d == f / 2 ? 2.0 * (f % 2) - 1.0 : 0.0;
        }
    }
    for (size_t k = 0; k < kRhs; ++k) bv[6 * k] = 3.0 * (k + 1);
    for (int handle = 0; handle < 8; ++handle) {   // which operator a tuner chooses may differ
        mhs_solver *s = nullptr;
        int rc = mhs_create(&s, 0, nullptr);
        if (!rc) rc = mhs_set_grid(s, 1, cells, 1, fp, nb, &vol, cc, area, fc, fn);
        if (!rc) rc = mhs_set_cell_ijk(s, ijk);
        if (!rc) rc = mhs_init_system_structure(s, bt, nullptr);
        if (!rc) rc = mhs_compute_inner_products(s, perm, g);
        mhs_solve_options o;
        mhs_default_options(&o);
        o.precision = MHS_MIXED;
        o.nrhs = (int)kRhs;
        o.maxit = 100;
        mhs_solve_report r{};
        for (int k = 0; !rc && k < 2; ++k) {
            rc = mhs_solve(s, &one, &half, src.data(), bt, bv.data(), &o, &r);
            std::printf("%d %d %d %d\n", rc, r.iterations, r.converged, r.element_operator);
        }
        if (rc) std::fprintf(stderr, "%s\n", mhs_last_error(s));
        mhs_destroy(s);
    }
    return 0;
}
