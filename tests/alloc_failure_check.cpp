// First solves of a handle whose device allocations fail part of the way, with
// this program's hipMalloc and hipFree in place of the runtime's (which they
// call); for test_gpu_alloc_failure.py.  Prints the bytes that a handle holds
// after a first solve without failures and after one that failed before, for
// each allocation that the solve makes.
#include <dlfcn.h>

#include <cstdio>
#include <map>
#include <vector>

#include "mimetic_hybrid.h"

static std::map<void *, size_t> g_live;
static size_t g_bytes = 0;
static int g_count = 0, g_fail_at = 0;

extern "C" int hipMalloc(void **p, size_t n) {
    static auto real = reinterpret_cast<int (*)(void **, size_t)>(dlsym(RTLD_NEXT, "hipMalloc"));
    if (++g_count == g_fail_at) {
        *p = nullptr;
        return 2;   // hipErrorOutOfMemory, without asking the runtime
    }
    const int e = real(p, n);
    if (e == 0) {
        g_live[*p] = n;
        g_bytes += n;
    }
    return e;
}
extern "C" int hipFree(void *p) {
    static auto real = reinterpret_cast<int (*)(void *)>(dlsym(RTLD_NEXT, "hipFree"));
    const auto it = g_live.find(p);
    if (it != g_live.end()) {
        g_bytes -= it->second;
        g_live.erase(it);
    }
    return real(p);
}

int main() {
    const int n[3] = {9, 8, 7}, step[3] = {1, 9, 72}, nc = 9 * 8 * 7;
    std::vector<int> fp{0}, nb, bt, ijk;
    std::vector<double> vol(nc, 1.0), cc, area, fc, fn, bv, perm(9 * nc, 0.0), one(nc, 1.0), zero(nc, 0.0);
    for (int c = 0; c < nc; ++c) {
        const int q[3] = {c % 9, c / 9 % 8, c / 72};
        for (int d = 0; d < 3; ++d) {
            ijk.push_back(q[d]);
            cc.push_back(q[d] + 0.5);
            perm[9 * c + 4 * d] = 1.0 + (c * 37 % 11);
        }
        for (int d = 0; d < 3; ++d)
            for (int up = 0; up < 2; ++up) {
                const bool in = up ? q[d] + 1 < n[d] : q[d] > 0;
                nb.push_back(in ? c + (up ? step[d] : -step[d]) : -1);
                bt.push_back(!in && d == 0 ? MHS_BC_DIRICHLET : MHS_BC_NEUMANN);
                bv.push_back(!in && d == 0 ? 1.0 - up : 0.0);
                area.push_back(1.0);
                for (int e = 0; e < 3; ++e) {
                    fc.push_back(q[e] + (e == d ? up : 0.5));
                    fn.push_back(e == d ? 2.0 * up - 1.0 : 0.0);
                }
            }
        fp.push_back((int)nb.size());
    }
    mhs_solve_options o;
    mhs_default_options(&o);
    o.autotune = 0;
    const double g[3] = {0.0, 0.0, 0.0};
    // a first solve whose fail_at-th allocation fails (0: none), tried again with the second failing, then without
    // failures; the bytes held, or -1 where even the last one fails
    auto first_solve = [&](int fail_at, int *made) -> long long {
        mhs_solver *s = nullptr;
        const size_t before = g_bytes;
        const int cells[2] = {0, nc};
        int rc = mhs_create(&s, 0, nullptr);
        if (!rc)
            rc = mhs_set_grid(s, 1, cells, nc, fp.data(), nb.data(), vol.data(), cc.data(), area.data(), fc.data(),
                              fn.data());
        if (!rc) rc = mhs_set_cell_ijk(s, ijk.data());
        if (!rc) rc = mhs_init_system_structure(s, bt.data(), nullptr);
        if (!rc) rc = mhs_compute_inner_products(s, perm.data(), g);
        for (int attempt = 0; !rc && attempt < (fail_at ? 4 : 1); ++attempt) {
            g_count = 0;
            g_fail_at = attempt == 3 || !fail_at ? 0 : attempt == 0 ? fail_at : 2;
            const int rs = mhs_solve(s, one.data(), zero.data(), zero.data(), bt.data(), bv.data(), &o, nullptr);
            if (attempt == 3 || !fail_at) rc = rs;
            if (made) *made = g_count;
        }
        g_fail_at = 0;
        const long long held = rc ? -1 : (long long)(g_bytes - before);
        if (rc) std::fprintf(stderr, "fail_at %d: %s\n", fail_at, mhs_last_error(s));
        mhs_destroy(s);
        return held;
    };
    int made = 0;
    const long long clean = first_solve(0, &made);
    std::printf("%d %lld\n", made, clean);
    for (int f = 1; f <= made; ++f) std::printf("%d %lld\n", f, first_solve(f, nullptr));
    return 0;
}
