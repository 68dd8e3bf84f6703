// Stands in for the runtime's hipFuncSetAttribute (accepting it, or refusing it
// when called with "refuse") and asks for the tail's LDS twice, as the
// hierarchies of two handles do; for test_cpu_amg_lists.py.
#include <cstdio>
#include <set>

#include "mhs_kernels.h"

static int g_calls = 0;
static bool g_refuse = false;
static std::set<const void *> g_kernels;

extern "C" hipError_t hipFuncSetAttribute(const void *func, hipFuncAttribute attr, int value) {
    if (attr != hipFuncAttributeMaxDynamicSharedMemorySize || value < 64 * 1024) return hipErrorInvalidValue;
    ++g_calls;
    g_kernels.insert(func);
    return g_refuse ? hipErrorInvalidValue : hipSuccess;
}

int main(int argc, char **) {
    g_refuse = argc > 1;
    for (int handle = 0; handle < 2; ++handle) {
        g_calls = 0;
        g_kernels.clear();
        const int limit = mhs::tail_lds_limit();
        std::printf("%d %d %zu\n", limit, g_calls, g_kernels.size());
    }
    return 0;
}
