// device_alloc_all (hip_util.hpp) with an allocator that fails at a chosen call: what was had is
// given back, no pointer is left and no error stays for the next call.
#include <cstdio>
#include <cstdlib>

#include "../ifgf_amd/csrc/hip_util.hpp"

static int calls = 0, fail_at = 0, live = 0;
static hipError_t last = hipSuccess;
extern "C" hipError_t hipMalloc(void** p, size_t n)
{
    if (++calls == fail_at)
        return last = hipErrorOutOfMemory;
    *p = std::malloc(n);
    live++;
    return hipSuccess;
}
extern "C" hipError_t hipFree(void* p)
{
    if (p)
        live--;
    std::free(p);
    return hipSuccess;
}
extern "C" hipError_t hipGetLastError()
{
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}

int main()
{
    for (int f = 0; f <= 3; f++)
    {
        void *a = nullptr, *b = nullptr, *c = nullptr;
        calls = 0;
        fail_at = f;
        const bool ok = ifgf::device_alloc_all({{&a, 8}, {&b, 16}, {&c, 24}});
        const bool good = f == 0 ? ok && a && b && c && live == 3
                                 : !ok && !a && !b && !c && live == 0 && calls == f;
        if (!good || last != hipSuccess)
        {
            std::printf("failing at call %d\n", f);
            return 1;
        }
        for (void* p : {a, b, c})
            (void)hipFree(p);
    }
    std::puts("ok");
    return 0;
}
