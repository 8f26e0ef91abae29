// The grouped upward tables (up_groups.hpp) against their definition, and with allocations that
// fail in the worker threads: the caller has to see the exception (at the C entry it becomes an
// error code), where an exception that leaves a thread ends the process.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <thread>

#include "../ifgf_amd/csrc/up_groups.hpp"

static std::atomic<long> budget{1L << 60}; // allocations left
static const std::thread::id first = std::this_thread::get_id();
static std::atomic<bool> workers_only{false};

void* operator new(std::size_t n)
{
    if ((!workers_only || std::this_thread::get_id() != first) && budget.fetch_sub(1) <= 0)
        throw std::bad_alloc();
    if (void* p = std::malloc(n ? n : 1))
        return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

struct Rec
{
    static constexpr int N = 2;
    int32_t cf, subd;
    uint32_t q01, pad;
    double x0[N], x1[N], x2[N], tr[N], ti[N];
};

#define CHECK(x)                                                                               \
    do                                                                                         \
        if (!(x))                                                                              \
        {                                                                                      \
            std::printf("line %d: %s\n", __LINE__, #x);                                        \
            std::exit(1);                                                                      \
        }                                                                                      \
    while (0)

int main()
{
    using namespace ifgf;
    constexpr int NHI = 9, CELLS = 1000; // sixteen jobs of 64 cells
    UpLevel U[2];
    uint32_t r = 7;
    for (UpLevel& u : U)
    {
        u.entries.resize(size_t(CELLS) * NHI * 8);
        for (UpEntry& E : u.entries)
        {
            r = r * 1664525u + 1013904223u;
            const int cf = int(r >> 28) - 2; // -1 and -2: no child cone there
            E = UpEntry{cf, cf, cf < 0 ? -1 : cf, int((r >> 20) & 1), {0, 0, 0}, {0, 0}};
        }
    }
    const std::vector<const UpLevel*> parts = {&U[0], &U[1]};
    std::vector<int64_t> cell0;
    const GroupTables<Rec> T = group_tables<Rec>(parts, NHI, cell0);
    CHECK(cell0.size() == 2 && cell0[0] == 0 && cell0[1] == CELLS);
    CHECK(T.goff.size() == 2 * CELLS * 8 + 1 && T.doff.size() == T.goff.size());
    for (int part = 0; part < 2; part++)
        for (int cell = 0; cell < CELLS; cell++)
            for (int c = 0; c < 8; c++)
            {
                const size_t row = (size_t(part) * CELLS + cell) * 8 + c;
                int seen = 0, want = 0;
                for (int q = 0; q < NHI; q++)
                    want += U[part].entries[(size_t(cell) * NHI + q) * 8 + c].cf >= 0;
                for (int32_t g = T.goff[row]; g < T.goff[row + 1]; g++)
                {
                    const int d = T.grp[g].subd >> 8, sub = T.grp[g].subd & 255;
                    CHECK(d < T.doff[row + 1] - T.doff[row]);
                    CHECK(T.dkey[2 * (T.doff[row] + d)] == T.grp[g].cf);
                    CHECK(T.dkey[2 * (T.doff[row] + d) + 1] == sub);
                    for (int k = 0; k < 2; k++)
                    {
                        const uint32_t q = (T.grp[g].q01 >> (16 * k)) & 0xffffu;
                        if (q == 0xffffu)
                            continue;
                        const UpEntry& E = U[part].entries[(size_t(cell) * NHI + q) * 8 + c];
                        CHECK(E.cf == T.grp[g].cf && E.sub == sub);
                        seen++;
                    }
                }
                CHECK(seen == want);
            }
    for (int workers = 0; workers < 2; workers++)
        for (long left : {0L, 1L, 5L, 40L, 300L})
        {
            std::vector<int64_t> cells;
            cells.reserve(2);
            bool thrown = false;
            workers_only = workers != 0;
            budget = left;
            try
            {
                group_tables<Rec>(parts, NHI, cells);
            }
            catch (const std::bad_alloc&)
            {
                thrown = true;
            }
            budget = 1L << 60;
            CHECK(thrown);
        }
    std::puts("ok");
    return 0;
}
