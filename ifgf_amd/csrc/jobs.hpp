// jobs.hpp -- independent jobs of the host code on several threads.
#pragma once

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <exception>
#include <thread>
#include <vector>

namespace ifgf
{
// fn(j) for j < n on the calling thread and up to nthreads - 1 others (fewer where no more can be
// started).  An exception that leaves a job ends the others early and is thrown here, the first one:
// one that left a thread, or the caller before the threads are joined, would end the process.
template <class Fn> void run_jobs(size_t n, size_t nthreads, const Fn& fn)
{
    std::atomic<size_t> next{0};
    std::atomic<bool> failed{false};
    std::exception_ptr error;
    auto work = [&]()
    {
        try
        {
            for (size_t j; !failed && (j = next++) < n;)
                fn(j);
        }
        catch (...)
        {
            if (!failed.exchange(true))
                error = std::current_exception();
        }
    };
    std::vector<std::thread> pool;
    try
    {
        nthreads = std::min(nthreads, n);
        pool.reserve(nthreads);
        for (size_t t = 1; t < nthreads; t++)
            pool.emplace_back(work);
    }
    catch (...) // the threads there are do the work
    {
    }
    work();
    for (auto& th : pool)
        th.join();
    if (error)
        std::rethrow_exception(error);
}
} // namespace ifgf
