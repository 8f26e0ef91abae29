// up_groups.hpp -- the upward tables regrouped by child cone (host code of the upload).
#pragma once

#include <algorithm>
#include <cstdint>
#include <stdexcept>
#include <type_traits>
#include <vector>

#include "jobs.hpp"
#include "plan.hpp"

namespace ifgf
{
// The upward tables regrouped by child cone: per (cell, octant) row the distinct child fine
// cones (cf, sub) its nodes fall into, in order of first appearance, and per child cone its
// nodes (ascending) in records of at most Rec::N.  Row r's cones are dkey[2 doff[r] ..], its
// records [goff[r], goff[r + 1]).
template <class Rec> struct GroupTables
{
    std::vector<Rec> grp;
    std::vector<int32_t> goff, doff, dkey;
};
// the rows of cells [c0, c1) of one part, appended to T
template <class Rec>
void group_cells(const UpLevel& U, int n_hi, int64_t c0, int64_t c1, GroupTables<Rec>& T)
{
    std::vector<int32_t> gcnt, gnode, nd(n_hi);
    for (int64_t cell = c0; cell < c1; cell++)
        for (int c = 0; c < 8; c++)
        {
            const UpEntry* row = &U.entries[size_t(cell) * n_hi * 8 + c]; // node q: row[8 q]
            const size_t k0 = T.dkey.size() / 2;
            T.doff.push_back(int32_t(k0));
            T.goff.push_back(int32_t(T.grp.size()));
            int last = -1; // neighbouring nodes mostly share the last cone found
            for (int q = 0; q < n_hi; q++)
            {
                const UpEntry& E = row[8 * q];
                nd[q] = -1;
                if (E.cf < 0)
                    continue;
                const int nk = int(T.dkey.size() / 2 - k0);
                auto is = [&](int i)
                { return T.dkey[2 * (k0 + i)] == E.cf && T.dkey[2 * (k0 + i) + 1] == E.sub; };
                int d = (last >= 0 && is(last)) ? last : -1;
                for (int i = 0; d < 0 && i < nk; i++)
                    if (is(i))
                        d = i;
                if (d < 0)
                {
                    d = nk;
                    T.dkey.push_back(E.cf);
                    T.dkey.push_back(E.sub);
                }
                nd[q] = last = d;
            }
            const int nk = int(T.dkey.size() / 2 - k0);
            gcnt.assign(size_t(nk) + 1, 0);
            for (int q = 0; q < n_hi; q++)
                if (nd[q] >= 0)
                    gcnt[size_t(nd[q]) + 1]++;
            for (int i = 0; i < nk; i++)
                gcnt[i + 1] += gcnt[i];
            gnode.assign(size_t(gcnt[nk]), 0);
            for (int q = 0; q < n_hi; q++)
                if (nd[q] >= 0)
                    gnode[size_t(gcnt[nd[q]]++)] = q;
            for (size_t i = 0; i < gnode.size();)
            {
                const int d = nd[gnode[i]];
                Rec G{};
                G.cf = row[8 * gnode[i]].cf;
                G.subd = row[8 * gnode[i]].sub | (d << 8);
                uint32_t qs[4] = {0xffffu, 0xffffu, 0xffffu, 0xffffu};
                for (int g = 0; g < Rec::N && i < gnode.size() && nd[gnode[i]] == d; g++, i++)
                {
                    using X = typename std::remove_reference<decltype(G.x0[0])>::type;
                    const UpEntry& E = row[8 * gnode[i]];
                    qs[g] = uint32_t(gnode[i]);
                    G.x0[g] = X(E.xi[0]);
                    G.x1[g] = X(E.xi[1]);
                    G.x2[g] = X(E.xi[2]);
                    G.tr[g] = X(E.tf[0]);
                    G.ti[g] = X(E.tf[1]);
                }
                G.q01 = qs[0] | (qs[1] << 16);
                if constexpr (Rec::N == 4)
                    G.q23 = qs[2] | (qs[3] << 16);
                T.grp.push_back(G);
            }
        }
}
// every part's rows, by up to 16 threads; part_cell[part]: the part's first cell
template <class Rec>
GroupTables<Rec> group_tables(const std::vector<const UpLevel*>& parts, int n_hi,
                              std::vector<int64_t>& part_cell)
{
    struct Job
    {
        const UpLevel* U;
        int64_t c0, c1;
    };
    std::vector<Job> jobs;
    int64_t cells = 0;
    for (const UpLevel* U : parts)
    {
        part_cell.push_back(cells);
        const int64_t n = int64_t(U->entries.size()) / (int64_t(n_hi) * 8);
        for (int64_t c = 0; c < n; c += 64)
            jobs.push_back({U, c, std::min<int64_t>(n, c + 64)});
        cells += n;
    }
    std::vector<GroupTables<Rec>> out(jobs.size());
    run_jobs(jobs.size(), 16, [&](size_t j)
             { group_cells(*jobs[j].U, n_hi, jobs[j].c0, jobs[j].c1, out[j]); });
    GroupTables<Rec> T;
    size_t ng = 0, nk = 0;
    for (const auto& o : out)
    {
        ng += o.grp.size();
        nk += o.dkey.size();
    }
    if (nk / 2 > size_t(INT32_MAX))
        throw std::runtime_error("upward tables: too many distinct child cones");
    if (ng > size_t(INT32_MAX))
        throw std::runtime_error("upward tables: too many node groups");
    T.grp.reserve(ng);
    T.dkey.reserve(nk);
    for (auto& o : out)
    {
        const int32_t g0 = int32_t(T.grp.size()), k0 = int32_t(T.dkey.size() / 2);
        for (int32_t v : o.goff)
            T.goff.push_back(g0 + v);
        for (int32_t v : o.doff)
            T.doff.push_back(k0 + v);
        T.grp.insert(T.grp.end(), o.grp.begin(), o.grp.end());
        T.dkey.insert(T.dkey.end(), o.dkey.begin(), o.dkey.end());
        o = GroupTables<Rec>();
    }
    T.goff.push_back(int32_t(T.grp.size()));
    T.doff.push_back(int32_t(T.dkey.size() / 2));
    return T;
}
} // namespace ifgf
