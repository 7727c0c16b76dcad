"""The decomposition writes every digit position that the sort reads: a walk of
its blocks and scalars over the planner's own plans (a small C++ program on the
library's make_plan), plain and window-shifted, whole and split into up to
eight parts, at sizes that do and do not fill their last sort tile."""
from plan_program import run_cpp

SOURCE = r"""
#include <stdio.h>
#include "engine.hpp"
using namespace zk;
int main() {
    int bad = 0, plans = 0;
    for (uint32_t n : {1u, 511u, 2048u, 5001u, 8192u, 70001u})
        for (uint32_t nmsm = 1; nmsm <= 3; nmsm++)
            for (uint32_t parts = 1; parts <= kMaxParts; parts++)
                for (uint32_t floor : {0u, 1u}) {
                    std::vector<uint32_t> ns(nmsm), cs(nmsm, 13);
                    for (uint32_t j = 0; j < nmsm; j++) ns[j] = n + 37 * j;
                    std::vector<uint64_t> t0(nmsm, 0);
                    const uint64_t stride = (2ull * ns.back() + kSortTile - 1) / kSortTile * kSortTile;
                    Plan pl;
                    if (make_plan(ns.data(), t0.data(), nmsm, cs.data(), pl, 0, 1u << 17, CurveId::Bn254, parts,
                                  floor ? stride : 0, 16, floor) != kOk)
                        return 2;
                    plans++;
                    std::vector<uint8_t> seen(pl.entries, 0);
                    for (const MsmDesc& m : pl.msms) {
                        if (padded(m) != (floor != 0)) bad++;
                        const uint64_t ntw = (2ull * m.n + kSortTile - 1) / kSortTile;
                        for (uint64_t i = 0; i < ntw * kSortTile / 2; i++) {
                            if (i >= m.n && !padded(m)) break;
                            for (uint32_t w = 0; w < m.nwin; w++) {
                                const SegDesc& s = pl.segs[m.seg0 + w / m.wps];
                                const uint64_t p = (w % m.wps) * ntw * kSortTile + 2 * i;
                                if (p + 1 >= s.len) { bad++; continue; }
                                seen[s.ent0 + p]++;
                                seen[s.ent0 + p + 1]++;
                            }
                        }
                    }
                    for (uint8_t c : seen) bad += c != 1;
                    // what a shifted window's digits address stays in the table
                    for (const SegDesc& s : pl.segs)
                        if (floor && s.wbase + (uint64_t)(s.ntiles / s.wtiles - 1) * s.wadj + s.len > 8 * stride) bad++;
                }
    printf("%d plans, %d faults\n", plans, bad);
    return bad != 0;
}
"""


def test_every_sorted_position_is_written(tmp_path):
    run_cpp(tmp_path, SOURCE)
