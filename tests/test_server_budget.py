"""The bytes a server charges for its requests cover what the planner lays out
for them: batches of one size and of mixed ones, plain and window-shifted, at
the built-in widths, by ws_sizes of the library's own plans."""
from plan_program import run_cpp

SOURCE = r"""
#include <stdio.h>
#include "engine.hpp"
#include "tuned_gfx950.hpp"
extern "C" uint64_t zkmsm_server_footprint(uint32_t n);
using namespace zk;
int main() {
    int bad = 0;
    auto check = [&](const std::vector<uint32_t>& ns) {
        uint64_t charged = 0, scalars = 0;
        std::vector<uint32_t> cs;
        std::vector<uint64_t> t0(ns.size(), 0);
        uint32_t top = 0;
        for (uint32_t n : ns) {
            charged += zkmsm_server_footprint(n);
            scalars += 32ull * n;
            top = std::max(top, n);
            uint32_t cls = 0;
            while ((1ull << cls) < n) cls++;
            cs.push_back((ns.size() > 1 ? kTunedBatch : kTunedPlain)[cls]);
        }
        const uint64_t stride = (2ull * top + kSortTile - 1) / kSortTile * kSortTile;
        Schedule sched{};
        for (int floor : {0, 1, 512, 4096}) {
            Plan pl;
            if (make_plan(ns.data(), t0.data(), ns.size(), cs.data(), pl, 0, 196608, CurveId::Bn254, 0,
                          floor ? stride : 0, Engine::kShiftC, floor, &sched) != kOk) {
                bad++;
                continue;
            }
            const uint64_t need = scalars + ws_sizes(pl, true).device;
            if (need > charged) {
                bad++;
                printf("%zu requests, first %u, shifted from %d: %lu > %lu\n", ns.size(), ns[0], floor,
                       (unsigned long)need, (unsigned long)charged);
            }
        }
    };
    for (uint32_t k = 0; k <= 22; k++)
        for (uint32_t n : {1u << k, (1u << k) + 1, 3u << k >> 1})
            for (uint32_t m : {1u, 2u, 64u})
                if (n && (uint64_t)n * m <= 1u << 24) check(std::vector<uint32_t>(m, n));
    check({1u << 16, 1024, 1024});
    check({1u << 20, 512, 600, 700, 5000, 300000});
    return bad != 0;
}
"""


def test_charge_covers_the_plans(tmp_path):
    run_cpp(tmp_path, SOURCE)
