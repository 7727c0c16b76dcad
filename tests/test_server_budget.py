"""The bytes a server charges a call of its requests cover what the planner
lays out for it: requests of one size and of mixed ones, on plain and
window-shifted tables, at the built-in widths and shift rules, by ws_sizes of
the library's own plans; and the published charge of a request covers its
charge alone."""
from plan_program import run_cpp

SOURCE = r"""
#include <stdio.h>
#include "server.hpp"
#include "tuned_gfx950.hpp"
extern "C" uint64_t zkmsm_server_footprint(uint32_t n);
using namespace zk;
int main() {
    int bad = 0;
    auto check = [&](const std::vector<uint32_t>& ns) {
        const uint32_t m = (uint32_t)ns.size();
        uint64_t scalars = 0;
        std::vector<uint32_t> cs;
        std::vector<uint64_t> t0(m, 0);
        uint32_t top = 0;
        for (uint32_t n : ns) {
            scalars += 32ull * n;
            top = std::max(top, n);
            uint32_t cls = 0;
            while ((1ull << cls) < n) cls++;
            const uint32_t b = kTunedBatch[cls];
            cs.push_back(m > 1 && b ? b : kTunedPlain[cls]);
            for (bool sh : {false, true}) bad += Server::charge(Server::load(n, sh)) > zkmsm_server_footprint(n);
        }
        const uint64_t stride = (2ull * top + kSortTile - 1) / kSortTile * kSortTile;
        // plain tables (-1), and the shift rules that a table with copies meets
        std::vector<int> floors{-1, 1};
        if (m > 64) floors.insert(floors.end(), {0, 4096});
        else if (m > 1 || top <= kShiftSingleMax) floors.push_back(512);
        else floors.insert(floors.end(), {0, 512});
        for (int floor : floors) {
            Server::Load sum{0, 0};
            for (uint32_t n : ns) {
                const Server::Load l = Server::load(n, floor >= 0);
                sum = Server::Load{sum.entries + l.entries, sum.bytes + l.bytes};
            }
            const uint64_t charged = Server::charge(sum);
            Plan pl;
            if (make_plan(ns.data(), t0.data(), m, cs.data(), pl, 0, 196608, CurveId::Bn254, 0,
                          floor >= 0 ? stride : 0, Engine::kShiftC, floor > 0 ? floor : 0) != kOk) {
                bad++;
                continue;
            }
            const uint64_t need = scalars + ws_sizes(pl, true).device;
            if (need > charged) {
                bad++;
                printf("%u requests, first %u, floor %d: %lu > %lu\n", m, ns[0], floor, (unsigned long)need,
                       (unsigned long)charged);
            }
        }
    };
    for (uint32_t k = 0; k <= 22; k++)
        for (uint32_t n : {1u << k, (1u << k) + 1, 3u << k >> 1})
            for (uint32_t m : {1u, 2u, 64u, 100u})
                if (n && (uint64_t)n * m <= 1u << 24) check(std::vector<uint32_t>(m, n));
    check({1u << 16, 1024, 1024});
    check({1u << 20, 512, 600, 700, 5000, 300000});
    return bad != 0;
}
"""


def test_charge_covers_the_plans(tmp_path):
    run_cpp(tmp_path, SOURCE)
