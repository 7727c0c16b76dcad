"""Device memory of a planned call: never more than with digits of four bytes, a
merge list as long as the record keys and bit planes in memory of their own,
so that a cap which left room for that leaves room for the call; and the
planes of a segment fit over its buckets, where the device keeps them."""
from plan_program import run_cpp

SOURCE = r"""
#include <stdio.h>
#include "engine.hpp"
#include "tuned_gfx950.hpp"
using namespace zk;
int main() {
    int bad = 0;
    for (uint32_t c = 2; c <= 16; c++) bad += c > 1u << (c - 1);
    auto up = [](uint64_t b) { return (b + 255) & ~uint64_t(255); };
    for (CurveId cv : {CurveId::Bn254, CurveId::Grumpkin, CurveId::Bn254G2})
        for (uint32_t n : {1u, 2u, 7u, 48u, 150u, 1000u, 1429u, 5000u, 20000u, 70000u, 300000u})
            for (uint32_t m : {1u, 4u, 15u, 62u}) {
                std::vector<uint32_t> ns(m, n), cs(m, 0);
                uint32_t cls = 0;
                while ((1ull << cls) < n) cls++;
                if (cv == CurveId::Bn254)
                    for (uint32_t& c : cs) c = m > 1 && kLeanBatch[cls] ? kLeanBatch[cls] : kLeanPlain[cls];
                std::vector<uint64_t> t0(m, 0);
                Plan pl;
                if ((uint64_t)n * m > 1u << 20) continue;
                if (make_plan(ns.data(), t0.data(), m, cs.data(), pl, 0, kTwoWaveLanes, cv) != kOk) return 1;
                const bool dev_tail = m >= 8 && cv != CurveId::Bn254G2;
                const WsSizes z = ws_sizes(pl, dev_tail);
                const uint64_t nseg = pl.segs.size(), own = dev_tail ? up(z.res) : 0;  // (results: host memory)
                const uint64_t former = up(z.desc) + up(4 * pl.entries) + 2 * up(z.keys) + 2 * up(z.vals) + up(z.hist) +
                                        up(z.part) + up(z.segvalid) + up(z.buckets) + 2 * up(z.rec_keys) +
                                        up(z.rec_pts) + up(z.rc) + up(nseg * 16 * host_point_bytes(cv)) + 256;
                if (z.device - own > former) {
                    bad++;
                    printf("curve %u, %u of %u points: %lu > %lu\n", (unsigned)cv, m, n,
                           (unsigned long)(z.device - own), (unsigned long)former);
                }
            }
    return bad != 0;
}
"""


def test_device_memory_of_small_and_lean_plans(tmp_path):
    run_cpp(tmp_path, SOURCE)
