"""The rule that splits a call in parts by its entries: one line per curve, not
beside a power of two, so that a call of one point more than 2^20 is planned
as one of 2^20 is."""
from plan_program import run_cpp

SOURCE = r"""
#include "engine.hpp"
using namespace zk;
int main() {
    int bad = 0;
    for (CurveId cv : {CurveId::Bn254, CurveId::Grumpkin, CurveId::Bn254G2}) {
        uint32_t last = 1;
        for (uint64_t e = 1; e < 1ull << 31; e += 1 + e / 64) {
            const uint32_t p = default_parts(e, cv);
            bad += p < last || p > kMaxParts;
            last = p;
        }
        for (uint32_t k = 16; k < 31; k++)  // a window of one more point, either way
            for (uint64_t d : {16u, 512u})
                bad += default_parts((1ull << k) + d, cv) != default_parts((1ull << k) - d, cv) ||
                       default_parts(1ull << k, cv) != default_parts((1ull << k) + d, cv);
        for (uint32_t n : {(1u << 20) - 1, 1u << 20, (1u << 20) + 1}) {
            Plan pl;
            const uint64_t t0 = 0;
            const uint32_t c = 16;
            bad += make_plan(&n, &t0, 1, &c, pl, 0, 196608, cv) != kOk || pl.nparts != 1;
        }
    }
    return bad;
}
"""


def test_parts_by_entries(tmp_path):
    run_cpp(tmp_path, SOURCE)
