"""Teams that leave the bit-plane kernel before its tree do so only where the
tree has no barrier (it stays within one wave), and then by whole waves that
hold no element, for every block and point count."""
from plan_program import run_cpp

SOURCE = r"""
#include <initializer_list>
#include "plan.hpp"
using namespace zk;
int main() {
    int bad = 0;
    for (uint32_t lanes : {team_lanes(CurveId::Bn254), team_lanes(CurveId::Bn254G2)}) {
        const uint32_t per_wave = 64 / lanes;
        for (uint32_t threads : {64u, 128u, 256u})
            for (uint32_t count = 1; count <= 256; count *= 2) {
                const uint32_t teams = threads / lanes, P = count < teams ? count : teams;
                bool leaves = false;
                for (uint32_t team = 0; team < teams; team++) {
                    const bool idle = tree_idle(P, team, per_wave);
                    leaves |= idle;
                    bad += idle && team < P;
                    bad += idle != tree_idle(P, team / per_wave * per_wave, per_wave);
                }
                bad += leaves && P / per_wave > 1;
            }
    }
    return bad;
}
"""


def test_no_team_leaves_before_a_barrier(tmp_path):
    run_cpp(tmp_path, SOURCE)
