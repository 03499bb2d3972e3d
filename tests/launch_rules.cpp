// The rules by which launches are chosen, for tests without a GPU: plain functions of a call's shape and the number of compute units.
#include "../turbogpt_amd/csrc/gemm_launch.h"
#include "../turbogpt_amd/csrc/width16_launch.h"

extern "C" {
int gemm_columns_of_256(int M, int N, int K, int mode, int units) {
    return columns_of_256(M, N, K, mode, units);
}
// teams of a block, blocks, waves of a team, whether the rows stay in LDS; passes: of the separate forward (1) and, 2, forward with gradient and
// backward launches
void w16_teams(int passes, int waves, int count, int depth, int flying, int units, int *out) {
    const w16::Teams t = passes ? w16::pass_teams(waves, depth, passes == 2, units) : w16::step_teams(waves, count, depth, flying, units);
    out[0] = t.teams, out[1] = t.blocks, out[2] = t.roles, out[3] = t.rows;
}
int w16_shares_launches(int depth, int K, int flying, int blocks, int steps, int units) {
    return w16::shares_launches(depth, K, flying, blocks, steps, units);
}
}
