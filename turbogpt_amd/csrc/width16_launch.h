// How the width-16 network's passes are cut into blocks (width16.hip), and what a block has in LDS.  Plain functions of the shape and
// of the number of compute units.
#pragma once
#include <algorithm>
#include <cstddef>
#include <initializer_list>

namespace w16 {

constexpr int W = 16, V = 256, MAX_DEPTH = 8;
constexpr int ROLES = 4; // waves of a team, which has sixteen tokens; or it is a lone wave
constexpr int block_waves(int roles) { return roles == 1 ? 8 : 16; } // they stage the weights, as many stay as are in teams

// What a team's own backward pass wants of a layer (cuda/types.cuh:40-44, cuda/model.cuh:25-29), a record of ROW_BYTES: tiles of
// block input, post-RoPE query, the winning key and value (head layout) and post-attention residual; a word a lane of
// GELU(top) and GELU'(top), a byte of the distance to the winner; a word a token of the two inverse norms.
enum RowTile { R_X, R_Q, R_KEY, R_VALUE, R_MIDDLE, ROW_TILES };
enum RowWord { R_GATE, R_SLOPE, ROW_WORDS };
constexpr int ROW_DISTANCE = ROW_TILES * 512 + ROW_WORDS * 256, ROW_INVERSE = ROW_DISTANCE + 64, ROW_BYTES = ROW_INVERSE + 2 * W * 4;

// The weights in LDS as first operands, a tile of 64 x 8 bytes each (lane 16 g + c: elements (row c, k = 4 j + g), j = 0..3):
// 13 tiles a layer - q, k, v, attention, gate x 3, up x 3, down x 3 - and the head's 16; and every RMSNorm scale in fp32.
// The order of a tile's rows makes the product's layout: row c of a feed tile is the matrix's row 4 (c % 4) + c / 4.
// Operands of dX = dY W (rows = inputs, k = outputs) are read from the same tiles with the transposing load, in feed
// layout; the attention projection's, which are wanted in head layout, are staged a second time, behind the head's.  Then
// comes the embedding as it is, so that a token's row is no further trip to memory behind the token's own; behind the first
// layer, which no wave passes before all have read theirs, its place is the teams' for the sums of the softmax.  Last, for
// each team, what its waves hand one another and, where they fit, the rows that the backward pass wants.
constexpr int LAYER_TILES = 13, HEAD_TILES = 16;
constexpr int staged_tiles(int depth) { return depth * (LAYER_TILES + 1) + HEAD_TILES; }
constexpr size_t embedding_at(int depth) { return size_t(staged_tiles(depth)) * 512 + size_t(2 * depth + 1) * W * 4; }
constexpr int EXCHANGE_BYTES = 16 * 1024 + 2 * ROLES * W * 4; // tiles, and a maximum and a picked logit of every role and token
constexpr size_t teams_at(int depth, int teams) {
    return embedding_at(depth) + (teams * 4096 > V * W * 2 ? teams * 4096 : V * W * 2);
}
constexpr size_t team_bytes(int depth, bool rows) { return EXCHANGE_BYTES + (rows ? depth * ROW_BYTES : 0); }
constexpr size_t lds_bytes(int depth, int teams, bool rows) { return teams_at(depth, teams) + teams * team_bytes(depth, rows); }
constexpr size_t lone_lds_bytes(int depth) { return embedding_at(depth) + V * W * 2; }
constexpr size_t LDS_BYTES = 160 * 1024;

// How a pass over `waves` teams in each of `count` batches is launched: the fewest teams a block that need no more than `places` blocks.
struct Teams {
    int teams, blocks, roles; // teams of a block
    size_t lds;
    bool rows; // stay in LDS
};
inline Teams teams_of(int waves, int count, int depth, int roles, bool rows, int places) {
    const auto lds = [&](int teams) { return roles == 1 ? lone_lds_bytes(depth) : lds_bytes(depth, teams, rows); };
    int teams = 1;
    while ((teams + 1) * roles <= block_waves(roles) && (waves + teams - 1) / teams * count > places && lds(teams + 1) <= LDS_BYTES)
        ++teams;
    return {teams, (waves + teams - 1) / teams, roles, lds(teams), rows};
}
// Lone waves with the units to themselves.  Two blocks fit a unit, and the next one starts where one ends: every block has the same share, as
// few blocks a unit as that takes, so that no unit has one more than another.  us forward, eight a block and so: depth 8, 73728 tokens (18 lone waves
// a unit, six a block) 120, 102; depth 4, context 5, 131072 (34, seven) 131, 118; depth 1 65536 (17, six) 59, 50; a step at depth 8: 40960 267, 231;
// 73728 424, 399.  With gradient and backward blocks of six are the slowest for their number (three waves a SIMD, two of them on one): at 10
// to 12 a unit three blocks of four, 49152 tokens at depth 8 102, 93 and 179, 173, a step 286, 269; depth 4 69, 61 and 105, 101, 162, 149; forward 81, 83.
inline Teams lone_teams(int waves, int depth, bool gradient, int units) {
    const bool of_four = gradient && waves > 10 * units && waves <= 12 * units;
    return teams_of(waves, 1, depth, 1, false, (of_four ? 3 : (waves + 8 * units - 1) / (8 * units)) * units);
}
// Teams of four waves while every one has a place on the units at once, with its rows in LDS where they fit.  Beyond that a lone wave
// does less in all: no handing over, two waves' arithmetic side by side on a SIMD.  us a step, teams and lone waves: 640 teams at depth 8
// (context 4) 87 and 106, 1280 (context 8) 171 and 145.  Where there are other batches a block takes four lone waves (K = 4, 640
// teams: 3, 4, 5, 8 a block 62, 59, 68, 67 us).
// `flying` such launches run side by side, on streams of their own, and a unit has room for one block of teams: they are cut so that all of
// them fit, their rows left out of LDS for more teams a block, and one's tail is another's start, so that teams are the better form for
// longer.  Depth 8, 64 blocks of four teams (256 teams a batch), calls of one step, us a step with one, two (rows in LDS) and four teams a block
// and on lone waves: two flying 54.8, 41.4, 44.6, 52; three 43.8, 31, 32.5, 38; four 45, 31, 31.5, 36.  96 blocks, one to four teams
// without rows, lone waves: two 65.5, 50.8, 47.8, 48.9, 57; four 63, 43.5, 37.7, 32.0, 40.3.  Two a block with rows may be an eighth too many
// (two flying, 72 blocks 42.7, three without 46.9).  Lone waves take over at some 220, 190 and 160 blocks, four teams a block against
// them: two flying 200 66.9, 70.0; 240 83.6, 80.2; three 180 61.8, 65.0; 200 70.8, 69.0; four 144 49.0, 51.4; 180 60.8, 59.8.  At depth 4 the lines
// lie further out, by differences of a tenth at most.
constexpr int STEP_TEAMS = 4; // of a unit
inline Teams step_teams(int waves, int count, int depth, int flying, int units, bool rows_in_lds = true) {
    for (const bool rows : {true, false}) {
        if (rows && !rows_in_lds)
            continue;
        if (flying > 1 ? waves * count * (flying + 2) > 14 * units : waves * count > STEP_TEAMS * units)
            break;
        const int places = flying > 1 ? (rows ? units * 9 / 8 : units) / flying : units;
        const Teams t = teams_of(waves, count, depth, ROLES, rows, places);
        if (t.blocks * count <= places || (flying > 1 && !rows))
            return t;
    }
    return count * flying > 1 ? teams_of(waves, count, depth, 1, false, (waves + 3) / 4 * count) : lone_teams(waves, depth, true, units);
}
// Whether the batches of a call of `steps` steps, K of them in flight, share their launches: by the lesser of two estimated times in
// us, for batches of `blocks` blocks of four teams' tokens at depth 4 or 8.  A shared launch's batches and their optimizer steps go as one
// (a launch's time, 4 us a batch, and the blocks of all of them in one, two or more rounds on the units), but the next launch stands
// behind it.  On streams a step costs the host 34 us, hides behind as many others as there are hardware queues (`flying`), and with those fills
// the units.  The constants are a fit to K = 2 to 16, calls of 1 to 32 steps and 1 to 512 blocks, 1372 points: the choice is within 0.3 % of
// the better one (geometric mean; beyond 10 % at six).  us a step, streams and shared:
//   depth 8, 1 block, calls of K: K = 2 35, 29; 3 34, 20; 4 34, 17; calls of one at K = 4 34, 54; of five 34, 25
//   depth 8, K = 4, calls of four: 96 blocks 35, 39; 128 42, 45   K = 2, calls of two: 96 48, 44; 128 52, 48; 160 59, 71
//   depth 4, 1 block, calls of K: K = 2 33, 20; 4 33, 12   K = 4, calls of four: 128 blocks 34, 27; 160 34, 34   calls of two: 40 34, 25; 160 33, 46
// A batch that fills three quarters of the units by itself stays on streams (depth 4, K = 8, 200 blocks 41, 42; depth 8 65, 70).
inline bool shares_launches(int depth, int K, int flying, int blocks, int steps, int units) {
    if (K == 1)
        return true;
    if (blocks > units * 3 / 4)
        return false;
    const double share = double(blocks) / units; // of the units that one batch fills
    const auto together = [&](int n) {
        const double all = n * share;
        const double time = depth == 4 ? (all <= 1 ? 34 + 26 * all : all <= 2 ? 66 + 17 * all : 54 + 33 * all)
                                       : (all <= 1 ? 50 + 44 * all : all <= 2 ? 95 + 33 * all : 80 + 64 * all);
        return time + 4 * n;
    };
    const double alone = depth == 4 ? std::max((26 + 84 * share) / flying, 46 * share) : std::max((62 + 90 * share) / flying, 82 * share);
    return steps / K * together(K) + (steps % K ? together(steps % K) : 0.) < steps * std::max(34., alone);
}
// The forward and the backward pass as launches of their own: by the same rule, and both alike, as a lone wave leaves its
// features' rows to the backward pass.  us forward, with gradient, and backward with the weight gradients at depth 8, context 8, teams;
// lone waves: 16384 tokens 35, 39, 70; (older kernels) 39, 44, 75   20480 66, 71, 107; 46, 57, 87   131072 258, 276, 549; 156, 222, 442
inline Teams pass_teams(int waves, int depth, bool gradient, int units) {
    const Teams t = step_teams(waves, 1, depth, 1, units, false);
    return t.roles > 1 ? t : lone_teams(waves, depth, gradient, units);
}

} // namespace w16
