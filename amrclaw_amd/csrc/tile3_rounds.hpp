// tile3_rounds.hpp -- the schedule of a sweep of the fused 3-D step
// (sweep3_tile.hpp) over the lines of a tile, on the host and the device.
#pragma once

namespace amrgpu {

// The schedule of a sweep over the (tq + 2) (tp + 2) lines through a tile and
// around it, in the order in which the shorter of the two axes across them runs
// fastest: chunks of 64 / (tr + 1) lines, dealt to the waves in blocks, one chunk
// a wave and round (wave w takes chunk w rounds + r in round r).  A line's
// increments reach the cells within one line of it, so two lines at least 2 n + 3
// apart in the order (n: the length of the fast axis) touch no cell of each
// other.  If that holds between the chunks of neighbouring waves, four waves add
// at once; if between those of waves two apart, in two phases, waves 0 and 2
// before 1 and 3; else (tiles of 4 cells and less) two waves work, one after the
// other.
struct Tile3Rounds {
    int rounds, waves, phases;
};
constexpr Tile3Rounds tile3_rounds(int tr, int tq, int tp) {
    const int lpw = 64 / (tr + 1), n = (tq < tp ? tq : tp) + 2;
    const int chunks = ((tq + 2) * (tp + 2) + lpw - 1) / lpw;
    const int four = (chunks + 3) / 4;
    if ((four - 1) * lpw + 1 >= 2 * n + 3) return {four, 4, 1};
    if ((2 * four - 1) * lpw + 1 >= 2 * n + 3) return {four, 4, 2};
    return {(chunks + 1) / 2, 2, 2};
}

}  // namespace amrgpu
