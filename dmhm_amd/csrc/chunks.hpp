// The inner chunks of a tile's contributions as one wave of the MFMA tile
// kernel walks them; plain index arithmetic, shared with host code.
#pragma once
#include <cstdint>
#include "hostdev.hpp"

namespace dmhm {

// Where a wave is: chunk p (inner indices p .. p + 15) of a contribution of
// inner dimension q. With byChunk the S waves of a workgroup are dealt the
// chunks of all contributions in turn; wave w takes every S-th one, and `turn`
// counts the chunks dealt.
template <int S>
struct ChunkWalk {
    int w;
    bool byChunk;
    int turn = 0;
    int q = 0, p = 0;

    // Starts over (turn goes on: the next contributions are dealt after these).
    DMHM_HD void start() { q = p = 0; }

    // Moves to the wave's next whole chunk (p + 16 <= q; TAIL: next remainder,
    // p < q) among the contributions in `left`, of inner dimension dim(i); a
    // contribution without one is passed over. enter(i) is called when the
    // chunk lies in contribution i and the one before did not. False at the
    // end, with q, p and what enter() set still those of the last chunk: it is
    // fetched once more, and its offset is in bounds for its own contribution
    // only.
    template <bool TAIL, typename Dim, typename Enter>
    DMHM_HD bool next(uint64_t& left, Dim dim, Enter enter)
    {
        int n = p + (S > 1 && byChunk ? 16 * S : 16);
        if (TAIL || n + 16 > q) {
            int i, nq;
            bool none = false;
            do {
                if (left == 0) return false;
                i = __builtin_ctzll(left);
                left &= left - 1;
                nq = dim(i);
                n = TAIL ? nq & ~15 : 0;
                if (S > 1 && byChunk) {
                    const int mine = (w - turn) & (S - 1);      // chunks dealt before this wave's first one
                    turn += TAIL ? 1 : nq >> 4;
                    none = TAIL ? mine != 0 : 16 * mine + 16 > nq;
                    if (!TAIL) n = 16 * mine;
                }
            } while (none);
            q = nq;
            enter(i);
        }
        p = n;
        return true;
    }
};

} // namespace dmhm
