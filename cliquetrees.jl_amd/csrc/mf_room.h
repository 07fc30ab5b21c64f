// mf_room.h — the order in which a solve takes its workspaces, apart from the
// allocations themselves, so that it can be run on the host against a memory
// that is too small.
#pragma once

#include <algorithm>
#include <cstdint>

namespace mf {

// Columns of a block of the blocked solves, and a count of columns in whole blocks.
constexpr int64_t ROOM_BLOCK = 16;
inline int64_t whole_blocks(int64_t cols) { return (cols + ROOM_BLOCK - 1) / ROOM_BLOCK * ROOM_BLOCK; }

// Workspaces of a solve of nrhs columns, of which `few` at a time need no room.
//   need()   what no form does without (the permuted columns and a staging copy)
//   room(c)  update vectors and solutions for c columns, a multiple of ROOM_BLOCK
//   small()  update vectors for min(nrhs, few) columns
//   drop()   gives back what room and small hold
// Room for all columns if it is there, else for half of them, a quarter, and so
// on, else none: what fails is given back before less is tried, so a solve that
// fits without room is never refused for it.  False: not even that fits.
template <typename Need, typename Room, typename Small, typename Drop>
bool take_room(int64_t nrhs, int64_t few, Need need, Room room, Small small, Drop drop) {
    if (!need()) {
        drop();
        if (!need()) return false;
    }
    for (int64_t c = nrhs > few ? whole_blocks(nrhs) : 0; c > 0; c = c > ROOM_BLOCK ? whole_blocks(c / 2) : 0) {
        if (room(c)) return true;
        drop();
    }
    if (small()) return true;
    drop();
    return small();
}

}  // namespace mf
