// Which kernel takes a problem, and what its loads may name: whole-number rules that host and device
// code share and a plain C++ compiler takes too, so that tests run them without a GPU.
#pragma once

#include <stdint.h>

namespace nc {

// The piece a prefetch of piece `at` of a table block of `pieces` reads: past the block's end its last
// one again (never used). A buffer load does not check its scalar offset against the buffer's size, so
// the index itself has to stay in the block, which may be the last of its allocation.
constexpr int head_piece(int at, int pieces) { return at < pieces ? at : pieces - 1; }

}  // namespace nc
