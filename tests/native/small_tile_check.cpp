/* Walks the LDS staging of the small-output GEMM's result tile
 * (flashvsr-sm89-ops_amd/csrc/small_tile.h): every row must lie within the
 * array of its slot, no two rows may share a byte, and the 32 rows that a wave
 * writes at a time must share a slot.  With ONE_SLOT defined all rows are placed
 * in slot 0, one behind the other, which must be reported.  Prints the rows
 * out of place per tile; exit status 1 if there are any. */
#include <cstdio>
#include <vector>

#include "../../flashvsr-sm89-ops_amd/csrc/small_tile.h"

template <class T, int S>
int check(const char* name) {
  std::vector<std::vector<char>> lds(S, std::vector<char>(T::kSlotBytes));
  int bad = 0;
  for (int r = 0; r < T::TM; ++r) {
#ifdef ONE_SLOT
    const int slot = 0, off = r * T::kRowBytes;
#else
    const int slot = T::stage_slot(r), off = T::stage_offset(r);
    bad += slot != T::stage_slot(r / 32 * 32);
#endif
    if (slot < 0 || slot >= S || off < 0 || off + T::kRowBytes > T::kSlotBytes) {
      ++bad;
      continue;
    }
    for (int b = 0; b < T::kRowBytes; ++b) bad += lds[slot][off + b]++ != 0;
  }
  std::printf("%s %d\n", name, bad);
  return bad;
}

int main() {
  return (check<SmallTile<1, 1, 4>, 4>("64x64") + check<SmallTile<1, 2, 3>, 3>("64x128") +
          check<SmallTile<2, 2, 4>, 4>("128x128") + check<SmallTile<2, 4, 3>, 3>("128x256")) != 0;
}
