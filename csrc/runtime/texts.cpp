// Packed texts laid out for an encoder (host C++ runtime).
#include <cstdint>
#include <cstring>

#define CFC_API extern "C" __attribute__((visibility("default")))

// What an encoder reads of n texts that lie side by side, text i at ids [cu[i], cu[i + 1]): the ids, their positions, where
// each text starts, and the text and first row of every tile of `tile` rows.  Five arrays in `out` (room for `room` values),
// each starting at a multiple of four.  sizes: tiles, the longest text.  One pass here takes the place of some twenty array
// operations of a microsecond each, which a short text waited for.  -1: starts that fall or lie outside the ids, or no room.
CFC_API int cfc_pack_texts(const int32_t* ids, int64_t n_ids, const int64_t* cu, int64_t n, int tile, int32_t* out,
                           int64_t room, int64_t* sizes) {
  if (n < 1 || tile < 1 || cu[0] < 0 || cu[n] > n_ids) return -1;
  const auto up = [](int64_t v) { return (v + 3) / 4 * 4; };
  int64_t tiles = 0, longest = 0;
  for (int64_t i = 0; i < n; ++i) {
    const int64_t len = cu[i + 1] - cu[i];
    if (len < 0 || cu[i + 1] > n_ids) return -1;
    tiles += (len + tile - 1) / tile;
    longest = len > longest ? len : longest;
  }
  const int64_t total = cu[n] - cu[0];
  if (total > INT32_MAX || 2 * up(total) + up(n + 1) + 2 * up(tiles) > room) return -1;
  int32_t *pos = out + up(total), *start = pos + up(total), *text = start + up(n + 1), *row = text + up(tiles);
  if (total) std::memcpy(out, ids + cu[0], total * sizeof(int32_t));
  start[0] = 0;
  for (int64_t i = 0; i < n; ++i) {
    const int32_t len = (int32_t)(cu[i + 1] - cu[i]);
    for (int32_t p = 0; p < len; ++p) *pos++ = p;
    start[i + 1] = (int32_t)(cu[i + 1] - cu[0]);
    for (int64_t r = 0; r < len; r += tile) *text++ = (int32_t)i, *row++ = (int32_t)r;
  }
  sizes[0] = tiles;
  sizes[1] = longest;
  return 0;
}
