// ixt_rounds.h -- blocks of a launch and the rounds in which they go through the chip, a block a CU.
#pragma once

#define IXT_CUS 256
// Of `tiles` tiles of `heads` blocks each: as many lie behind the last whole round, in whole units of `unit` tiles unless it is all of them.  Rounded up: what stays in front is whole rounds at most.
constexpr int tiles_behind_rounds(int tiles, int heads, int unit) {
  const int left = (int)((long)tiles * heads % IXT_CUS), need = (left + heads - 1) / heads, over = (need + unit - 1) / unit * unit;
  return over < tiles ? over : tiles;
}
// Prompt attention, heads of 128, more than 1024 keys (mtile_attn_t): so many tiles go by scores ahead and two blocks a value.  All of them where they are half a round at most: 264 launches of 2 to 40 kv
// heads, 64 to 500 rows and 1100 to 2040 keys, 0.70 to 0.97 of the time.  Else those behind the last whole round, half of one at most, where their rows, the call's first, have 2560 keys in front of them:
// 115 launches 0.94 of the time in the mean, the worst one 1.006.  With fewer the round that falls away is cheaper than the two launches: 16 heads, us, 296 rows at <= 1100 keys 61 -> 75, 828 at <= 1500
// 137 -> 146 and at <= 2300 210 -> 213; at <= 3064 / 3900 282 -> 274 and 393 -> 374.
constexpr int tiles_split(int tiles, int heads, int unit, int keys_in_front) {
  const int over = tiles_behind_rounds(tiles, heads, unit);
  return (long)over * heads <= IXT_CUS / 2 && (over == tiles || keys_in_front >= 2560) ? over : 0;
}
