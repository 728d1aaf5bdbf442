// ixt_tile_attn.hip -- launches of k_attn_mtile (an object of its own: it compiles beside the others).
#include "ixt_rounds.h"
#include "ixt_tile_attn.h"

#include <algorithm>

template <int HD, int GQ, int NW, int NR, bool GIVEN = false, int VW = mtile_width(HD)>
static void mtile_launch(const dim3& grid, const TileAttnArgs& ta, hipStream_t st) {
  constexpr size_t lds = mtile_lds(HD, NW, NR, VW);
  if (lds_room<&k_attn_mtile<HD, GQ, NW, NR, GIVEN, VW>>(lds) != hipSuccess) return;  // (the runtime's last error, which the caller looks at)
  hipLaunchKernelGGL((k_attn_mtile<HD, GQ, NW, NR, GIVEN, VW>), grid, dim3(NW * 64), lds, st, ta);
}
// rows of one page group whose blocks leave half of the CUs idle: the scores by a launch of their own on all CUs, a value's columns by several blocks
template <int HD, int GQ, int VW>
static void mtile_split_t(const dim3& grid, const TileAttnArgs& ta, hipStream_t st) {
  hipLaunchKernelGGL((k_attn_mscores<HD, GQ>), dim3(grid.x, grid.y, std::min(8, std::max(2, 256 / (int)(grid.x * grid.y)))), dim3(512), 0, st, ta);
  if (ta.lmax <= 1024) mtile_launch<HD, GQ, 8, 1, true, VW>(grid, ta, st);
  else if (ta.lmax <= 2048) mtile_launch<HD, GQ, 8, 2, true, VW>(grid, ta, st);
  else if (ta.lmax <= 3072) mtile_launch<HD, GQ, 8, 3, true, VW>(grid, ta, st);
  else mtile_launch<HD, GQ, 8, 4, true, VW>(grid, ta, st);
}
// The smallest form that holds the call's longest prefix (ta.lmax keys, at most 4096).
template <int HD, int GQ>
static void mtile_attn_t(TileAttnArgs ta, hipStream_t st) {
  constexpr int TQ = 16 / GQ;
  const int tiles = (ta.R + TQ - 1) / TQ, blocks = ta.g.nkv * tiles;
  // half of the CUs idle: the halves of a value side by side; still half of them: the page groups of a tile, too.  A tile of a prompt has one, and the other blocks
  // end at once (64 and 100 rows: the same time); one of a mixed step's decoded tokens has up to TQ, and one behind the other 64 rows at 128 keys with heads of 256
  // took 2.40 ms a step of four sub-layers (per-vector units: 2.35), dealt out 1.84; 16 heads of 128, four layers: 64 keys 2.45 -> 1.77, 1500 keys 4.50 -> 2.58
  ta.parts = HD > 128 && blocks <= 128 ? HD / 128 : 1;
  dim3 grid(ta.g.nkv, tiles, ta.parts * std::min(TQ, std::max(1, 256 / (blocks * ta.parts))));
  // two blocks a value and rows of one page group: the scores once, by a launch of their own on all CUs (256 rows, 8 heads of 256 on 4, <= 1024 / 2048 / 3072 keys: 45.6,
  // 74.3, 112 us, now 22.0, 33.6, 54.6 and the scores before them, 27.0 in the mean; at <= 512 keys the second launch costs what it gives)
  if constexpr (HD > 128) {
    if (ta.parts > 1 && ta.scores != nullptr && ta.lmax > 512) {
      mtile_split_t<HD, GQ, 128>(grid, ta, st);
      return;
    }
  }
  // Heads of 128, a block a CU (below): what is left behind the last whole round of 256 blocks, at most half of one, goes by two blocks a value and scores ahead, too (tiles_split): the
  // first rows, whose keys are the fewest.  16 heads, us: 100 rows at <= 1124 / 2148 / 3172 keys 44.8 / 69.7 / 100.4, now 25.5 / 39.0 / 61.0 and the scores before them 14.5 / 20.0 / 25.9; 828
  // rows at <= 3900 keys, 3 rounds and 64 blocks, 345, now 281 + 44 + 10.  The other rows by moved pointers: a first row as the kernel's argument spills 36 bytes more, 330 instead of 316.
  if constexpr (HD == 128) {
    constexpr int PER16 = 16 / TQ;                       // tiles of 16 rows, the unit of `out`
    const int over = ta.scores != nullptr && ta.lmax > 1024 ? tiles_split(tiles, ta.g.nkv, PER16, ta.lmax - ta.R) : 0;
    if (over > 0) {
      TileAttnArgs rest = ta;
      rest.parts = 2;
      rest.R = std::min(ta.R, over * TQ);
      mtile_split_t<HD, GQ, 64>(dim3(ta.g.nkv, over, 2), rest, st);
      if (over == tiles) return;
      const int row0 = over * TQ;
      ta.row_slot += row0; ta.row_pos += row0; ta.row_active += row0;
      ta.qbuf += (size_t)row0 * ta.g.nq * HD; ta.out += xidx(row0, 0, ta.g.nq * HD);
      ta.R -= row0;
      grid.y = tiles - over;
    }
  }
  if (ta.lmax <= 256) mtile_launch<HD, GQ, 2, 1>(grid, ta, st);
  else if (ta.lmax <= 512) mtile_launch<HD, GQ, 4, 1>(grid, ta, st);
  // more than one block a CU: two of four waves side by side (256 registers a wave; one block's softmax and exchange under the other's products), else all the waves a CU has room
  // for in one.  16 heads of 128 at <= 1024 keys, us of <8, 1> / <4, 2>: 256 blocks 32.0 / 37.8, 320 61.2 / 57.9, 512 64.0 / 58.1, 1024 105 / 88.  With twice the keys two blocks' scores
  // take every register: level
  else if (ta.lmax <= 1024 && (int)(grid.x * grid.y * ta.parts) > 256) mtile_launch<HD, GQ, 4, 2>(grid, ta, st);
  else if (ta.lmax <= 1024) mtile_launch<HD, GQ, 8, 1>(grid, ta, st);
  else if (ta.lmax <= 2048) mtile_launch<HD, GQ, 8, 2>(grid, ta, st);
  // (the scores of three rounds leave registers that those of four do not: 1024 rows at <= 3072 keys 322 -> 302 us)
  else if (ta.lmax <= 3072) mtile_launch<HD, GQ, 8, 3>(grid, ta, st);
  else mtile_launch<HD, GQ, 8, 4>(grid, ta, st);
}
bool launch_mtile_attn(const TileAttnArgs& ta, int hd, int gq, hipStream_t st) {
#define ATT(HD_, GQ_) if (hd == HD_ && gq == GQ_) { mtile_attn_t<HD_, GQ_>(ta, st); return true; }
  ATT(128, 1) ATT(128, 2) ATT(128, 4) ATT(64, 1) ATT(64, 2) ATT(64, 4) ATT(256, 1) ATT(256, 2) ATT(256, 4)
#undef ATT
  return false;
}
