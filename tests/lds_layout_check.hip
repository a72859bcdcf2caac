// Host-side check of index arithmetic the kernels and launchers share (compiled for the host only and
// run on the CPU by tests/test_lds_layout.py): the workgroup -> (head, tile) mapping with its head
// groups, and the LDS tile layout.  For every padded head dimension it walks all lanes, waves and
// wave-loads of a 64-row tile and verifies that
//   * the slot an LDS-direct load writes is where the fragment readers (swz_off) look for the chunk
//     the loader fetched into it, and every (row, chunk) of the tile is written exactly once;
//   * the loader's shortcut holds: the chunk does not depend on the load index, except with rows of
//     256 halves, where odd loads take the even load's chunk with bit 1 flipped;
//   * both read patterns are free of bank conflicts on 64 banks of 4 bytes: 16 consecutive rows at
//     one logical chunk (ds_read_b128) and 4 consecutive rows x 4 consecutive chunks (transposing read).
#include <cstdio>
#include <set>
#include <vector>

#include "fa2_common.hpp"
#include "fa2_launch.hpp"

template <int DP>
int check() {
  constexpr int ROWS = 64, NW = 4;
  using TL = TileLoader<DP, ROWS, NW, false>;
  constexpr int LP = TL::LP, CPR = TL::CPR, RPL = TL::RPL;
  int bad = 0;
  std::vector<int> seen(ROWS * CPR, 0);
  for (int i = 0; i < TL::LOADS; i++)
    for (int wave = 0; wave < NW; wave++)
      for (int lane = 0; lane < 64; lane++) {
        const int row = i * NW * RPL + wave * RPL + lane / CPR;
        const int chunk = TL::chunk_of(lane, wave, i);
        const int written = ((i * NW + wave) * 1024 + 16 * lane) / 2;  // element offset of the slot
        if (row >= ROWS || chunk < 0 || chunk >= CPR) { bad++; continue; }
        if (written != swz_off<LP>(row, chunk)) bad++;
        seen[row * CPR + chunk]++;
        const int c0 = TL::chunk_of(lane, wave, 0);
        if (chunk != ((TL::BY_PARITY && (i & 1)) ? (c0 ^ 2) : c0)) bad++;
      }
  for (int v : seen) bad += v != 1;
  auto banks_distinct = [&](const std::vector<int> &slot_offsets) {  // 16-byte slots, element offsets
    std::set<int> banks;
    for (int off : slot_offsets)
      for (int w = 0; w < 4; w++) banks.insert(((off * 2) / 4 + w) % 64);
    return banks.size() == slot_offsets.size() * 4;
  };
  for (int r0 = 0; r0 < ROWS; r0 += 16)
    for (int c = 0; c < CPR; c++) {
      std::vector<int> offs;
      for (int j = 0; j < 16; j++) offs.push_back(swz_off<LP>(r0 + j, c));
      bad += !banks_distinct(offs);
    }
  for (int r0 = 0; r0 < ROWS; r0 += 4)
    for (int c0 = 0; c0 + 4 <= CPR; c0 += 4) {
      std::vector<int> offs;
      for (int j = 0; j < 4; j++)
        for (int c = 0; c < 4; c++) offs.push_back(swz_off<LP>(r0 + j, c0 + c));
      bad += !banks_distinct(offs);
    }
  printf("DP %3d: row pitch %3d, %2d slots per row, %d wave-loads per wave, by parity %d: %s\n", DP, LP, CPR, TL::LOADS,
         (int)TL::BY_PARITY, bad ? "FAILED" : "ok");
  return bad;
}

// Workgroup index -> (head, tile rank) with the head groups the launchers compute: every pair is
// visited exactly once, ranks never decrease inside a group (heaviest tile first), group sizes are
// multiples of 8, and with a head count that is a multiple of 8 all workgroups of a head have the
// same index modulo 8, that is, land on one XCD.
int check_mapping() {
  int bad = 0, cases = 0;
  for (int table_group : {32, 64})
    for (int heads : {1, 3, 8, 16, 24, 33, 48, 63, 64, 72, 80, 96, 100, 128, 129, 192, 2048})
      for (int tiles : {1, 2, 7, 32}) {
        const int group = fa2::equal_head_groups(table_group, heads);
        if (group % 8 != 0 || group < 8) bad++;
        if (heads >= 2 * table_group && group > 2 * table_group) bad++;  // groups stay near the table's size
        std::vector<int> seen(heads * tiles, 0), xcd(heads, -1);
        int last_rank = 0, last_group = -1;
        for (int i = 0; i < heads * tiles; i++) {
          int bh = -1, rank = -1;
          fa2::map_workgroup(i, heads, tiles, group, bh, rank);
          if (bh < 0 || bh >= heads || rank < 0 || rank >= tiles) { bad++; continue; }
          seen[bh * tiles + rank]++;
          const int g = bh / group;
          if (g == last_group && rank < last_rank) bad++;
          if (g < last_group) bad++;  // groups are walked in order
          last_group = g;
          last_rank = rank;
          if (heads % 8 == 0) {
            if (xcd[bh] < 0) xcd[bh] = i % 8;
            else if (xcd[bh] != i % 8) bad++;
          }
        }
        for (int v : seen) bad += v != 1;
        cases++;
      }
  printf("workgroup mapping, %d cases: %s\n", cases, bad ? "FAILED" : "ok");
  return bad;
}

// balanced_index on every grid of up to four rounds: a permutation of the grid that keeps a workgroup's index modulo 8
// (the XCD a head stays on) and its round, and walks the second and fourth round backwards.
int check_balanced_index() {
  int bad = 0;
  for (int total = 1; total <= 4 * fa2::kCUs; total++) {
    std::vector<int> seen(total, 0);
    for (int i = 0; i < total; i++) {
      const int j = fa2::balanced_index(i, total);
      if (j < 0 || j >= total) { bad++; continue; }
      seen[j]++;
      bad += j % 8 != i % 8 || j / fa2::kCUs != i / fa2::kCUs;
      if (!(i / fa2::kCUs & 1)) bad += j != i;
    }
    for (int v : seen) bad += v != 1;
    for (int base = fa2::kCUs; base + 16 <= total; base += 2 * fa2::kCUs)  // its first steps take its last tiles
      bad += fa2::balanced_index(base, total) <= fa2::balanced_index(base + 8, total);
  }
  printf("balanced index, %d grids: %s\n", 4 * fa2::kCUs, bad ? "FAILED" : "ok");
  return bad;
}

// Grids that are reordered by balanced_index are ordered heaviest tile first as a whole, and a head stays on its XCD where
// the heads divide by 8.
int check_resident_walk() {
  int bad = 0, walked = 0;
  for (int group : {32, 64})
    for (int heads = 1; heads <= 4 * fa2::kCUs; heads++)
      for (int tiles = 1; tiles * heads <= 4 * fa2::kCUs; tiles++) {
        const fa2::ResidentWalk walk = fa2::resident_walk(group, heads);
        if (!walk.balanced) {
          bad += heads % 8 == 0 || heads < 2 * group;
          continue;
        }
        walked++;
        int last = 0;
        for (int i = 0; i < tiles * heads; i++) {
          int bh, rank;
          fa2::map_workgroup(i, heads, tiles, walk.head_group, bh, rank);
          bad += rank < last || bh < 0 || bh >= heads || rank >= tiles || (heads % 8 == 0 && bh % 8 != i % 8);
          last = rank;
        }
      }
  printf("resident walk, %d grids: %s\n", walked, bad ? "FAILED" : "ok");
  return bad;
}

// The paired dK/dV kernel has twice the workgroups of the others: it is not picked where only they make a grid
// that can be launched.
int check_launchable_grids() {
  int bad = 0, cases = 0;
  for (int dp : {32, 64, 96, 128, 192, 256})
    for (int seqlen : {1, 64, 65, 128, 129, 4096, 100000})
      for (int64_t wgs : {int64_t(512), int64_t(fa2::kMaxWorkgroups) / 2, int64_t(fa2::kMaxWorkgroups) / 2 + 1, int64_t(fa2::kMaxWorkgroups)}) {
        fa2::BwdParams p{};
        p.headdim = dp;
        p.vec = 1;
        p.batch = (int)(wgs / ((seqlen + fa2::kDkvBlockKV - 1) / fa2::kDkvBlockKV));
        p.nheads = 1;
        p.seqlen_q = p.seqlen_k = seqlen;
        if (p.batch == 0) continue;
        const int keys = fa2::dkdv_block_kv(dp, p);
        if ((int64_t)((seqlen + keys - 1) / keys) * p.batch > fa2::kMaxWorkgroups) bad++;
        if (dp == 96 && fa2::dkdv_direct_ok(dp, p)) bad++;  // there is no such kernel
        cases++;
      }
  printf("launchable grids, %d cases: %s\n", cases, bad ? "FAILED" : "ok");
  return bad;
}

// The columns a row's kernels multiply: enough for every head dimension, in one of the counts printed here.
int check_columns() {
  int bad = 0, below = 0;
  for (int dp : {32, 64, 96, 128, 192, 256}) {
    std::set<int> counts;
    for (int d = 8; d <= dp; d += 8) {
      const int cols = fa2::direct_columns(dp, d);
      if (cols < d || cols > dp || cols % 16) bad++;
      if (d > below) counts.insert(cols);  // (smaller ones come to this row only by its id)
      else if (cols != fa2::direct_columns(dp, below + 8)) bad++;
    }
    printf("columns %d:", dp);
    for (int c : counts) printf(" %d", c);
    printf("\n");
    below = dp;
  }
  return bad;
}

int main() {
  int bad = check_mapping();
  bad += check_balanced_index();
  bad += check_resident_walk();
  bad += check_launchable_grids();
  bad += check_columns();
  bad += check<32>();
  bad += check<64>();
  bad += check<96>();
  bad += check<128>();
  bad += check<192>();
  bad += check<256>();
  return bad ? 1 : 0;
}
