// speedy_workspace.hpp -- how a call's workspace (include/speedy_abi.h) is laid out, and
// the tags of the words that workgroups exchange inside a launch.  Host code (the
// constexpr functions also run on the GPU).
//
//   0                words: [0] generation, [1] error, from kArrivedWord the members'
//                    counts of arrived blocks (zero between calls)
//   kHeaderBytes     tagged words of the single launch: level bits, then partials of the
//                    parameter gradients
//   from there on    last_s[nmember], level-set chunk words, parameter and budget
//                    partials, a single call's argument block: places by the grid
//
// A workspace serves calls on several grids, and a block of the single launch takes a
// word for this call's by its tag alone.  So the tagged words lie where no grid's layout
// has anything else: a word there is zero, or was written with the generation of its own
// call, and a generation comes back only after 2^32 - 1 single launches.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace speedy {

constexpr int kBlock = 256;                  // columns of a workgroup
constexpr int kParamParts = 5;               // floats of a parameter partial
constexpr int kBudParts = 7;                 // doubles of a budget partial: the budgets and the weight sum
constexpr uint32_t kArrivedWord = 2, kMergedMembers = 62;
// Blocks of a single launch at most: its kernels take more than 170 registers a lane, so
// a CU holds two workgroups, and the GPU has 256 CUs.
constexpr uint32_t kFusedBlocks = 512;

constexpr size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

constexpr size_t kHeaderBytes = 256;
constexpr size_t kWordBytes = sizeof(uint64_t) * 2 * kFusedBlocks;                    // two members a block
constexpr size_t kTagBytes = kWordBytes + sizeof(uint64_t) * 2 * kFusedBlocks * kParamParts;
static_assert(kHeaderBytes >= sizeof(uint32_t) * (kArrivedWord + kMergedMembers), "header");

// Generations run from 0 to 2^32 - 2; a call's tag is never that of a zeroed word.
constexpr uint32_t call_tag(uint32_t gen) { return gen + 1u; }
constexpr uint32_t next_generation(uint32_t gen) { return gen + 2u == 0u ? 0u : gen + 1u; }
constexpr uint64_t tagged_word(uint32_t tag, uint32_t value) { return (uint64_t)tag << 32 | value; }

// Polls of a wait inside a launch, for the whole of it, before the call gives up and sets
// the error word: about a minute, nearly all of them 4 us apart.  Other work may hold the
// GPU that long before a call's last block runs; a wait that lasts longer waits for a word
// that cannot come (calls that overlap on one workspace).
constexpr uint32_t kSpinLimit = 1u << 24;
constexpr uint32_t kShortPolls = 256;   // the first ones: about 1 us apart

// The N words w[i] = load(i), all read again until each carries `tag`.  Takes its polls from
// `left`; with none left it reads them once and returns false where one has not come.
template <int N, typename Load, typename Pause>
constexpr bool await_words(uint32_t tag, uint32_t& left, Load load, Pause pause, uint64_t (&w)[N]) {
  for (;;) {
    for (int i = 0; i < N; ++i) w[i] = load(i);
    uint32_t stale = 0u;
    for (int i = 0; i < N; ++i) stale |= (uint32_t)(w[i] >> 32) ^ tag;
    if (!stale) return true;
    if (left == 0u) return false;
    pause(kSpinLimit - left-- < kShortPolls);
  }
}

struct Grid {
  uint32_t ncol, ntot, nblk, ls_blocks, chunk, jmax;
};

inline Grid make_grid(int64_t nlon, int64_t nlat, int64_t nmember) {
  Grid g;
  g.ncol = (uint32_t)(nlon * nlat);
  g.ntot = (uint32_t)(nlon * nlat * nmember);
  g.nblk = (g.ntot + kBlock - 1) / kBlock;
  // At most 512 level-set chunks, two workgroups a CU: more make the gather of a
  // member's chunk words longer than they make the level-set pass shorter, and at T425
  // 256 chunks take that pass from 25 to 33 us.
  const uint32_t lsb = g.nblk < 512u ? g.nblk : 512u;
  g.chunk = ((g.ntot + lsb - 1) / lsb + kBlock - 1) / kBlock * kBlock;
  g.ls_blocks = (g.ntot + g.chunk - 1) / g.chunk;
  g.jmax = (g.chunk - 1) / g.ncol + 2;
  return g;
}

struct WsLayout {
  size_t last_s, partial, prm, bud, desc, total;
};

// tag_bytes: kTagBytes, or 0 for a workspace that single launches never use.
inline WsLayout ws_layout(const Grid& g, int32_t nmember, size_t desc_bytes, size_t tag_bytes = kTagBytes) {
  const bool wide = g.ncol >= (uint32_t)kBlock;
  WsLayout L;
  L.last_s = kHeaderBytes + tag_bytes;
  L.partial = L.last_s + align256(sizeof(uint32_t) * (size_t)nmember);
  L.prm = L.partial + align256(sizeof(uint32_t) * (size_t)g.ls_blocks * g.jmax);
  const size_t nprm = wide ? (size_t)g.nblk * 2 : (size_t)g.ntot;        // block and member slot, or column
  L.bud = L.prm + align256(sizeof(float) * kParamParts * nprm);
  const size_t nbud = wide ? (size_t)g.nblk + nmember : (size_t)g.ntot;  // block plus member, or column
  L.desc = L.bud + align256(sizeof(double) * kBudParts * nbud);
  L.total = L.desc + align256(desc_bytes);
  return L;
}

}  // namespace speedy
