// workspace_host.cpp -- TEST HARNESS ONLY: the workspace layout and the tags of the
// single launch (jax-gcm_amd/csrc/speedy_workspace.hpp) for the host, so that the CPU
// test suite can check them without a GPU.
#include "../../jax-gcm_amd/csrc/speedy_workspace.hpp"

using namespace speedy;

extern "C" {

// kHeaderBytes, kWordBytes, kTagBytes, kFusedBlocks, kBlock, kParamParts, kBudParts, kArrivedWord, kMergedMembers
void ws_constants(uint64_t* out) {
  const uint64_t c[] = {kHeaderBytes, kWordBytes,  kTagBytes, kFusedBlocks, (uint64_t)kBlock, (uint64_t)kParamParts,
                        (uint64_t)kBudParts, kArrivedWord, kMergedMembers};
  for (uint64_t x : c) *out++ = x;
}

// nblk, ls_blocks, jmax, then WsLayout
void ws_grid(int64_t nlon, int64_t nlat, int32_t nmember, uint64_t desc_bytes, uint64_t tag_bytes, uint64_t* out) {
  const Grid g = make_grid(nlon, nlat, nmember);
  const WsLayout L = ws_layout(g, nmember, desc_bytes, tag_bytes);
  const uint64_t c[] = {g.nblk, g.ls_blocks, g.jmax, L.last_s, L.partial, L.prm, L.bud, L.desc, L.total};
  for (uint64_t x : c) *out++ = x;
}

uint32_t ws_call_tag(uint32_t gen) { return call_tag(gen); }
uint32_t ws_next_generation(uint32_t gen) { return next_generation(gen); }
uint64_t ws_tagged_word(uint32_t tag, uint32_t value) { return tagged_word(tag, value); }


// await_words on three words, the middle one of which carries `tag` from its polls-th
// second read on: {came, reads, short pauses, polls left}
void ws_await(uint32_t tag, uint32_t left, uint64_t polls, uint64_t* out) {
  uint64_t reads = 0, brief = 0, w[3] = {};
  const bool came = await_words(
      tag, left,
      [&](int i) {
        if (i == 0) ++reads;
        return tagged_word(i == 1 && reads <= polls ? tag - 1u : tag, 7u);
      },
      [&](bool b) { brief += b; }, w);
  out[0] = came; out[1] = reads; out[2] = brief; out[3] = left;
}
uint32_t ws_spin_limit() { return kSpinLimit; }

}  // extern "C"
