// stubs.h -- a HIP runtime and kernel launchers in host memory, to run
// bsattn_capi.cpp (the page pool, the metadata and the launch order) without
// a GPU.  "Device" memory is the host's; a launch that patches the metadata
// applies its patches, the others do nothing.  launches_left makes a launch
// fail.
#pragma once

#include <hip/hip_runtime_api.h>
#include <stdint.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

#include "../../include/bsattn.h"
#include "../../mlx-swift-lm_amd/csrc/bsattn_internal.h"

namespace stub {
inline int launches_left = -1;  // launches that succeed before the next one fails (-1: all)
inline bool applies = false;    // whether the failing launch still writes the metadata
inline bsattn::Geometry last{};     // geometry of the last launch

// events: `done` says whether the work before the last record has finished
struct Event {
  bool done = true;
  int records = 0;
};
inline std::vector<std::pair<hipStream_t, Event*>> waits;  // hipStreamWaitEvent on unfinished work
inline hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
inline std::map<void*, size_t> memory;                     // device allocations
inline size_t memory_limit = SIZE_MAX;                     // largest allocation that succeeds
struct Prefill {
  float* ws;
  Event* done;
  int nsplit;
};
inline std::vector<Prefill> prefills;
inline int splits = 1;  // what prefill_splits answers
inline std::mutex mu;

// one launch: its patches, and whether it fails
inline hipError_t run(const bsattn::Geometry& g, const bsattn::PatchBatch* pb) {
  last = g;
  const bool fails = launches_left == 0;
  if (launches_left >= 0) --launches_left;
  if (pb && (!fails || applies))
    for (int i = 0; i < pb->n; ++i) g.meta[pb->idx[i]] = pb->val[i];
  return fails ? hipErrorLaunchFailure : hipSuccess;
}
}  // namespace stub

#define CHECK(cond)                                                     \
  do {                                                                  \
    if (!(cond)) {                                                      \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #cond);            \
      std::exit(1);                                                     \
    }                                                                   \
  } while (0)

// the device's length, capacity and block table of a sequence are the host's
inline void check_meta(bsattn_cache* c, int seq, int len) {
  const bsattn::Geometry& g = stub::last;
  int32_t host_len = -1, n = 0, pages[4096];
  CHECK(bsattn_seq_len(c, seq, &host_len) == BSATTN_OK && host_len == len);
  CHECK(bsattn_seq_pages(c, seq, pages, 4096, &n) == BSATTN_OK);
  CHECK(g.meta[seq] == len);
  CHECK(g.meta[g.cap_off + seq] == n * g.tb);
  for (int i = 0; i < n; ++i) CHECK(g.meta[g.bt_off + seq * g.mbps + i] == pages[i]);
}

inline bsattn_desc small_desc(int seqs, int blocks) {
  bsattn_desc d{};
  d.max_seqs = seqs;
  d.num_q_heads = 8;
  d.num_kv_heads = 2;
  d.head_dim = 128;
  d.block_size = 32;
  d.dtype = BSATTN_F16;
  d.top_k = 4;
  d.sink_blocks = 1;
  d.recent_blocks = 1;
  d.max_blocks_per_seq = blocks;
  return d;
}
