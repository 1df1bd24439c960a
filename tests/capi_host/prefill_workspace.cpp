// prefill_workspace.cpp -- the workspaces of split prefills: a GPU's caches
// share them, no two unfinished calls of different streams write one without
// a wait between them, captured calls have the cache's own, and all are given
// back with the last cache.
#include <thread>

#include "stubs.h"

static uint16_t kv[1];
static const size_t kSpace = (size_t)bsattn::kPrefillRows * (bsattn::kHeadDim + 2) * sizeof(float);

static bsattn_cache* filled() {
  const bsattn_desc d = small_desc(1, 16);
  bsattn_cache* c = nullptr;
  CHECK(bsattn_cache_create(&d, &c) == BSATTN_OK);
  CHECK(bsattn_append(c, kv, kv, nullptr, 1, 40, nullptr) == BSATTN_OK);
  return c;
}
static int prefill(bsattn_cache* c, hipStream_t s) { return bsattn_prefill(c, kv, nullptr, 1, 20, 1.f, kv, s); }
static stub::Prefill call(bsattn_cache* c, hipStream_t s) {
  CHECK(prefill(c, s) == BSATTN_OK);
  return stub::prefills.back();
}
static int spaces() {
  int n = 0;
  for (const auto& m : stub::memory) n += m.second == kSpace;
  return n;
}
static hipStream_t stream(int i) { return (hipStream_t)(uintptr_t)(16 + i); }

int main() {
  std::vector<bsattn_cache*> layers;
  for (int i = 0; i < 6; ++i) layers.push_back(filled());
  // unsplit: no workspace
  CHECK(call(layers[0], nullptr).ws == nullptr && spaces() == 0);
  stub::splits = 4;
  // the layers of a model on one stream: one workspace
  const stub::Prefill first = call(layers[0], stream(0));
  CHECK(first.ws && first.done && first.nsplit == 4 && first.done->records == 1);
  for (bsattn_cache* c : layers) CHECK(call(c, stream(0)).ws == first.ws);
  CHECK(spaces() == 1);
  // another stream while that is under way: another workspace, no wait
  stub::waits.clear();
  const stub::Prefill second = call(layers[1], stream(1));
  CHECK(second.ws != first.ws && second.done != first.done && spaces() == 2 && stub::waits.empty());
  // its own again, and the first one's once that has finished
  CHECK(call(layers[1], stream(1)).ws == second.ws);
  first.done->done = true;
  stub::waits.clear();
  CHECK(call(layers[2], stream(2)).ws == first.ws && spaces() == 2 && stub::waits.empty());
  // (the stream that used it before takes another, or waits)
  CHECK(call(layers[0], stream(0)).ws != first.ws && spaces() == 3);
  // no more than four: the next ones wait on their streams
  CHECK(call(layers[3], stream(3)).ws && spaces() == 4);
  for (int i = 4; i < 12; ++i) {
    stub::waits.clear();
    const stub::Prefill p = call(layers[i % 6], stream(i));
    CHECK(spaces() == 4 && stub::waits.size() == 1);
    CHECK(stub::waits[0] == std::make_pair(stream(i), p.done));
  }
  // a launch that fails part of the way still ends with the event
  for (const auto& p : stub::prefills)
    if (p.done) p.done->done = true;
  stub::launches_left = 0;
  CHECK(prefill(layers[0], stream(40)) == BSATTN_ERR_HIP);
  stub::launches_left = -1;
  CHECK(!stub::prefills.back().done->done);
  // captured: the cache's own, of the call's size, and again the same
  stub::capture = hipStreamCaptureStatusActive;
  const stub::Prefill g0 = call(layers[0], stream(0)), g1 = call(layers[1], stream(0));
  CHECK(g0.ws && g1.ws && g0.ws != g1.ws && !g0.done && g0.nsplit == 4 && spaces() == 4);
  CHECK(stub::memory.at(g0.ws) == 4u * 8 * 20 * (bsattn::kHeadDim + 2) * sizeof(float));
  CHECK(call(layers[0], stream(0)).ws == g0.ws);
  stub::splits = 8;  // (a larger one beside it: the graph keeps its address)
  CHECK(call(layers[0], stream(0)).ws != g0.ws && stub::memory.count(g0.ws) == 1);
  stub::capture = hipStreamCaptureStatusNone;
  for (bsattn_cache* c : layers) bsattn_cache_destroy(c);
  CHECK(stub::memory.empty());
  // no memory: unsplit
  layers = {filled()};
  stub::memory_limit = 1000;
  const stub::Prefill none = call(layers[0], stream(0));
  CHECK(none.ws == nullptr && none.nsplit == 1);
  stub::capture = hipStreamCaptureStatusActive;
  CHECK(call(layers[0], stream(0)).ws == nullptr);
  stub::capture = hipStreamCaptureStatusNone;
  stub::memory_limit = SIZE_MAX;
  // threads, each with its cache and stream
  std::vector<std::thread> th;
  for (int t = 0; t < 8; ++t)
    th.emplace_back([t] {
      for (int i = 0; i < 50; ++i) {
        bsattn_cache* c = nullptr;
        const bsattn_desc d = small_desc(1, 16);
        CHECK(bsattn_cache_create(&d, &c) == BSATTN_OK);
        CHECK(bsattn_append(c, kv, kv, nullptr, 1, 40, stream(t)) == BSATTN_OK);
        for (int k = 0; k < 5; ++k) CHECK(prefill(c, stream(t)) == BSATTN_OK);
        bsattn_cache_destroy(c);
      }
    });
  for (auto& t : th) t.join();
  CHECK(spaces() <= 4);
  bsattn_cache_destroy(layers[0]);
  CHECK(stub::memory.empty());
  std::puts("ok");
  return 0;
}
