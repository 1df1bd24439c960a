// failed_launch.cpp -- a launch that fails leaves the cache as it was, and the
// device's lengths, capacities and block tables follow the host's from the
// next call on: an append that is tried again, and the decode after it, see
// every page the host holds.
#include <algorithm>

#include "stubs.h"

static uint16_t kv[1];

static bsattn_cache* filled(int seqs, int blocks, int len) {
  const bsattn_desc d = small_desc(seqs, blocks);
  bsattn_cache* c = nullptr;
  CHECK(bsattn_cache_create(&d, &c) == BSATTN_OK);
  CHECK(bsattn_append(c, kv, kv, nullptr, seqs, len, nullptr) == BSATTN_OK);
  for (int s = 0; s < seqs; ++s) check_meta(c, s, len);
  return c;
}

static int decode(bsattn_cache* c, int n) { return bsattn_decode(c, kv, nullptr, n, 1.f, kv, nullptr, nullptr); }
static int append_decode(bsattn_cache* c, int n) {
  return bsattn_append_decode(c, kv, kv, kv, nullptr, n, 1.f, kv, nullptr, nullptr);
}

// an append of n_tokens that fails at its launch number `at`, then `between`
// (a decode: what it reads must be the old state), then the append again
static void append_fails(int seqs, int len, int n_tokens, int at, bool applies, bool step) {
  bsattn_cache* c = filled(seqs, 16, len);
  auto call = [&] { return step ? append_decode(c, seqs) : bsattn_append(c, kv, kv, nullptr, seqs, n_tokens, nullptr); };
  for (int tries = 0; tries < 2; ++tries) {  // (a second failure loses nothing either)
    stub::launches_left = at;
    stub::applies = applies;
    CHECK(call() == BSATTN_ERR_HIP);
    stub::launches_left = -1;
  }
  CHECK(decode(c, seqs) == BSATTN_OK);
  for (int s = 0; s < seqs; ++s) check_meta(c, s, len);
  stub::launches_left = std::min(at, 2);  // (the pages are held by now: fewer patches)
  CHECK(call() == BSATTN_ERR_HIP);
  stub::launches_left = -1;
  CHECK(call() == BSATTN_OK);
  for (int s = 0; s < seqs; ++s) check_meta(c, s, len + n_tokens);
  CHECK(append_decode(c, seqs) == BSATTN_OK);
  for (int s = 0; s < seqs; ++s) check_meta(c, s, len + n_tokens + 1);
  bsattn_cache_destroy(c);
}

int main() {
  for (bool applies : {false, true}) {
    append_fails(2, 31, 5, 0, applies, false);     // new pages, patched by the append's launch
    append_fails(2, 32, 1, 0, applies, true);      // the same in a decode step's launch
    append_fails(3, 10, 1, 0, applies, true);      // no new page
    append_fails(100, 30, 40, 0, applies, false);  // patches in launches of their own: the first fails,
    append_fails(100, 30, 40, 1, applies, false);  // the second,
    append_fails(100, 30, 40, 3, applies, false);  // the second batch's append
    append_fails(70, 31, 1, 2, applies, true);     // a step of two calls
  }
  // not into a graph: its replays would set the words back
  {
    bsattn_cache* g = filled(2, 16, 31);
    stub::launches_left = 0;
    stub::applies = false;
    CHECK(bsattn_append(g, kv, kv, nullptr, 2, 5, nullptr) == BSATTN_ERR_HIP);
    stub::launches_left = -1;
    stub::capture = hipStreamCaptureStatusActive;
    CHECK(decode(g, 2) == BSATTN_ERR_INVALID && append_decode(g, 2) == BSATTN_ERR_INVALID);
    CHECK(stub::last.meta[stub::last.cap_off] == 32);  // (nothing was sent)
    stub::capture = hipStreamCaptureStatusNone;
    CHECK(decode(g, 2) == BSATTN_OK);
    check_meta(g, 0, 31);
    stub::capture = hipStreamCaptureStatusActive;
    CHECK(decode(g, 2) == BSATTN_OK);
    stub::capture = hipStreamCaptureStatusNone;
    bsattn_cache_destroy(g);
  }
  // patches that a reserve, a trim and a reset could not send
  bsattn_cache* c = filled(2, 16, 40);
  stub::launches_left = 0;
  stub::applies = false;
  CHECK(bsattn_reserve(c, nullptr, 2, 100, nullptr) == BSATTN_ERR_HIP);
  stub::launches_left = -1;
  CHECK(bsattn_append_step(c, kv, kv, nullptr, 2, nullptr) == BSATTN_OK);
  CHECK(bsattn_sync(c, nullptr) == BSATTN_OK);
  for (int s = 0; s < 2; ++s) check_meta(c, s, 40);
  stub::launches_left = 0;
  CHECK(bsattn_trim(c, nullptr, 2, 20, nullptr, nullptr) == BSATTN_ERR_HIP);
  stub::launches_left = -1;
  CHECK(bsattn_prefill(c, kv, nullptr, 2, 17, 1.f, kv, nullptr) == BSATTN_OK);
  for (int s = 0; s < 2; ++s) check_meta(c, s, 20);
  stub::launches_left = 0;
  CHECK(bsattn_reset(c, nullptr, 1, nullptr) == BSATTN_ERR_HIP);
  stub::launches_left = -1;
  bsattn_cache* copy = nullptr;  // (a copy takes the words over as well)
  CHECK(bsattn_copy(c, &copy, nullptr) == BSATTN_OK);
  for (bsattn_cache* x : {c, copy}) {
    CHECK(decode(x, 2) == BSATTN_OK);
    check_meta(x, 0, 0);
    check_meta(x, 1, 20);
    bsattn_cache_destroy(x);
  }
  std::puts("ok");
  return 0;
}
