// When to try again what other work on the device made fail: after the k-th
// failure in a row the next 2^(k-1) chances are passed over, at most
// BACKOFF_MAX; a success forgets them.  Plain arithmetic, checked on the host.
#pragma once

namespace dmrg {

constexpr int BACKOFF_MAX = 64;

struct Backoff {
  int skip = 0, last = 0;   // chances still to pass over, passed over last
  bool allowed() {
    if (skip == 0) return true;
    --skip;
    return false;
  }
  void failed() {
    last = last == 0 ? 1 : (2 * last < BACKOFF_MAX ? 2 * last : BACKOFF_MAX);
    skip = last;
  }
  void succeeded() { skip = last = 0; }
};

}  // namespace dmrg
