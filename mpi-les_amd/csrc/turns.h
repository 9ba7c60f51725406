// The order of the streams' work on one device around work that needs the
// whole of it.
#pragma once

#include <algorithm>
#include <vector>

namespace les {

// A step whose pressure solve runs in one launch (k_sor_res) needs every
// compute unit its boxes were cut for at once: beside work of another stream
// its blocks hold units while they wait for units that work holds.  Such a
// step runs after everything enqueued before it, and everything enqueued later
// runs after it.  Other steps are not ordered among themselves.  Work is told
// to take its turn whether or not any domain solves in one launch yet: a step
// enqueued before the first such domain exists may still wait to run when that
// domain's first step comes.
template <class Stream>
class Turns {
 public:
  // Work is about to be enqueued on s; that of earlier calls is enqueued.
  // after(t, s) has what is enqueued on s from now on run after all that is
  // enqueued on t (nonzero: it failed, and so does this call).
  template <class After>
  int take(Stream s, bool whole, After after) {
    const bool seen = std::find(since_.begin(), since_.end(), s) != since_.end();
    if (!whole && seen) return 0;  // came after the last whole-device work already
    int rc = 0;
    if (any_ && last_ != s) rc = after(last_, s);
    if (!whole) {
      if (!rc) since_.push_back(s);
      return rc;
    }
    for (const Stream& t : since_)
      if (!rc && t != s && !(any_ && t == last_)) rc = after(t, s);
    if (rc) return rc;
    since_.clear();
    any_ = true;
    last_ = s;
    return 0;
  }
  // The stream goes away, its work complete.
  void forget(Stream s) {
    since_.erase(std::remove(since_.begin(), since_.end(), s), since_.end());
    if (any_ && last_ == s) any_ = false;
  }

 private:
  bool any_ = false;
  Stream last_{};              // the stream of the last whole-device work
  std::vector<Stream> since_;  // streams with other work since
};

}  // namespace les
