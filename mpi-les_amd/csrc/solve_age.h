// How long the words of a workspace of the one-launch SOR can be told apart.
#pragma once

namespace les {

// A word of a workspace (k_sor_res) carries the number of its domain's solve in
// 19 bits of its tag.  One left from 2^19 solves ago would pass for this solve's: a
// workspace need not be written in between, for a domain has two (its own and a
// batch's) and solves by other kernels count too.  So a workspace is cleared
// when its oldest words may be kMaxAge solves old.  The host counts no fewer
// solves than the device: those of a press are 1, in mode 1 one more per outer step.
class SolveAge {
 public:
  static constexpr long long kMaxAge = 1LL << 18;
  // Solves up to number `last` of the domain are about to use the workspace,
  // `count` of them.  True: it has to be cleared before.
  bool use(long long last, long long count) {
    if (last - born_ <= kMaxAge) return false;
    born_ = last - count;
    return true;
  }
  void cleared(long long last) { born_ = last; }

 private:
  long long born_ = 0;  // the number of the last solve before it was cleared
};

}  // namespace les
