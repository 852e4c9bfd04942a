// At which Picard iterates the separate residual test is worth taking (see ReState::step). The test of an iterate
// that fails is a pass for nothing, and the storm steps that fail it at h^m mostly do so again in the next step: there
// the system is stored and solved at once. What is known of a step is kept for the next one only: which
// iterates before the one that ended the loop failed their test.
#pragma once

namespace frehg {

class PicardChecks {
 public:
  bool expect_fail(int m) const { return (failed_ & bit(m)) != 0; }
  // The residual test of h^m failed.
  void failed(int m) { failed_ |= bit(m); }
  // The loop ended at h^m, by whichever test: h^m did not need the solve that an expected failure stands for,
  // and no later iterate was met.
  void ended(int m) {
    if (m < 32) failed_ &= bit(m) - 1u;
  }
  void clear() { failed_ = 0; }

 private:
  static unsigned int bit(int m) { return m < 32 ? 1u << m : 0u; }
  unsigned int failed_ = 0;
};

}  // namespace frehg
