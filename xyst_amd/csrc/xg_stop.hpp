// Device state of a Krylov solve and the words through which its launches
// learn of the stop.
//
// An iteration's first launch tests for the stop: every workgroup takes the
// same sums, so all find it alike, and the first one records it.  The launches
// after it ask stop_found, and the last of the iteration passes the word on
// for the next iterations' first launches, which ask stop_past.  So no launch
// reads a word that it writes: the waves of a workgroup, which ask each for
// itself, cannot differ.
#pragma once

namespace xg {

struct CgState {
  double normb, rho0, rr;
  long long it;
  int found;       // written by the launch that tests
  int past;        // written by an iteration's last launch
  int converged;
};

constexpr void stop_clear(CgState& s) {
  s.it = 0;
  s.found = 0;
  s.past = 0;
  s.converged = 0;
}
constexpr void stop_record(CgState& s, long long it, double rr, int converged) {
  s.it = it;
  s.rr = rr;
  s.converged = converged;
  s.found = 1;
}
constexpr bool stop_found(const CgState& s) { return s.found != 0; }
constexpr void stop_pass(CgState& s) { s.past = 1; }
constexpr bool stop_past(const CgState& s) { return s.past != 0; }

}  // namespace xg
