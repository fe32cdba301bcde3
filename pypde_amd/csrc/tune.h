// The autotuner's decisions on its trials' times.
#pragma once

namespace pypde {

// The fastest of n launch variants.
inline int fastest(const double* ms, int n) {
  int b = 0;
  for (int i = 1; i < n; i++)
    if (ms[i] < ms[b]) b = i;
  return b;
}

// The predictor schedule: 0 one kernel, 1.. the split's builds.  Trials step from
// the run's state, usually its first, while the cells that the split computes
// twice grow in number as the run goes on, so a tie goes to the one kernel and
// the split has to be 5 % faster (1D reactive run, order 4: 156.6 against 156.3
// us in the trial, 153 against 225 us a step over the first 20 steps).
inline int predictor_schedule(const double* ms, int n) {
  const int b = fastest(ms, n);
  return b > 0 && ms[b] < 0.95 * ms[0] ? b : 0;
}

}  // namespace pypde
