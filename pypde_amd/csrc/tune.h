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

// The most V x V matrices (V > 8) in a face-flux launch, two per face point, up to
// which one wavefront per matrix is the faster form; above, one lane per matrix.
// A wavefront hides the latency of a lane's chain but works for one matrix, 20
// ns each at V = 9 and 77 at 17; lanes take as long for one wavefront's 64 matrices
// as for a GPU full of them.  Measured, 1D order 2, us of wavefront / lane:
//   V = 9   8,000 matrices  221 / 230      80,000   1659 / 232      800,000  16070 / 982
//   V = 10  8,000           261 / 232      80,000   1930 / 244
//   V = 12  8,000           376 / 531      80,000   3094 / 545      800,000  30184 / 2653
//   V = 14  8,000           446 / 1200     80,000   3746 / 1339     800,000  36301 / 8299
//   V = 17  8,000           754 / 2681     80,000   6322 / 3762     800,000  61787 / 23939
//   V = 17 (GPR)            80,000  1938-2847 / 1893-2944           400,000  9166-13870 / 5254-10952
// At 17 variables a lane's matrix lies in scratch and the lane form takes minutes to
// compile, so the line stays where the GPR model has it.
inline long wide_matrices(int V) {
  return V <= 11 ? 9000 : V <= 13 ? 14000 : V <= 15 ? 27000 : 90000;
}

}  // namespace pypde
