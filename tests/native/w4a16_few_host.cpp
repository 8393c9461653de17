// w4a16_few_host.cpp -- the host-side rules of csrc/w4a16_few.hpp for the CPU
// tests.  TEST INFRASTRUCTURE.
#include "../../cudaforge_amd/csrc/w4a16_few.hpp"

extern "C" int few_takes(int M, int N, int K) { return cfa::w4few::takes(M, N, K) ? 1 : 0; }

extern "C" uint32_t few_group(uint32_t sl, uint32_t d) {
  return cfa::w4few::slice_group(sl, cfa::w4few::slice_div(d));
}

// The first slice of [lo, hi) whose group is not sl / d, or hi.
extern "C" uint32_t few_group_wrong(uint32_t lo, uint32_t hi, uint32_t d) {
  const cfa::w4few::SliceDiv v = cfa::w4few::slice_div(d);
  for (uint32_t sl = lo; sl < hi; ++sl)
    if (cfa::w4few::slice_group(sl, v) != sl / d) return sl;
  return hi;
}
