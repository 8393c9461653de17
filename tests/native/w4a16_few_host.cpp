// w4a16_few_host.cpp -- the host-side rules of csrc/w4a16_few.hpp for the CPU
// tests.  TEST INFRASTRUCTURE.
#include "../../cudaforge_amd/csrc/w4a16_few.hpp"

extern "C" int few_takes(int M, int N, int K) { return cfa::w4few::takes(M, N, K) ? 1 : 0; }
