// Prints the LDS slots that the 20-state walks get (netrax_amd/csrc/
// schedule.cpp) and the dynamic LDS of their workgroups.
//
// Input (stdin): lines "categories fp32 padded_sites".
// Output: per line "forward_slots forward_bytes reverse_slots reverse_bytes".
#include <cstdio>

#include "../netrax_amd/csrc/schedule.hpp"

using namespace nrx;

int main() {
  int C, fp32;
  long long sites;
  while (std::scanf("%d %d %lld", &C, &fp32, &sites) == 3) {
    const AaSlots s = aa_walk_slots(C, fp32 != 0, sites);
    std::printf("%d %zu %d %zu\n", s.fwd, fp32 ? forward_lds_aa32(C, s.fwd) : forward_walk_lds_aa(C, s.fwd), s.adj,
                fp32 ? adjoint_lds_aa32(s.adj) : adjoint_walk_lds_aa(s.adj));
  }
  return 0;
}
