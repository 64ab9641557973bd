// What tests call of hrn_args.h, the arithmetic that launches and kernels share.
#include "../heron_amd/csrc/hrn_args.h"

extern "C" {

// quotients of ns by d as the kernels compute them
void div_all(const uint32_t* ns, uint32_t* out, int count, uint32_t d) {
    const HrnDiv by(d);
    for (int i = 0; i < count; ++i) out[i] = by(ns[i]);
}

int pair_of(int block, int pairs) { return hrn_pair_of(block, pairs); }
}
