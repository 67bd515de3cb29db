// Host-side exhaustive check of the library's definition of the fp32 -> bf16 narrowing
// (xfastertransformer_amd/csrc/bf16_convert.h: the host's conversion, and what bf16_device_sweep.hip holds
// the device's against) against the oracle's restatement of the reference conversion, over all 2^32 bit patterns.
// Built and run by tests/test_oracle_pins.py; prints the number of mismatches.
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include "bf16_convert.h"

extern "C" uint16_t orc_f32_to_bf16(float f);

int main() {
    unsigned long long bad = 0;
#pragma omp parallel for reduction(+ : bad) schedule(static)
    for (long long i = 0; i < (1LL << 32); ++i) {
        const uint32_t u = (uint32_t)i;
        float f;
        memcpy(&f, &u, 4);
        bad += xfthip::f32_bits_to_bf16_ref(u) != orc_f32_to_bf16(f);
    }
    printf("mismatches %llu\n", bad);
    return bad ? 1 : 0;
}
