// Quantization by the host's vector units.
#pragma once

#include <stdint.h>

namespace vtlhip {

// Codes and scales as the device's quantizer makes them; rows of codes start `row` bytes apart, with zeros behind the codes.
struct HostQuantizer {
    // each row with a scale of its own
    void (*rows)(const float *x, int64_t rows, int64_t cols, int8_t *codes, int64_t row, float *scales);
    // with one given scale, that of an absmax which covers them
    void (*scaled)(const float *x, int64_t rows, int64_t cols, int8_t *codes, int64_t row, float scale);
    float (*absmax)(const float *x, int64_t count);
    float (*scale)(float absmax);
};

// For this machine's processors; nullptr: none that keeps up with a copy.
const HostQuantizer *host_quantizer();

}  // namespace vtlhip
