// Weight type tags, for device and plain host code.
#pragma once

namespace jamhip {

// ggml / jam dtype tags (jam/jam-native/include/jam.h:59-77).
enum Dtype : int {
    F32 = 0, F16 = 1, Q4_0 = 2, Q8_0 = 8, Q4_K = 12, Q5_K = 13, Q6_K = 14, BF16 = 30, MXFP4 = 39, NVFP4 = 40, Q1_0 = 41
};

}  // namespace jamhip
