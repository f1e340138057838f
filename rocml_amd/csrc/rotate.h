// Rotation of a part of a row by tabled angles.
#pragma once
#include "common.h"

// Number e of a part whose first `dims` numbers turn: pairs (e, e + dims/2), or with pairing 1 (2i, 2i + 1), by the
// angle whose cosine and sine stand in c and s.
__device__ __forceinline__ float turned(const float* __restrict__ v, int e, int dims, int pairing, const float* __restrict__ c,
                                        const float* __restrict__ s) {
    if (e >= dims) return v[e];
    if (pairing == 1) {
        int i = e >> 1;
        return (e & 1) ? v[e] * c[i] + v[e - 1] * s[i] : v[e] * c[i] - v[e + 1] * s[i];
    }
    int half = dims / 2;
    return e < half ? v[e] * c[e] - v[e + half] * s[e] : v[e] * c[e - half] + v[e - half] * s[e - half];
}
