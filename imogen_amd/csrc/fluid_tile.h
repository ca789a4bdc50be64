// fluid_tile.h -- chunk loads and stores shared by the fluid sweep kernels.
#pragma once

#include "imh_common.h"

namespace imh {

// K consecutive cells as 16-byte (or one 8-byte) vector accesses; p is aligned to
// K * sizeof(T) bytes.
template <typename T, int K>
__device__ __forceinline__ void chunk_load(const T* p, T (&out)[K]) {
    constexpr int B = K * int(sizeof(T));
    if constexpr (B % 16 == 0) {
        constexpr int L = 16 / int(sizeof(T));
        typedef T V __attribute__((ext_vector_type(L)));
#pragma unroll
        for (int j = 0; j < K / L; ++j) {
            const V x = *gmem(reinterpret_cast<const V*>(p + j * L));
#pragma unroll
            for (int l = 0; l < L; ++l) out[j * L + l] = x[l];
        }
    } else if constexpr (B == 8 && K == 2) {
        typedef T V __attribute__((ext_vector_type(2)));
        const V x = *gmem(reinterpret_cast<const V*>(p));
        out[0] = x[0];
        out[1] = x[1];
    } else {
#pragma unroll
        for (int k = 0; k < K; ++k) out[k] = gmem(p)[k];
    }
}

template <typename T, int K>
__device__ __forceinline__ void chunk_store(T* p, const T (&in)[K]) {
    constexpr int B = K * int(sizeof(T));
    if constexpr (B % 16 == 0) {
        constexpr int L = 16 / int(sizeof(T));
        typedef T V __attribute__((ext_vector_type(L)));
#pragma unroll
        for (int j = 0; j < K / L; ++j) {
            V x;
#pragma unroll
            for (int l = 0; l < L; ++l) x[l] = in[j * L + l];
            *gmem(reinterpret_cast<V*>(p + j * L)) = x;
        }
    } else if constexpr (B == 8 && K == 2) {
        typedef T V __attribute__((ext_vector_type(2)));
        V x;
        x[0] = in[0];
        x[1] = in[1];
        *gmem(reinterpret_cast<V*>(p)) = x;
    } else {
#pragma unroll
        for (int k = 0; k < K; ++k) gmem(p)[k] = in[k];
    }
}

}  // namespace imh
