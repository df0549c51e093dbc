// Wrap-around embedding of a table of offsets on a torus.
#pragma once

#include <hip/hip_runtime.h>

namespace aspher {

// The table offset that index i of a torus of side n holds: 0 .. Ns-1 from the
// front, their mirror images Ns-1 .. 1 from the end, and -1 (a zero) between
// them. n may be any side of at least 2 Ns - 1; at 2 Ns the only zero is i = Ns.
__host__ __device__ __forceinline__ int embed_offset(int i, int Ns, int n) {
    const int d = i < Ns ? i : n - i;
    return d < Ns ? d : -1;
}

} // namespace aspher
