// The sum of the fp32 partial results that the workgroups of a split product leave behind.
#pragma once
#include "lowbit_mfma.h"

namespace lowbit {

// U more parts, their loads in flight together, added in order.
template <int U> __device__ inline void add_parts(f32x4 &a, const f32x4 *__restrict__ part, int64_t stride) {
    f32x4 v[U];
#pragma unroll
    for (int j = 0; j < U; j++) v[j] = part[j * stride];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < U; j++) a += v[j];
}

// part[0] + part[stride] + ... in that order, `splits` terms (the same for every thread of the launch).
//
// Up to nine loads are in flight at a time: a thread that waited for each part in turn spent a memory latency per part, which is
// what such a launch takes where tiles are few and splits many (214 rows on [592 x 6144] in sym_int4, both launches, 18.3 -> 16.3
// us; row-major 40 rows on [745 x 10176] in nf4 17.4 -> 14.9).  As many loads as parts, none for a round number's sake: with up to
// four splits the launch is bound by their bytes.
__device__ inline f32x4 sum_splits(const f32x4 *__restrict__ part, int64_t stride, int splits) {
    f32x4 a = *part;
    part += stride;
    int left = splits - 1;
    for (; left >= 8; left -= 8, part += 8 * stride) add_parts<8>(a, part, stride);
    switch (left) {
    case 1: add_parts<1>(a, part, stride); break;
    case 2: add_parts<2>(a, part, stride); break;
    case 3: add_parts<3>(a, part, stride); break;
    case 4: add_parts<4>(a, part, stride); break;
    case 5: add_parts<5>(a, part, stride); break;
    case 6: add_parts<6>(a, part, stride); break;
    case 7: add_parts<7>(a, part, stride); break;
    }
    return a;
}

}  // namespace lowbit
