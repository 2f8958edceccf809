// exchange.h -- words through which running blocks hand values to each other, and the wave
// sums of their reductions (device code of the resident kernels).
//
// A word holds the mark, a signalling NaN that no arithmetic produces (results are quiet NaNs),
// until its owner posts the value; a reader peeks until it is not the mark.  Both are relaxed
// atomics of agent scope: all XCDs see them without cache writebacks or invalidations.
#pragma once

#include <hip/hip_runtime.h>

namespace prism_hip {

namespace {

template <typename T> struct Word;
template <> struct Word<double> {
    using U = unsigned long long;
    static constexpr U MARK = 0x7FF4A11C0DE5EED1ull;  // a signalling NaN
};
template <> struct Word<float> {
    using U = unsigned int;
    static constexpr U MARK = 0x7FA5EED1u;
};

template <typename T>
__device__ inline T asValue(typename Word<T>::U u) {
    T v;
    __builtin_memcpy(&v, &u, sizeof(T));
    return v;
}
template <typename T>
__device__ inline typename Word<T>::U asWord(T v) {
    typename Word<T>::U u;
    __builtin_memcpy(&u, &v, sizeof(T));
    return u;
}
template <typename U>
__device__ inline U peek(const U* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename U>
__device__ inline void post(U* p, U v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Published vectors are reached through a buffer descriptor: one 32-bit offset per lane beside
// scalar registers, and an offset past the end reads zero and stores nothing, without a
// branch (FAR marks such offsets).  Cache policy 16 is the agent scope of peek and post.
constexpr unsigned FAR = 0x80000000u;
constexpr int AGENT = 16;
using U2 = unsigned int __attribute__((ext_vector_type(2)));
template <typename U, int POLICY = AGENT>
__device__ inline U bufPeek(__amdgpu_buffer_rsrc_t b, unsigned at, unsigned base) {
    if constexpr (sizeof(U) == 8) {
        const U2 v = __builtin_amdgcn_raw_buffer_load_b64(b, at, base, POLICY);
        return (unsigned long long)v.y << 32 | v.x;
    } else {
        return __builtin_amdgcn_raw_buffer_load_b32(b, at, base, POLICY);
    }
}
template <typename U>
__device__ inline void bufPost(__amdgpu_buffer_rsrc_t b, unsigned at, unsigned base, U v) {
    if constexpr (sizeof(U) == 8) {
        const U2 w = {(unsigned)v, (unsigned)(v >> 32)};
        __builtin_amdgcn_raw_buffer_store_b64(w, b, at, base, AGENT);
    } else {
        __builtin_amdgcn_raw_buffer_store_b32(v, b, at, base, AGENT);
    }
}

// Sums over the wavefront of K = 2 or 4 values at once, each with the additions of the
// butterfly over lane distances 32, 16, 8, 4, 2, 1 (krylov.hip's waveSum: the same bits).  The
// halves, and then the row pairs, of two values are swapped and added, which leaves each of
// the K values on its own 64 / K lanes; DPP row rotations sum those: 7 additions for K = 4
// instead of 24, and no moves through LDS.  The total of value k is in lane sumLane<K>(k).
template <int CTRL>
__device__ inline double rotAdd(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
    return v + __hiloint2double(hi, lo);
}
__device__ inline double swapAdd32(double a, double b) {  // lanes 0-31: a's sums at distance 32, 32-63: b's
    const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
    return __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
}
__device__ inline double swapAdd16(double a, double b) {  // even rows: a's sums at distance 16, odd rows: b's
    const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false, false);
    return __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
}
template <int K>
__device__ inline double waveSums(const double (&v)[K]) {
    static_assert(K == 2 || K == 4);
    double s = swapAdd32(v[0], v[1]);
    if constexpr (K == 4) s = swapAdd16(s, swapAdd32(v[2], v[3]));  // rows 0 to 3: values 0, 2, 1, 3
    else s = swapAdd16(s, s);
    s = rotAdd<0x128>(s);  // row_ror:8
    s = rotAdd<0x124>(s);  // row_ror:4
    s = rotAdd<0x122>(s);  // row_ror:2
    return rotAdd<0x121>(s);  // row_ror:1
}
template <int K>
__device__ constexpr int sumLane(int k) {
    return K == 2 ? 32 * k : 16 * (k == 1 ? 2 : k == 2 ? 1 : k);
}
__device__ inline double laneValue(double v, int lane) {
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), lane);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), lane);
    return __hiloint2double(hi, lo);
}

// A bounded wait: true while it may go on.  A wait that ran out, here or in another block
// (looked up now and then), raises the block's flag.
__device__ inline bool keepWaiting(unsigned& polls, unsigned limit, int* stuck, int* fail) {
    ++polls;
    if (polls >= limit || ((polls & 255) == 0 && peek(stuck) != 0)) {
        post(stuck, 1);
        *fail = 1;
        return false;
    }
    return true;
}

}  // namespace

}  // namespace prism_hip
