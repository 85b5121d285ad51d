// cast_kernel.hip -- the wire codec on one tensor: fp32 -> bf16 for sending (ProcessGroupMCCL.cpp:131-132)
// and bf16 -> fp32 on arrival (:179-183), the bits that the fold kernels give these plans.
//
// HBM-bound: 6 bytes an element.  The fold kernels fetch a descriptor, pick their segment and work out the
// head of its packet grid in every block, 0.3 us of a small launch and a sixth of what a wave of a cast lives
// for; here the host has done that and a block has three scalar operations in front of its loads.  That also
// makes several packets a lane worth it (in the fold kernels they are not): where one generation of
// waves covers the tensor, all its loads come in front of all its stores, 26 MB written behind
// 13 MB read instead of among them, and a wave has one store under way at a time (without that wait a
// decode of 6.5 M elements takes 9.0 us, with it 7.8).  Decode and encode of 0.2 M elements 2.5 -> 2.2 and 2.3 -> 2.1 us,
// of 2.5 M 4.4 -> 3.6 and 4.7 -> 3.9, of 6.5 M 8.7 -> 7.8 and 8.7 -> 8.4, of 48 M 45.9 -> 46.0 and 45.8 -> 44.0.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "fold_launch.h"
#include "wire_codec.h"

namespace mcclx {
namespace {
#define MCCLX_GLOBAL __attribute__((address_space(1)))
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
// element alignment is all the kernels may assume
typedef u32x4 F32Pack __attribute__((aligned(4)));
typedef u32x2 WirePack __attribute__((aligned(2)));

// s_waitcnt vmcnt(0), the other counters as they are: all loads of the wave are back, and its last store has arrived.
constexpr int kVmcnt0 = 0x0F70;

// Packets of four elements; `dst` and `src` point at packet 0, `head` elements lie in front of it and `tail`
// behind the last.
template <bool DECODE, int B, int T>
__global__ void __launch_bounds__(B) cast_kernel(void* dst, const void* src, uint32_t packets, uint32_t head, uint32_t tail) {
    constexpr uint32_t kIn = DECODE ? 8 : 16, kOut = DECODE ? 16 : 8;  // bytes a packet
    using Raw = std::conditional_t<DECODE, u32x2, u32x4>;
    const uint32_t first = blockIdx.x * (uint32_t)(B * T), left = packets - first;
    const MCCLX_GLOBAL uint8_t* in = (const MCCLX_GLOBAL uint8_t*)src + (uint64_t)first * kIn;
    MCCLX_GLOBAL uint8_t* out = (MCCLX_GLOBAL uint8_t*)dst + (uint64_t)first * kOut;
    auto load = [&](uint32_t p) -> Raw {
        if constexpr (DECODE) return __builtin_nontemporal_load((const MCCLX_GLOBAL WirePack*)(in + p * kIn));
        else return __builtin_nontemporal_load((const MCCLX_GLOBAL F32Pack*)(in + p * kIn));
    };
    auto store = [&](uint32_t p, const Raw& v) {
        if constexpr (DECODE)
            __builtin_nontemporal_store((u32x4{v[0] << 16, v[0] & 0xFFFF0000u, v[1] << 16, v[1] & 0xFFFF0000u}),
                                        (MCCLX_GLOBAL F32Pack*)(out + p * kOut));
        else
            __builtin_nontemporal_store((u32x2{bf16_encode_pair(__uint_as_float(v[0]), __uint_as_float(v[1])),
                                               bf16_encode_pair(__uint_as_float(v[2]), __uint_as_float(v[3]))}),
                                        (MCCLX_GLOBAL WirePack*)(out + p * kOut));
    };
    Raw v[T];
    if (left >= (uint32_t)(B * T)) {
#pragma unroll
        for (int u = 0; u < T; ++u) v[u] = load(u * B + threadIdx.x);
#pragma unroll
        for (int u = 0; u < T; ++u) {
            if constexpr (T > 1) __builtin_amdgcn_s_waitcnt(kVmcnt0);
            store(u * B + threadIdx.x, v[u]);
        }
    } else {  // (all loads first here too: this block is the last to start)
#pragma unroll
        for (int u = 0; u < T; ++u)
            if (u * B + threadIdx.x < left) v[u] = load(u * B + threadIdx.x);
#pragma unroll
        for (int u = 0; u < T; ++u)
            if (u * B + threadIdx.x < left) store(u * B + threadIdx.x, v[u]);
    }
    if (blockIdx.x == 0) {
        auto edge = [&](int64_t i) {
            if constexpr (DECODE)
                ((MCCLX_GLOBAL uint32_t*)dst)[i] = (uint32_t)((const MCCLX_GLOBAL uint16_t*)src)[i] << 16;
            else
                ((MCCLX_GLOBAL uint16_t*)dst)[i] = (uint16_t)(bf16_round_bits(((const MCCLX_GLOBAL float*)src)[i]) >> 16);
        };
        if (threadIdx.x < head) edge((int64_t)threadIdx.x - head);
        if (threadIdx.x < tail) edge((int64_t)packets * 4 + threadIdx.x);
    }
}

template <bool DECODE, int B, int T>
hipError_t go(hipStream_t st, void* dst, const void* src, uint32_t packets, uint32_t head, uint32_t tail) {
    const uint32_t blocks = (uint32_t)(((uint64_t)packets + B * T - 1) / (B * T));
    cast_kernel<DECODE, B, T><<<dim3(blocks ? blocks : 1), dim3(B), 0, st>>>(dst, src, packets, head, tail);
    return hipGetLastError();
}
}  // namespace

// Packets a lane, by the waves of one packet a lane in generations of the device (8192 waves on 256 CUs).
// Decode, us at 1 / 2 / 4 / 8 packets in blocks of four wavefronts and at 2 in blocks of one:
// 1.5 M elements (0.7 generations) 2.9 / 2.9 / 3.2 / - / 3.5, 4 M (1.9) 5.9 / 4.9 / 5.0 / - / 5.8, 5 M (2.4) 7.4 / 6.6 / 6.2 /
// 6.3 / 6.8, 6.5 M (3.1) 9.1 / 8.5 / 7.9 / 7.8 / 8.6, 10 M (4.8) 12.4 / 12.6 / 13.1 / 11.3 / 11.9, 14 M (6.7) 16.3 / 16.6 / 16.8 /
// 15.7 / 15.9, 16 M (7.6) 18.0 / 18.5 / 18.7 / 17.7 / 17.4.  Encode at 1 / 2 in blocks of four and at 1 in blocks of one: 1.5 M
// 3.1 / 3.3 / 3.6, 2.5 M (1.2) 4.4 / 3.9 / 4.5, 4 M 5.7 / 6.0 / 5.7, 6.5 M 9.2 / 8.9 / 8.4, 16 M 19.3 / 18.1 / 16.9.
// Off the lines a decode of 1.5 M takes 3.6 us at 1 and 3.1 at 2, which are level on them: 2 from 0.6 generations on.
// An encode from off the lines of 3.4 / 4 M takes 5.6 / 6.1 us at 1 in blocks of one and 5.4 / 5.9 in blocks of four (on the
// lines 5.3 / 5.7 and 5.4 / 5.8).
// One store under way per wave is not enough for a result in host memory (6.5 M decoded into pinned memory 536 us at 2
// in blocks of one and 561 at 8): `far`.
hipError_t launch_cast(hipStream_t st, bool decode, void* dst, const void* src, uint64_t count, int cus, bool far) {
    // packets start on a 128-byte line of the output
    const uint32_t size = decode ? 4 : 2, mis = (uint32_t)(reinterpret_cast<uintptr_t>(dst) & 127u);
    const uint64_t peel = mis ? (128u - mis) / size : 0;
    const uint32_t head = (uint32_t)(count < peel ? count : peel), tail = (uint32_t)((count - head) % 4);
    const uint64_t whole = (count - head) / 4;
    if (whole >> 31) return hipErrorInvalidValue;
    const uint32_t packets = (uint32_t)whole;
    dst = static_cast<char*>(dst) + (uint64_t)head * size;
    src = static_cast<const char*>(src) + (uint64_t)head * (6 - size);
    const uint64_t waves = whole / 64, gen = 32 * (uint64_t)cus;
    if (decode) {
        if (waves * 5 <= 3 * gen) return go<true, 256, 1>(st, dst, src, packets, head, tail);
        if (waves <= 2 * gen) return go<true, 256, 2>(st, dst, src, packets, head, tail);
        if (waves <= 3 * gen && !far) return go<true, 256, 4>(st, dst, src, packets, head, tail);
        if (waves <= 7 * gen && !far) return go<true, 256, 8>(st, dst, src, packets, head, tail);
        return go<true, 64, 2>(st, dst, src, packets, head, tail);
    }
    if (waves <= gen) return go<false, 256, 1>(st, dst, src, packets, head, tail);
    if (waves * 2 <= 3 * gen) return go<false, 256, 2>(st, dst, src, packets, head, tail);
    if (waves <= 2 * gen && (reinterpret_cast<uintptr_t>(src) & 127u)) return go<false, 256, 1>(st, dst, src, packets, head, tail);
    return go<false, 64, 1>(st, dst, src, packets, head, tail);
}

}  // namespace mcclx
