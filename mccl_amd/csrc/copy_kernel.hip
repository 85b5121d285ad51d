// copy_kernel.hip -- streaming device copies on the reduce queue: the allgather
// legs (AllreduceAlgos.cpp:77-86, ProcessGroupMCCL.cpp:232-273) and the
// unstage copy (MPSInterop.mm:408-435); a few copies travel by value in the
// kernel arguments and run as one grid, thousands go through a table.  Also the
// known-traffic kernel the memory counters are calibrated against, and the
// read-only / write-only probes a launch's footprint is measured against.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fold_launch.h"

namespace mcclx {
namespace {
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
#define MCCLX_GLOBAL __attribute__((address_space(1)))
// every byte is touched once: non-temporal loads and stores
#define COPY_LD(p) __builtin_nontemporal_load(p)
#define COPY_ST(p, v) __builtin_nontemporal_store((v), (p))
// 16-byte packets at any address (gfx950 global accesses are alignment-agnostic)
typedef u32x4 Packet __attribute__((aligned(1)));
constexpr int kBlock = 256;

constexpr int kOneWave = 64, kFourWaves = 256;  // threads per block of a launch by value, see kOneWaveBlocksFrom
constexpr uint32_t kXcds = 8;
constexpr uint32_t kSpreadTile = kFourWaves * 32;  // bytes a block of copy_spread_kernel moves

// Up to kFewCopies copies with their descriptors in the kernel arguments:
// blockIdx.y picks the copy, blockIdx.x one tile of B packets of 16 bytes, one
// per lane; block 0 of a copy also moves the bytes in front of its first and
// behind its last whole packet.  Packets start on a 128-byte boundary of the
// first destination: a stream of full lines, where an odd-sized chunk of an
// allgather would otherwise write every line in two parts.
// One tile per block and no loop, like the fold kernels: a uniform 64-bit base
// plus a 32-bit lane offset per access, and a short path to the first load.
// The number of destinations is a compile-time constant and every field a block
// needs is fetched in one batch of scalar loads (as the fold kernels do): with few
// waves on a CU what a wave waits for in front of its load is not hidden by others.
// MIXED: copies of different numbers of destinations, up to N, share the launch.
template <int N, int B, bool MIXED = false>
__global__ void __launch_bounds__(B) copy_few_kernel(CopyFew a) {
    const CopyDesc& d = a.d[blockIdx.y];
    const void* src = d.src;
    uint64_t nbytes = d.nbytes;
    const int n = MIXED ? (int)d.n : N;
    void* dst[N];
#pragma unroll
    for (int f = 0; f < N; ++f) dst[f] = d.dst[f];
    asm volatile("" : "+s"(src), "+s"(nbytes));
#pragma unroll
    for (int f = 0; f < N; ++f) asm volatile("" : "+s"(dst[f]));
    const uint32_t mis = (0u - (uint32_t)reinterpret_cast<uintptr_t>(dst[0])) & 127u;
    const uint32_t head = nbytes < mis ? (uint32_t)nbytes : mis;
    const uint64_t P = (nbytes - head) / 16;
    const uint64_t first = (uint64_t)blockIdx.x * B;
    const uint64_t at = head + first * 16;
    if (first < P) {
        if (threadIdx.x < P - first) {
            const uint32_t off = threadIdx.x * 16u;
            const u32x4 v = COPY_LD((const MCCLX_GLOBAL Packet*)((const MCCLX_GLOBAL uint8_t*)src + at + off));
#pragma unroll
            for (int f = 0; f < N; ++f)
                if (!MIXED || f < n) COPY_ST((MCCLX_GLOBAL Packet*)((MCCLX_GLOBAL uint8_t*)dst[f] + at + off), v);
        }
    }
    if (blockIdx.x == 0) {
        auto byte = [&](uint64_t i) {
            const uint8_t x = ((const MCCLX_GLOBAL uint8_t*)src)[i];
#pragma unroll
            for (int f = 0; f < N; ++f)
                if (!MIXED || f < n) ((MCCLX_GLOBAL uint8_t*)dst[f])[i] = x;
        };
        for (uint32_t i = threadIdx.x; i < head; i += B) byte(i);
        const uint64_t i = head + P * 16 + threadIdx.x;  // fewer than 16 bytes remain
        if (i < nbytes) byte(i);
    }
}

// One source to N destinations, one destination after another.  copy_few_kernel reads a packet once and
// stores it N times: N + 1 streams at a time, and the memory channels switch rows between them.  Here a
// piece of the source goes to its first destination, then to the next, and then the next piece
// follows: the first pass brings the piece into the L2 caches, the others read it there (ordinary loads; a
// tile's number within the piece decides its XCD, for every destination alike), and memory sees one
// stream of writes.  Bound by those: writes alone run at 6.6-7.2 TB/s, eight streams of them beside one read
// at 6.2.  Eight to eight, us: 8 x 1 MiB 15.9 -> 12.6, 8 x 8 MiB 105 -> 90, 8 x 16 MiB 212 -> 183, 8 x 64 MiB 774 -> 744.
// blockIdx.x is the tile of the piece, blockIdx.y copy and destination, blockIdx.z the piece.  An XCD takes
// 2^group tiles in a row (blocks go to the XCDs in turn): 64 tiles, 512 KiB, 737 us, in turn 773.
template <int N>
__global__ void __launch_bounds__(kFourWaves) copy_spread_kernel(CopyFew a, uint64_t piece, uint32_t group) {
    const uint32_t c = blockIdx.y / N, f = blockIdx.y - c * N;
    const void* src = a.d[c].src;
    void* dst = a.d[c].dst[f];
    uint64_t nbytes = a.d[c].nbytes;
    asm volatile("" : "+s"(src), "+s"(dst), "+s"(nbytes), "+s"(piece), "+s"(group));
    const uint32_t xcd = blockIdx.x % kXcds, n = blockIdx.x / kXcds;
    const uint32_t tile = (((n >> group) * kXcds + xcd) << group) + (n & ((1u << group) - 1));
    const uint32_t mis = (0u - (uint32_t)reinterpret_cast<uintptr_t>(dst)) & 127u;  // packets start on a line of this destination
    const uint32_t head = nbytes < mis ? (uint32_t)nbytes : mis;
    const uint64_t whole = (nbytes - head) / 16 * 16;
    const uint64_t first = blockIdx.z * piece + (uint64_t)tile * kSpreadTile;
    const MCCLX_GLOBAL uint8_t* gs = (const MCCLX_GLOBAL uint8_t*)src;
    MCCLX_GLOBAL uint8_t* gd = (MCCLX_GLOBAL uint8_t*)dst;
    if (first < whole) {
        const MCCLX_GLOBAL uint8_t* ps = gs + head + first;
        MCCLX_GLOBAL uint8_t* pd = gd + head + first;
        constexpr uint32_t half = kSpreadTile / 2;
        const uint32_t off = threadIdx.x * 16u;
        if (whole - first >= kSpreadTile) {
            const u32x4 v0 = *(const MCCLX_GLOBAL Packet*)(ps + off), v1 = *(const MCCLX_GLOBAL Packet*)(ps + half + off);
            COPY_ST((MCCLX_GLOBAL Packet*)(pd + off), v0);
            COPY_ST((MCCLX_GLOBAL Packet*)(pd + half + off), v1);
        } else {
            const uint32_t left = (uint32_t)(whole - first);
            if (off < left) COPY_ST((MCCLX_GLOBAL Packet*)(pd + off), *(const MCCLX_GLOBAL Packet*)(ps + off));
            if (half + off < left)
                COPY_ST((MCCLX_GLOBAL Packet*)(pd + half + off), *(const MCCLX_GLOBAL Packet*)(ps + half + off));
        }
    }
    if (blockIdx.x == 0 && blockIdx.z == 0) {
        if (threadIdx.x < head) gd[threadIdx.x] = gs[threadIdx.x];
        const uint64_t i = head + whole + threadIdx.x;  // fewer than 16 bytes remain
        if (i < nbytes) gd[i] = gs[i];
    }
}

// One-directional streams with the copy kernel's access shape: what a launch
// that only reads, or only writes, nbytes costs.  The read keeps its loads alive
// through a store no input takes (packet XOR == magic, into the buffer's first
// word).
template <bool WRITE>
__global__ void __launch_bounds__(kBlock) stream_probe_kernel(uint8_t* buf, uint64_t nbytes, uint32_t magic) {
    typedef Packet V;
    MCCLX_GLOBAL uint8_t* g = (MCCLX_GLOBAL uint8_t*)buf;
    const uint64_t P = nbytes / 16;
    const uint64_t p = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    if (p >= P) return;
    if (WRITE) {
        const uint32_t w = (uint32_t)p * 2654435761u;
        COPY_ST((MCCLX_GLOBAL V*)(g + p * 16), (u32x4{w, w ^ magic, ~w, w + magic}));
    } else {
        u32x4 v = COPY_LD((const MCCLX_GLOBAL V*)(g + p * 16));
        const uint32_t x = v[0] ^ v[1] ^ v[2] ^ v[3];
        if (x == magic) *(MCCLX_GLOBAL uint32_t*)g = x;
    }
}

// The mark of mcclx_queue_wait: the number travels in the arguments, so the one wave that runs reads
// no memory.  Bound by the store's way over the link (4 us in a trace, to its acknowledgement; the host
// sees the number before that).
__global__ void __launch_bounds__(64) word_kernel(uint64_t* word, uint64_t number) {
    if (threadIdx.x == 0) __hip_atomic_store(word, number, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

__device__ __forceinline__ uint32_t uni32(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ uint64_t uni64(uint64_t v) {
    return ((uint64_t)uni32((uint32_t)(v >> 32)) << 32) | uni32((uint32_t)v);
}

// Many copies, one launch: work item w is tile (w - first_item[c]) of copy c.
// A tile is kManyU * kBlock packets of 16 bytes (16 KiB); tile 0 also moves the
// bytes behind the last whole packet.  The loop bound is fixed at launch.
constexpr int kManyU = 4;

// Up to kCopyDsts destinations a copy (FAN), or one.
template <bool FAN>
__global__ void __launch_bounds__(kBlock) copy_many_kernel(CopyTable t) {
    constexpr int D = FAN ? kCopyDsts : 1;
    const uint64_t span = (uint64_t)kManyU * kBlock;
    for (uint32_t w = blockIdx.x; w < t.total_items; w += gridDim.x) {
        uint32_t c, tile;
        if (t.uniform_items) {  // every copy has the same number of tiles: no search
            c = w / t.uniform_items;
            tile = w - c * t.uniform_items;
        } else if (t.item_map) {
            const uint2 m = t.item_map[w];
            c = m.x;
            tile = m.y;
        } else {
            uint32_t lo = 0, hi = t.n;  // first_item[lo] <= w < first_item[hi]
            while (hi - lo > 1) {
                uint32_t mid = (lo + hi) >> 1;
                if ((uint32_t)t.first_item[mid] <= w) lo = mid; else hi = mid;
            }
            c = lo;
            tile = w - (uint32_t)t.first_item[c];
        }
        c = uni32(c);
        tile = uni32(tile);
        const CopyDesc* __restrict__ d = t.descs + c;
        const MCCLX_GLOBAL uint8_t* gs = (const MCCLX_GLOBAL uint8_t*)uni64(reinterpret_cast<uint64_t>(d->src));
        const uint32_t n = FAN ? uni32((uint32_t)d->n) : 1u;
        MCCLX_GLOBAL uint8_t* gd[D];
#pragma unroll
        for (int f = 0; f < D; ++f) gd[f] = (MCCLX_GLOBAL uint8_t*)uni64(reinterpret_cast<uint64_t>(d->dst[f]));
        auto deliver = [&](uint64_t off, u32x4 v) {
            COPY_ST((MCCLX_GLOBAL Packet*)(gd[0] + off), v);
            if constexpr (FAN) {
#pragma unroll
                for (uint32_t f = 1; f < (uint32_t)kCopyDsts; ++f)
                    if (f < n) COPY_ST((MCCLX_GLOBAL Packet*)(gd[f] + off), v);
            }
        };
        const uint64_t nbytes = uni64(d->nbytes);
        const uint64_t P = nbytes / 16;
        const uint64_t base = (uint64_t)tile * span;
        if (base + span <= P) {
            u32x4 v[kManyU];
#pragma unroll
            for (int u = 0; u < kManyU; ++u)
                v[u] = COPY_LD((const MCCLX_GLOBAL Packet*)(gs + (base + (uint64_t)u * kBlock + threadIdx.x) * 16));
#pragma unroll
            for (int u = 0; u < kManyU; ++u) deliver((base + (uint64_t)u * kBlock + threadIdx.x) * 16, v[u]);
        } else {
            for (uint64_t p = base + threadIdx.x; p < P; p += kBlock)
                deliver(p * 16, COPY_LD((const MCCLX_GLOBAL Packet*)(gs + p * 16)));
        }
        if (tile == 0) {
            const uint64_t i = P * 16 + threadIdx.x;
            if (i < nbytes) {
                const uint8_t x = gs[i];
#pragma unroll
                for (int f = 0; f < D; ++f)
                    if ((uint32_t)f < n) gd[f][i] = x;
            }
        }
    }
}
}  // namespace

uint64_t copy_items(uint64_t nbytes) {
    const uint64_t span = (uint64_t)kManyU * kBlock * 16;
    uint64_t n = (nbytes + span - 1) / span;
    return n ? n : (nbytes ? 1 : 0);
}

hipError_t launch_copy_many(hipStream_t st, const CopyTable& t, int most, uint32_t max_blocks) {
    if (t.total_items == 0) return hipSuccess;
    const dim3 grid(t.total_items < max_blocks ? t.total_items : max_blocks), block(kBlock);
    if (most > 1)
        copy_many_kernel<true><<<grid, block, 0, st>>>(t);
    else
        copy_many_kernel<false><<<grid, block, 0, st>>>(t);
    return hipGetLastError();
}

hipError_t launch_word(hipStream_t st, uint64_t* word, uint64_t number) {
    word_kernel<<<dim3(1), dim3(64), 0, st>>>(word, number);
    return hipGetLastError();
}

hipError_t launch_stream_probe(hipStream_t st, void* buf, uint64_t nbytes, bool write) {
    const uint64_t g = (nbytes / 16 + kBlock - 1) / kBlock;
    if (g == 0) return hipSuccess;
    if (g >> 31) return hipErrorInvalidValue;
    uint8_t* b = static_cast<uint8_t*>(buf);
    if (write)
        stream_probe_kernel<true><<<dim3((uint32_t)g), dim3(kBlock), 0, st>>>(b, nbytes, 0x9E3779B9u);
    else
        stream_probe_kernel<false><<<dim3((uint32_t)g), dim3(kBlock), 0, st>>>(b, nbytes, 0x9E3779B9u);
    return hipGetLastError();
}

namespace {
template <int N, bool MIXED = false>
hipError_t launch_copy_few_n(hipStream_t st, const CopyFew& a) {
    uint64_t longest = 0, moved = 0;
    for (uint32_t i = 0; i < a.n; ++i) {
        longest = a.d[i].nbytes > longest ? a.d[i].nbytes : longest;
        moved += a.d[i].nbytes * (1 + a.d[i].n);
    }
    if (longest == 0) return hipSuccess;
    const uint64_t waves = (longest + 1023) / 1024;
    // (a source off the lines of its one destination: neighbours share lines, as off_lines of the folds
    // says: 120 MB out of pinned host memory 2497 -> 2307 us, level in HBM)
    bool off = false;
    if constexpr (N == 1)
        for (uint32_t i = 0; i < a.n; ++i)
            off |= ((reinterpret_cast<uintptr_t>(a.d[i].src) ^ reinterpret_cast<uintptr_t>(a.d[i].dst[0])) & 127u) != 0;
    const bool four = off || waves * a.n < kOneWaveBlocksFrom;
    const uint64_t g = four ? (waves + 3) / 4 : waves;
    if (g * (four ? kFourWaves : kOneWave) >> 32) return hipErrorInvalidValue;
    const dim3 grid((uint32_t)g, a.n);
    // Where copies of different numbers of destinations share the launch, few blocks have all N: the
    // waves that copies of three destinations get are right for every mixture tried (67 MB from nine
    // ranks to all nine, eight destinations and one in turn, 1465 -> 1065 us; twelve ranks, eight and
    // four, 609 -> 450).
    const uint32_t lds = resident_lds(moved, MIXED ? 16 * (3 + 1) : 16 * (N + 1), N, kLaneBytesCopy, kResidentMinBytesCopy);
    if (four)
        copy_few_kernel<N, kFourWaves, MIXED><<<grid, dim3(kFourWaves), lds, st>>>(a);
    else
        copy_few_kernel<N, kOneWave, MIXED><<<grid, dim3(kOneWave), lds, st>>>(a);
    return hipGetLastError();
}

// Four blocks a CU: their writes lie close together (16 / 12 / 8 waves a CU, 8 x 64 MiB to eight: 735 / 734 / 763 us, two
// copies of 8 MiB to two 8.7 / 8.9 / 9.3).
constexpr uint32_t kSpreadLds = 163840 / 4;

// Pieces of 8 to 12 MiB (1 to 1.5 MiB of each XCD's L2; 8 x 64 MiB to eight with 4 / 8 / 16 MiB: 755 / 737 / 735 us, 4 x 32 MiB
// to four 97.0 / 95.2 / 95.2).  A source is cut where all pieces have one length and the XCDs take long runs of tiles, with at
// most one block in sixteen without work; the shortest, of fewer than 16 tiles, have up to seven tiles beside theirs.
constexpr uint64_t kSpreadTiles = (8u << 20) / kSpreadTile;
struct SpreadShape {
    uint64_t pieces, tiles;  // tiles of a piece
    uint32_t group;
};
SpreadShape spread_shape(uint64_t need) {  // tiles of the longest source, one at least
    constexpr uint32_t kGroup = 6;
    if (need > 16 * kSpreadTiles) return {(need + kSpreadTiles - 1) / kSpreadTiles, kSpreadTiles, kGroup};
    const uint64_t most = (need + kSpreadTiles - 1) / kSpreadTiles, least = (2 * need + 3 * kSpreadTiles - 1) / (3 * kSpreadTiles);
    for (uint32_t g = kGroup;; --g)
        for (uint64_t p = most; p >= least; --p) {
            const uint64_t step = kXcds << g, tiles = ((need + p - 1) / p + step - 1) / step * step;
            if (g == 0 || (p * tiles - need) * 16 <= need) return {p, tiles, g};
        }
}
// From 6 MB moved on pieces are 0.97-1.3 times as fast on the device, one, two or a rank's number of sources to two to eight
// destinations, 1.1 times on average; below that 0.86-1.2 times, worst where many small sources leave blocks without work
// (eight of 16 KB to eight 2.14 and 2.46 us).  Looking up where the memory lies takes the host 0.3 to 0.7 us, so whole calls
// gain from 20 MB on (allgathers of 8 x 20 / 128 / 256 KB 17.6 / 18.0 / 18.9 us without, 18.0 / 18.5 / 18.7 with; of 8 x 1 / 2 / 4 MB
// 29.2 / 42.4 / 65.1 and 26.4 / 35.9 / 56.8).
// To two or three, pieces pay while the launch is small: 50 / 100 / 200 / 400 MB moved to two 1.2 / 1.12 / 0.95 / 0.94 times as
// fast, to three 1.19 / 1.19 / 0.99 / 1.0; to four and more 1.0-1.26 times up to 5.6 GB.
constexpr uint64_t kSpreadFrom = 20'000'000, kSpreadToThree = 150'000'000;

template <int N>
hipError_t launch_copy_spread(hipStream_t st, const CopyFew& a) {
    uint64_t longest = 0;
    for (uint32_t i = 0; i < a.n; ++i) longest = a.d[i].nbytes > longest ? a.d[i].nbytes : longest;
    if (longest == 0) return hipSuccess;
    const SpreadShape p = spread_shape((longest + kSpreadTile - 1) / kSpreadTile);
    if (p.pieces > 65535) return hipErrorInvalidValue;
    copy_spread_kernel<N><<<dim3((uint32_t)p.tiles, N * a.n, (uint32_t)p.pieces), dim3(kFourWaves), kSpreadLds, st>>>(
        a, p.tiles * kSpreadTile, p.group);
    return hipGetLastError();
}
}  // namespace

bool copy_spread_pays(const CopyFew& a) {
    if (a.n == 0 || a.d[0].n < 2) return false;
    uint64_t moved = 0;
    for (uint32_t i = 0; i < a.n; ++i) {
        if (a.d[i].n != a.d[0].n) return false;
        moved += a.d[i].nbytes * (1 + a.d[i].n);
    }
    return moved >= kSpreadFrom && (a.d[0].n >= 4 || moved < kSpreadToThree);
}

hipError_t launch_copy_few(hipStream_t st, const CopyFew& a, bool spread) {
    if (a.n == 0 || a.n > (uint32_t)kFewCopies) return a.n ? hipErrorInvalidValue : hipSuccess;
    for (uint32_t i = 1; i < a.n; ++i)
        if (a.d[i].n != a.d[0].n) return launch_copy_few_n<kCopyDsts, true>(st, a);
    if (spread) switch (a.d[0].n) {
        case 2: return launch_copy_spread<2>(st, a);
        case 3: return launch_copy_spread<3>(st, a);
        case 4: return launch_copy_spread<4>(st, a);
        case 5: return launch_copy_spread<5>(st, a);
        case 6: return launch_copy_spread<6>(st, a);
        case 7: return launch_copy_spread<7>(st, a);
        case 8: return launch_copy_spread<8>(st, a);
        default: return hipErrorInvalidValue;
    }
    switch (a.d[0].n) {
        case 1: return launch_copy_few_n<1>(st, a);
        case 2: return launch_copy_few_n<2>(st, a);
        case 3: return launch_copy_few_n<3>(st, a);
        case 4: return launch_copy_few_n<4>(st, a);
        case 5: return launch_copy_few_n<5>(st, a);
        case 6: return launch_copy_few_n<6>(st, a);
        case 7: return launch_copy_few_n<7>(st, a);
        case 8: return launch_copy_few_n<8>(st, a);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_copy(hipStream_t st, void* dst, const void* src, uint64_t nbytes) {
    CopyFew a;
    a.d[0] = CopyDesc{src, nbytes, 1, {dst}};
    a.n = 1;
    return launch_copy_few(st, a, false);
}

}  // namespace mcclx
