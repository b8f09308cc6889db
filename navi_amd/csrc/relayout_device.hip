// relayout_device.hip — the record layout and the cell tables (see relayout.cpp)
// made on the GPU from DAG words that are already there: scene loading without
// the copy of the words back to the host, the conversion there and the upload
// of its result.
//
// Records are numbered as relayout.cpp numbers them, breadth-first with a
// node's children in octant order, so both give the same arrays bit for bit.
// One level of the tree is three kernels over its candidates (record, octant):
// every candidate that names an unnumbered internal word bids for it with its
// own position (an atomic minimum: the first in the host's order wins), the
// winners are counted per workgroup, and every workgroup adds up the counts of
// those before it and numbers its own. The level's bounds stay in device
// memory, so kLevels levels are enqueued at once and the host reads the result
// once; levels past the last one find an empty range.
//
// What bounds it: each level waits for its predecessor, three launches of 3 to
// 5 us; the last levels hold most records and read a node, a table word and a
// child word per slot (scattered, 12 bytes used of three 64-byte lines). A
// 1024^3 scene (4.3 M words, 610 K records) with its cell table: 0.5 ms, where
// the host took 81 ms; the words' upload before it takes 1.3 ms.
//
// DAGs that this does not cover are left to the host: a one-leaf DAG, leaves of
// semantic 0x7fff or above (they need the leaf table, in order of first sight),
// more than kLevels levels, and records reached from two levels (the longest
// chain, which decides what an out-of-range child means, is then not the level
// count).
#include <hip/hip_runtime.h>

#include <cstdint>

#include "navi_trace.h"

namespace navi {

int set_error(int code, const char* fmt, ...);

namespace {

constexpr uint32_t kSlotVoid = 0x7fffffffu;
constexpr uint32_t kSlotFault = 0x7ffffffeu;
constexpr uint32_t kSlotBadChild = 0x7ffffffdu;  // lowest terminal slot value
constexpr uint32_t kUnassigned = 0xffffffffu;
constexpr uint32_t kBid = 0x80000000u;  // a bid (record * 8 + octant) for a word, not its record yet
// levels of records: 31 leave every slot at depth 31 or less, above the 32-level
// limit of kernel.cu:136, where a bad child index is a fault
constexpr uint32_t kLevels = 31;
constexpr uint32_t kBlocks = 1024, kThreads = 256;  // of the kernels of a level: four workgroups per CU

// words of the caller's state buffer
enum : uint32_t {
    kStateBounds = 0,  // [kLevels + 2]: first record of each level, then the record count
    kStateFlags = 40,  // kSeen* bits
    kStateRoot = 41,   // the root word's bit 63
    kStateCounts = 64  // [kBlocks]: the level's winners per workgroup
};
constexpr uint32_t kStateWords = kStateCounts + kBlocks;
static_assert(kStateWords <= NAVI_RELAYOUT_STATE_WORDS, "the header's state size");
enum : uint32_t { kSeenNegative = 1u, kSeenTableLeaf = 2u, kSeenCross = 4u };

__device__ __forceinline__ void raise(uint32_t* state, uint32_t bits) {
    if ((__hip_atomic_load(state + kStateFlags, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & bits) != bits)
        atomicOr(state + kStateFlags, bits);
}

// The candidate `oct` of a node word: its slot when that is terminal, or the
// child's word index in *child (returned kSlotBadChild - 1, which no slot is).
constexpr uint32_t kInternal = kSlotBadChild - 1u;
__device__ __forceinline__ uint32_t candidate(const uint64_t* __restrict__ words, uint32_t n_words, uint64_t node,
                                              uint32_t oct, uint32_t& child) {
    const uint32_t mask = static_cast<uint32_t>(node >> 55) & 0xffu;
    if (!(mask >> oct & 1u)) return kSlotVoid;
    const uint32_t tab = static_cast<uint32_t>(node) + __popc(mask & ((1u << oct) - 1u));  // as kernel.cu:197
    if (tab >= n_words) return kSlotFault;
    child = static_cast<uint32_t>(words[tab]);
    if (child >= n_words) return kSlotBadChild;
    const uint64_t w = words[child];
    if (w >> 63) return 0x80000000u | (static_cast<uint32_t>(w) & 0x7fffffffu);
    return kInternal;
}

__global__ __launch_bounds__(kThreads) void relayout_init_kernel(const uint64_t* __restrict__ words, uint32_t n_words,
                                                                 uint32_t* __restrict__ mark,
                                                                 uint32_t* __restrict__ order, uint32_t* state) {
    const uint32_t i0 = blockIdx.x * kThreads + threadIdx.x;
    for (uint32_t i = i0; i < n_words; i += gridDim.x * kThreads) mark[i] = i == 0u ? 0u : kUnassigned;
    if (blockIdx.x == 0) {
        const bool leaf = (words[0] >> 63) != 0u;
        if (threadIdx.x <= kLevels + 1u) state[kStateBounds + threadIdx.x] = threadIdx.x == 0u || leaf ? 0u : 1u;
        if (threadIdx.x == 0) {
            order[0] = 0u;
            state[kStateFlags] = 0u;
            state[kStateRoot] = leaf ? 1u : 0u;
        }
    }
}

// The workgroup's run of candidates of level `level`: [lo, hi) of record * 8 + octant.
__device__ __forceinline__ void candidates_of(const uint32_t* state, uint32_t level, uint32_t& lo, uint32_t& hi) {
    const uint32_t r0 = 8u * state[kStateBounds + level], r1 = 8u * state[kStateBounds + level + 1u];
    const uint32_t per = ((r1 - r0 + kBlocks - 1u) / kBlocks + kThreads - 1u) & ~(kThreads - 1u);
    lo = r0 + min(blockIdx.x * per, r1 - r0);
    hi = r0 + min((blockIdx.x + 1u) * per, r1 - r0);
}

// Every unnumbered internal word of the level's candidates takes the lowest
// bid. A word that an earlier level numbered keeps its record (no bid lies
// below a record) and raises kSeenCross.
__global__ __launch_bounds__(kThreads) void relayout_bid_kernel(const uint64_t* __restrict__ words, uint32_t n_words,
                                                                uint32_t* mark, const uint32_t* __restrict__ order,
                                                                uint32_t* state, uint32_t level) {
    uint32_t lo, hi;
    candidates_of(state, level, lo, hi);
    uint32_t seen = 0u;
    for (uint32_t c = lo + threadIdx.x; c < hi; c += kThreads) {
        uint32_t child;
        const uint32_t slot = candidate(words, n_words, words[order[c >> 3]], c & 7u, child);
        if (slot == kInternal) {
            const uint32_t old = atomicMin(mark + child, kBid | c);
            if (!(old & kBid)) seen |= kSeenCross;
        } else if (slot & 0x80000000u) {
            if (slot & 0x8000u) seen |= kSeenNegative;
            if ((slot & 0x7fff0000u) == 0x7fff0000u) seen |= kSeenTableLeaf;
            // (a semantic of 0x8000 or above has its top bit under the slot's bit 31)
            if (words[child] & 0x80000000ull) seen |= kSeenTableLeaf;
        }
    }
    if (seen) raise(state, seen);
}

// The workgroup's winners, [lo, hi) walked in rounds of kThreads.
__global__ __launch_bounds__(kThreads) void relayout_count_kernel(const uint64_t* __restrict__ words, uint32_t n_words,
                                                                  const uint32_t* __restrict__ mark,
                                                                  const uint32_t* __restrict__ order, uint32_t* state,
                                                                  uint32_t level) {
    uint32_t lo, hi;
    candidates_of(state, level, lo, hi);
    __shared__ uint32_t total;
    if (threadIdx.x == 0) total = 0u;
    __syncthreads();
    uint32_t n = 0u;
    for (uint32_t c = lo + threadIdx.x; c < hi; c += kThreads) {
        uint32_t child;
        const uint32_t slot = candidate(words, n_words, words[order[c >> 3]], c & 7u, child);
        n += slot == kInternal && mark[child] == (kBid | c) ? 1u : 0u;
    }
    if (n) atomicAdd(&total, n);
    __syncthreads();
    if (threadIdx.x == 0) state[kStateCounts + blockIdx.x] = total;
}

// Numbers the winners: records from the level's end on, in candidate order.
// The last workgroup writes the next level's end. (A loser of the level reads
// a winner's bid or its record, neither of which is its own bid.)
__global__ __launch_bounds__(kThreads) void relayout_number_kernel(const uint64_t* __restrict__ words, uint32_t n_words,
                                                                   uint32_t* mark, uint32_t* order, uint32_t* state,
                                                                   uint32_t level) {
    uint32_t lo, hi;
    candidates_of(state, level, lo, hi);
    __shared__ uint32_t before, waves[kThreads / 64u];
    if (threadIdx.x == 0) before = 0u;
    __syncthreads();
    uint32_t mine = 0u;
    for (uint32_t b = threadIdx.x; b < blockIdx.x; b += kThreads) mine += state[kStateCounts + b];
    if (mine) atomicAdd(&before, mine);
    __syncthreads();
    uint32_t next = state[kStateBounds + level + 1u] + before;
    if (blockIdx.x == kBlocks - 1u && threadIdx.x == 0)
        state[kStateBounds + level + 2u] = next + state[kStateCounts + blockIdx.x];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    for (uint32_t c0 = lo; c0 < hi; c0 += kThreads) {
        const uint32_t c = c0 + threadIdx.x;
        uint32_t child = 0u;
        const bool wins = c < hi &&
                          candidate(words, n_words, words[order[c >> 3]], c & 7u, child) == kInternal &&
                          mark[child] == (kBid | c);
        const uint64_t m = __ballot(wins);
        if (lane == 0u) waves[wave] = static_cast<uint32_t>(__popcll(m));
        __syncthreads();
        uint32_t at = next;
        for (uint32_t w = 0; w < kThreads / 64u; ++w) {
            if (w < wave) at += waves[w];
            next += waves[w];
        }
        if (wins) {
            at += __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(m >> 32),
                                            __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), 0u));
            mark[child] = at;
            order[at] = child;
        }
        __syncthreads();
    }
}

// The records: one lane per slot, child records as pool indices from `base` on.
__global__ __launch_bounds__(kThreads) void relayout_emit_kernel(const uint64_t* __restrict__ words, uint32_t n_words,
                                                                 const uint32_t* __restrict__ mark,
                                                                 const uint32_t* __restrict__ order, uint32_t n_slots,
                                                                 uint32_t base, uint32_t* __restrict__ records) {
    const uint32_t c = blockIdx.x * kThreads + threadIdx.x;
    if (c >= n_slots) return;
    uint32_t child;
    const uint32_t slot = candidate(words, n_words, words[order[c >> 3]], c & 7u, child);
    records[c] = slot == kInternal ? base + mark[child] : (slot == kSlotBadChild ? kSlotFault : slot);
}

// One lane per cell: what a descent from the root reaches within D levels
// (fill_cells of relayout.cpp).
__global__ __launch_bounds__(kThreads) void cell_table_kernel(const uint32_t* __restrict__ records, uint32_t n_records,
                                                              uint32_t root, uint32_t D, uint64_t* __restrict__ table) {
    const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
    if (i >> (3u * D)) return;
    const uint32_t x = i & ((1u << D) - 1u), y = i >> D & ((1u << D) - 1u), z = i >> (2u * D);
    uint32_t slot = root, d = 0u;
    while (d < D && slot < kSlotBadChild) {
        const uint32_t b = D - 1u - d;
        const uint32_t oct = (x >> b & 1u) | (y >> b & 1u) << 1 | (z >> b & 1u) << 2;
        slot = slot < n_records ? records[8ull * slot + oct] : kSlotFault;
        ++d;
    }
    if (slot == kSlotBadChild) slot = kSlotFault;
    table[i] = static_cast<uint64_t>(slot) | static_cast<uint64_t>(d) << 32;
}

int launched(const char* what) {
    const hipError_t err = hipGetLastError();
    return err == hipSuccess ? NAVI_OK : set_error(NAVI_E_LAUNCH, "%s: %s", what, hipGetErrorString(err));
}

}  // namespace
}  // namespace navi

extern "C" int navi_relayout_device(const uint64_t* words, uint64_t n_words, uint32_t* mark, uint32_t* order,
                                    uint32_t* state, navi_device_layout* layout, void* stream) {
    using namespace navi;
    if (!words || n_words == 0) return set_error(NAVI_E_ARG, "dag must hold at least one word");
    if (!mark || !order || !state || !layout) return set_error(NAVI_E_ARG, "null argument");
    *layout = navi_device_layout{};
    const hipStream_t s = static_cast<hipStream_t>(stream);
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    hipError_t err = hipStreamIsCapturing(s, &status);
    if (err != hipSuccess || status != hipStreamCaptureStatusNone)
        return set_error(NAVI_E_LAUNCH, "a conversion waits for its stream, which is capturing");
    // bids are 31-bit positions of at most n_words records' slots
    if (n_words >= (1ull << 28)) return NAVI_OK;
    const uint32_t n = static_cast<uint32_t>(n_words);
    const dim3 grid(kBlocks), block(kThreads);
    hipLaunchKernelGGL(relayout_init_kernel, grid, block, 0, s, words, n, mark, order, state);
    uint32_t host[kStateCounts] = {};
    // most DAGs end within kFirst levels; the rest are enqueued when they do not
    constexpr uint32_t kFirst = 12;
    uint32_t level = 0;
    const uint32_t* bounds = host + kStateBounds;
    do {
        for (const uint32_t end = level == 0u ? kFirst : kLevels; level < end; ++level) {
            hipLaunchKernelGGL(relayout_bid_kernel, grid, block, 0, s, words, n, mark, order, state, level);
            hipLaunchKernelGGL(relayout_count_kernel, grid, block, 0, s, words, n, mark, order, state, level);
            hipLaunchKernelGGL(relayout_number_kernel, grid, block, 0, s, words, n, mark, order, state, level);
        }
        const int code = launched("relayout");
        if (code != NAVI_OK) return code;
        err = hipMemcpyAsync(host, state, sizeof host, hipMemcpyDeviceToHost, s);
        if (err == hipSuccess) err = hipStreamSynchronize(s);
        if (err != hipSuccess) return set_error(NAVI_E_LAUNCH, "relayout: %s", hipGetErrorString(err));
    } while (level < kLevels && bounds[level] != bounds[level + 1u]);
    if (host[kStateRoot] != 0u || bounds[level] != bounds[level + 1u] ||
        (host[kStateFlags] & (kSeenTableLeaf | kSeenCross)) != 0u)
        return NAVI_OK;
    uint32_t levels = 0;
    while (bounds[levels] != bounds[levels + 1u]) ++levels;
    layout->converted = 1u;
    layout->n_records = bounds[levels];
    layout->max_depth = levels - 1u;
    layout->flags = (host[kStateFlags] & kSeenNegative) ? 0u : NAVI_SCENE_NONNEG_LEAVES;
    return NAVI_OK;
}

extern "C" int navi_relayout_device_records(const uint64_t* words, uint64_t n_words, const uint32_t* mark,
                                            const uint32_t* order, uint32_t n_records, uint32_t rec_offset,
                                            uint32_t* out_records, void* stream) {
    using namespace navi;
    if (!words || !mark || !order || !out_records) return set_error(NAVI_E_ARG, "null argument");
    if (n_words >= (1ull << 28) || n_records == 0u || n_records > n_words)
        return set_error(NAVI_E_ARG, "n_words and n_records must be those of navi_relayout_device");
    const uint32_t slots = 8u * n_records;
    hipLaunchKernelGGL(relayout_emit_kernel, dim3((slots + kThreads - 1u) / kThreads), dim3(kThreads), 0,
                       static_cast<hipStream_t>(stream), words, static_cast<uint32_t>(n_words), mark, order, slots,
                       rec_offset, out_records);
    return launched("records");
}

extern "C" int navi_build_cell_table_device(const uint32_t* records, uint64_t n_records, uint32_t root_slot,
                                            int32_t depth, uint64_t* out_table, void* stream) {
    using namespace navi;
    if (!out_table || (!records && n_records)) return set_error(NAVI_E_ARG, "null argument");
    if (depth < 4 || depth > 7) return set_error(NAVI_E_ARG, "table depth must be in [4, 7]");
    if (n_records > kSlotBadChild) return set_error(NAVI_E_ARG, "record pool exceeds the slot values");
    hipLaunchKernelGGL(cell_table_kernel, dim3(1u << (3 * depth) >> 8), dim3(kThreads), 0,
                       static_cast<hipStream_t>(stream), records, static_cast<uint32_t>(n_records), root_slot,
                       static_cast<uint32_t>(depth), out_table);
    return launched("cell table");
}
