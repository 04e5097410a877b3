// LogUp multiplicities: how often each table entry was looked up (prover/kernels/gl_extras.cuh:118-150).
//
// Counting with one global atomic per look-up runs at 20 G per second whatever the table (1.5 M look-ups in a 2^16 table:
// 77 us) and slower the more look-ups share an entry.  Here a workgroup counts its share of the look-ups in LDS, for a
// slice of up to 32768 entries, leaves its counts as one row of a workspace, and a second launch adds up the rows: 13 us
// for the same call.  A table of up to 1024 entries is kept several times over, one copy per group of lanes, so that
// look-ups of one entry do not queue up.
//
// A table that is not literally 0 .. T-1 is first turned into a hash table (linear probing, at most half full) of
// entry -> first index that holds it; a look-up then costs a probe or two where the search from the front costs half the
// table.
#include "common.hpp"
#include "gl_field.hpp"

namespace {

constexpr int BLOCK = 256;
constexpr int COUNT_THREADS = 1024;
constexpr int SLICE = 32768;                   // counters of a workgroup: 128 KiB of LDS
constexpr int MAX_COPIES = 32;
constexpr i64 MAX_GROUPS = 256;                // rows of the workspace per slice
constexpr u32 EMPTY = 0xFFFFFFFFu;

struct Slot {                                  // one entry of the hash table
    u64 key;
    u32 index, unused;
};

// Fibonacci hashing into 2^bits slots
__device__ __forceinline__ u32 slot_of(u64 key, int bits) { return (u32)((key * 0x9E3779B97F4A7C15ull) >> (64 - bits)); }

__global__ __launch_bounds__(BLOCK) void k_clear_slots(Slot *slots, i64 n) {
    const i64 stride = (i64)gridDim.x * BLOCK;
    for (i64 i = (i64)blockIdx.x * BLOCK + threadIdx.x; i < n; i += stride) slots[i].index = EMPTY;
}

// A slot belongs to the first index that claims it; later indices of the same entry lower it to the smallest.  The entry
// of a claimed slot is read from the table (every index it ever holds has the same one).  Ends after at most 2^bits
// probes, and half of the slots stay empty.
__global__ __launch_bounds__(BLOCK) void k_insert(const u64 *__restrict__ table, i64 n_table, Slot *slots, int bits) {
    const i64 stride = (i64)gridDim.x * BLOCK;
    const u32 mask = (1u << bits) - 1;
    for (i64 j = (i64)blockIdx.x * BLOCK + threadIdx.x; j < n_table; j += stride) {
        const u64 key = table[j];
        u32 h = slot_of(key, bits);
        for (u32 probes = 0; probes <= mask; ++probes, h = (h + 1) & mask) {
            const u32 was = atomicCAS(&slots[h].index, EMPTY, (u32)j);
            if (was == EMPTY) {
                slots[h].key = key;
                break;
            }
            if (table[was] == key) {
                atomicMin(&slots[h].index, (u32)j);
                break;
            }
        }
    }
}

__global__ __launch_bounds__(BLOCK) void k_clear_counts(u64 *mult, i64 n) {
    const i64 stride = (i64)gridDim.x * BLOCK;
    for (i64 i = (i64)blockIdx.x * BLOCK + threadIdx.x; i < n; i += stride) mult[i] = 0;
}

// the index a value counts for, or at least n_table for none
template <bool RANGE>
__device__ __forceinline__ u64 index_of(u64 x, const Slot *__restrict__ slots, int bits) {
    if (RANGE) return x;
    const u32 mask = (1u << bits) - 1;
    u32 h = slot_of(x, bits);
    for (u32 probes = 0; probes <= mask; ++probes, h = (h + 1) & mask) {
        const ulonglong2 s = *reinterpret_cast<const ulonglong2 *>(slots + h);
        if ((u32)s.y == EMPTY) break;
        if (s.x == x) return (u32)s.y;
    }
    return ~0ull;
}

// Workgroup (slice, group): counts of the entries slice * SLICE .. of the group's share of x.  `copies` (a power of two)
// interleaved counters per entry.  rows: the group's row of n_table counts, or null when there is one group: the counts go
// straight to mult.
template <bool RANGE>
__global__ __launch_bounds__(COUNT_THREADS) void k_count(const u64 *__restrict__ x, i64 n_x, i64 per_group, const Slot *__restrict__ slots, int bits,
                                                         i64 n_table, int copies, u32 *rows, u64 *mult, int accumulate) {
    extern __shared__ u32 counts[];
    const int tid = threadIdx.x;
    const i64 base = (i64)blockIdx.x * SLICE, group = blockIdx.y;
    const int mine = n_table - base < SLICE ? (int)(n_table - base) : SLICE;
    const int n_counts = mine * copies;
    // the launch's LDS is a whole number of 16-byte words
    for (int i = tid; i < (n_counts + 3) / 4; i += COUNT_THREADS) reinterpret_cast<uint4 *>(counts)[i] = make_uint4(0, 0, 0, 0);
    __syncthreads();
    const i64 lo = group * per_group, hi = lo + per_group < n_x ? lo + per_group : n_x;
    const int copy = tid & (copies - 1);
    constexpr int UN = 4;                      // look-ups of a thread in flight
    for (i64 i0 = lo + tid; i0 < hi; i0 += UN * COUNT_THREADS) {
        u64 v[UN];
#pragma unroll
        for (int u = 0; u < UN; ++u) v[u] = i0 + u * COUNT_THREADS < hi ? x[i0 + u * COUNT_THREADS] : 0;
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            if (i0 + u * COUNT_THREADS < hi) {
                const u64 at = index_of<RANGE>(v[u], slots, bits) - (u64)base;
                if (at < (u64)mine) atomicAdd(&counts[(int)at * copies + copy], 1u);
            }
        }
    }
    __syncthreads();
    if (rows && copies == 1 && (mine & 3) == 0 && (n_table & 3) == 0) {        // 16-byte aligned rows
        uint4 *to = reinterpret_cast<uint4 *>(rows + group * n_table + base);
        for (int i = tid; i < mine / 4; i += COUNT_THREADS) to[i] = reinterpret_cast<const uint4 *>(counts)[i];
        return;
    }
    for (int i = tid; i < mine; i += COUNT_THREADS) {
        u32 c = 0;
        for (int k = 0; k < copies; ++k) c += counts[i * copies + ((k + tid) & (copies - 1))];
        if (rows) rows[group * n_table + base + i] = c;
        else mult[base + i] = accumulate ? mult[base + i] + c : (u64)c;
    }
}

// mult[j] (+)= sum over the rows: 64 entries per workgroup, the rows dealt over its four wavefronts, eight in flight
__global__ __launch_bounds__(BLOCK) void k_add_rows(const u32 *__restrict__ rows, int groups, i64 n_table, u64 *mult, int accumulate) {
    __shared__ u64 part[BLOCK / 64][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const i64 j = (i64)blockIdx.x * 64 + lane;
    u64 sum = 0;
    if (j < n_table) {
        constexpr int UN = 8;
        for (int g0 = w; g0 < groups; g0 += UN * (BLOCK / 64)) {
            u32 c[UN];
#pragma unroll
            for (int u = 0; u < UN; ++u) {
                const int g = g0 + u * (BLOCK / 64);
                c[u] = g < groups ? rows[(i64)g * n_table + j] : 0;
            }
#pragma unroll
            for (int u = 0; u < UN; ++u) sum += c[u];
        }
    }
    part[w][lane] = sum;
    __syncthreads();
    if (w == 0 && j < n_table) {
        sum = part[0][lane] + part[1][lane] + part[2][lane] + part[3][lane];
        mult[j] = accumulate ? mult[j] + sum : sum;
    }
}

// one global atomic per look-up, through the hash table where there is one
template <bool RANGE>
__global__ __launch_bounds__(BLOCK) void k_count_global(const u64 *__restrict__ x, i64 n_x, const Slot *__restrict__ slots, int bits, i64 n_table,
                                                        unsigned long long *__restrict__ mult) {
    const i64 stride = (i64)gridDim.x * BLOCK;
    for (i64 i = (i64)blockIdx.x * BLOCK + threadIdx.x; i < n_x; i += stride) {
        const u64 at = index_of<RANGE>(x[i], slots, bits);
        if (at < (u64)n_table) atomicAdd(&mult[at], 1ULL);
    }
}

// the same without a hash table, the table searched from the front: no workspace
__global__ __launch_bounds__(BLOCK) void k_lookup_mult(const u64 *__restrict__ x, i64 n_x, const u64 *__restrict__ table, i64 n_table,
                                                       i64 t_len_range, unsigned long long *__restrict__ mult) {
    const i64 stride = (i64)gridDim.x * BLOCK;
    for (i64 i = (i64)blockIdx.x * BLOCK + threadIdx.x; i < n_x; i += stride) {
        const u64 xi = x[i];
        if (t_len_range > 0) {
            if (xi < (u64)t_len_range) atomicAdd(&mult[xi], 1ULL);
            continue;
        }
        for (i64 j = 0; j < n_table; ++j) {
            if (table[j] == xi) {
                atomicAdd(&mult[j], 1ULL);
                break;
            }
        }
    }
}

inline unsigned capped_grid(i64 work_items) {
    i64 b = (work_items + BLOCK - 1) / BLOCK;
    return (unsigned)(b < 1 ? 1 : (b > 256 * 32 ? 256 * 32 : b));
}

struct Plan {
    bool direct;                               // one global atomic per look-up
    i64 slices, groups;
    int copies, bits;
    size_t slot_bytes, row_bytes;
};

Plan make_plan(i64 n_x, i64 n_table, bool range) {
    Plan L = {};
    L.bits = 1;
    while (((i64)1 << L.bits) < 2 * n_table) ++L.bits;
    L.slot_bytes = range ? 0 : sizeof(Slot) << L.bits;
    L.slices = (n_table + SLICE - 1) / SLICE;
    // Few look-ups, spread over many entries: 30000 in a 2^16 table take 3.6 us and 2.5 us for clearing the counts, 11 us
    // through the histogram.  And a table of many slices: all of them read all look-ups, 10 us a slice for 2^24 of them
    // against 711 us of atomics in all.
    L.direct = (range && n_table >= 8192 && n_x <= 131072) || L.slices > 64;
    if (L.direct) return L;
    // a workgroup per CU, but no more rows than look-ups are worth: clearing and storing a slice's counters takes as long
    // as some eight thousand look-ups
    L.groups = (n_x + 8191) / 8192;
    if (L.groups * L.slices > MAX_GROUPS) L.groups = MAX_GROUPS / L.slices;
    if (L.groups < (n_x >> 31) + 1) L.groups = (n_x >> 31) + 1;        // a group's counters have 32 bits
    L.copies = 1;
    while (L.copies < MAX_COPIES && n_table * L.copies * 2 <= SLICE) L.copies *= 2;
    L.row_bytes = L.groups > 1 ? (size_t)L.groups * n_table * sizeof(u32) : 0;
    return L;
}

}  // namespace

extern "C" {

int vi_lookup_multiplicities(const uint64_t *x, int64_t n_x, const uint64_t *table, int64_t n_table, int table_is_range,
                             uint64_t *mult, void *stream) {
    if (n_x < 0 || n_table < 0) return vi::fail(VI_EINVAL, "vi_lookup_multiplicities: n_x = %lld, n_table = %lld", (long long)n_x, (long long)n_table);
    if (n_x == 0 || n_table == 0) return VI_OK;
    if (!x || !mult || (!table_is_range && !table)) return vi::fail(VI_EINVAL, "vi_lookup_multiplicities: null pointer");
    hipLaunchKernelGGL(k_lookup_mult, dim3(capped_grid(n_x)), dim3(BLOCK), 0, (hipStream_t)stream, x, (i64)n_x, table, (i64)n_table,
                       (i64)(table_is_range ? n_table : 0), (unsigned long long *)mult);
    VI_LAUNCH_CHECK("k_lookup_mult");
    return VI_OK;
}

size_t vi_lookup_histogram_workspace_bytes(int64_t n_x, int64_t n_table, int table_is_range) {
    if (n_x <= 0 || n_table <= 0) return 0;
    const Plan L = make_plan(n_x, n_table, table_is_range != 0);
    return L.slot_bytes + L.row_bytes;
}

int vi_lookup_histogram(const uint64_t *x, int64_t n_x, const uint64_t *table, int64_t n_table, int table_is_range, int accumulate,
                        uint64_t *mult, void *ws, size_t ws_bytes, void *stream) {
    if (n_x < 0 || n_table < 0 || n_table > ((int64_t)1 << 30))
        return vi::fail(VI_EINVAL, "vi_lookup_histogram: n_x = %lld, n_table = %lld", (long long)n_x, (long long)n_table);
    if (n_table == 0 || (n_x == 0 && accumulate)) return VI_OK;
    if ((n_x > 0 && !x) || !mult || (!table_is_range && !table)) return vi::fail(VI_EINVAL, "vi_lookup_histogram: null pointer");
    const Plan L = make_plan(n_x, n_table, table_is_range != 0);
    const size_t need = L.slot_bytes + L.row_bytes;
    if (need && (!ws || ws_bytes < need)) return vi::fail(VI_ENOMEM, "vi_lookup_histogram: workspace below %zu bytes", need);
    hipStream_t s = (hipStream_t)stream;
    Slot *slots = (Slot *)ws;
    u32 *rows = L.row_bytes ? (u32 *)((char *)ws + L.slot_bytes) : nullptr;
    if (!table_is_range) {
        hipLaunchKernelGGL(k_clear_slots, dim3(capped_grid((i64)1 << L.bits)), dim3(BLOCK), 0, s, slots, (i64)1 << L.bits);
        VI_LAUNCH_CHECK("k_clear_slots");
        hipLaunchKernelGGL(k_insert, dim3(capped_grid(n_table)), dim3(BLOCK), 0, s, table, (i64)n_table, slots, L.bits);
        VI_LAUNCH_CHECK("k_insert");
    }
    if (L.direct) {
        if (!accumulate) {
            hipLaunchKernelGGL(k_clear_counts, dim3(capped_grid(n_table)), dim3(BLOCK), 0, s, mult, (i64)n_table);
            VI_LAUNCH_CHECK("k_clear_counts");
        }
        if (n_x == 0) return VI_OK;
        if (table_is_range)
            hipLaunchKernelGGL(k_count_global<true>, dim3(capped_grid(n_x)), dim3(BLOCK), 0, s, x, (i64)n_x, (const Slot *)slots, L.bits, (i64)n_table, (unsigned long long *)mult);
        else
            hipLaunchKernelGGL(k_count_global<false>, dim3(capped_grid(n_x)), dim3(BLOCK), 0, s, x, (i64)n_x, (const Slot *)slots, L.bits, (i64)n_table, (unsigned long long *)mult);
        VI_LAUNCH_CHECK("k_count_global");
        return VI_OK;
    }
    const i64 per = (n_x + L.groups - 1) / L.groups;
    const i64 in_slice = n_table < SLICE ? n_table : SLICE;
    const size_t lds = ((size_t)in_slice * L.copies * sizeof(u32) + 15) & ~(size_t)15;
    const dim3 grid((unsigned)L.slices, (unsigned)L.groups);
    // more than 64 KiB of dynamic LDS has to be asked for, once per device and kernel
    static std::atomic<unsigned long long> asked{0};
    int dev = 0;
    VI_HIP(hipGetDevice(&dev));
    const unsigned long long bit = 1ull << (dev & 63);
    if (!(asked.load(std::memory_order_acquire) & bit)) {
        VI_HIP(hipFuncSetAttribute((const void *)k_count<true>, hipFuncAttributeMaxDynamicSharedMemorySize, SLICE * (int)sizeof(u32)));
        VI_HIP(hipFuncSetAttribute((const void *)k_count<false>, hipFuncAttributeMaxDynamicSharedMemorySize, SLICE * (int)sizeof(u32)));
        asked.fetch_or(bit, std::memory_order_release);
    }
    if (table_is_range)
        hipLaunchKernelGGL(k_count<true>, grid, dim3(COUNT_THREADS), lds, s, x, (i64)n_x, per, (const Slot *)slots, L.bits, (i64)n_table, L.copies, rows, mult, accumulate);
    else
        hipLaunchKernelGGL(k_count<false>, grid, dim3(COUNT_THREADS), lds, s, x, (i64)n_x, per, (const Slot *)slots, L.bits, (i64)n_table, L.copies, rows, mult, accumulate);
    VI_LAUNCH_CHECK("k_count");
    if (rows) {
        hipLaunchKernelGGL(k_add_rows, dim3((unsigned)((n_table + 63) / 64)), dim3(BLOCK), 0, s, (const u32 *)rows, (int)L.groups, (i64)n_table, mult, accumulate);
        VI_LAUNCH_CHECK("k_add_rows");
    }
    return VI_OK;
}

}  // extern "C"
