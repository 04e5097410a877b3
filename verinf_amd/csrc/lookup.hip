// LogUp multiplicities: how often each table entry was looked up (prover/kernels/gl_extras.cuh:118-150).
//
// Counting with one global atomic per look-up runs at about 22 G per second whatever the table (1.5 M look-ups in a 2^16
// table: 65 us) and slower the more look-ups share an entry.  Here a workgroup counts its share of the look-ups in LDS, for a
// slice of up to 32768 entries, leaves its counts as one row of a workspace, and a second launch adds up the rows.  Small
// tables are kept several times over, one copy per group of lanes, so that look-ups of one entry do not queue up.
//
// A table that is literally 0 .. T-1 is indexed; of any other one the entries that are not their own index go into a hash
// table (linear probing, at most half full) of entry -> first index that holds it, and a look-up costs a probe or two where
// the search from the front costs half the table.  Which of the two a table is, is looked at in every call, on the device: up
// to 4096 entries by every workgroup for itself (k_count_small: table and hash in LDS), beyond by a launch over the table
// (k_survey), whose findings the counting workgroups read.  us per call in a queue of them, 1.5 M look-ups: 10 in 2^6 entries,
// 12.0 in 2^12, 17.9 in 2^16, 51 in 2^20 (48 for the last when the caller promises a range); 10^6 look-ups in 3003
// values 12.6, in 40000 31.
#include <algorithm>

#include "common.hpp"
#include "gl_field.hpp"

namespace {

constexpr int BLOCK = 256;
constexpr int COUNT_THREADS = 1024;
constexpr int SLICE = 32768;                   // counters of a workgroup: 128 KiB of LDS
constexpr int MAX_COPIES = 32;
constexpr i64 MAX_HALF = 0xFFFF;               // look-ups of a group that counts in 16 bits
constexpr i64 MAX_GROUPS = 256;                // rows of the workspace per slice
constexpr u32 EMPTY = 0xFFFFFFFFu;
constexpr i64 MAX_HASHED = (i64)1 << 30;       // entries of a hash table
constexpr u64 INDEX_BITS = MAX_HASHED - 1;
constexpr int SMALL_TABLE = 4096;              // entries of a table that every workgroup takes into its LDS
constexpr int SMALL_COUNTERS = 16384;          // counters beside it
constexpr int SURVEYORS = 256;                 // workgroups of k_survey at most

// Fibonacci hashing into 2^bits slots
__device__ __forceinline__ u32 slot_of(u64 key, int bits) { return (u32)((key * 0x9E3779B97F4A7C15ull) >> (64 - bits)); }

// One slot of the hash table in memory: an index of the table under the tag of the call (any other tag: unused).
typedef unsigned long long Slot;

// How a look-up finds its entry.
struct Finder {
    const u64 *table;
    i64 n_table;
    Slot *slots;
    int bits;                                  // log2 of the slots, 0: no hash table
    u64 tag;                                   // of this call, in the bits above an index
    u32 *found;                                // what each workgroup of the survey saw
    int n_found;                               // 0: the caller promises a range
};
constexpr u32 OFF = 1, DIAGONAL = 2;           // entries that are not, and that are, their own index
constexpr u32 LOST = 4;                        // an entry that found no slot: the table is searched from the front
constexpr u32 MAX_PROBES = 1 << 14;

// A slot belongs to the first index that claims it; later indices of the same entry lower it to the smallest (every index it
// ever holds has the same entry, which is read from the table).  Slots need no emptying: what lies there from before has
// another tag, unless by an accident of one in 2^33.  Even then it is met like a claim: the index it names is compared with the
// table, here and by the look-ups, so it can stand in the way but not be taken for another entry, and an entry that finds no
// slot within MAX_PROBES is reported.  Half of the slots and more stay unused.
__device__ __forceinline__ bool insert(const Finder &F, u64 j, u64 key) {
    const u32 mask = (1u << F.bits) - 1;
    u32 h = slot_of(key, F.bits);
    for (u32 probes = 0; probes <= mask && probes < MAX_PROBES; ++probes, h = (h + 1) & mask) {
        Slot was = __hip_atomic_load(&F.slots[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if ((was & ~INDEX_BITS) != F.tag) {
            const Slot now = atomicCAS(&F.slots[h], was, (Slot)(F.tag | j));
            if (now == was) return true;
            was = now;                         // another thread of this call was faster
        }
        const u64 other = was & INDEX_BITS;
        if (other < (u64)F.n_table && F.table[other] == key) {
            atomicMin(&F.slots[h], (Slot)(F.tag | j));
            return true;
        }
    }
    return false;
}

// Goes over the table: notes in found[workgroup] whether there are entries that are, and that are not, their own index, and puts
// the latter into the hash table; a range puts nothing.  When single look-ups are going to be added to the result it is zeroed
// here (the launch that would do this is saved).  Costs a call over a range 2 us up to 2^18 entries, 3 at 2^20.
__global__ __launch_bounds__(COUNT_THREADS) void k_survey(const Finder F, u64 *clear) {
    const i64 first = (i64)blockIdx.x * COUNT_THREADS + threadIdx.x, stride = (i64)gridDim.x * COUNT_THREADS;
    __shared__ u32 seen;
    if (threadIdx.x == 0) seen = 0;
    __syncthreads();
    bool off = false, diagonal = false, lost = false;
    for (i64 j = first; j < F.n_table; j += stride) {
        const u64 key = F.table[j];
        if (clear) clear[j] = 0;
        if (key == (u64)j) diagonal = true;
        else {
            off = true;
            if (F.bits && !insert(F, (u64)j, key)) lost = true;
        }
    }
    const u32 mine = (__any(off) ? OFF : 0) | (__any(diagonal) ? DIAGONAL : 0) | (__any(lost) ? LOST : 0);
    if ((threadIdx.x & 63) == 0) atomicOr(&seen, mine);
    __syncthreads();
    if (threadIdx.x == 0) F.found[blockIdx.x] = seen;
}

// the survey's result: a thread's part of it, which may be asked for early, and the whole, the same for every thread of a
// workgroup (which all call this)
__device__ __forceinline__ u32 found_part(const Finder &F) { return (int)threadIdx.x < F.n_found ? F.found[threadIdx.x] : 0; }
__device__ __forceinline__ bool found_any(u32 part, u32 what) { return __syncthreads_or((part & what) != 0); }

__global__ __launch_bounds__(BLOCK) void k_clear_slots(Slot *slots, i64 n) {
    const i64 stride = (i64)gridDim.x * BLOCK;
    for (i64 i = (i64)blockIdx.x * BLOCK + threadIdx.x; i < n; i += stride) slots[i] = 0;
}

__global__ __launch_bounds__(BLOCK) void k_clear_counts(u64 *mult, i64 n) {
    const i64 stride = (i64)gridDim.x * BLOCK;
    for (i64 i = (i64)blockIdx.x * BLOCK + threadIdx.x; i < n; i += stride) mult[i] = 0;
}

// The index a value counts for, or at least n_table for none: the smaller one of its own, where the table holds it there, and of
// the one in the hash table.
__device__ __forceinline__ u64 index_of(u64 x, const Finder &F, bool diagonal, bool search) {
    if (search) {                              // from the front
        i64 j = 0;
        while (j < F.n_table && F.table[j] != x) ++j;
        return (u64)j;
    }
    u64 own = ~0ull;
    if (diagonal && x < (u64)F.n_table && F.table[x] == x) own = x;
    const u32 mask = (1u << F.bits) - 1;
    u32 h = slot_of(x, F.bits);
    for (u32 probes = 0; probes <= mask && probes < MAX_PROBES; ++probes, h = (h + 1) & mask) {
        const Slot slot = F.slots[h];
        if ((slot & ~INDEX_BITS) != F.tag) break;
        const u64 at = slot & INDEX_BITS;
        if (at < (u64)F.n_table && F.table[at] == x) return at < own ? at : own;
    }
    return own;
}

// counts of the entries base .. base + mine - 1 among x[lo .. hi - 1], each at(value) an index of the table; `copies` (a power
// of two) interleaved counters per entry, so that look-ups of one entry do not queue up.  HALF: counters of 16 bits, two to a word.
template <bool HALF, class F>
__device__ __forceinline__ void count(const u64 *__restrict__ x, i64 lo, i64 hi, u64 base, int mine, int copies, u32 *counts, F at) {
    const int copy = threadIdx.x & (copies - 1);
    constexpr int UN = HALF ? 8 : 4;           // look-ups of a thread in flight
    for (i64 i0 = lo + threadIdx.x; i0 < hi; i0 += UN * COUNT_THREADS) {
        u64 v[UN];
        // requested together: as loads behind a test each they were waited for one by one.  In the place of those past the end the first.
        // 2^24 look-ups in 2^20 entries 337 -> 295 us, 1.5 M in 2^20 51.7 -> 48.  (Those of the next trip as well: 253 and 44.7, but in tables of
        // one slice 3 % more, 1.5 M in 2^16 17.9 and 18.5.)
#pragma unroll
        for (int u = 0; u < UN; ++u) v[u] = x[i0 + u * COUNT_THREADS < hi ? i0 + u * COUNT_THREADS : lo];
        VI_SCHED_FENCE();
        u32 times[UN];
#pragma unroll
        for (int u = 0; u < UN; ++u) times[u] = i0 + u * COUNT_THREADS < hi ? 1 : 0;
        if (HALF) {
            // with few copies or none, look-ups of a thread that equal its first go as one (1.5 M look-ups of one entry of 2^16: 34.5 us
            // without this, 17.1 with it, 27.1 with 32-bit counters)
#pragma unroll
            for (int u = 1; u < UN; ++u) {
                const bool same = v[u] == v[0];
                times[0] += same ? times[u] : 0;
                times[u] = same ? 0 : times[u];
            }
        }
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            if (times[u]) {
                const u64 j = at(v[u]) - base;
                if (j >= (u64)mine) continue;
                if (HALF) atomicAdd(&counts[((int)j >> 1) * copies + copy], times[u] << (16 * ((int)j & 1)));
                else atomicAdd(&counts[(int)j * copies + copy], 1u);
            }
        }
    }
}

// mult = c, or mult += c: an atomic one, as calls on other streams may be adding to the same counts
__device__ __forceinline__ void put(u64 *mult, u64 c, int accumulate) {
    if (!accumulate) *mult = c;
    else if (c) atomicAdd((unsigned long long *)mult, (unsigned long long)c);
}

// a workgroup's counts to its row, or straight to the result where there are no rows.  Two or four copies are one LDS read (1.5 M look-ups
// in a range of 2^13 12.0 us a copy at a time, 11.0 this way).
__device__ __forceinline__ void put_counts(const u32 *counts, int mine, int copies, u32 *row, bool aligned, u64 *mult, int accumulate) {
    const int tid = threadIdx.x;
    if (row && copies == 1 && aligned && (mine & 3) == 0) {
        uint4 *to = reinterpret_cast<uint4 *>(row);
        for (int i = tid; i < mine / 4; i += COUNT_THREADS) to[i] = reinterpret_cast<const uint4 *>(counts)[i];
        return;
    }
    if (row && (copies == 2 || copies == 4)) {
        for (int i = tid; i < mine; i += COUNT_THREADS) {
            if (copies == 4) {
                const uint4 c = reinterpret_cast<const uint4 *>(counts)[i];
                row[i] = c.x + c.y + c.z + c.w;
            } else {
                const uint2 c = reinterpret_cast<const uint2 *>(counts)[i];
                row[i] = c.x + c.y;
            }
        }
        return;
    }
    for (int i = tid; i < mine; i += COUNT_THREADS) {
        u32 c = 0;
        for (int k = 0; k < copies; ++k) c += counts[i * copies + ((k + tid) & (copies - 1))];
        if (row) row[i] = c;
        else put(&mult[i], c, accumulate);
    }
}

// Workgroup (slice, group): counts of the entries slice * SLICE .. of the group's share of x.  rows: the group's row of n_table
// counts, or null when there is one group: the counts go straight to mult.  HALF: slices of 2 SLICE entries and rows of 16-bit counts, an
// even number of them; there is more than one group, and none has more than MAX_HALF look-ups.
// Over a range only the first range_groups groups count, with a larger share each.
template <bool HALF>
__global__ __launch_bounds__(COUNT_THREADS) void k_count(const u64 *__restrict__ x, i64 n_x, i64 per_group, const Finder F, int copies, u32 *rows,
                                                         u64 *mult, int accumulate, int range_groups) {
    extern __shared__ uint4 lds_counts[];
    u32 *counts = reinterpret_cast<u32 *>(lds_counts);
    constexpr int MOST = HALF ? 2 * SLICE : SLICE;
    const i64 base = (i64)blockIdx.x * MOST, group = blockIdx.y;
    const int mine = F.n_table - base < MOST ? (int)(F.n_table - base) : MOST, words = HALF ? (mine + 1) / 2 : mine;
    const u32 part = found_part(F);
    // the launch's LDS is a whole number of 16-byte words
    for (int i = threadIdx.x; i < (words * copies + 3) / 4; i += COUNT_THREADS) lds_counts[i] = make_uint4(0, 0, 0, 0);
    const bool range = !found_any(part, OFF);  // a barrier as well
    if (HALF && range) {
        if (group >= range_groups) return;
        per_group = (n_x + range_groups - 1) / range_groups;
    }
    const i64 lo = group * per_group, hi = lo + per_group < n_x ? lo + per_group : n_x;
    if (range) count<HALF>(x, lo, hi, (u64)base, mine, copies, counts, [](u64 v) { return v; });
    else {
        const bool diagonal = found_any(part, DIAGONAL), search = found_any(part, LOST) || F.bits == 0;
        count<HALF>(x, lo, hi, (u64)base, mine, copies, counts, [&](u64 v) { return index_of(v, F, diagonal, search); });
    }
    __syncthreads();
    if (HALF) {
        const i64 row_words = (F.n_table + 1) / 2;
        put_counts(counts, words, copies, rows + group * row_words + base / 2, (row_words & 3) == 0, nullptr, 0);
        return;
    }
    put_counts(counts, words, copies, rows ? rows + group * F.n_table + base : nullptr, (F.n_table & 3) == 0, mult + base, accumulate);
}

// The same for a table of up to SMALL_TABLE entries that nothing is known of: every workgroup takes it into its LDS, sees
// whether it is a range and, if not, makes its own hash table beside it.  One launch where the survey of a longer table takes
// one more (1.5 M look-ups in 2^12 entries 12.0 us, in 2^13 through the survey 16.6); 32 KiB of table per workgroup come
// from the L2.
__global__ __launch_bounds__(COUNT_THREADS) void k_count_small(const u64 *__restrict__ x, i64 n_x, i64 per_group, const u64 *__restrict__ table,
                                                               int n_table, int bits, int copies, u32 *rows, u64 *mult, int accumulate) {
    extern __shared__ uint4 lds_counts[];
    const int tid = threadIdx.x, words = (n_table * copies + 3) / 4, n_slots = 1 << bits;
    u32 *counts = reinterpret_cast<u32 *>(lds_counts);
    u64 *keys = reinterpret_cast<u64 *>(lds_counts + words);
    u32 *index = reinterpret_cast<u32 *>(keys + n_table);
    int odd = 0;
    for (int j = tid; j < n_table; j += COUNT_THREADS) {
        const u64 key = table[j];
        keys[j] = key;
        odd |= key != (u64)j;
    }
    for (int i = tid; i < words; i += COUNT_THREADS) lds_counts[i] = make_uint4(0, 0, 0, 0);
    for (int i = tid; i < n_slots; i += COUNT_THREADS) index[i] = EMPTY;
    odd = __syncthreads_or(odd);
    const i64 group = blockIdx.x, lo = group * per_group, hi = lo + per_group < n_x ? lo + per_group : n_x;
    if (!odd) count<false>(x, lo, hi, 0, n_table, copies, counts, [](u64 v) { return v; });
    else {
        for (int j = tid; j < n_table; j += COUNT_THREADS) {
            const u64 key = keys[j];
            u32 h = slot_of(key, bits);
            for (int probes = 0; probes < n_slots; ++probes, h = (h + 1) & (n_slots - 1)) {
                const u32 was = atomicCAS(&index[h], EMPTY, (u32)j);
                if (was == EMPTY) break;
                if (keys[was] == key) {
                    atomicMin(&index[h], (u32)j);
                    break;
                }
            }
        }
        __syncthreads();
        count<false>(x, lo, hi, 0, n_table, copies, counts, [&](u64 v) -> u64 {
            u32 h = slot_of(v, bits);
            for (int probes = 0; probes < n_slots; ++probes, h = (h + 1) & (n_slots - 1)) {
                const u32 at = index[h];
                if (at == EMPTY) break;
                if (keys[at] == v) return at;
            }
            return ~0ull;
        });
    }
    __syncthreads();
    put_counts(counts, n_table, copies, rows ? rows + group * n_table : nullptr, (n_table & 3) == 0, mult, accumulate);
}

// mult[j] (+)= sum over the rows: 64 words of the rows per workgroup, the rows dealt over its four wavefronts, eight in flight.
// HALF: two 16-bit counts to a word, fewer rows over a range (k_count).
template <bool HALF>
__global__ __launch_bounds__(BLOCK) void k_add_rows(const u32 *__restrict__ rows, int groups, i64 n_table, u64 *mult, int accumulate, const u32 *found,
                                                    int n_found, int range_groups) {
    constexpr int PER = HALF ? 2 : 1;
    __shared__ u64 part[PER][BLOCK / 64][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const i64 at = (i64)blockIdx.x * 64 + lane, row_words = (n_table + PER - 1) / PER;
    u64 sum[PER] = {};
    if (HALF && !found_any((int)threadIdx.x < n_found ? found[threadIdx.x] : 0, OFF)) groups = range_groups;
    if (at < row_words) {
        constexpr int UN = 8;
        for (int g0 = w; g0 < groups; g0 += UN * (BLOCK / 64)) {
            u32 c[UN];
#pragma unroll
            for (int u = 0; u < UN; ++u) {
                const int g = g0 + u * (BLOCK / 64);
                c[u] = g < groups ? rows[(i64)g * row_words + at] : 0;
            }
#pragma unroll
            for (int u = 0; u < UN; ++u) {
                sum[0] += HALF ? c[u] & 0xFFFF : c[u];
                if (HALF) sum[PER - 1] += c[u] >> 16;
            }
        }
    }
#pragma unroll
    for (int q = 0; q < PER; ++q) part[q][w][lane] = sum[q];
    __syncthreads();
    // the workgroup's 64 PER counts in the order of the table
    const i64 j = (i64)blockIdx.x * 64 * PER + threadIdx.x;
    if (threadIdx.x < 64 * PER && j < n_table) {
        const int q = threadIdx.x % PER, word = threadIdx.x / PER;
        put(&mult[j], part[q][0][word] + part[q][1][word] + part[q][2][word] + part[q][3][word], accumulate);
    }
}

// one global atomic per look-up
__global__ __launch_bounds__(BLOCK) void k_count_global(const u64 *__restrict__ x, i64 n_x, const Finder F, unsigned long long *__restrict__ mult) {
    const i64 stride = (i64)gridDim.x * BLOCK, first = (i64)blockIdx.x * BLOCK + threadIdx.x;
    const u32 part = found_part(F);
    if (!found_any(part, OFF)) {
        for (i64 i = first; i < n_x; i += stride) {
            const u64 at = x[i];
            if (at < (u64)F.n_table) atomicAdd(&mult[at], 1ULL);
        }
    } else {
        const bool diagonal = found_any(part, DIAGONAL), search = found_any(part, LOST) || F.bits == 0;
        for (i64 i = first; i < n_x; i += stride) {
            const u64 at = index_of(x[i], F, diagonal, search);
            if (at < (u64)F.n_table) atomicAdd(&mult[at], 1ULL);
        }
    }
}

// the same without a workspace, a table that is not promised to be a range searched from the front
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
    bool small, direct, half;                  // k_count_small; one global atomic per look-up; 16-bit counters
    i64 slices, groups, range_groups;          // groups: with 16-bit counters of another table, range_groups of a range
    int copies, bits, surveyors;
    size_t slot_bytes, found_bytes, row_bytes;
    size_t bytes() const {
        const size_t used = slot_bytes + found_bytes + row_bytes;
        return used ? used + vi::WS_SLACK : 0;
    }
};

// promised: the caller says that the table is a range
Plan make_plan(i64 n_x, i64 n_table, bool promised) {
    Plan L = {};
    L.small = !promised && n_table <= SMALL_TABLE;
    if (!promised) {
        // slots have 32-bit indices: a longer table is searched
        if (n_table <= MAX_HASHED) {
            L.bits = 1;
            while (((i64)1 << L.bits) < 2 * n_table) ++L.bits;
        }
        if (!L.small) {
            const i64 shares = (n_table + COUNT_THREADS - 1) / COUNT_THREADS;
            L.surveyors = (int)(shares < SURVEYORS ? shares : SURVEYORS);
            if (L.bits) L.slot_bytes = sizeof(Slot) << L.bits;
            L.found_bytes = SURVEYORS * sizeof(u32);
        }
    }
    L.slices = (n_table + SLICE - 1) / SLICE;
    // Few look-ups, spread over many entries: 30000 in a 2^16 table take 3.6 us and 2.5 us for clearing the counts, 11 us
    // through the histogram.  And a table of many slices: all of them read all look-ups, 10 us a slice for 2^24 of them
    // against 711 us of atomics in all.
    L.direct = (n_table >= 8192 && n_x <= 131072) || L.slices > 64;
    if (L.direct) return L;
    // a workgroup per CU, but no more rows than look-ups are worth: clearing and storing a slice's counters takes as long
    // as some eight thousand look-ups
    L.groups = (n_x + 8191) / 8192;
    if (L.groups * L.slices > MAX_GROUPS) L.groups = MAX_GROUPS / L.slices;
    if (L.groups < (n_x >> 31) + 1) L.groups = (n_x >> 31) + 1;        // a group's counters have 32 bits
    // From 8192 entries on 16-bit counters: half the bytes go through the rows, and half the slices read the look-ups, as long as no group
    // has more look-ups than such a counter holds.  Over a range a group's look-ups cost less than its row: from 64 groups on they are
    // larger (1.5 M in a range of 2^16: 21.0 us with 32-bit counters, 21.6 with 184 groups, 17.9 with 62; 10^6 in 40000 other entries
    // 35.6, 49 with 41 groups, 30.7 with 123; 1.5 M in 2^14 20.1 -> 14.4).
    if (n_table >= 8192) {
        const i64 slices = (n_table + 2 * SLICE - 1) / (2 * SLICE), most = MAX_GROUPS / slices;
        const i64 groups = std::min((n_x + 8191) / 8192, most), range_groups = std::min(std::max(std::min(groups, (i64)64), (n_x + 24575) / 24576), most);
        if (range_groups > 1 && (n_x + range_groups - 1) / range_groups <= MAX_HALF) {
            L.half = true;
            L.slices = slices;
            L.groups = groups;
            L.range_groups = range_groups;
            // as many copies as 32-bit counters would have: 4 of 8192 entries (1.5 M look-ups of eight entries 16.7 us with one, 11.2; 16 M 38.8
            // and 28.5; 14.3 and 29.0 with 32-bit counters, 1.5 M of any entry 13.8, 10.7 and 11.0), 2 of 16384 (17.5, 14.1; 39.3,
            // 29.8).  From 32768 on there is one: 1.5 M look-ups of eight entries of 2^16 take 21.6, of 32-bit counters in twice the groups 18.5.
            L.copies = 1;
            while (n_table * L.copies * 2 <= SLICE) L.copies *= 2;
            L.row_bytes = (size_t)groups * ((n_table + 1) / 2) * sizeof(u32);
            return L;
        }
    }
    const i64 counters = L.small ? SMALL_COUNTERS : SLICE;
    L.copies = 1;
    while (L.copies < MAX_COPIES && n_table * L.copies * 2 <= counters) L.copies *= 2;
    L.row_bytes = L.groups > 1 ? (size_t)L.groups * n_table * sizeof(u32) : 0;
    return L;
}

// The tag of a call, in the 34 bits above an index.  The top bit is set, as it is in no emptied slot, count or other small number
// that scratch may hold; the others take all values in turn, scattered so that no run of calls meets a common pattern.
u64 next_tag() {
    static std::atomic<u64> calls{0};
    const u64 n = calls.fetch_add(1, std::memory_order_relaxed) * 0x9E3779B97F4A7C15ull & (((u64)1 << 33) - 1);
    return ((u64)1 << 63) | n << 30;
}

// more than 64 KiB of dynamic LDS has to be asked for, once per device and kernel
int ask_for_lds() {
    static std::atomic<unsigned long long> asked{0};
    int dev = 0;
    VI_HIP(hipGetDevice(&dev));
    const unsigned long long bit = 1ull << (dev & 63);
    if (asked.load(std::memory_order_acquire) & bit) return VI_OK;
    VI_HIP(hipFuncSetAttribute((const void *)k_count<true>, hipFuncAttributeMaxDynamicSharedMemorySize, SLICE * (int)sizeof(u32)));
    VI_HIP(hipFuncSetAttribute((const void *)k_count<false>, hipFuncAttributeMaxDynamicSharedMemorySize, SLICE * (int)sizeof(u32)));
    VI_HIP(hipFuncSetAttribute((const void *)k_count_small, hipFuncAttributeMaxDynamicSharedMemorySize,
                               SMALL_COUNTERS * (int)sizeof(u32) + SMALL_TABLE * (int)(sizeof(u64) + 2 * sizeof(u32))));
    asked.fetch_or(bit, std::memory_order_release);
    return VI_OK;
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
    return make_plan(n_x, n_table, table_is_range != 0).bytes();
}

int vi_lookup_histogram(const uint64_t *x, int64_t n_x, const uint64_t *table, int64_t n_table, int table_is_range, int accumulate,
                        uint64_t *mult, void *ws, size_t ws_bytes, void *stream) {
    if (n_x < 0 || n_table < 0) return vi::fail(VI_EINVAL, "vi_lookup_histogram: n_x = %lld, n_table = %lld", (long long)n_x, (long long)n_table);
    if (n_table == 0 || (n_x == 0 && accumulate)) return VI_OK;
    if ((n_x > 0 && !x) || !mult || (!table_is_range && !table)) return vi::fail(VI_EINVAL, "vi_lookup_histogram: null pointer");
    hipStream_t s = (hipStream_t)stream;
    if (n_x == 0) {
        hipLaunchKernelGGL(k_clear_counts, dim3(capped_grid(n_table)), dim3(BLOCK), 0, s, mult, (i64)n_table);
        VI_LAUNCH_CHECK("k_clear_counts");
        return VI_OK;
    }
    const Plan L = make_plan(n_x, n_table, table_is_range != 0);
    if (L.bytes() && (!ws || ws_bytes < L.bytes())) return vi::fail(VI_ENOMEM, "vi_lookup_histogram: workspace below %zu bytes", L.bytes());
    if (int rc = ask_for_lds()) return rc;
    ws = vi::align16(ws);
    Finder F = {};
    F.table = table;
    F.n_table = n_table;
    F.slots = (Slot *)ws;
    F.bits = L.bits;
    F.found = (u32 *)((char *)ws + L.slot_bytes);
    F.n_found = L.surveyors;
    u32 *rows = L.row_bytes ? (u32 *)((char *)ws + L.slot_bytes + L.found_bytes) : nullptr;
    if (L.surveyors) {
        // a replay has the tag of the capture, so a captured call empties the slots
        F.tag = next_tag();
        bool captured = false;
        if (int rc = vi::capturing(s, &captured)) return rc;
        if (captured && L.bits) {
            hipLaunchKernelGGL(k_clear_slots, dim3(capped_grid((i64)1 << L.bits)), dim3(BLOCK), 0, s, F.slots, (i64)1 << L.bits);
            VI_LAUNCH_CHECK("k_clear_slots");
        }
        hipLaunchKernelGGL(k_survey, dim3((unsigned)L.surveyors), dim3(COUNT_THREADS), 0, s, F, L.direct && !accumulate ? mult : nullptr);
        VI_LAUNCH_CHECK("k_survey");
    } else if (L.direct && !accumulate) {
        hipLaunchKernelGGL(k_clear_counts, dim3(capped_grid(n_table)), dim3(BLOCK), 0, s, mult, (i64)n_table);
        VI_LAUNCH_CHECK("k_clear_counts");
    }
    if (L.direct) {
        hipLaunchKernelGGL(k_count_global, dim3(capped_grid(n_x)), dim3(BLOCK), 0, s, x, (i64)n_x, F, (unsigned long long *)mult);
        VI_LAUNCH_CHECK("k_count_global");
        return VI_OK;
    }
    const i64 per = (n_x + L.groups - 1) / L.groups;
    const i64 in_slice = n_table < SLICE ? n_table : SLICE;
    size_t lds = ((size_t)in_slice * L.copies * sizeof(u32) + 15) & ~(size_t)15;
    if (L.small) {
        lds += (size_t)n_table * sizeof(u64) + (sizeof(u32) << L.bits);
        hipLaunchKernelGGL(k_count_small, dim3((unsigned)L.groups), dim3(COUNT_THREADS), lds, s, x, (i64)n_x, per, table, (int)n_table, L.bits, L.copies,
                           rows, mult, accumulate);
        VI_LAUNCH_CHECK("k_count_small");
    } else {
        const dim3 grid((unsigned)L.slices, (unsigned)L.groups);
        if (L.half) lds = (size_t)SLICE * sizeof(u32);
        if (L.half) hipLaunchKernelGGL(k_count<true>, grid, dim3(COUNT_THREADS), lds, s, x, (i64)n_x, per, F, L.copies, rows, mult, accumulate, (int)L.range_groups);
        else hipLaunchKernelGGL(k_count<false>, grid, dim3(COUNT_THREADS), lds, s, x, (i64)n_x, per, F, L.copies, rows, mult, accumulate, 0);
        VI_LAUNCH_CHECK("k_count");
    }
    if (rows) {
        const unsigned adders = (unsigned)((n_table + (L.half ? 127 : 63)) / (L.half ? 128 : 64));
        if (L.half)
            hipLaunchKernelGGL(k_add_rows<true>, dim3(adders), dim3(BLOCK), 0, s, (const u32 *)rows, (int)L.groups, (i64)n_table, mult, accumulate,
                               (const u32 *)F.found, F.n_found, (int)L.range_groups);
        else
            hipLaunchKernelGGL(k_add_rows<false>, dim3(adders), dim3(BLOCK), 0, s, (const u32 *)rows, (int)L.groups, (i64)n_table, mult, accumulate,
                               (const u32 *)nullptr, 0, 0);
        VI_LAUNCH_CHECK("k_add_rows");
    }
    return VI_OK;
}

}  // extern "C"
