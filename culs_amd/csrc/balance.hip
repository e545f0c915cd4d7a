// Balance (`b`) on the device.
//
// Semantics of balancePerformV2 (src/algorithms/balance.cu:912-1382) with
// sortDecId = 1, made exact:
//   1. covers: from every root AND node a DFS (fanin0 first) collects the
//      cover's inputs: literals that are complemented, not AND nodes, have
//      more than one fanout (POs count), or sit at the stack / size limits
//      (128 / 1024); a repeated input is dropped and an input seen in both
//      polarities makes the cover constant FALSE (balance.cu:666-750).
//      Roots are found level by level from the POs; a root's level is the
//      last (deepest) level it appears at (balance.cu:958-1037, 753-834).
//   2. reconstruction, deepest level first, covers of a level in id order,
//      in batches of 32768 (balance.cu:1129-1229): a cover's inputs are
//      sorted by (level desc, literal desc); then, step by step over the whole
//      batch, the last input may be swapped with an earlier one of the same
//      level that already forms an AND with the last (sharedNodeDrivenPermute,
//      :187-247); the last two inputs are popped and their AND is looked up
//      (trivial rules, then the table, :113-185); new ANDs take id
//      counter + cover index, the smallest id wins among equal keys, the
//      counter moves past the largest id (:1188-1210); the result goes back
//      into the cover in level order unless already present (:429-467).
//   3. created nodes are renumbered in id order (:1237-1262); POs follow
//      their cover's result (:882-910).
// Literal values decide ties in the input order; there the reference's own
// values are used (lit 0 = TRUE, common.h:285-286), not the AIGER ones.
//
// Mapping to MI355X.  Only the order of the created ids matters, so a step's
// new nodes take consecutive ids by a prefix sum over its covers: the ids are
// then the output's, levels travel with the literals and the table's values,
// and nothing is renumbered.  Which ANDs are roots is a property of their
// fanout edges, so all covers are computed in one launch; one sweep over
// them in id order tells which ones a PO reaches, and their levels.  The sweep,
// and the reconstruction of a level that fits its LDS, run in one persistent workgroup
// per member of a batched arena (one in all for a single AIG): a step is bound
// by the latency of its lookups, and the members do not depend on each other.
// Other levels run each phase of a step as a grid-wide kernel.
#include "gls_internal.h"
#include "dev_common.h"
#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_reduce.hpp>
#include <rocprim/device/device_scan.hpp>
#include <rocprim/device/device_select.hpp>
#include <rocprim/iterator/counting_iterator.hpp>
#include <algorithm>
#include <chrono>
#include <vector>

namespace {

constexpr int kB = 256;
constexpr int BAL_STACK = 128;        // DFS_COVER_STACK_SIZE, balance.cu:18
constexpr int BAL_MAX_COVER = 1024;   // MAX_LOCAL_COVER_SIZE, balance.cu:17
constexpr int BAL_BATCH = 32768;      // iterLen, balance.cu:1129
constexpr int BAL_WG = 1024;          // threads of the persistent workgroups
constexpr int COVER_THREADS = 65536;  // most threads of a cover launch (each owns COVER_SCRATCH slots)
// the size limit is checked before an expansion, so a cover can end up to a
// few inputs above BAL_MAX_COVER: room for that
constexpr int COVER_SCRATCH = BAL_MAX_COVER + 64;
constexpr int COVER_FAST = 16;        // first inputs of a cover, kept in LDS during its DFS
constexpr uint32_t UNSET = 0xFFFFFFFFu;
constexpr unsigned long long EMPTY64 = ~0ull;

inline int nblocks(int64_t n) { return (int)std::max<int64_t>(1, std::min<int64_t>((n + kB - 1) / kB, 1 << 20)); }

__device__ __forceinline__ uint32_t culs_val(uint32_t l) { return l < 2u ? 1u - l : l; }

// Literal and level of a signal, as one word.
__device__ __forceinline__ unsigned long long sig(uint32_t lit, uint32_t lev) {
    return (unsigned long long)lev << 32 | lit;
}
__device__ __forceinline__ uint32_t sig_lit(unsigned long long s) { return (uint32_t)s; }
__device__ __forceinline__ uint32_t sig_lev(unsigned long long s) { return (uint32_t)(s >> 32); }

// ---------------------------------------------------------------------------
// table of created nodes: key lit0 << 32 | lit1 (lit0 < lit1) -> positive
// literal and level of the node (open addressing, linear probing; keys and
// values apart, because most lookups miss).  Written with atomics and read past
// the L1, so a workgroup sees its own insertions after a wait and a barrier.
// ---------------------------------------------------------------------------
struct NodeTable {
    unsigned long long *k, *v;
    uint64_t mask;
};

__device__ __forceinline__ unsigned long long t_load(const unsigned long long *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// first slot of a key: three 32-bit products, because a wavefront that hashes
// its candidates is bound by issue
__device__ __forceinline__ uint64_t t_hash(const NodeTable &t, unsigned long long key) {
    uint32_t h = (uint32_t)(key >> 32) * 0x9E3779B1u + (uint32_t)key * 0x85EBCA77u;
    h = (h ^ h >> 16) * 0xC2B2AE3Du;
    return (h ^ h >> 15) & t.mask;
}

// the node of a key that is there: it may be on its way still (the workgroup
// that inserts does not wait for it)
__device__ __forceinline__ unsigned long long t_node(const NodeTable &t, uint64_t s) {
    unsigned long long v;
    do v = t_load(&t.v[s]);
    while (v == EMPTY64);
    return v;
}

// the node with this key, or EMPTY64; k is the key word at its first slot s
__device__ __forceinline__ unsigned long long t_find_at(const NodeTable &t, unsigned long long key, uint64_t s,
                                                        unsigned long long k) {
    for (uint64_t probes = 0; probes <= t.mask; probes++) {
        if (k == key) return t_node(t, s);
        if (k == EMPTY64) return EMPTY64;
        s = (s + 1) & t.mask;
        k = t_load(&t.k[s]);
    }
    return EMPTY64;
}

__device__ __forceinline__ unsigned long long t_find(const NodeTable &t, unsigned long long key) {
    const uint64_t s = t_hash(t, key);
    return t_find_at(t, key, s, t_load(&t.k[s]));
}

__device__ __forceinline__ unsigned long long t_cas(const NodeTable &t, uint64_t s, unsigned long long key) {
    unsigned long long prev = EMPTY64;
    __hip_atomic_compare_exchange_strong(&t.k[s], &prev, key, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
    return prev;
}

// slot of the key, inserted if it is new; UNSET if the table is full
__device__ __forceinline__ uint32_t t_slot(const NodeTable &t, unsigned long long key) {
    uint64_t s = t_hash(t, key);
    for (uint64_t probes = 0; probes <= t.mask; probes++, s = (s + 1) & t.mask) {
        const unsigned long long prev = t_cas(t, s, key);
        if (prev == EMPTY64 || prev == key) return (uint32_t)s;
    }
    return UNSET;
}

// trivial AND rules (hash_table.h:435-449) in AIGER literals; EMPTY64 if none.
// The result is one of the two signals or the constant (level 0).
__device__ __forceinline__ unsigned long long and_trivial(unsigned long long a, unsigned long long b) {
    const uint32_t x = sig_lit(a), y = sig_lit(b);
    if ((x ^ y) > 1u && min(x, y) > 1u) return EMPTY64;
    if (x == y) return a;
    if (x == (y ^ 1u)) return 0ull;
    if (x == 1u) return b;
    if (y == 1u) return a;
    if (x == 0u || y == 0u) return 0ull;
    return EMPTY64;
}

__device__ __forceinline__ unsigned long long and_key_of(uint32_t x, uint32_t y) {
    return x < y ? (unsigned long long)x << 32 | y : (unsigned long long)y << 32 | x;
}

// LDS that other wavefronts write (a volatile pointer would make these FLAT
// loads, which wait for all memory)
template <class T> __device__ __forceinline__ T lds_load(const T *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// ---------------------------------------------------------------------------
// phase 1: covers
// ---------------------------------------------------------------------------
enum : uint8_t { RM_STOP = 1, RM_PO = 2 };      // marks of a node: a complemented edge or a PO stops a cover there; a PO

__global__ void k_fanouts(int32_t n, int32_t nPIs, const uint32_t *__restrict__ f0, const uint32_t *__restrict__ f1,
                          int32_t nPOs, const uint32_t *__restrict__ pos, uint32_t *nFo, uint32_t *mark) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t v = nPIs + 1 + blockIdx.x * (int64_t)blockDim.x + threadIdx.x; v < n; v += stride) {
        const uint32_t a = f0[v], b = f1[v];
        atomicAdd(&nFo[LID(a)], 1u);
        atomicAdd(&nFo[LID(b)], 1u);
        if (LC(a)) mark[LID(a)] = RM_STOP;
        if (LC(b)) mark[LID(b)] = RM_STOP;
    }
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < nPOs; i += stride)
        atomicAdd(&nFo[LID(pos[i])], 1u);
}

__global__ void k_po_marks(int32_t nPOs, const uint32_t *__restrict__ pos, uint32_t *mark) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < nPOs; i += stride)
        mark[LID(pos[i])] = RM_STOP | RM_PO;
}

// The ANDs at which every cover that meets them stops: their covers are
// needed if any cover or PO reaches them.
__global__ void k_root_flags(int32_t n, int32_t nPIs, const uint32_t *__restrict__ nFo,
                             const uint32_t *__restrict__ mark, uint8_t *flag) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t v = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; v < n; v += stride)
        flag[v] = v > nPIs && (nFo[v] > 1u || mark[v] != 0u);
}

struct CoverArgs {
    const uint32_t *f0, *f1, *nFo;
    int32_t nPIs;
    uint2 *cover;                    // per root: first input in pool, inputs
    uint32_t *pool, *poolNext;
    uint64_t poolCap;
    uint32_t *scratch;               // COVER_SCRATCH entries per thread
    uint8_t *isRoot;
    uint32_t *extra, *extraLen;      // roots met at the stack / size limits
    uint32_t *disorder;              // an AND input's id is not below its cover's root
    uint32_t *err;                   // 1: cover pool full
};

// a cover's inputs during its DFS
struct CoverIn {
    uint32_t *fast;      // column of an LDS array [COVER_FAST][kB]
    uint32_t *slow;
    __device__ __forceinline__ uint32_t &operator[](uint32_t i) const {
        return i < (uint32_t)COVER_FAST ? fast[i * kB] : slow[i];
    }
};

// localCoverTravToTable (balance.cu:666-750) of root v into in[]; returns len
// (0 = constant FALSE)
__device__ uint32_t cover_dfs(const CoverArgs &a, uint32_t v, const CoverIn &in) {
    uint32_t stack[BAL_STACK];
    int top = -1;
    uint32_t len = 0;
    const uint32_t rootLit = 2u * v;
    stack[++top] = rootLit;
    while (top != -1) {
        const uint32_t cur = stack[top--];
        bool rep = false;
        for (uint32_t i = 0; i < len; i++) {
            const uint32_t x = in[i];
            if (x == cur) { rep = true; break; }
            if (x == (cur ^ 1u)) return 0u;
        }
        if (rep) continue;
        const uint32_t id = cur >> 1;
        if (cur != rootLit && ((cur & 1u) || (int32_t)id <= a.nPIs || a.nFo[id] > 1u || top + 2 >= BAL_STACK ||
                               (int)len + 2 * (top + 1) + 1 >= BAL_MAX_COVER)) {
            in[len++] = cur;
            continue;
        }
        stack[++top] = a.f1[id];
        stack[++top] = a.f0[id];
    }
    return len;
}

// The covers of the listed roots.
__global__ void __launch_bounds__(kB) k_covers(CoverArgs a, uint32_t nList, const uint32_t *__restrict__ list) {
    __shared__ uint32_t s_in[COVER_FAST * kB];
    const int64_t tid = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, stride = (int64_t)gridDim.x * blockDim.x;
    const CoverIn in{s_in + threadIdx.x, a.scratch + (size_t)tid * COVER_SCRATCH};
    const int64_t lane = threadIdx.x & 63;
    // the wavefront runs the same number of iterations (its first lane's
    // index decides), so the pool reservation sees all 64 lanes
    for (int64_t k = tid; k - lane < (int64_t)nList; k += stride) {
        const bool has = k < (int64_t)nList;
        const uint32_t v = has ? list[k] : 0u;
        const uint32_t len = has ? cover_dfs(a, v, in) : 0u;
        const uint32_t off = wave_reserve(a.poolNext, len);
        if (!has) continue;
        if ((uint64_t)off + len > a.poolCap) {
            atomicOr(a.err, 1u);
            a.cover[v] = make_uint2(0u, 0u);
            continue;
        }
        for (uint32_t i = 0; i < len; i++) {
            const uint32_t lit = in[i], id = lit >> 1;
            a.pool[off + i] = lit;
            if ((int32_t)id > a.nPIs) {
                if (id >= v) *a.disorder = 1u;
                // an AND that is no root by its edges: a limit cut the cover there
                if (a.isRoot[id] == 0) {
                    uint32_t *word = reinterpret_cast<uint32_t *>(a.isRoot + (id & ~3u));
                    const uint32_t bit = 1u << (8u * (id & 3u));
                    if (!(atomicOr(word, bit) & bit)) a.extra[atomicAdd(a.extraLen, 1u)] = id;
                }
            }
        }
        a.cover[v] = make_uint2(off, len);
    }
}

// ---- the levels of the covers.  Fanins have smaller ids than their AND, so a
// cover's inputs have smaller ids than its root.  Roots are laid
// out by falling id, per segment, so covers stand before their inputs: one
// workgroup per segment goes over them in chunks of 1024, and a root hands its
// level to its cover's inputs.  A level is 1 above the reference's (0: no PO
// reaches the root), so a root's level is the largest value handed to it.
//
// What bounds it is the chain of dependent roots within a chunk (an LDS
// round trip and two LDS atomics a step), so nothing else is waited for there:
// the levels of the next ID_RING - 1 chunks are in LDS, and so are the chunk's
// inputs, read a chunk ahead; only a root that is further away is handed its
// level by an atomic in memory.  A root counts the parents in its own chunk
// that are still to come (counted by k_id_pack); those of earlier chunks are
// done at the barrier.  LDS is double buffered, so a chunk has one barrier.
// 2M random ANDs (1.2M covers, 1795 levels): 2.5 ms; 15.2 for a level at a
// time, where each of a level's four dependent accesses was a miss in memory.
// With the inputs read from LDS after the root is known, 3.5.
constexpr uint32_t ID_CHUNK = BAL_WG;
constexpr uint32_t ID_RING = 16;         // chunks
constexpr uint32_t ID_INPUTS = 6144;     // inputs of a chunk in LDS; the rest is read from memory
constexpr uint32_t IDQ_IN = ID_INPUTS / ID_CHUNK;
constexpr uint32_t ID_NEAR = 4;          // inputs of a root that are in registers

struct IdSweepArgs {
    const uint32_t *segFirst, *segCnt;   // positions of a segment
    const uint32_t *off, *in;            // per position its cover's inputs, as positions (UNSET: no AND)
    const uint32_t *pend;                // parents within the position's chunk
    uint32_t *val;                       // 1 for a PO driver, else 0; becomes the level + 1
    uint32_t *rounds;                    // per segment: levels
};

// positions by falling id within the segment (order: roots by segment and id)
__global__ void k_id_place(uint32_t m, const uint32_t *__restrict__ order, const uint32_t *__restrict__ tag,
                           const uint32_t *__restrict__ segFirst, const uint32_t *__restrict__ segCnt,
                           const uint2 *__restrict__ cover, const uint32_t *__restrict__ mark, uint32_t *rootAt,
                           uint32_t *place, uint32_t *len, uint32_t *pend, uint32_t *val) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i <= m; i += stride) {
        if (i == m) { len[m] = 0; continue; }
        const uint32_t v = order[i], s = tag ? tag[v] : 0u, first = segFirst[s];
        const uint32_t p = first + (segCnt[s] - 1u - ((uint32_t)i - first));
        rootAt[p] = v;
        place[v] = p;
        len[p] = cover[v].y;
        pend[p] = 0;
        val[p] = mark[v] & RM_PO ? 1u : 0u;
    }
}

__global__ void k_id_pack(uint32_t m, const uint32_t *__restrict__ rootAt, const uint32_t *__restrict__ tag,
                          const uint32_t *__restrict__ segFirst, const uint2 *__restrict__ cover,
                          const uint32_t *__restrict__ pool, const uint32_t *__restrict__ place, int32_t nPIs,
                          const uint32_t *__restrict__ off, uint32_t *in, uint32_t *pend) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < m; p += stride) {
        const uint32_t v = rootAt[p], first = segFirst[tag ? tag[v] : 0u], chunk = ((uint32_t)p - first) / ID_CHUNK;
        const uint2 c = cover[v];
        for (uint32_t j = 0; j < c.y; j++) {
            const uint32_t id = pool[c.x + j] >> 1, q = (int32_t)id > nPIs ? place[id] : UNSET;
            in[off[p] + j] = q;
            if (q != UNSET && (q - first) / ID_CHUNK == chunk) atomicAdd(&pend[q], 1u);
        }
    }
}

__global__ void __launch_bounds__(ID_CHUNK) k_id_sweep(IdSweepArgs a) {
    __shared__ uint32_t s_val[ID_RING * ID_CHUNK];
    __shared__ uint32_t s_in[2][ID_INPUTS];
    __shared__ uint32_t s_pend[2][ID_CHUNK];
    __shared__ uint32_t s_most;
    const uint32_t tid = threadIdx.x, first = a.segFirst[blockIdx.x], cnt = a.segCnt[blockIdx.x];
    const uint32_t nChunk = (cnt + ID_CHUNK - 1) / ID_CHUNK;
    // a chunk's words, one root per thread
    struct Chunk {
        uint32_t base, end;                  // its inputs
        uint32_t off, stop, pend, val, in[IDQ_IN];
    };
    auto chunk_off = [&](uint32_t c) -> uint32_t { return c <= nChunk ? a.off[first + min(c * ID_CHUNK, cnt)] : 0u; };
    auto load_chunk = [&](uint32_t c, uint32_t base, uint32_t end, Chunk &x) {
        const uint32_t k = c * ID_CHUNK + tid;
        const bool has = k < cnt;
        x.base = base;
        x.end = end;
        x.off = has ? a.off[first + k] : 0u;
        x.stop = has ? a.off[first + k + 1] : 0u;
        x.pend = has ? a.pend[first + k] : 0u;
        x.val = has ? __hip_atomic_load(&a.val[first + k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0u;
#pragma unroll
        for (uint32_t q = 0; q < IDQ_IN; q++) {
            const uint32_t i = base + tid + q * ID_CHUNK;
            x.in[q] = i < end ? a.in[i] : 0u;
        }
    };
    for (uint32_t i = tid; i < ID_RING * ID_CHUNK; i += ID_CHUNK) s_val[i] = 0;
    if (tid == 0) s_most = 0;
    Chunk cur;
    uint32_t end1 = chunk_off(1), end2 = chunk_off(2), most = 0;
    if (nChunk != 0) load_chunk(0, chunk_off(0), end1, cur);
    __syncthreads();
    for (uint32_t c = 0; c < nChunk; c++) {
        const uint32_t b = c & 1u, k = c * ID_CHUNK + tid;
        // this chunk's words; atomics of the chunk before are in memory too
        __builtin_amdgcn_s_waitcnt(0x0F70);     // vmcnt(0)
        uint32_t *own = &s_val[(c % ID_RING) * ID_CHUNK + tid];
        s_pend[b][tid] = cur.pend;
        if (cur.val) atomicMax(own, cur.val);
#pragma unroll
        for (uint32_t q = 0; q < IDQ_IN; q++)
            if (cur.base + tid + q * ID_CHUNK < cur.end) s_in[b][tid + q * ID_CHUNK] = cur.in[q];
        const uint32_t off = cur.off, stop = cur.stop, base = cur.base;
        __syncthreads();
        const uint32_t nextBase = end1, nextEnd = end2;
        end1 = end2;
        end2 = chunk_off(c + 3);
        if (c + 1 < nChunk) load_chunk(c + 1, nextBase, nextEnd, cur);
        bool wait = k < cnt;
        uint32_t v = 0;
        // the first inputs are in registers before the root's level is known
        auto input = [&](uint32_t i) -> uint32_t {
            if (i >= stop) return UNSET;
            return i - base < ID_INPUTS ? s_in[b][i - base] : a.in[i];
        };
        uint32_t near[ID_NEAR];
#pragma unroll
        for (uint32_t j = 0; j < ID_NEAR; j++) near[j] = input(off + j);
        auto hand = [&](uint32_t q) {
            if (q == UNSET) return;
            const uint32_t d = (q - first) / ID_CHUNK, t = (q - first) % ID_CHUNK;
            if (v) {
                if (d - c < ID_RING - 1) atomicMax(&s_val[(d % ID_RING) * ID_CHUNK + t], v + 1u);
                else atomicMax(&a.val[q], v + 1u);
            }
            asm volatile("" ::: "memory");       // handed over before it is counted
            if (d == c) atomicSub(&s_pend[b][t], 1u);
        };
        while (__ballot(wait) != 0) {
            const uint32_t left = lds_load(&s_pend[b][tid]);
            asm volatile("" ::: "memory");       // the level is read after the count
            const uint32_t x = lds_load(own);
            if (!wait || left != 0) continue;
            wait = false;
            v = x;
#pragma unroll
            for (uint32_t j = 0; j < ID_NEAR; j++) hand(near[j]);
            for (uint32_t i = off + ID_NEAR; i < stop; i++) hand(input(i));
        }
        if (k < cnt) a.val[first + k] = v;
        most = max(most, v);
        *own = 0;                                // of the chunk that takes its place
    }
    atomicMax(&s_most, most);
    __syncthreads();
    if (tid == 0) a.rounds[blockIdx.x] = s_most;
}

__global__ void k_id_levels(uint32_t m, const uint32_t *__restrict__ rootAt, const uint32_t *__restrict__ val,
                            uint32_t *lastLevel) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < m; p += stride)
        if (val[p]) lastLevel[rootAt[p]] = val[p] - 1u;
}

__global__ void k_taken_flags(int32_t n, const uint32_t *__restrict__ lastLevel, uint8_t *flag) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t v = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; v < n; v += stride) flag[v] = lastLevel[v] != UNSET;
}

__global__ void __launch_bounds__(kBlock) k_count_tags(uint32_t m, const uint32_t *__restrict__ roots,
                                                       const uint32_t *__restrict__ tag, uint32_t *cnt) {
    __shared__ uint32_t s_bins[TAG_BINS];
    TagBins tb{s_bins};
    tb.init();
    int64_t b, e;
    tag_chunk(0, m, b, e);
    for (int64_t i = b + threadIdx.x; i < e; i += blockDim.x) tb.add(cnt, tag[roots[i]], 1u);
    tb.flush_add(cnt, 0xFFFFFFFFu);
}

__global__ void k_gather_tags(uint32_t m, const uint32_t *__restrict__ roots, const uint32_t *__restrict__ tag,
                              uint32_t *keys) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < m; i += stride) keys[i] = tag[roots[i]];
}

// sort key of every root: its level, after the levels of the segments before
// its own (levOff) where they are given
__global__ void k_level_keys(uint32_t m, const uint32_t *__restrict__ roots, const uint32_t *__restrict__ lastLevel,
                             const uint32_t *__restrict__ tag, const uint32_t *__restrict__ levOff, uint32_t *keys) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < m; i += stride)
        keys[i] = lastLevel[roots[i]] + (levOff ? levOff[tag[roots[i]]] : 0u);
}

// first position of every key (each occurs), and one past the last
__global__ void k_key_starts(uint32_t m, const uint32_t *__restrict__ keys, uint32_t nKeys, uint32_t *starts) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i <= m; i += stride) {
        if (i == m) starts[nKeys] = m;
        else if (i == 0 || keys[i] != keys[i - 1]) starts[keys[i]] = (uint32_t)i;
    }
}

constexpr uint32_t SRC_MEM = 0xFFFFu;

// every root's place, its cover's inputs, and the most ANDs it can create (none from a constant)
__global__ void k_cover_lens(uint32_t m, const uint32_t *__restrict__ roots, const uint2 *__restrict__ cover,
                             uint32_t *len, uint32_t *most, uint32_t *place) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i <= m; i += stride) {
        const uint32_t k = i < m ? cover[roots[i]].y : 0u;
        if (i < m) place[roots[i]] = (uint32_t)i;
        len[i] = k;
        most[i] = k ? k - 1u : 0u;
    }
}

// the covers' inputs in the order in which they are rebuilt
__global__ void k_pack_inputs(uint32_t m, const uint32_t *__restrict__ roots, const uint2 *__restrict__ cover,
                              const uint32_t *__restrict__ pool, const uint32_t *__restrict__ off,
                              const uint32_t *__restrict__ keys, const uint32_t *__restrict__ starts,
                              const uint32_t *__restrict__ lastLevel, const uint32_t *__restrict__ place, int32_t nPIs,
                              uint32_t *in, uint32_t *src) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < m; i += stride) {
        const uint32_t v = roots[i], lv = lastLevel[v], key = keys[i], cov = ((uint32_t)i - starts[key]) & 0xFFFFu;
        const uint2 c = cover[v];
        for (uint32_t j = 0; j < c.y; j++) {
            const uint32_t lit = pool[c.x + j], id = lit >> 1;
            uint32_t at = SRC_MEM;
            if ((int32_t)id > nPIs && lastLevel[id] == lv + 1u) at = min(place[id] - starts[key + 1u], SRC_MEM);
            in[off[i] + j] = lit;
            src[off[i] + j] = at << 16 | cov;
        }
    }
}

// largest level: covers, inputs, ANDs it can create; and per level its extent
struct alignas(16) LevelRec {
    uint32_t s, nb, in0, T;           // first root, roots, first input, inputs
    uint32_t most, pad[3];            // ANDs it can create
};

__global__ void k_level_sizes(uint32_t nKeys, const uint32_t *__restrict__ starts, const uint32_t *__restrict__ off,
                              const uint32_t *__restrict__ newOff, LevelRec *rec, uint32_t *most) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < nKeys; k += stride) {
        const uint32_t a = starts[k], b = starts[k + 1];
        const LevelRec z = {a, b - a, off[a], off[b] - off[a], newOff[b] - newOff[a], {}};
        rec[k] = z;
        atomicMax(&most[0], z.nb);
        atomicMax(&most[1], z.T);
        atomicMax(&most[2], z.most);
    }
}

// ---------------------------------------------------------------------------
// phase 2: reconstruction
// ---------------------------------------------------------------------------
struct RecArgs {
    NodeTable t;
    int32_t nPIs;
    const uint32_t *roots;            // roots by (segment, level, id)
    const uint32_t *off, *in;         // their covers' inputs
    const uint32_t *src;              // per input: place of its root in the level before << 16 (SRC_MEM: not there) | cover
    const LevelRec *lev;              // per (segment, level)
    const uint32_t *starts;           // first root of every (segment, level)
    unsigned long long *newSig;       // per root id: the result
    uint32_t *of0, *of1;              // fanins of the created nodes, by id
    uint32_t *tagOut;                 // optional: their tags (where a segment holds several)
    const uint32_t *tagIn;
    uint32_t *err;                    // 2: table full
    uint32_t shuffle;                 // 1: `b -s` input order (sortDecId = 0)
    // grid-wide phases: a batch's covers and their state
    unsigned long long *arr;          // inputs, packed as in `in` from the batch's first
    uint32_t *alen;
    uint8_t *mask;
    unsigned long long *skey, *sres;
    uint32_t *slot, *bcnt;
    uint32_t *counter;                // next id, alternating between two words by step
};

// thrust::shuffle(thrust::seq, ..., default_random_engine(seed)) as an index
// map, the tie-break of `b -s` (balance.cu:301, 404-411).  The algorithm is
// thrust's (rocThrust thrust/system/detail/generic/shuffle.inl, ROCm 7.2): a
// 24-round Feistel bijection over the next power of two (at least 16) with
// round keys from minstd_rand seeded by `seed` (0 taken as 1); position k of
// the shuffled sequence holds the input whose index is the k-th value below
// len that the bijection yields for 0, 1, 2, ...
struct ThrustShuffle {
    uint32_t key[24];
    uint32_t lb, rb, lmask, rmask, span;
    __device__ ThrustShuffle(uint32_t len, uint32_t seed) {
        uint32_t x = seed % 2147483647u;
        if (x == 0) x = 1;
        uint32_t bits = 4;
        if (len > 16) {
            bits = 0;
            for (uint32_t m = len - 1; m; m >>= 1) bits++;
        }
        lb = bits / 2;
        rb = bits - lb;
        lmask = (1u << lb) - 1u;
        rmask = (1u << rb) - 1u;
        span = 1u << bits;
        for (int i = 0; i < 24; i++) {
            x = (uint32_t)(((uint64_t)x * 48271u) % 2147483647u);
            key[i] = x;
        }
    }
    __device__ uint32_t operator()(uint32_t j) const {
        uint32_t s0 = j >> rb, s1 = j & rmask;
        for (int r = 0; r < 24; r++) {
            const uint64_t prod = 0xD2B74407B1CE6E93ull * (uint64_t)s0;
            const uint32_t hi = (uint32_t)(prod >> 32);
            const uint32_t lo = ((uint32_t)prod << (rb - lb)) | (s1 >> lb);
            s0 = ((hi ^ key[r]) ^ s1) & lmask;
            s1 = lo & rmask;
        }
        return (s0 << rb) | s1;
    }
};

// the input before which another one stands: level descending, then (`b`) the
// reference's literal value descending; equal ones keep their order
__device__ __forceinline__ bool sorts_before(uint32_t shuffle, unsigned long long a, unsigned long long b) {
    if (sig_lev(a) != sig_lev(b)) return sig_lev(a) > sig_lev(b);
    return !shuffle && culs_val(sig_lit(a)) > culs_val(sig_lit(b));
}

// the same as a number: a stands before b if its key is larger
__device__ __forceinline__ unsigned long long order_key(uint32_t shuffle, unsigned long long a) {
    return (unsigned long long)sig_lev(a) << 32 | (shuffle ? 0u : culs_val(sig_lit(a)));
}

__device__ __forceinline__ unsigned long long input_sig(const RecArgs &r, uint32_t lit) {
    const uint32_t id = lit >> 1;
    return (int32_t)id <= r.nPIs ? sig(lit, 0u) : r.newSig[id] ^ (lit & 1u);
}

// ---- one workgroup per segment, levels within its LDS
constexpr uint32_t LT_INPUTS = 4096;      // inputs of a level
constexpr uint32_t LT_COVERS = BAL_LDS_COVERS;   // covers of a level
constexpr uint32_t LT_NEW = 3072;         // ANDs that a level can create
constexpr uint32_t LT_HASH = 4096;        // entries of the level's own node table
constexpr uint32_t LQ_IN = LT_INPUTS / BAL_WG, LQ_COV = LT_COVERS / BAL_WG, LQ_NEW = LT_NEW / BAL_WG;
constexpr uint32_t LN_FINAL = 0x80000000u, LS_NONE = 0xFFFFu;

// Rebuilds levels lFirst, lFirst - 1, .., lLast of its segment (levOff: the
// segments' first levels in starts; levels beyond the segment's are skipped).
// A level's cover inputs and the nodes it creates live in LDS; the table in
// memory holds the nodes of the levels before.  A pair of a cover's inputs is
// looked up there once, before the steps: the partner that the permutation may
// try for input j has the level of input j - 1 (the list is consumed from its
// end, and what a step puts back does not separate inputs of one level), so
// each input tries those, four at a time, and the ones that exist enter the
// level's own table.  The steps then look up in LDS only, except a cover whose
// pair was found once: what came back may be an older node, and the permutation
// may have changed which inputs meet, so its later pairs are looked up in
// memory as well.  A step has three barriers: keys inserted; winners (the
// smallest cover index of a key) counted; ids given; and once 64 covers at most
// have a pair left, one wavefront takes the remaining steps without any.
// What bounds it is latency, so little is left between two levels: results of
// the level before come from LDS, other inputs are read during its steps, its
// table insertions are under way until the lookups, and only used entries of
// the level's table are cleared.  The 128 registers of a thread matter: what is
// spilled is waited for, and the insertions with it, so the next level's words
// are read after the sort.  The table in memory is at most a quarter full: a
// wavefront waits for the longest of its lanes' probe chains.  2M random ANDs
// (1786 levels of 668 covers and 1523 inputs): 37.2 ms; 38.8 with each step's
// pairs and nodes handed on through LDS, 45.1 before that with the next
// level read at the start (spilled) and a table twice as full, 63 with every
// lookup made at its step in memory.  The 64-bit multiplier (a level has 77
// covers, 161 inputs): 2.5 ms for 414 levels, 3.4 before.
__global__ void __launch_bounds__(BAL_WG) k_rec_lds(RecArgs r, const uint32_t *__restrict__ levOff,
                                                    const uint32_t *__restrict__ idBase, uint32_t *made, int32_t lFirst,
                                                    int32_t lLast) {
    __shared__ unsigned long long s_key[LT_HASH];
    __shared__ uint32_t s_val[LT_HASH];              // smallest cover index, then LN_FINAL | node
    __shared__ unsigned long long s_arr[LT_INPUTS];  // the covers' current inputs
    __shared__ unsigned long long s_node[LT_NEW];    // nodes: created from 0 up, found in memory from the top down
    __shared__ unsigned long long s_res[LT_COVERS];  // the covers' results, for the next level
    __shared__ uint16_t s_ent[LT_NEW];               // the nodes' entries in s_key, LS_NONE: another one has it
    __shared__ uint16_t s_perm[LT_INPUTS];           // `b -s`: the shuffled inputs
    __shared__ uint16_t s_off[LT_COVERS + 1], s_len[LT_COVERS], s_act[64];
    __shared__ uint8_t s_mem[LT_COVERS];             // the cover's pairs are looked up in memory too
    __shared__ uint32_t s_cnt[LQ_COV][BAL_WG / 64], s_over;
    __shared__ int32_t s_top;
    const uint32_t tid = threadIdx.x, seg = blockIdx.x, wave = tid >> 6, lane = tid & 63u;
    const uint32_t lev0 = levOff[seg], nLev = levOff[seg + 1] - lev0, base0 = idBase[seg];
    uint32_t counter = base0 + made[seg];            // next id
    // a level's extent, its inputs (one per thread and LQ_IN), its covers' first
    // inputs and roots.  Extents are read a level before they are used, into
    // vector registers: in scalar ones they would be waited for at once
    struct Extent {
        uint4 x;
        uint32_t most;
    };
    struct Level {
        LevelRec e;
        uint32_t lit[LQ_IN], src[LQ_IN], off[LQ_COV], root[LQ_COV];
        unsigned long long sig[LQ_IN];
    };
    auto load_extent = [&](int32_t l) -> Extent {
        uint32_t k = lev0 + (uint32_t)max(l, 0);
        asm volatile("" : "+v"(k));
        return {*reinterpret_cast<const uint4 *>(&r.lev[k]), r.lev[k].most};
    };
    auto first_lane = [](uint32_t x) -> uint32_t { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); };
    auto load_level = [&](int32_t l, const Extent &x, Level &v) {
        LevelRec e = {};
        if (l >= lLast) e = {first_lane(x.x.x), first_lane(x.x.y), first_lane(x.x.z), first_lane(x.x.w), first_lane(x.most), {}};
        v.e = e;
#pragma unroll
        for (uint32_t q = 0; q < LQ_IN; q++) {
            const uint32_t i = tid + q * BAL_WG;
            v.lit[q] = i < e.T ? r.in[e.in0 + i] : 0u;
            v.src[q] = i < e.T ? r.src[e.in0 + i] : 0u;
        }
#pragma unroll
        for (uint32_t q = 0; q < LQ_COV; q++) {
            const uint32_t c = tid + q * BAL_WG;
            v.off[q] = c < e.nb ? r.off[e.s + c] : 0u;
            v.root[q] = c < e.nb ? r.roots[e.s + c] : 0u;
        }
    };
    // the inputs that are not results of the level before (first: all), without
    // their complement: nothing is to wait for them here
    auto load_inputs = [&](bool first, Level &v) {
#pragma unroll
        for (uint32_t q = 0; q < LQ_IN; q++) {
            v.sig[q] = 0;
            if (tid + q * BAL_WG >= v.e.T) continue;
            if (first) v.src[q] |= SRC_MEM << 16;
            const uint32_t id = v.lit[q] >> 1;
            if ((int32_t)id <= r.nPIs) v.sig[q] = sig(2u * id, 0u);
            else if (v.src[q] >> 16 == SRC_MEM) v.sig[q] = r.newSig[id];
        }
    };
    for (uint32_t i = tid; i < LT_HASH; i += BAL_WG) { s_key[i] = EMPTY64; s_val[i] = UNSET; }
    int32_t l = min(lFirst, (int32_t)nLev - 1);
    Level cur, next;
    load_level(l, load_extent(l), cur);
    Extent ahead = load_extent(l - 1);
    load_inputs(true, cur);
    // (also before the first level: a wait that the loop shares with it would include the insertions)
    auto arrived = [&](Level &v) {
#pragma unroll
        for (uint32_t q = 0; q < LQ_IN; q++) asm volatile("" : "+v"(v.sig[q]), "+v"(v.lit[q]), "+v"(v.src[q]));
#pragma unroll
        for (uint32_t q = 0; q < LQ_COV; q++) asm volatile("" : "+v"(v.off[q]), "+v"(v.root[q]));
    };
    arrived(cur);
    // the level before's nodes, on their way into the table
    unsigned long long newKey[LQ_NEW], newPrev[LQ_NEW];
    uint32_t newSlot[LQ_NEW];
#pragma unroll
    for (uint32_t q = 0; q < LQ_NEW; q++) newKey[q] = EMPTY64;
    auto finish_inserts = [&]() {
#pragma unroll
        for (uint32_t q = 0; q < LQ_NEW; q++) {
            if (newKey[q] == EMPTY64) continue;
            uint64_t probes = 0;
            while (newPrev[q] != EMPTY64 && newPrev[q] != newKey[q] && probes++ <= r.t.mask) {
                newSlot[q] = (uint32_t)((newSlot[q] + 1ull) & r.t.mask);
                newPrev[q] = t_cas(r.t, newSlot[q], newKey[q]);
            }
            if (newPrev[q] != EMPTY64 && newPrev[q] != newKey[q]) { atomicOr(r.err, 2u); continue; }
            // (its place in s_node is taken by this level's nodes only later)
            __hip_atomic_store(&r.t.v[newSlot[q]], s_node[tid + q * BAL_WG], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    };
    for (; l >= lLast; l--) {
        const uint32_t nb = cur.e.nb, T = cur.e.T, most = cur.e.most, levBase = counter;
#pragma unroll
        for (uint32_t q = 0; q < LQ_COV; q++) {
            const uint32_t c = tid + q * BAL_WG;
            if (c < nb) { s_off[c] = (uint16_t)(cur.off[q] - cur.e.in0); s_mem[c] = 0; }
        }
        if (tid == 0) { s_off[nb] = (uint16_t)T; s_top = (int32_t)LT_NEW; s_over = 0; }
        unsigned long long mine[LQ_IN];
#pragma unroll
        for (uint32_t q = 0; q < LQ_IN; q++) {
            mine[q] = cur.sig[q];
            if (tid + q * BAL_WG >= T) continue;
            if (cur.src[q] >> 16 != SRC_MEM) mine[q] = s_res[cur.src[q] >> 16];
            mine[q] ^= cur.lit[q] & 1u;
            s_arr[tid + q * BAL_WG] = mine[q];
        }
        __syncthreads();
        if (r.shuffle) {
            // `b -s`: the inputs in the order of the shuffle seeded with the
            // cover's index in its batch
            for (uint32_t c = tid; c < nb; c += BAL_WG) {
                const uint32_t o = s_off[c], n = s_off[c + 1] - o;
                if (n == 0) continue;
                const ThrustShuffle sh(n, c);
                uint32_t k = 0;
                for (uint32_t j = 0; j < sh.span && k < n; j++) {
                    const uint32_t src = sh(j);
                    if (src < n) s_perm[o + k++] = (uint16_t)(o + src);
                }
            }
            __syncthreads();
#pragma unroll
            for (uint32_t q = 0; q < LQ_IN; q++)
                if (tid + q * BAL_WG < T) mine[q] = s_arr[s_perm[tid + q * BAL_WG]];
            __syncthreads();
#pragma unroll
            for (uint32_t q = 0; q < LQ_IN; q++)
                if (tid + q * BAL_WG < T) s_arr[tid + q * BAL_WG] = mine[q];
            __syncthreads();
        }
        // each input's place by its rank among the cover's
        uint32_t place[LQ_IN];
#pragma unroll
        for (uint32_t q = 0; q < LQ_IN; q++) {
            const uint32_t i = tid + q * BAL_WG;
            place[q] = UNSET;
            if (i >= T) continue;
            const uint32_t c = cur.src[q] & 0xFFFFu, o = s_off[c], e = s_off[c + 1];
            const unsigned long long x = order_key(r.shuffle, mine[q]);
            uint32_t p = o;
            for (uint32_t j = o; j < e; j += 2) {
                const unsigned long long y0 = order_key(r.shuffle, s_arr[j]);
                const unsigned long long y1 = order_key(r.shuffle, s_arr[min(j + 1, e - 1)]);
                p += y0 > x || (y0 == x && j < i) ? 1u : 0u;
                p += j + 1 < e && (y1 > x || (y1 == x && j + 1 < i)) ? 1u : 0u;
            }
            place[q] = p;
        }
        __syncthreads();
#pragma unroll
        for (uint32_t q = 0; q < LQ_IN; q++)
            if (place[q] != UNSET) s_arr[place[q]] = mine[q];
        for (uint32_t c = tid; c < nb; c += BAL_WG) s_len[c] = (uint16_t)(s_off[c + 1] - s_off[c]);
        finish_inserts();                       // the keys are there; the nodes are not waited for
        __syncthreads();
        // the next level's words set out (not earlier: they take registers, and what
        // does not fit is spilled to memory)
        load_level(l - 1, ahead, next);
        ahead = load_extent(l - 2);
        // the level's own table
        auto hash = [](unsigned long long key) -> uint32_t {
            const uint32_t h = (uint32_t)(key >> 32) * 0x9E3779B1u + (uint32_t)key;
            return (h ^ h >> 15) & (LT_HASH - 1);
        };
        auto level_slot = [&](unsigned long long key, bool &isNew) -> uint32_t {
            for (uint32_t h = hash(key);; h = (h + 1) & (LT_HASH - 1)) {
                unsigned long long prev = EMPTY64;
                __hip_atomic_compare_exchange_strong(&s_key[h], &prev, key, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_WORKGROUP);
                isNew = prev == EMPTY64;
                if (isNew || prev == key) return h;
            }
        };
        // its node with this key, or EMPTY64; k is the key at its first entry h
        auto level_find = [&](unsigned long long key, uint32_t h, unsigned long long k) -> unsigned long long {
            for (;;) {
                if (k == EMPTY64) return EMPTY64;
                if (k == key) {
                    const uint32_t v = lds_load(&s_val[h]);
                    // inserted in this step: not there yet
                    return v == UNSET || !(v & LN_FINAL) ? EMPTY64 : s_node[v & ~LN_FINAL];
                }
                h = (h + 1) & (LT_HASH - 1);
                k = lds_load(&s_key[h]);
            }
        };
        // pairs of inputs that exist: two of a thread's inputs at a time, two
        // candidates of each
#pragma unroll
        for (uint32_t g = 0; g < LQ_IN; g += 2) {
            if (g * BAL_WG >= T) break;
            uint32_t o[2], left[2], border[2];       // candidates [o, left)
            unsigned long long x[2];
#pragma unroll
            for (int p = 0; p < 2; p++) {
                const uint32_t j = tid + (g + p) * BAL_WG;
                o[p] = left[p] = border[p] = 0;
                x[p] = 0;
                if (j >= T) continue;
                // position j's cover is input j's: the order is within covers
                o[p] = s_off[cur.src[g + p] & 0xFFFFu];
                left[p] = j;
                x[p] = s_arr[j];
                border[p] = j > o[p] ? sig_lev(s_arr[j - 1]) : 0u;
            }
            while (__ballot(left[0] > o[0] || left[1] > o[1]) != 0) {
                unsigned long long key[4];
                uint64_t slot[4];
                uint32_t wait = 0;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int p = q >> 1;
                    key[q] = EMPTY64;
                    slot[q] = 0;
                    if (left[p] <= o[p]) continue;
                    const unsigned long long y = s_arr[left[p] - 1];
                    if (sig_lev(y) != border[p]) { left[p] = o[p]; continue; }
                    left[p]--;
                    if (and_trivial(x[p], y) != EMPTY64) continue;
                    key[q] = and_key_of(sig_lit(x[p]), sig_lit(y));
                    slot[q] = t_hash(r.t, key[q]);
                    wait |= 1u << q;
                }
                while (__ballot(wait != 0) != 0) {
                    unsigned long long k[4];
#pragma unroll
                    for (int q = 0; q < 4; q++) k[q] = (wait >> q) & 1u ? t_load(&r.t.k[slot[q]]) : EMPTY64;
                    uint32_t hit = 0;
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        if (k[q] == EMPTY64) wait &= ~(1u << q);
                        if (k[q] == key[q] && ((wait >> q) & 1u)) hit |= 1u << q;
                        slot[q] = (slot[q] + 1) & r.t.mask;
                    }
                    wait &= ~hit;
                    while (hit) {
                        const int q = __ffs((int)hit) - 1;
                        hit &= hit - 1u;
                        const unsigned long long kq = q < 2 ? (q == 0 ? key[0] : key[1]) : (q == 2 ? key[2] : key[3]);
                        const uint64_t sq = q < 2 ? (q == 0 ? slot[0] : slot[1]) : (q == 2 ? slot[2] : slot[3]);
                        // nodes found and created together at most LT_NEW (so the table has room)
                        const int32_t at = atomicSub(&s_top, 1) - 1;
                        if (at < (int32_t)most) { s_over = 1; continue; }
                        bool isNew = false;
                        const uint32_t h = level_slot(kq, isNew);
                        s_ent[at] = isNew ? (uint16_t)h : (uint16_t)LS_NONE;
                        if (isNew) {
                            s_node[at] = t_node(r.t, (sq - 1) & r.t.mask);
                            s_val[h] = LN_FINAL | (uint32_t)at;
                        }
                    }
                }
            }
        }
        __builtin_amdgcn_s_waitcnt(0x0F70);     // vmcnt(0): the level before's results are written
        __syncthreads();
        load_inputs(false, next);
        const bool over = s_over != 0;       // not all of them fit: every cover looks up in memory too
        // sharedNodeDrivenPermute and prepareDataToInsert (balance.cu:113-247)
        // of a cover with two inputs at least: takes its last two; returns the
        // existing signal, or EMPTY64, the inserted key, its slot (+ 1) and the
        // level of its node
        struct Pair {
            unsigned long long key;
            uint32_t slot, lev;
        };
        auto prepare = [&](uint32_t c, uint32_t o, uint32_t L, Pair &pair) -> unsigned long long {
            const uint32_t right = o + L - 2;
            const unsigned long long l1 = s_arr[right + 1], l2 = s_arr[right];
            const uint32_t x1 = sig_lit(l1), border = sig_lev(l2);
            const bool old1 = (over || s_mem[c] != 0) && (x1 >> 1) < levBase;
            unsigned long long found = EMPTY64, l3 = l2;
            for (uint32_t i = right;;) {
                const unsigned long long before = s_arr[i > o ? i - 1 : o], key = and_key_of(x1, sig_lit(l3));
                const uint32_t h = hash(key);
                const unsigned long long k = lds_load(&s_key[h]);
                found = and_trivial(l1, l3);
                if (found == EMPTY64 && k != EMPTY64) found = level_find(key, h, k);
                if (found == EMPTY64 && old1 && (sig_lit(l3) >> 1) < levBase) found = t_find(r.t, key);
                if (found != EMPTY64) {
                    s_arr[i] = l2;           // the partner goes next to last; the order by level stays
                    break;
                }
                if (i == o || sig_lev(before) != border) break;
                i--;
                l3 = before;
            }
            pair.slot = 0;
            if (found == EMPTY64) {
                bool isNew;
                pair.key = and_key_of(x1, sig_lit(l2));
                pair.lev = (sig_lev(l1) > border ? sig_lev(l1) : border) + 1u;
                const uint32_t h = level_slot(pair.key, isNew);
                atomicMin(&s_val[h], c);
                pair.slot = h + 1;
            } else {
                s_mem[c] = 1;
            }
            return found;
        };
        // the winner of a key becomes node `at` of the level
        auto create = [&](uint32_t c, const Pair &pair, uint32_t at) -> unsigned long long {
            const uint32_t id = levBase + at;
            const unsigned long long x = sig(2u * id, pair.lev);
            s_node[at] = x;
            s_val[pair.slot - 1] = LN_FINAL | at;
            s_ent[at] = (uint16_t)(pair.slot - 1);
            r.of0[id] = (uint32_t)(pair.key >> 32);
            r.of1[id] = (uint32_t)pair.key;
            if (r.tagOut) r.tagOut[id] = r.tagIn[r.roots[cur.e.s + c]];
            return x;
        };
        // addBackLocalArrays (balance.cu:429-467); returns the new length.  The
        // last four inputs are read together: a step waits for these reads, and
        // most covers have no more.
        auto add_back = [&](uint32_t o, uint32_t L, unsigned long long x) -> uint32_t {
            unsigned long long y[4];
            bool there = false;
#pragma unroll
            for (uint32_t k = 0; k < 4; k++) y[k] = s_arr[o + (L > k ? L - 1 - k : 0)];
#pragma unroll
            for (uint32_t k = 0; k < 4; k++) there |= k < L && sig_lit(y[k]) == sig_lit(x);
            for (uint32_t i = 4; i < L; i += 2)
                there |= sig_lit(s_arr[o + L - 1 - i]) == sig_lit(x) || sig_lit(s_arr[o + (L > i + 1 ? L - 2 - i : 0)]) == sig_lit(x);
            if (there) return L;
            uint32_t i = L;
            bool stop = false;
#pragma unroll
            for (uint32_t k = 0; k < 4; k++) {
                stop |= k >= L || sig_lev(x) <= sig_lev(y[k]);
                if (stop) continue;
                s_arr[o + i] = y[k];
                i--;
            }
            while (!stop && i > 0) {
                const unsigned long long z = s_arr[o + i - 1];
                if (sig_lev(x) <= sig_lev(z)) break;
                s_arr[o + i] = z;
                i--;
            }
            s_arr[o + i] = x;
            return L + 1;
        };
        // ---- steps by all wavefronts, while more than 64 covers have a pair left
        uint32_t nAct = nb;
        if (nb <= 64u && tid < 64u) s_act[tid] = (uint16_t)tid;
        while (nAct > 64u) {
            Pair pair[LQ_COV];
            uint32_t len[LQ_COV];
            unsigned long long became[LQ_COV];        // what the pair became
#pragma unroll
            for (uint32_t q = 0; q < LQ_COV; q++) {
                const uint32_t c = tid + q * BAL_WG;
                pair[q].slot = 0;
                len[q] = c < nb ? s_len[c] : 0u;
                if (len[q] <= 1) continue;
                const uint32_t o = s_off[c];
                const unsigned long long f = prepare(c, o, len[q], pair[q]);
                len[q] = pair[q].slot ? len[q] - 2 : add_back(o, len[q] - 2, f);
            }
            __syncthreads();
            // winners, counted in cover order
            uint32_t rank[LQ_COV];
#pragma unroll
            for (uint32_t q = 0; q < LQ_COV; q++) {
                const uint32_t c = tid + q * BAL_WG;
                const bool win = pair[q].slot != 0 && s_val[pair[q].slot - 1] == c;
                const uint64_t m = __ballot(win);
                rank[q] = win ? (uint32_t)__popcll(m & ((1ull << lane) - 1ull)) : UNSET;
                if (lane == 0) s_cnt[q][wave] = (uint32_t)__popcll(m);
            }
            __syncthreads();
            uint32_t total = 0;
#pragma unroll
            for (uint32_t q = 0; q < LQ_COV; q++) {
                uint32_t before = total;
#pragma unroll
                for (uint32_t w = 0; w < BAL_WG / 64; w++) {
                    const uint32_t x = s_cnt[q][w];
                    before += w < wave ? x : 0u;
                    total += x;
                }
                if (rank[q] != UNSET) became[q] = create(tid + q * BAL_WG, pair[q], counter - levBase + before + rank[q]);
            }
            counter += total;
            __syncthreads();
            // results back; the covers that still have a pair, counted
            uint64_t am[LQ_COV];
#pragma unroll
            for (uint32_t q = 0; q < LQ_COV; q++) {
                const uint32_t c = tid + q * BAL_WG;
                if (pair[q].slot != 0) {
                    if (rank[q] == UNSET) became[q] = s_node[s_val[pair[q].slot - 1] & ~LN_FINAL];
                    len[q] = add_back(s_off[c], len[q], became[q]);
                }
                if (c < nb) s_len[c] = (uint16_t)len[q];
                am[q] = __ballot(len[q] > 1);
                if (lane == 0) s_cnt[q][wave] = (uint32_t)__popcll(am[q]);
            }
            __syncthreads();
            nAct = 0;
            uint32_t before[LQ_COV];
#pragma unroll
            for (uint32_t q = 0; q < LQ_COV; q++) {
                before[q] = nAct;
#pragma unroll
                for (uint32_t w = 0; w < BAL_WG / 64; w++) {
                    const uint32_t x = s_cnt[q][w];
                    before[q] += w < wave ? x : 0u;
                    nAct += x;
                }
            }
            if (nAct > 64u) continue;
#pragma unroll
            for (uint32_t q = 0; q < LQ_COV; q++)
                if ((am[q] >> lane) & 1ull)
                    s_act[before[q] + (uint32_t)__popcll(am[q] & ((1ull << lane) - 1ull))] = (uint16_t)(tid + q * BAL_WG);
        }
        __syncthreads();
        // ---- the others by the first wavefront: its lanes hold the covers in order
        if (nAct != 0) {
            if (wave == 0) {
                const bool has = lane < nAct;
                const uint32_t c = has ? s_act[lane] : 0u, o = s_off[c];
                uint32_t L = has ? s_len[c] : 0u;
                while (__ballot(L > 1) != 0) {
                    Pair pair = {};
                    unsigned long long f = EMPTY64;
                    const bool act = L > 1;
                    if (act) {
                        f = prepare(c, o, L, pair);
                        L -= 2;
                    }
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    const bool win = pair.slot != 0 && lds_load(&s_val[pair.slot - 1]) == c;
                    const uint64_t m = __ballot(win);
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    if (win) f = create(c, pair, counter - levBase + (uint32_t)__popcll(m & ((1ull << lane) - 1ull)));
                    counter += (uint32_t)__popcll(m);
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    if (pair.slot != 0 && !win) f = s_node[lds_load(&s_val[pair.slot - 1]) & ~LN_FINAL];
                    if (act) L = add_back(o, L, f);
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                }
                if (has) s_len[c] = (uint16_t)L;
                if (lane == 0) s_cnt[0][0] = counter;
            }
            __syncthreads();
            counter = s_cnt[0][0];
        }
        // the next level's loads have arrived: the waits for them stand here, where
        // they do not include the insertions
        arrived(next);
        // the level's nodes set out for the table; its own table is cleared
#pragma unroll
        for (uint32_t q = 0; q < LQ_NEW; q++) {
            const uint32_t i = tid + q * BAL_WG;
            newKey[q] = EMPTY64;
            if (i >= counter - levBase) continue;
            const uint32_t h = s_ent[i];
            newKey[q] = s_key[h];
            s_key[h] = EMPTY64;
            s_val[h] = UNSET;
            newSlot[q] = (uint32_t)t_hash(r.t, newKey[q]);
            newPrev[q] = t_cas(r.t, newSlot[q], newKey[q]);
        }
        for (int32_t i = (int32_t)(LT_NEW - 1 - tid), end = max(s_top, (int32_t)most); i >= end; i -= (int32_t)BAL_WG) {
            const uint32_t h = s_ent[i];
            if (h == LS_NONE) continue;
            s_key[h] = EMPTY64;
            s_val[h] = UNSET;
        }
        // results
#pragma unroll
        for (uint32_t q = 0; q < LQ_COV; q++) {
            const uint32_t c = tid + q * BAL_WG;
            if (c >= nb) continue;
            const unsigned long long x = s_len[c] == 0 ? 0ull : s_arr[s_off[c]];
            s_res[c] = x;
            r.newSig[cur.root[q]] = x;
        }
        cur = next;
        __syncthreads();
    }
    finish_inserts();
    if (tid == 0) made[seg] = counter - base0;
}

// ---- wide levels: a batch of covers, one kernel per phase of a step

// prepareReconstructArrays (balance.cu:272-427)
__global__ void k_rec_gather(RecArgs r, uint32_t s, uint32_t nb) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    const uint32_t in0 = r.off[s];
    for (int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; c < nb; c += stride) {
        const uint32_t o = r.off[s + c], len = r.off[s + c + 1] - o;
        unsigned long long *A = r.arr + (o - in0);
        r.alen[c] = len;
        if (r.shuffle) {
            // `b -s`: the inputs in the order of the shuffle seeded with the
            // cover's index in its batch
            if (len > 0) {
                const ThrustShuffle sh(len, (uint32_t)c);
                uint32_t k = 0;
                for (uint32_t j = 0; j < sh.span && k < len; j++) {
                    const uint32_t src = sh(j);
                    if (src < len) A[k++] = input_sig(r, r.in[o + src]);
                }
            }
        } else {
            for (uint32_t i = 0; i < len; i++) A[i] = input_sig(r, r.in[o + i]);
        }
        // insertion sort keeps equal keys in order, as thrust's sequential sort does
        for (uint32_t i = 1; i < len; i++) {
            const unsigned long long x = A[i];
            int j = (int)i - 1;
            while (j >= 0 && sorts_before(r.shuffle, x, A[j])) {
                A[j + 1] = A[j];
                j--;
            }
            A[j + 1] = x;
        }
    }
}

// sharedNodeDrivenPermute then prepareDataToInsert: mask 0 done, 1 a new key
// (skey, its level in sres), 2 an existing signal (sres)
__global__ void k_rec_prepare(RecArgs r, uint32_t s, uint32_t nb) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    const uint32_t in0 = r.off[s];
    auto lookup = [&](unsigned long long a, unsigned long long b) -> unsigned long long {
        const unsigned long long t = and_trivial(a, b);
        return t != EMPTY64 ? t : t_find(r.t, and_key_of(sig_lit(a), sig_lit(b)));
    };
    for (int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; c < nb; c += stride) {
        unsigned long long *A = r.arr + (r.off[s + c] - in0);
        const uint32_t L = r.alen[c];
        if (L <= 1) { r.mask[c] = 0; continue; }
        const int right = (int)L - 2;
        int left = right;
        const unsigned long long l1 = A[right + 1], l2 = A[right];
        while (left > 0 && sig_lev(A[left - 1]) == sig_lev(l2)) left--;
        unsigned long long found = EMPTY64;
        for (int i = right; i >= left && found == EMPTY64; i--) {
            found = lookup(l1, A[i]);
            if (found != EMPTY64) A[i] = l2;        // the partner goes next to last
        }
        r.alen[c] = L - 2;
        if (found != EMPTY64) {
            r.mask[c] = 2;
            r.sres[c] = found;
            continue;
        }
        r.mask[c] = 1;
        r.skey[c] = and_key_of(sig_lit(l1), sig_lit(l2));
        r.sres[c] = (sig_lev(l1) > sig_lev(l2) ? sig_lev(l1) : sig_lev(l2)) + 1u;
    }
}

__global__ void k_rec_insert(RecArgs r, uint32_t nb) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; c < nb; c += stride) {
        if (r.mask[c] != 1) continue;
        const uint32_t slot = t_slot(r.t, r.skey[c]);
        r.slot[c] = slot;
        if (slot == UNSET) { atomicOr(r.err, 2u); r.mask[c] = 0; continue; }
        atomicMin(&r.t.v[slot], (unsigned long long)c);
    }
}

// winners (the smallest cover index of a key) of every workgroup's kB covers
__global__ void __launch_bounds__(kB) k_rec_winners(RecArgs r, uint32_t nb) {
    const uint32_t c = blockIdx.x * kB + threadIdx.x;
    const bool win = c < nb && r.mask[c] == 1 && r.t.v[r.slot[c]] == (unsigned long long)c;
    const int n = __syncthreads_count(win);
    if (c < nb && win) r.mask[c] = 3;
    if (threadIdx.x == 0) r.bcnt[blockIdx.x] = (uint32_t)n;
}

// ids of the winners: the counter, the winners of the workgroups before, the
// rank inside the workgroup
__global__ void __launch_bounds__(kB) k_rec_ids(RecArgs r, uint32_t s, uint32_t nb, uint32_t step) {
    __shared__ uint32_t s_sum, s_w[kB / 64];
    if (threadIdx.x == 0) s_sum = 0;
    __syncthreads();
    uint32_t x = 0;
    for (uint32_t b = threadIdx.x; b < blockIdx.x; b += kB) x += r.bcnt[b];
    if (x) atomicAdd(&s_sum, x);
    const uint32_t c = blockIdx.x * kB + threadIdx.x, lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const bool win = c < nb && r.mask[c] == 3;
    const uint64_t m = __ballot(win);
    if (lane == 0) s_w[wave] = (uint32_t)__popcll(m);
    __syncthreads();
    uint32_t id = r.counter[step & 1u] + s_sum + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
    for (uint32_t w = 0; w < wave; w++) id += s_w[w];
    if (win) {
        const unsigned long long key = r.skey[c];
        r.of0[id] = (uint32_t)(key >> 32);
        r.of1[id] = (uint32_t)key;
        if (r.tagOut) r.tagOut[id] = r.tagIn[r.roots[s + c]];
        r.t.v[r.slot[c]] = sig(2u * id, (uint32_t)r.sres[c]);
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
        uint32_t n = r.counter[step & 1u] + s_sum;
        for (uint32_t w = 0; w < kB / 64; w++) n += s_w[w];
        r.counter[(step & 1u) ^ 1u] = n;
    }
}

// addBackLocalArrays (balance.cu:429-467)
__global__ void k_rec_add_back(RecArgs r, uint32_t s, uint32_t nb) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    const uint32_t in0 = r.off[s];
    for (int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; c < nb; c += stride) {
        const uint8_t m = r.mask[c];
        if (m == 0) continue;
        unsigned long long *A = r.arr + (r.off[s + c] - in0);
        const unsigned long long x = m == 2 ? r.sres[c] : r.t.v[r.slot[c]];
        const uint32_t L = r.alen[c];
        bool there = false;
        for (uint32_t i = 0; i < L; i++) there |= sig_lit(A[i]) == sig_lit(x);
        if (there) continue;
        uint32_t i = L;
        while (i > 0 && sig_lev(x) > sig_lev(A[i - 1])) {
            A[i] = A[i - 1];
            i--;
        }
        A[i] = x;
        r.alen[c] = L + 1;
    }
}

__global__ void k_rec_record(RecArgs r, uint32_t s, uint32_t nb) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    const uint32_t in0 = r.off[s];
    for (int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; c < nb; c += stride)
        r.newSig[r.roots[s + c]] = r.alen[c] == 0 ? 0ull : r.arr[r.off[s + c] - in0];
}

// ---------------------------------------------------------------------------
// phase 3: output.  A segment's ids are consecutive; they move down by its gap
// (its first id less the first of its output) behind the segments before it.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint32_t moved(uint32_t lit, int32_t nPIs, uint32_t gap) {
    return (int32_t)(lit >> 1) <= nPIs ? lit : lit - 2u * gap;
}

__global__ void k_out_emit(uint32_t m, int32_t nPIs, uint32_t nSeg, const uint32_t *__restrict__ outOff,
                           const uint32_t *__restrict__ idBase, const uint32_t *__restrict__ if0,
                           const uint32_t *__restrict__ if1, uint32_t *of0, uint32_t *of1, uint32_t *olevel,
                           const uint32_t *__restrict__ tagIn, const uint32_t *__restrict__ itag, uint32_t *otag) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < m; q += stride) {
        uint32_t lo = 0, hi = nSeg - 1;          // the segment whose output holds q
        while (lo < hi) {
            const uint32_t mid = (lo + hi + 1) >> 1;
            if (outOff[mid] <= (uint32_t)q) lo = mid;
            else hi = mid - 1;
        }
        const uint32_t gap = idBase[lo] - (uint32_t)(nPIs + 1) - outOff[lo];
        const uint32_t o = (uint32_t)(nPIs + 1) + (uint32_t)q, v = o + gap;
        of0[o] = moved(if0[v], nPIs, gap);
        of1[o] = moved(if1[v], nPIs, gap);
        olevel[o] = 0;
        if (otag) otag[o] = itag ? itag[v] : lo;
    }
    for (int64_t v = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; v <= nPIs; v += stride) {
        of0[v] = 0;
        of1[v] = 0;
        olevel[v] = 0;
        if (otag) otag[v] = tagIn[v];
    }
}

__global__ void k_out_pos(int32_t nPOs, int32_t nPIs, const uint32_t *__restrict__ pos,
                          const unsigned long long *__restrict__ newSig, const uint32_t *__restrict__ segTag,
                          const uint32_t *__restrict__ outOff, const uint32_t *__restrict__ idBase, uint32_t *opos) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < nPOs; i += stride) {
        const uint32_t l = pos[i], id = l >> 1;
        if ((int32_t)id <= nPIs) { opos[i] = l; continue; }
        const uint32_t seg = segTag ? segTag[id] : 0u;
        opos[i] = moved(sig_lit(newSig[id]), nPIs, idBase[seg] - (uint32_t)(nPIs + 1) - outOff[seg]) ^ (l & 1u);
    }
}

// (level << 32 | tag) of every root in level order, for the batch-split check
__global__ void k_level_tag_keys(uint32_t nRoots, const uint32_t *__restrict__ levels,
                                 const uint32_t *__restrict__ roots, const uint32_t *__restrict__ tag,
                                 unsigned long long *keys) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < nRoots; i += stride)
        keys[i] = (unsigned long long)levels[i] << 32 | tag[roots[i]];
}

// In sorted (level, tag) keys, a key equal to the one BAL_BATCH places
// before it belongs to a tag with more than BAL_BATCH covers on that level:
// its tag goes to the list (at most cap entries; *count counts them all).
__global__ void k_split_tags(uint32_t nRoots, const unsigned long long *__restrict__ sortedKeys, uint32_t *list,
                             uint32_t cap, uint32_t *count) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)BAL_BATCH + blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < nRoots; i += stride) {
        const unsigned long long k = sortedKeys[i];
        // the first place of each offending run past the limit reports it
        if (k == sortedKeys[i - BAL_BATCH] && (i == BAL_BATCH || sortedKeys[i - BAL_BATCH - 1] != k)) {
            const uint32_t q = atomicAdd(count, 1u);
            if (q < cap) list[q] = (uint32_t)k;
        }
    }
}

// steps of every reconstruction batch of the wide levels: the largest
// (cover length - 1) of its roots; batchOff[l] = first batch of level l
// (UNSET for a level that the persistent workgroup takes)
__global__ void k_batch_steps(uint32_t nRoots, const uint32_t *__restrict__ levels, const uint32_t *__restrict__ off,
                              const uint32_t *__restrict__ starts, const uint32_t *__restrict__ batchOff,
                              uint32_t batchLimit, uint32_t *steps) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < nRoots; i += stride) {
        const uint32_t l = levels[i], bo = batchOff[l];
        if (bo == UNSET) continue;
        const uint32_t len = off[i + 1] - off[i];
        const uint32_t st = len > 1 ? len - 1 : 0u;
        // most roots of a batch see a maximum at least as large already: the
        // atomic is taken only by those that raise it
        uint32_t *dst = &steps[bo + ((uint32_t)i - starts[l]) / batchLimit];
        if (st > __hip_atomic_load(dst, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(dst, st);
    }
}

// the wide levels' counter from the nodes made so far, or (to = 0) back
__global__ void k_counter_made(uint32_t *counter, uint32_t *made, uint32_t firstId, uint32_t to) {
    if (to) *made = *counter - firstId;
    else *counter = firstId + *made;
}

struct Tmp {
    gls_ctx *ctx;
    std::vector<void *> ptrs;
    bool ok = true;
    template <class T> T *get(size_t n) {
        T *p = pool_get<T>(ctx, std::max<size_t>(n, 1));
        if (p) ptrs.push_back(p);
        else ok = false;
        return p;
    }
    ~Tmp() {
        for (void *p : ptrs) pool_put(ctx, p);
    }
};

uint32_t bits_of(uint32_t x) {
    uint32_t b = 1;
    while (b < 32 && (x >> b) != 0) ++b;
    return b;
}

} // namespace

int dev_balance(gls_ctx *ctx, const DevGraph &in, DevGraph &out, gls_op_info *info, const uint32_t *tagIn,
                uint32_t **tagOut, std::vector<uint32_t> *splitTags, int sortDecId, int32_t nTags) {
    const bool tagged = tagIn && tagOut;
    if (sortDecId != 0 && sortDecId != 1) return gls_fail(ctx, GLS_ERR_ARG, "balance: sortDecId must be 0 or 1");
    // the shuffle is seeded with a cover's index in its batch, which in a
    // batched arena is not its index when balanced alone
    if (sortDecId == 0 && tagged) return gls_fail(ctx, GLS_ERR_ARG, "balance: `b -s` is not batched");
    if (tagged && nTags <= 0) return gls_fail(ctx, GLS_ERR_INTERNAL, "balance: tags without their number");
    const int32_t n = in.nObjs, nPIs = in.nPIs, nPOs = in.nPOs;
    const uint32_t nSeg = tagged ? (uint32_t)nTags : 1u;
    const uint32_t narrowMax = (uint32_t)tuning_for(ctx, n).balance_narrow_max;
    hipStream_t st = ctx->stream;
    Tmp t{ctx};
    const auto t0 = std::chrono::steady_clock::now();
    // ---- phase 1: covers
    uint32_t *nFo = t.get<uint32_t>(n), *mark = t.get<uint32_t>(n), *place = t.get<uint32_t>(n);
    uint2 *cover = t.get<uint2>(n);
    uint32_t *lastLevel = t.get<uint32_t>(n), *roots = t.get<uint32_t>(n), *rootsSorted = t.get<uint32_t>(n);
    uint8_t *flag = t.get<uint8_t>((size_t)n + 4), *flag2 = t.get<uint8_t>(n);
    uint32_t *extra = t.get<uint32_t>(n);
    // [0] pool next, [1] error, [2] extra roots, [3] roots, [4..6] largest level, [7] ids out of order, [8..9] counter
    uint32_t *ctr = t.get<uint32_t>(16);
    const uint64_t poolCap = 2ull * (uint64_t)n + 64;   // cover inputs are distinct fanin edges
    uint32_t *pool = t.get<uint32_t>(poolCap);
    const int coverThreads = (int)std::min<int64_t>(COVER_THREADS, (int64_t)nblocks(n) * kB);
    uint32_t *scratch = t.get<uint32_t>((size_t)coverThreads * COVER_SCRATCH);
    uint32_t *segInfo = t.get<uint32_t>(3 * (size_t)nSeg);
    if (!t.ok) return gls_fail(ctx, GLS_ERR_NOMEM, "balance: allocation (n=%d)", n);
    uint32_t *segFirst = segInfo, *segRound = segInfo + nSeg, *segCnt = segRound + nSeg;
    GLS_TRY(Fills(ctx)
                .add(nFo, 0, sizeof(uint32_t) * n)
                .add(mark, 0, sizeof(uint32_t) * n)
                .add(lastLevel, 0xFF, sizeof(uint32_t) * n)
                .add(ctr, 0, sizeof(uint32_t) * 16)
                .add(segInfo, 0, sizeof(uint32_t) * 3 * (size_t)nSeg)
                .run());
    k_fanouts<<<nblocks(n), kB, 0, st>>>(n, nPIs, in.f0, in.f1, nPOs, in.pos, nFo, mark);
    if (nPOs > 0) k_po_marks<<<nblocks(nPOs), kB, 0, st>>>(nPOs, in.pos, mark);
    k_root_flags<<<nblocks(n), kB, 0, st>>>(n, nPIs, nFo, mark, flag);
    GLS_HIP(ctx, hipGetLastError());
    rocprim::counting_iterator<uint32_t> ids(0u);
    size_t tb = 0;
    GLS_HIP(ctx, rocprim::select(nullptr, tb, ids, flag, roots, &ctr[3], (size_t)n, st));
    void *tmp = t.get<uint8_t>(tb);
    if (!tmp) return gls_fail(ctx, GLS_ERR_NOMEM, "balance: select storage");
    auto select_ids = [&](const uint8_t *f, uint32_t &count) -> int {
        GLS_HIP(ctx, rocprim::select(tmp, tb, ids, f, roots, &ctr[3], (size_t)n, st));
        return stream_copy(ctx, &count, &ctr[3], sizeof(uint32_t), hipMemcpyDeviceToHost);
    };
    uint32_t nCand = 0;
    GLS_TRY(select_ids(flag, nCand));
    const CoverArgs ca{in.f0, in.f1, nFo, nPIs, cover, pool, &ctr[0], poolCap, scratch, flag, extra, &ctr[2], &ctr[7],
                       &ctr[1]};
    // covers of the roots by their edges; then of those a limit made, until
    // no cover meets another one
    uint32_t misc[8] = {};
    bool limited = false;
    const uint32_t *list = roots;
    for (uint32_t todo = nCand, done = 0; todo > 0;) {
        k_covers<<<(int)std::min<int64_t>(nblocks(todo), coverThreads / kB), kB, 0, st>>>(ca, todo, list);
        GLS_HIP(ctx, hipGetLastError());
        GLS_TRY(stream_copy(ctx, misc, ctr, sizeof(misc), hipMemcpyDeviceToHost));
        if (misc[1]) return gls_fail(ctx, GLS_ERR_INTERNAL, "balance: cover pool overflow");
        if (misc[7]) return gls_fail(ctx, GLS_ERR_INTERNAL, "balance: input not topological");
        list = extra + done;
        todo = misc[2] - done;
        done = misc[2];
        limited |= todo > 0;
    }
    const uint32_t poolUsed = misc[0];
    if (limited) GLS_TRY(select_ids(flag, nCand));
    // ---- levels
    if (tagged && nCand > 0) {
        k_count_tags<<<tag_grid(nCand), kBlock, 0, st>>>(nCand, roots, tagIn, segCnt);
        size_t tbs = 0;
        GLS_HIP(ctx, rocprim::exclusive_scan(nullptr, tbs, segCnt, segFirst, 0u, (size_t)nSeg, rocprim::plus<uint32_t>(), st));
        void *ts = t.get<uint8_t>(std::max<size_t>(tbs, 1));
        if (!ts) return gls_fail(ctx, GLS_ERR_NOMEM, "balance: scan storage");
        GLS_HIP(ctx, rocprim::exclusive_scan(ts, tbs, segCnt, segFirst, 0u, (size_t)nSeg, rocprim::plus<uint32_t>(), st));
    }
    const size_t room = std::max(nCand, 1u);
    uint32_t *keys = t.get<uint32_t>(room), *keysSorted = t.get<uint32_t>(room);
    uint32_t *off = t.get<uint32_t>(room + 1), *len = t.get<uint32_t>(room + 1);
    uint32_t *newLen = t.get<uint32_t>(room + 1), *newOff = t.get<uint32_t>(room + 1);
    uint32_t *inputs = t.get<uint32_t>(std::max<size_t>(poolUsed, 1)), *inSrc = t.get<uint32_t>(std::max<size_t>(poolUsed, 1));
    if (!t.ok) return gls_fail(ctx, GLS_ERR_NOMEM, "balance: order allocation");
    std::vector<uint32_t> segLevels(nSeg, 0);
    auto levels_by_id = [&]() -> int {
        const uint32_t *ordered = roots;
        size_t tbs = 0, tbk = 0;
        GLS_HIP(ctx, rocprim::exclusive_scan(nullptr, tbs, len, off, 0u, (size_t)nCand + 1, rocprim::plus<uint32_t>(), st));
        GLS_HIP(ctx, rocprim::radix_sort_pairs(nullptr, tbk, keys, keysSorted, roots, rootsSorted, (size_t)nCand, 0u,
                                               bits_of(nSeg), st));
        void *ts = t.get<uint8_t>(std::max<size_t>(std::max(tbs, tbk), 1));
        if (!ts) return gls_fail(ctx, GLS_ERR_NOMEM, "balance: level storage");
        if (tagged) {
            k_gather_tags<<<nblocks(nCand), kB, 0, st>>>(nCand, roots, tagIn, keys);
            GLS_HIP(ctx, rocprim::radix_sort_pairs(ts, tbk, keys, keysSorted, roots, rootsSorted, (size_t)nCand, 0u,
                                                   bits_of(nSeg), st));
            ordered = rootsSorted;
        } else {
            GLS_TRY(stream_copy(ctx, segCnt, &nCand, sizeof(uint32_t), hipMemcpyHostToDevice));
        }
        uint32_t *rootAt = extra, *pend = newLen, *val = newOff;
        const uint32_t *tags = tagged ? tagIn : nullptr;
        k_id_place<<<nblocks((int64_t)nCand + 1), kB, 0, st>>>(nCand, ordered, tags, segFirst, segCnt, cover, mark, rootAt,
                                                             place, len, pend, val);
        GLS_HIP(ctx, rocprim::exclusive_scan(ts, tbs, len, off, 0u, (size_t)nCand + 1, rocprim::plus<uint32_t>(), st));
        k_id_pack<<<nblocks(nCand), kB, 0, st>>>(nCand, rootAt, tags, segFirst, cover, pool, place, nPIs, off, inputs, pend);
        k_id_sweep<<<nSeg, ID_CHUNK, 0, st>>>(IdSweepArgs{segFirst, segCnt, off, inputs, pend, val, segRound});
        k_id_levels<<<nblocks(nCand), kB, 0, st>>>(nCand, rootAt, val, lastLevel);
        GLS_HIP(ctx, hipGetLastError());
        return GLS_OK;
    };
    uint32_t nRoots = 0, levels = 0;
    if (nCand > 0) {
        GLS_TRY(levels_by_id());
        GLS_TRY(stream_copy(ctx, segLevels.data(), segRound, sizeof(uint32_t) * nSeg, hipMemcpyDeviceToHost));
        for (uint32_t x : segLevels) levels = std::max(levels, x);
        k_taken_flags<<<nblocks(n), kB, 0, st>>>(n, lastLevel, flag2);
        GLS_TRY(select_ids(flag2, nRoots));
    }
    // ---- roots in the order in which they are rebuilt: by (segment, level,
    // id) where every level fits the persistent workgroup's LDS, else by (level,
    // id).  Levels that do not fit go to the grid-wide kernels; one workgroup
    // that reads them from memory takes longer.  30 levels of 2500 covers of 3
    // inputs 1.95 ms / 5.6, of 4000 of 3 2.5 / 7.6, of 4000 of 6 4.6 / 21.3.  One
    // member with such a level puts a whole batch in that order: 15 members of 20k
    // ANDs 1.6 ms alone, 9.9 with it (18.3 where all members share one workgroup).
    const uint32_t fitCovers = std::min<uint32_t>(narrowMax, LT_COVERS);
    uint32_t *d_starts = nullptr, *d_levOff = nullptr;
    LevelRec *d_lev = nullptr;
    uint32_t most[3] = {};
    std::vector<uint32_t> levOff;
    auto order = [&](bool bySeg) -> int {
        const uint32_t ns = bySeg ? nSeg : 1u;
        levOff.assign(ns + 1, 0);
        for (uint32_t k = 0; k < ns; k++) levOff[k + 1] = levOff[k] + (bySeg ? segLevels[k] : levels);
        const uint32_t nKeys = levOff[ns];
        d_levOff = t.get<uint32_t>(ns + 1);
        d_starts = t.get<uint32_t>((size_t)nKeys + 1);
        d_lev = t.get<LevelRec>((size_t)nKeys + 1);
        if (!d_levOff || !d_starts || !d_lev) return gls_fail(ctx, GLS_ERR_NOMEM, "balance: levels");
        GLS_TRY(stream_copy(ctx, d_levOff, levOff.data(), sizeof(uint32_t) * (ns + 1), hipMemcpyHostToDevice));
        k_level_keys<<<nblocks(nRoots), kB, 0, st>>>(nRoots, roots, lastLevel, tagIn,
                                                     bySeg && tagged ? d_levOff : nullptr, keys);
        size_t tb2 = 0, tb3 = 0;
        const uint32_t eb = bits_of(nKeys);
        GLS_HIP(ctx, rocprim::radix_sort_pairs(nullptr, tb2, keys, keysSorted, roots, rootsSorted, (size_t)nRoots, 0u,
                                               eb, st));
        GLS_HIP(ctx, rocprim::exclusive_scan(nullptr, tb3, len, off, 0u, (size_t)nRoots + 1, rocprim::plus<uint32_t>(), st));
        void *tmp2 = t.get<uint8_t>(std::max<size_t>(std::max(tb2, tb3), 1));
        if (!tmp2) return gls_fail(ctx, GLS_ERR_NOMEM, "balance: sort storage");
        GLS_HIP(ctx, rocprim::radix_sort_pairs(tmp2, tb2, keys, keysSorted, roots, rootsSorted, (size_t)nRoots, 0u,
                                               eb, st));
        k_key_starts<<<nblocks((int64_t)nRoots + 1), kB, 0, st>>>(nRoots, keysSorted, nKeys, d_starts);
        k_cover_lens<<<nblocks((int64_t)nRoots + 1), kB, 0, st>>>(nRoots, rootsSorted, cover, len, newLen, place);
        GLS_HIP(ctx, rocprim::exclusive_scan(tmp2, tb3, len, off, 0u, (size_t)nRoots + 1, rocprim::plus<uint32_t>(), st));
        GLS_HIP(ctx, rocprim::exclusive_scan(tmp2, tb3, newLen, newOff, 0u, (size_t)nRoots + 1,
                                             rocprim::plus<uint32_t>(), st));
        GLS_TRY(Fills(ctx).add(&ctr[4], 0, sizeof(uint32_t) * 3).run());
        k_level_sizes<<<nblocks(nKeys), kB, 0, st>>>(nKeys, d_starts, off, newOff, d_lev, &ctr[4]);
        k_pack_inputs<<<nblocks(nRoots), kB, 0, st>>>(nRoots, rootsSorted, cover, pool, off, keysSorted, d_starts, lastLevel, place,
                                                      nPIs, inputs, inSrc);
        GLS_HIP(ctx, hipGetLastError());
        return stream_copy(ctx, most, &ctr[4], sizeof(most), hipMemcpyDeviceToHost);
    };
    bool bySeg = true, fits = true;
    if (nRoots > 0) {
        GLS_TRY(order(true));
        fits = most[0] <= fitCovers && most[1] <= LT_INPUTS && most[2] <= LT_NEW;
        if (!fits && tagged) {
            // Batches: 32768 covers of a level at a time.  With tags (a union of
            // independent AIGs) a level is one batch, which gives every AIG the
            // batches it gets alone as long as none has more than 32768 covers
            // on a level: the (level, tag) keys of the roots are sorted on the
            // device, and a tag with a longer run is reported to the caller
            // (splitTags), which balances it alone.
            bySeg = false;
            GLS_TRY(order(false));
            if (nRoots > (uint32_t)BAL_BATCH) {
                unsigned long long *gk = t.get<unsigned long long>(nRoots), *gkS = t.get<unsigned long long>(nRoots);
                uint32_t *lst = t.get<uint32_t>(1024), *lcnt = t.get<uint32_t>(1);
                if (!t.ok) return gls_fail(ctx, GLS_ERR_NOMEM, "balance: split check");
                k_level_tag_keys<<<nblocks(nRoots), kB, 0, st>>>(nRoots, keysSorted, rootsSorted, tagIn, gk);
                size_t tbk = 0;
                GLS_HIP(ctx, rocprim::radix_sort_keys(nullptr, tbk, gk, gkS, (size_t)nRoots, 0u, 64u, st));
                void *tmpk = t.get<uint8_t>(tbk);
                if (!tmpk) return gls_fail(ctx, GLS_ERR_NOMEM, "balance: split check sort");
                GLS_HIP(ctx, rocprim::radix_sort_keys(tmpk, tbk, gk, gkS, (size_t)nRoots, 0u, 64u, st));
                GLS_TRY(Fills(ctx).add(lcnt, 0, sizeof(uint32_t)).run());
                k_split_tags<<<nblocks(nRoots), kB, 0, st>>>(nRoots, gkS, lst, 1024u, lcnt);
                GLS_HIP(ctx, hipGetLastError());
                uint32_t nsplit = 0;
                GLS_TRY(stream_copy(ctx, &nsplit, lcnt, sizeof(uint32_t), hipMemcpyDeviceToHost));
                if (nsplit > 0) {
                    if (splitTags) {
                        splitTags->assign(std::min<uint32_t>(nsplit, 1024u), 0u);
                        GLS_TRY(stream_copy(ctx, splitTags->data(), lst, sizeof(uint32_t) * splitTags->size(),
                                            hipMemcpyDeviceToHost));
                        if (nsplit > 1024u) splitTags->clear();   // too many to list: the caller splits them all
                    }
                    return GLS_ERR_BATCH_SPLIT;
                }
            }
        }
    }
    const uint32_t ns = bySeg ? nSeg : 1u;
    const uint32_t batchLimit = tagged ? 0xFFFFFFFFu : (uint32_t)BAL_BATCH;

    // ---- phase 2: reconstruction
    const uint64_t cap = balance_table_slots(poolUsed);
    const size_t idEnd = (size_t)nPIs + 1 + poolUsed;
    unsigned long long *tabK = t.get<unsigned long long>(cap), *tabV = t.get<unsigned long long>(cap), *newSig = t.get<unsigned long long>(n);
    uint32_t *cf0 = t.get<uint32_t>(idEnd), *cf1 = t.get<uint32_t>(idEnd);
    uint32_t *ctag = tagged && !bySeg ? t.get<uint32_t>(idEnd) : nullptr;     // by segment: the segment
    uint32_t *segIds = t.get<uint32_t>(3 * (size_t)ns + 3);
    if (!t.ok) return gls_fail(ctx, GLS_ERR_NOMEM, "balance: reconstruction allocation");
    uint32_t *d_idBase = segIds, *d_made = segIds + ns, *d_outOff = segIds + 2 * (size_t)ns;
    GLS_TRY(Fills(ctx)
                .add(tabK, 0xFF, sizeof(unsigned long long) * cap)
                .add(tabV, 0xFF, sizeof(unsigned long long) * cap)
                .run());
    std::vector<uint32_t> idBase(ns, (uint32_t)nPIs + 1u), made(ns, 0u);
    if (bySeg && ns > 1 && nRoots > 0) {
        // a segment's ids start after room for all that those before it can create
        std::vector<LevelRec> hl(levOff[ns]);
        GLS_TRY(stream_copy(ctx, hl.data(), d_lev, sizeof(LevelRec) * hl.size(), hipMemcpyDeviceToHost));
        uint32_t sum = (uint32_t)nPIs + 1u;
        for (uint32_t k = 0; k < ns; k++) {
            idBase[k] = sum;
            for (uint32_t l = levOff[k]; l < levOff[k + 1]; l++) sum += hl[l].most;
        }
    }
    GLS_TRY(stream_copy(ctx, d_idBase, idBase.data(), sizeof(uint32_t) * ns, hipMemcpyHostToDevice));
    GLS_TRY(Fills(ctx).add(d_made, 0, sizeof(uint32_t) * ns).run());
    RecArgs ra{NodeTable{tabK, tabV, cap - 1}, nPIs, rootsSorted, off, inputs, inSrc, d_lev, d_starts, newSig, cf0, cf1, ctag, tagIn, &ctr[1],
               sortDecId == 0 ? 1u : 0u, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, &ctr[8]};
    if (nRoots > 0 && fits) {
        k_rec_lds<<<ns, BAL_WG, 0, st>>>(ra, d_levOff, d_idBase, d_made, (int32_t)levels - 1, 0);
        GLS_HIP(ctx, hipGetLastError());
    } else if (nRoots > 0) {
        std::vector<uint32_t> starts((size_t)levels + 1);
        std::vector<LevelRec> size(levels);
        GLS_TRY(stream_copy(ctx, starts.data(), d_starts, sizeof(uint32_t) * ((size_t)levels + 1), hipMemcpyDeviceToHost));
        GLS_TRY(stream_copy(ctx, size.data(), d_lev, sizeof(LevelRec) * levels, hipMemcpyDeviceToHost));
        // a level goes to the persistent workgroup if it fits its LDS (it is
        // one batch then)
        auto narrow = [&](uint32_t l) {
            return starts[l + 1] - starts[l] <= fitCovers && size[l].T <= LT_INPUTS && size[l].most <= LT_NEW;
        };
        // the wide levels' batches and their step counts
        std::vector<uint32_t> batchOff(levels + 1, UNSET), batchSteps;
        uint32_t nBatches = 0, maxBatch = 1;
        for (uint32_t l = 0; l < levels; l++) {
            const uint32_t cnt = starts[l + 1] - starts[l], per = std::min(cnt, batchLimit);
            if (narrow(l)) continue;
            batchOff[l] = nBatches;
            nBatches += (cnt + per - 1) / per;
            maxBatch = std::max(maxBatch, per);
        }
        uint32_t *d_off = t.get<uint32_t>(levels + 1), *d_steps = t.get<uint32_t>(std::max(nBatches, 1u));
        ra.arr = t.get<unsigned long long>(most[1]);
        ra.alen = t.get<uint32_t>(maxBatch);
        ra.mask = t.get<uint8_t>(maxBatch);
        ra.skey = t.get<unsigned long long>(maxBatch);
        ra.sres = t.get<unsigned long long>(maxBatch);
        ra.slot = t.get<uint32_t>(maxBatch);
        ra.bcnt = t.get<uint32_t>((size_t)nblocks(maxBatch));
        if (!t.ok) return gls_fail(ctx, GLS_ERR_NOMEM, "balance: wide levels");
        GLS_TRY(stream_copy(ctx, d_off, batchOff.data(), sizeof(uint32_t) * (levels + 1), hipMemcpyHostToDevice));
        GLS_TRY(Fills(ctx).add(d_steps, 0, sizeof(uint32_t) * std::max(nBatches, 1u)).run());
        k_batch_steps<<<nblocks(nRoots), kB, 0, st>>>(nRoots, keysSorted, off, d_starts, d_off, batchLimit, d_steps);
        GLS_HIP(ctx, hipGetLastError());
        batchSteps.resize(nBatches);
        if (nBatches > 0)
            GLS_TRY(stream_copy(ctx, batchSteps.data(), d_steps, sizeof(uint32_t) * nBatches, hipMemcpyDeviceToHost));
        const uint32_t firstId = (uint32_t)nPIs + 1u;
        uint32_t step = 0;               // counter[step & 1] is the next id of the wide levels
        GLS_TRY(stream_copy(ctx, &ctr[8], &firstId, sizeof(uint32_t), hipMemcpyHostToDevice));
        int32_t l = (int32_t)levels - 1;
        while (l >= 0) {
            // a run of narrow levels goes to the persistent workgroup
            int32_t e = l;
            while (e >= 0 && narrow((uint32_t)e)) e--;
            if (e < l) {
                k_counter_made<<<1, 1, 0, st>>>(&ctr[8 + (step & 1u)], d_made, firstId, 1u);
                k_rec_lds<<<1, BAL_WG, 0, st>>>(ra, d_levOff, d_idBase, d_made, l, e + 1);
                k_counter_made<<<1, 1, 0, st>>>(&ctr[8 + (step & 1u)], d_made, firstId, 0u);
                GLS_HIP(ctx, hipGetLastError());
                l = e;
                continue;
            }
            // one wide level, in batches, one kernel per phase
            uint32_t bi = batchOff[l];
            for (uint32_t b0 = starts[l]; b0 < starts[l + 1]; b0 += std::min<uint32_t>(starts[l + 1] - b0, batchLimit)) {
                const uint32_t nb = std::min<uint32_t>(starts[l + 1] - b0, batchLimit);
                const uint32_t steps = batchSteps[bi++];
                const int gb = (int)((nb + kB - 1) / kB);
                k_rec_gather<<<gb, kB, 0, st>>>(ra, b0, nb);
                for (uint32_t s2 = 0; s2 < steps; s2++, step++) {
                    k_rec_prepare<<<gb, kB, 0, st>>>(ra, b0, nb);
                    k_rec_insert<<<gb, kB, 0, st>>>(ra, nb);
                    k_rec_winners<<<gb, kB, 0, st>>>(ra, nb);
                    k_rec_ids<<<gb, kB, 0, st>>>(ra, b0, nb, step);
                    k_rec_add_back<<<gb, kB, 0, st>>>(ra, b0, nb);
                    GLS_HIP(ctx, hipGetLastError());
                }
                k_rec_record<<<gb, kB, 0, st>>>(ra, b0, nb);
                GLS_HIP(ctx, hipGetLastError());
            }
            l--;
        }
        k_counter_made<<<1, 1, 0, st>>>(&ctr[8 + (step & 1u)], d_made, firstId, 1u);
        GLS_HIP(ctx, hipGetLastError());
    }
    uint32_t herr = 0;
    GLS_TRY(stream_copy(ctx, &herr, &ctr[1], sizeof(uint32_t), hipMemcpyDeviceToHost));
    if (herr) return gls_fail(ctx, GLS_ERR_INTERNAL, "balance: table overflow (%u)", herr);

    // ---- phase 3: output
    GLS_TRY(stream_copy(ctx, made.data(), d_made, sizeof(uint32_t) * ns, hipMemcpyDeviceToHost));
    std::vector<uint32_t> outOff(ns + 1, 0u);
    for (uint32_t k = 0; k < ns; k++) outOff[k + 1] = outOff[k] + made[k];
    const uint32_t m = outOff[ns];
    GLS_TRY(stream_copy(ctx, d_outOff, outOff.data(), sizeof(uint32_t) * (ns + 1), hipMemcpyHostToDevice));
    if ((int64_t)nPIs + 1 + m > 0x7FFFFFF0LL) return gls_fail(ctx, GLS_ERR_ARG, "balance: result too large");
    GLS_TRY(dev_graph_alloc(ctx, out, nPIs + 1 + (int32_t)m, nPIs, nPOs));
    uint32_t *tags = nullptr;
    if (tagged) {
        tags = pool_get<uint32_t>(ctx, (size_t)nPIs + 1 + m);
        if (!tags) { dev_graph_free(ctx, out); return gls_fail(ctx, GLS_ERR_NOMEM, "balance: tags"); }
        *tagOut = tags;
    }
    k_out_emit<<<nblocks(std::max<int64_t>(m, nPIs + 1)), kB, 0, st>>>(m, nPIs, ns, d_outOff, d_idBase, cf0, cf1, out.f0,
                                                                     out.f1, out.level, tagIn, ctag, tags);
    if (nPOs > 0)
        k_out_pos<<<nblocks(nPOs), kB, 0, st>>>(nPOs, nPIs, in.pos, newSig, bySeg && tagged ? tagIn : nullptr, d_outOff,
                                                d_idBase, out.pos);
    GLS_HIP(ctx, hipGetLastError());
    GLS_HIP(ctx, hipStreamSynchronize(st));
    if (info) {
        info->total_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
        info->levels_enumerated = levels;
        info->new_nodes = m;
        info->candidates = nRoots;
    }
    return GLS_OK;
}
