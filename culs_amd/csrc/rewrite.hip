// DAG-aware rewriting with 4-input cuts on the device.
//
// Stages (reference in parentheses, paths relative to the CULS tree):
//   reorder   level-major renumbering, ties by id (rewrite.cu:1245-1279)
//   cuts      per-level 4-feasible cut enumeration, 16-bit truth tables, support
//             minimisation, CULS slot policy (rewrite.cu:49-294)
//   table     strash table of the current AND nodes (replaces the chained
//             table of rewrite.cu:328-367, 450-471)
//   eval      MFFC size within the cut, NPN class, library matching, nodes
//             added per subgraph root, best (gain, root level) (rewrite.cu:296-447)
//   plan      the chosen replacement of every candidate: deleted set W (root +
//             MFFC), leaves L, reused existing nodes M, nodes to create
//   select    greedy conflict-free selection by priority (gain desc, id asc),
//             computed in rounds of local maxima with atomicMax claims; it
//             replaces the reference's sequential host choice pass
//             (rewrite.cu:811-897), which cannot run in parallel
//   build     new nodes for the selected plans, ids by prefix sum, fanin
//             substitution of replaced roots, then the device strash.
//
// Everything is exact integer work and independent of thread timing: every
// shared decision goes through a prefix sum, a min/max atomic or a stable sort.
#include "gls_internal.h"
#include "dev_common.h"
#include "rwlib_forest.h"
#include "tt_place.h"
#include <hip/hip_cooperative_groups.h>
#include <hip/hip_ext.h>
#include <cstdlib>
#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_reduce.hpp>
#include <rocprim/device/device_scan.hpp>
#include <rocprim/device/device_select.hpp>
#include <rocprim/iterator/counting_iterator.hpp>

namespace {

constexpr int NCUT = 8;
constexpr int MFFC_TAB = 8;
constexpr int NMATCH = 54;
constexpr int EVAL_BLOCK = 64;
constexpr int32_t EVAL_FEW = 49152;
constexpr int PLAN_MAXM = 16;

struct Lib {
    const uint32_t *npn;     // phase | perm << 5 | cls << 10
    const uint8_t *perms4;
    const uint16_t *nodes, *nodeOff, *rootOff;
    const uint8_t *roots;
};

// complement of library input a: only the 4 cut inputs carry one (the
// reference keeps these bits in a 64-bit word, rewrite.cu:388-395)
__device__ __forceinline__ uint32_t isc_bit(uint32_t isC, int a) { return a < 4 ? (isC >> a) & 1u : 0u; }
__device__ __forceinline__ int lib_nn(const Lib &L, int c) { return L.nodeOff[c + 1] - L.nodeOff[c]; }
__device__ __forceinline__ int lib_nr(const Lib &L, int c) { return L.rootOff[c + 1] - L.rootOff[c]; }
__device__ __forceinline__ int lib_root(const Lib &L, int c, int k) { return L.roots[L.rootOff[c] + k]; }
__device__ __forceinline__ uint32_t lib_word(const Lib &L, int c, int j) { return L.nodes[L.nodeOff[c] + j]; }

// ------------------------------------------------------------------------
// cut enumeration
// ------------------------------------------------------------------------
struct DCut {
    uint32_t leaves[4];
    uint32_t tt, value;
    int32_t nLeaves, used;
};

// the reference counts of a cut's leaves, all four loads in flight at once;
// absent leaves read node 0's entry
__device__ __forceinline__ void leaf_refs(const DCut &c, const int32_t *nRef, int (&r)[4]) {
#pragma unroll
    for (int i = 0; i < 4; i++) r[i] = nRef[i < c.nLeaves ? c.leaves[i] : 0u];
}

// CutFindValue (rewrite.cu:49-61)
__device__ __forceinline__ uint32_t cut_value(const DCut &c, const int32_t *nRef) {
    int r[4];
    leaf_refs(c, nRef, r);
    int value = 0, nOnes = 0;
#pragma unroll
    for (int i = 0; i < 4; i++)
        if (i < c.nLeaves) {
            value += r[i];
            nOnes += (r[i] == 1);
        }
    if (c.nLeaves < 2) return 1001;
    if (value > 1000) value = 1000;
    if (nOnes > 3) value = 5 - nOnes;
    return (uint32_t)value;
}

// Reduction of truth-table variables (tt_place.h): the swaps of each phase.
__constant__ uint64_t kTtPlace[16] = {
    tt_place_entry(0),  tt_place_entry(1),  tt_place_entry(2),  tt_place_entry(3),
    tt_place_entry(4),  tt_place_entry(5),  tt_place_entry(6),  tt_place_entry(7),
    tt_place_entry(8),  tt_place_entry(9),  tt_place_entry(10), tt_place_entry(11),
    tt_place_entry(12), tt_place_entry(13), tt_place_entry(14), tt_place_entry(15)};

__device__ void store_cuts(uint32_t *out, const DCut *cs) {
    for (int s = 0; s < NCUT; s++) {
        const DCut &c = cs[s];
        uint32_t *o = out + 5 * s;
        for (int i = 0; i < 4; i++) o[i] = (c.used && i < c.nLeaves) ? c.leaves[i] : 0u;
        o[4] = c.used ? ((c.tt & 0xFFFF) | (c.value & 0x7FF) << 16 | (uint32_t)(c.nLeaves & 7) << 27 | 1u << 30) : 0u;
    }
}

__global__ void k_cuts_pi(int32_t nPIs, const int32_t *__restrict__ nRef, uint32_t *cuts) {
    int64_t v = 1 + blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (v > nPIs) return;
    DCut c[NCUT];
    for (int s = 0; s < NCUT; s++) { c[s].used = 0; c[s].nLeaves = 0; c[s].tt = 0; c[s].value = 0; }
    c[0].used = 1; c[0].tt = 0xAAAA; c[0].nLeaves = 1; c[0].leaves[0] = (uint32_t)v;
    c[0].value = cut_value(c[0], nRef);
    store_cuts(cuts + (size_t)v * NCUT * 5, c);
}

// One wavefront per node.  A node's candidate cuts are the pairs (cut i of
// fanin 0, cut j of fanin 1) that pass the signature prefilter, inserted one
// by one in (i, j) order with an order-dependent slot policy (FindCut evicts,
// CutFilter drops dominated cuts, rewrite.cu:84-193, 268-294).
//   - lane 4 s + k (+ 32 for fanin 1) loads leaf k of the fanin's slot s; the
//     signatures are an OR over the quad, lane 8 i + j tests pair (i, j);
//   - the candidates (about 10 of the 64 pairs on most graphs, 2 on most nodes
//     of the 10M deep AIG) are compacted to one quad of lanes each, 16 at a
//     time: lane k of a quad holds leaf k of both cuts, ranks its leaves in the
//     union, computes bits 4 k .. 4 k + 3 of the truth table and tests variable
//     k for support;
//   - on most nodes no two candidates compare, so the containment tests are
//     made up front, all candidates against one per step, and the candidates
//     before the first comparable pair take their slots by rank (or, with every
//     slot in use, by the smallest eviction key);
//   - the others are inserted one by one, slot s's leaf k in lane 4 s + k and
//     the slot's state in its quad.  A free slot's key is below every used
//     one's, so the slot a candidate takes, free or evicted, is the smallest
//     key, and a failed merge is the insertion of an empty slot.  The number of
//     slot leaves that the new cut holds decides containment both ways: the
//     smaller cut lies in the larger one when it equals the smaller leaf count.
// What bounds it is the length of one wavefront's instruction stream: a
// level's nodes are far fewer than the SIMDs, and the next level waits for
// the slowest.  Measured on a lone wavefront: 4 cycles an instruction, 16 more
// where a scalar instruction reads what a vector one wrote, about 14 a branch,
// 60 a lane permute.  One insertion in turn costs about 300 cycles, a
// containment step about 50.
constexpr int CUTW_BLOCK = 256;
// the per-level kernel runs one wavefront per workgroup: a level's ~200 nodes
// then spread over as many CUs, each wavefront with its own L1 and memory
// pipeline (4 wavefronts per workgroup measured 10% slower on the 10M AIG)
constexpr int CUTL_BLOCK = 64;

__device__ __forceinline__ int rl(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
__device__ __forceinline__ uint32_t bperm(uint32_t byteAddr, uint32_t v) {
    return (uint32_t)__builtin_amdgcn_ds_bpermute((int)byteAddr, (int)v);
}
// the lanes where x holds, from the comparison's own lane mask, and back
__device__ __forceinline__ uint64_t lanes_of(bool x) { return __builtin_amdgcn_ballot_w64(x); }
__device__ __forceinline__ bool in_lanes(uint64_t m) { return __builtin_amdgcn_inverse_ballot_w64(m); }

// lane j of the quad, to its four lanes; the quad's OR and sum
template <int CTRL> __device__ __forceinline__ uint32_t quad_perm(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, true);
}
template <int J> __device__ __forceinline__ uint32_t quad_lane(uint32_t v) { return quad_perm<J * 0x55>(v); }
__device__ __forceinline__ uint32_t quad_or(uint32_t v) {
    v |= quad_perm<0xB1>(v);
    return v | quad_perm<0x4E>(v);
}
__device__ __forceinline__ uint32_t quad_add(uint32_t v) {
    v += quad_perm<0xB1>(v);
    return v + quad_perm<0x4E>(v);
}

// Minimum over lanes 0..31 (in each of them), and over the wavefront, of v,
// which is the same in a quad: row rotations by 4 and 8 within 16 lanes, then
// the other rows.
__device__ __forceinline__ uint32_t min_quads32(uint32_t v) {
    v = min(v, (uint32_t)__builtin_amdgcn_update_dpp((int)0xFFFFFFFF, (int)v, 0x124, 0xF, 0xF, false));
    v = min(v, (uint32_t)__builtin_amdgcn_update_dpp((int)0xFFFFFFFF, (int)v, 0x128, 0xF, 0xF, false));
    const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return min((uint32_t)r[0], (uint32_t)r[1]);
}
__device__ __forceinline__ uint32_t min_quads(uint32_t v) {
    v = min_quads32(v);
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return min((uint32_t)r[0], (uint32_t)r[1]);
}

// Fence-free record format of the dataflow schedule: every 64-bit word of a
// slot carries a valid bit, so a reader polls the words themselves with
// relaxed device-scope atomics and needs no ordering between words.
//   w0 = leaf0 | leaf1 << 31 | V,  w1 = leaf2 | leaf3 << 31 | V,  w2 = meta | V
constexpr unsigned long long TAG_V = 1ull << 63;
constexpr uint32_t DF_SPIN_LIMIT = 1u << 22;

__device__ __forceinline__ unsigned long long load_tagged(const unsigned long long *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store_tagged(unsigned long long *p, unsigned long long v) {
    __hip_atomic_store(p, v | TAG_V, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// cut_node record modes
enum : int { REC_PLAIN = 0, REC_TAGGED = 1 };

// leaf words that are no leaf: of a slot, of a candidate (never equal)
constexpr uint32_t SLOT_PAD = 0xFFFFFFFEu, CAND_PAD = 0xFFFFFFFFu;
constexpr uint64_t QUAD_LANE0 = 0x1111111111111111ull;
// state of a slot, and what a candidate brings to it: leaf count << 24 |
// SLOT_NEW (its meta word is still with the candidate) | SLOT_USED | candidate
// << 16 | category << 14 | value << 3.  The bits of SLOT_KEY with the slot's
// index order the slots for eviction, free ones first.
constexpr uint32_t SLOT_FREE = 15u << 24, SLOT_NEW = 1u << 21, SLOT_USED = 1u << 20, SLOT_KEY = 0x10FFFFu;

// Cut set of node idx (fanin literals l0, l1), computed by one whole wavefront
// (lane = thread lane).  MODE REC_PLAIN: the fanins' 8-slot records (20 bytes
// per slot) start at ra and rb, in global memory or LDS, and the result goes to
// out in the same format (and to out2 as well when it is not null).  MODE
// REC_TAGGED: fanin cut sets are polled in the fence-free format and the result
// is written in it (tcuts, 24 bytes per slot).
// Returns false if a poll exceeded its bound (*err set), true otherwise.
template <int MODE>
__device__ __forceinline__ bool cut_node(const int idx, const uint32_t lane, const uint32_t l0, const uint32_t l1,
                                         const uint32_t *ra, const uint32_t *rb, uint32_t *out,
                                         const int32_t *__restrict__ nRef, unsigned long long *tcuts, uint32_t *err,
                                         const uint8_t *__restrict__ sigBits, uint32_t *out2 = nullptr) {
    const uint32_t k = lane & 3u, slot = (lane >> 2) & 7u, quad0 = lane & 60u, k4 = 4u * k;
    uint32_t leaf, meta;
    if (MODE == REC_TAGGED) {
        const unsigned long long *r = tcuts + ((size_t)(lane < 32 ? LID(l0) : LID(l1)) * NCUT + slot) * 3;
        uint32_t spins = 0;
        unsigned long long wl, wm;
        for (;;) {
            wl = load_tagged(r + (k >> 1));
            wm = load_tagged(r + 2);
            if (lanes_of(!(wl & wm & TAG_V)) == 0) break;
            if (++spins > DF_SPIN_LIMIT ||
                ((spins & 1023u) == 0 && __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
                if (lane == 0) atomicOr(err, 4u);
                return false;
            }
            __builtin_amdgcn_s_sleep(1);
        }
        leaf = (uint32_t)((k & 1u) ? wl >> 31 : wl) & 0x7FFFFFFFu;
        meta = (uint32_t)wm;
    } else {
        const uint32_t *r = (lane < 32 ? ra : rb) + slot * 5;
        leaf = r[k];
        meta = r[4];
    }
    // lane constants: the quad's lanes before this one, pext(k, 0..3) in 2 bits
    // each, the table entries with variable k clear
    const uint32_t below = (1u << k) - 1u, ext = k << 6 | (k >> 1) << 4 | (k & 1u) << 2;
    const uint32_t vmask = (uint32_t)(0x00FF0F0F33335555ull >> (16u * k)) & 0xFFFFu;
    // leaf signatures of the reference (rewrite.cu:68, 262: bit leaf & 31).  In
    // a batched pass sigBits holds each node's bit as it would be in its own
    // AIG (its id there & 31), so that the prefilter of rewrite.cu:283 sees the
    // same signatures as when that AIG is rewritten alone.  An empty slot gets
    // all bits, so that no pair with it passes.
    const bool has = k < ((meta >> 27) & 7u);
    const uint32_t bit = sigBits ? (uint32_t)sigBits[has ? leaf : 0u] : leaf & 31u;
    uint32_t sig = quad_or(has ? 1u << bit : 0u);
    sig = (meta >> 30) & 1u ? sig : 0xFFFFFFFFu;
    const uint32_t sa = bperm((lane >> 3) * 16u, sig), sb = bperm(128u + (lane & 7u) * 16u, sig);
    bool cand = __popc(sa | sb) <= 4;
    uint64_t todo = lanes_of(cand);
    // the slots, slot 0 holding the trivial cut; sval: their meta words
    uint32_t sl = lane == 0 ? (uint32_t)idx : SLOT_PAD;
    uint32_t st = lane < 4 ? 1u << 24 | SLOT_USED | 2u << 14 | 1001u << 3 : SLOT_FREE;
    uint32_t sval = 1u << 30 | 1u << 27 | 1001u << 16 | 0xAAAAu;
    const uint32_t keyLow = lane < 32 ? slot : 0xFFFFFFFFu;     // lanes 32 and up hold no slot
    bool first = true;
    while (todo) {
        // ---- the next 16 candidates, one quad of lanes each
        const uint32_t order = __builtin_amdgcn_mbcnt_hi((uint32_t)(todo >> 32),
                                                         __builtin_amdgcn_mbcnt_lo((uint32_t)todo, 0u));
        const uint32_t cnt = min((uint32_t)__popcll(todo), 16u);
        const bool now = cand && order < 16u;
        cand = cand && !now;
        // lane 1 takes what the lanes without a candidate send
        const uint32_t pair = quad_lane<0>((uint32_t)__builtin_amdgcn_ds_permute(now ? (int)(order * 16u) : 4, (int)lane));
        todo = lanes_of(cand);
        const uint32_t pa = (pair & 56u) * 2u + k4, pb = 128u + (pair & 7u) * 16u + k4;
        const uint32_t a = bperm(pa, leaf), b = bperm(pb, leaf), ma = bperm(pa, meta), mb = bperm(pb, meta);
        // sorted union (rewrite.cu:112-163): a leaf's position is the number
        // of distinct leaves before it (ids are below 2^31 - 16)
        const uint32_t na = (ma >> 27) & 7u, nb = (mb >> 27) & 7u;
        const uint32_t aa = k < na ? a : 0x7FFFFFFFu, bb = k < nb ? b : 0x7FFFFFFEu;
        const uint32_t b0 = quad_lane<0>(bb), b1 = quad_lane<1>(bb), b2 = quad_lane<2>(bb), b3 = quad_lane<3>(bb);
        const bool common = min(min(aa ^ b0, aa ^ b1), min(aa ^ b2, aa ^ b3)) == 0;
        const uint32_t both = quad_or((common ? 1u : 0u) << k);
        const uint32_t rank = k + ((b0 - aa) >> 31) + ((b1 - aa) >> 31) + ((b2 - aa) >> 31) + ((b3 - aa) >> 31) -
                              (uint32_t)__popc(both & below);
        const uint32_t n = na + nb - (uint32_t)__popc(both);
        const bool ok = (lane >> 2) < cnt && n <= 4u;
        // positions that hold a's leaves, and (high half) those that only a has
        const uint32_t kind = common ? 1u : 0x10001u;
        const uint32_t pos = quad_or((k < na ? kind : 0u) << (rank & 15u));
        const uint32_t phA = pos & 15u, phB = ~(pos >> 16) & ((1u << n) - 1u) & 15u;
        const uint32_t la = bperm(4u * (quad0 + (uint32_t)__popc(phA & below)), a);
        const uint32_t lb = bperm(4u * (quad0 + (uint32_t)__popc(phB & below)), b);
        // truth table over the union, four bits per lane
        const uint32_t ta = (ma ^ (0u - LC(l0))) & 0xFFFFu, tb = (mb ^ (0u - LC(l1))) & 0xFFFFu;
        const uint32_t tt = quad_or((tt_nibble(ta, phA, ext) & tt_nibble(tb, phB, ext)) << k4);
        const uint32_t m = (phA >> k) & 1u ? la : lb;
        // support reduction (rewrite.cu:223-266): fm, fn, ftt the final cut, the
        // leaves that the table does not depend on dropped, the others moved down
        const bool dep = ((tt ^ (tt >> (1u << k))) & vmask) != 0;
        uint32_t fm = m, ftt = tt, fn = n;
        if (lanes_of(ok && k < n && !dep) != 0) {      // some candidate shrinks
            const uint32_t keep = quad_or((k < n && dep ? 1u : 0u) << k);
            fn = (uint32_t)__popc(keep);
            // the kept leaves first, in order, then the dropped ones
            const uint32_t before = (uint32_t)__popc(keep & below);
            const uint32_t to = (keep >> k) & 1u ? before : fn + k - before;
            fm = (uint32_t)__builtin_amdgcn_ds_permute((int)(4u * (quad0 + to)), (int)m);
            ftt = tt_place_shrink(tt, kTtPlace[keep]) & 0xFFFFu;
        }
        // the final leaves' reference counts are in flight meanwhile: only an
        // eviction and the end of the batch need the values
        int ref = nRef[k < fn ? fm : 0u];
        const uint32_t cat = fn > 2u ? 0u : fn == 2u ? 1u : 2u;
        uint32_t info = ok ? fn << 24 | SLOT_NEW | SLOT_USED | (lane >> 2) << 16 | cat << 14 : SLOT_FREE;
        uint32_t fmeta = 0;
        bool valued = false;
        auto value = [&]() {            // meta words: CutFindValue (rewrite.cu:49-61)
            asm volatile("" : "+v"(ref));       // the load is waited for here, not before a branch to here
            const int sum = (int)quad_add(k < fn ? (uint32_t)ref : 0u);
            const uint32_t ones = quad_add(k < fn && ref == 1 ? 1u : 0u);
            uint32_t v = (uint32_t)(sum > 1000 ? 1000 : sum);
            v = ones > 3u ? 5u - ones : v;
            v = fn < 2u ? 1001u : v;
            fmeta = ftt | (v & 0x7FFu) << 16 | (fn & 7u) << 27 | 1u << 30;
            info |= ok ? (v & 0x7FFu) << 3 : 0u;
            const uint32_t g = bperm((st >> 12) & 0xF0u, info);
            st = st & SLOT_NEW ? g : st;
            valued = true;
        };
        const uint64_t okm = lanes_of(ok) & QUAD_LANE0;
        // candidates that shrink or end the insertions
        uint64_t odd = lanes_of(ok && (fn != n || fn < 2u)) & QUAD_LANE0;
        const uint32_t cl = ok && k < n ? m : CAND_PAD;
        uint32_t c = 0;
        if (!first) {
            value();
        } else if (cnt > 2u) {
            // ---- the candidates before the first odd one, and of these the
            // ones before the later of the first two that compare
            const uint32_t quad = lane >> 2;
            uint32_t end = odd ? (uint32_t)__builtin_ctzll(odd) >> 2 : cnt;
            // bit q of sub: candidate q's leaves all lie in this quad's cut
            const uint32_t m0 = quad_lane<0>(m);
            const uint32_t c0 = ok ? (k < n ? m : m0) : CAND_PAD;
            const uint32_t c1 = quad_perm<0x39>(c0), c2 = quad_perm<0x4E>(c0), c3 = quad_perm<0x93>(c0);
            uint32_t sub = 0;
            for (uint32_t q = (end + 3u) & ~3u; q; q -= 4) {
                const uint32_t at = 16u * q - 64u + k4;
                uint32_t d[4];
#pragma unroll
                for (uint32_t j = 0; j < 4; j++) d[j] = bperm(at + 16u * j, c0);
#pragma unroll
                for (uint32_t j = 0; j < 4; j++)
                    d[j] = quad_or(min(min(c0 ^ d[j], c1 ^ d[j]), min(c2 ^ d[j], c3 ^ d[j])));
#pragma unroll
                for (int j = 3; j >= 0; j--) sub = 2u * sub + (d[j] == 0 ? 1u : 0u);
            }
            const uint32_t early = (1u << quad) - 1u;
            sub = ok && quad < end ? sub & ((1u << end) - 1u) & ~(1u << quad) : 0u;
            if (lanes_of(sub != 0) != 0)
                end = (uint32_t)__builtin_amdgcn_readfirstlane(
                    (int)min_quads(sub == 0 ? 255u : sub & early ? quad : (uint32_t)__builtin_ctz(sub)));
            // the first seven that merged, to slots 1..7
            const uint64_t take = okm & (end < 16u ? (1ull << (4u * end)) - 1ull : ~0ull);
            const uint32_t r = quad_lane<0>(__builtin_amdgcn_mbcnt_hi((uint32_t)(take >> 32),
                                                                      __builtin_amdgcn_mbcnt_lo((uint32_t)take, 0u)));
            const bool slotted = ok && quad < end && r < (uint32_t)(NCUT - 1);
            const int to = (int)(slotted ? 16u * r + 16u + k4 : 128u + k4);    // lanes 32 and up take the rest
            const uint32_t nTake = (uint32_t)__popcll(take);
            const uint32_t pl = (uint32_t)__builtin_amdgcn_ds_permute(to, (int)cl);
            const uint32_t pi = (uint32_t)__builtin_amdgcn_ds_permute(to, (int)info);
            const bool filled = slot >= 1u && slot <= nTake && lane < 32;
            sl = filled ? min(pl, SLOT_PAD) : sl;
            st = filled ? pi : st;
            c = end;
            if (nTake >= (uint32_t)(NCUT - 1)) {
                // every slot is in use: each further one evicts (also if it
                // failed to merge), FindCut (rewrite.cu:84-109)
                c = (uint32_t)__builtin_ctzll(lanes_of(slotted && r == (uint32_t)(NCUT - 2))) / 4u + 1u;
                if (c < end) {
                    value();
                    uint32_t inf = bperm(16u * c, info);
                    for (; c < end; c++) {
                        const uint32_t next = bperm(16u * c + 16u, info);
                        const uint32_t key = (st & SLOT_KEY) | keyLow;
                        st = key == min_quads32(key) ? inf : st;
                        inf = next;
                        asm volatile("" : "+v"(inf));      // moved before the loop's branch
                    }
                    const uint32_t gl = bperm(((st >> 12) & 0xF0u) + k4, cl);
                    sl = st & SLOT_NEW ? min(gl, SLOT_PAD) : st & SLOT_USED ? sl : SLOT_PAD;
                }
            }
            if (!valued && nTake + (cnt - c) >= (uint32_t)NCUT && c < cnt) value();
        }
        first = false;
        // ---- the others one by one.
        // CutFilter (rewrite.cu:178-193) of a cut (leaf k in x, nn leaves)
        // against the slots where `hit` holds: scanning slots in order, a
        // larger slot that contains it is dropped; the first slot of no more
        // leaves that it contains drops it and ends the scan.  True if dropped.
        auto shared_with = [&](uint32_t x) -> uint32_t {
            const uint32_t d = min(min(sl ^ x, sl ^ quad_perm<0x39>(x)), min(sl ^ quad_perm<0x4E>(x), sl ^ quad_perm<0x93>(x)));
            return quad_add(d == 0 ? 1u : 0u);
        };
        auto filter = [&](uint32_t hit, uint32_t nn) -> bool {
            const uint32_t drops = hit & (uint32_t)lanes_of((st >> 24) <= nn);
            const uint32_t gone = hit & ~drops & ((drops & (0u - drops)) - 1u);     // before the first that drops it
            const bool g = in_lanes((uint64_t)gone);
            sl = g ? SLOT_PAD : sl;
            st = g ? SLOT_FREE : st;
            return drops != 0;
        };
        bool stop = false;
        uint32_t x = bperm(16u * c + k4, cl), inf = bperm(16u * c, info);
        odd &= c < 16u ? ~0ull << (4u * c) : 0ull;
        while (c < cnt) {
            const uint32_t end = odd ? (uint32_t)__builtin_ctzll(odd) >> 2 : cnt;
            for (; c < end; c++) {
                const uint32_t nx = bperm(16u * c + 16u + k4, cl), ninf = bperm(16u * c + 16u, info);
                // FindCut (rewrite.cu:84-109): the smallest key
                const uint32_t key = (st & SLOT_KEY) | keyLow;
                const bool here = key == min_quads32(key);
                const uint32_t nn = inf >> 24;
                const uint32_t shared = shared_with(x) + (here ? 64u : 0u);
                const uint32_t hit = (uint32_t)lanes_of(shared == min(st >> 24, nn));
                if (hit != 0 && filter(hit, nn)) {
                    x = CAND_PAD;
                    inf = SLOT_FREE;
                }
                sl = here ? min(x, SLOT_PAD) : sl;
                st = here ? inf : st;
                x = nx;
                inf = ninf;
                asm volatile("" : "+v"(x), "+v"(inf));     // moved before the loop's branch
            }
            if (c == cnt) break;
            const uint32_t key = (st & SLOT_KEY) | keyLow;
            const bool here = key == min_quads32(key);
            const uint32_t n1 = (uint32_t)rl((int)n, (int)(4u * c)), n2 = (uint32_t)rl((int)fn, (int)(4u * c));
            auto hits = [&](uint32_t y, uint32_t nn) {
                const uint32_t shared = shared_with(y) + (here ? 64u : 0u);
                return (uint32_t)lanes_of(shared == min(st >> 24, nn)) & (uint32_t)lanes_of((st & SLOT_USED) != 0);
            };
            bool dropped = filter(hits(x, n1), n1);
            if (!dropped) {
                if (n2 != n1) {
                    x = bperm(16u * c + k4, k < fn ? fm : CAND_PAD);
                    dropped = filter(hits(x, n2), n2);
                }
                stop = n2 < 2u;
            }
            sl = here ? (dropped ? SLOT_PAD : min(x, SLOT_PAD)) : sl;
            st = here ? (dropped ? SLOT_FREE : inf) : st;
            if (stop) break;
            odd &= odd - 1;
            c++;
            x = bperm(16u * c + k4, cl);
            inf = bperm(16u * c, info);
        }
        if (!valued) value();
        const uint32_t g = bperm((st >> 12) & 0xF0u, fmeta);
        sval = st & SLOT_NEW ? g : sval;
        st &= ~SLOT_NEW;
        if (stop) break;
    }
    // ---- lanes 0..31 store the slots
    if (lane < 32) {
        const uint32_t o = sl == SLOT_PAD ? 0u : sl;
        const uint32_t om = st & SLOT_USED ? sval : 0u;
        if (MODE == REC_TAGGED) {
            const uint32_t o1 = quad_perm<0xB1>(o);
            unsigned long long *q = tcuts + ((size_t)idx * NCUT + slot) * 3;
            if (!(k & 1u)) store_tagged(q + (k >> 1), (unsigned long long)o | (unsigned long long)o1 << 31);
            else if (k == 1u) store_tagged(q + 2, om);
        } else {
            out[slot * 5 + k] = o;
            if (k == 0) out[slot * 5 + 4] = om;
            if (out2) {
                out2[slot * 5 + k] = o;
                if (k == 0) out2[slot * 5 + 4] = om;
            }
        }
    }
    return true;
}

// Cut set of node idx from the records of its fanins in `cuts`, into `cuts`.
__device__ __forceinline__ void cut_node_global(const int idx, const int lane, const uint32_t *__restrict__ f0,
                                                const uint32_t *__restrict__ f1, const int32_t *__restrict__ nRef,
                                                uint32_t *cuts, const uint8_t *__restrict__ sigBits) {
    const uint32_t l0 = f0[idx], l1 = f1[idx];
    cut_node<REC_PLAIN>(idx, lane, l0, l1, cuts + (size_t)LID(l0) * NCUT * 5, cuts + (size_t)LID(l1) * NCUT * 5,
                        cuts + (size_t)idx * NCUT * 5, nRef, nullptr, nullptr, sigBits);
}

__global__ void __launch_bounds__(CUTL_BLOCK) k_cuts_level(int32_t start, int32_t count,
                                                           const uint32_t *__restrict__ f0,
                                                           const uint32_t *__restrict__ f1,
                                                           const int32_t *__restrict__ nRef, uint32_t *cuts,
                                                           const uint8_t *__restrict__ sigBits) {
    const int k = blockIdx.x * (CUTL_BLOCK / 64) + (threadIdx.x >> 6);
    if (k >= count) return;    // uniform per wavefront
    cut_node_global(start + k, threadIdx.x & 63, f0, f1, nRef, cuts, sigBits);
}

// Two levels in one launch.  Workgroups 0..n0-1 compute the nodes of the first
// level (ids s0..s0+n0-1) as k_cuts_level does.  Workgroup n0 + k takes node
// s1 + k of the second level: wavefront w first recomputes the cut set of
// fanin w if that fanin lies on the first level (its own fanins are on earlier
// levels, whose records are complete), into LDS; after the barrier wavefront 0
// computes the node from those LDS records and the global records of fanins on
// earlier levels.  Every computation is the deterministic cut_node, so the
// recomputed sets equal the stored ones, and one launch replaces two dependent
// ones (a dependent launch costs about as much as a node's whole computation).
constexpr int CUTP_BLOCK = 128;
__global__ void __launch_bounds__(CUTP_BLOCK) k_cuts_pair(int32_t s0, int32_t n0, int32_t s1,
                                                          const uint32_t *__restrict__ f0,
                                                          const uint32_t *__restrict__ f1,
                                                          const int32_t *__restrict__ nRef, uint32_t *cuts,
                                                          const uint8_t *__restrict__ sigBits) {
    __shared__ uint32_t s_rec[2][NCUT * 5];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int k = (int)blockIdx.x;
    if (k < n0) {                       // uniform per workgroup
        if (w == 0) cut_node_global(s0 + k, lane, f0, f1, nRef, cuts, sigBits);
        return;
    }
    const int v = s1 + (k - n0);
    const uint32_t l0 = f0[v], l1 = f1[v];
    const uint32_t in0 = LID(l0), in1 = LID(l1);
    const uint32_t mine = w == 0 ? in0 : in1;
    if (mine >= (uint32_t)s0) {         // on the first level (fanins of v are below s1)
        const uint32_t g0 = f0[mine], g1 = f1[mine];
        cut_node<REC_PLAIN>((int)mine, lane, g0, g1, cuts + (size_t)LID(g0) * NCUT * 5,
                            cuts + (size_t)LID(g1) * NCUT * 5, s_rec[w], nRef, nullptr, nullptr, sigBits);
    }
    __syncthreads();
    if (w == 0) {
        const uint32_t *ra = in0 >= (uint32_t)s0 ? s_rec[0] : cuts + (size_t)in0 * NCUT * 5;
        const uint32_t *rb = in1 >= (uint32_t)s0 ? s_rec[1] : cuts + (size_t)in1 * NCUT * 5;
        cut_node<REC_PLAIN>(v, lane, l0, l1, ra, rb, cuts + (size_t)v * NCUT * 5, nRef, nullptr, nullptr, sigBits);
    }
}

// Three levels in one launch (ids s0..s1-1, s1..s2-1, s2..e-1), one workgroup
// per node.  A node of the first level is computed as in k_cuts_level, one of
// the second as in k_cuts_pair.  A node v of the third level recomputes its
// cone in its workgroup: the bottom nodes (first-level fanins of v and of v's
// second-level fanins, at most 4, one wavefront each), then the middle nodes
// (v's second-level fanins, at most 2), then v, with a barrier between the
// steps and the recomputed sets held in LDS.  Fanins below the launch are read
// from the global records, which earlier launches completed.
constexpr int CUT3_BLOCK = 256;
__device__ __forceinline__ const uint32_t *rec_or_lds(uint32_t x, const uint32_t *cuts, uint32_t (*s_rec)[NCUT * 5],
                                                      uint32_t b0, uint32_t b1, uint32_t b2, uint32_t m0,
                                                      uint32_t m1, uint32_t s0, uint32_t s1) {
    if (x >= s1) return s_rec[x == m0 ? 4 : 5];
    if (x >= s0) return s_rec[x == b0 ? 0 : x == b1 ? 1 : x == b2 ? 2 : 3];
    return cuts + (size_t)x * NCUT * 5;
}

__global__ void __launch_bounds__(CUT3_BLOCK) k_cuts_triple(int32_t s0_, int32_t s1_, int32_t s2_, uint32_t n,
                                                            const uint32_t *__restrict__ f0,
                                                            const uint32_t *__restrict__ f1,
                                                            const int32_t *__restrict__ nRef, uint32_t *cuts,
                                                            const uint8_t *__restrict__ sigBits) {
    __shared__ uint32_t s_rec[6][NCUT * 5];     // bottom nodes 0..3, middle nodes 4..5
    const uint32_t s0 = (uint32_t)s0_, s1 = (uint32_t)s1_, s2 = (uint32_t)s2_;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint32_t v = s0 + blockIdx.x;
    // issue priority by chain length: a third-level node's workgroup runs three
    // dependent steps and bounds the launch, a first-level node's runs one
    if (v < s1) {                               // uniform per workgroup
        __builtin_amdgcn_s_setprio(0);
        if (w == 0) {
            cut_node_global((int)v, lane, f0, f1, nRef, cuts, sigBits);
        } else if (w == 1) {
            // the next launch's fanins into this XCD's L2 (workgroups go round
            // the 8 XCDs; a line holds 32 nodes): a cone walk there starts with
            // three dependent loads of them
            const uint32_t q = s0 + gridDim.x + (blockIdx.x >> 3) * 32u;
            if (lane < 2 && q < n) {
                const uint32_t l = lane == 0 ? f0[q] : f1[q];
                if (l == 0xFFFFFFFFu) cuts[0] = 0u;     // no literal: keeps the load
            }
        }
        return;
    }
    if (v >= s2) __builtin_amdgcn_s_setprio(2);
    else __builtin_amdgcn_s_setprio(1);
    const uint32_t l0 = f0[v], l1 = f1[v];
    const uint32_t a = LID(l0), b = LID(l1);
    const uint32_t NONE = 0xFFFFFFFFu;
    // middle nodes (second level) and bottom nodes (first level) of the cone
    uint32_t m0 = NONE, m1 = NONE, ml0 = 0u, ml1 = 0u, ml2 = 0u, ml3 = 0u;    // fanin literals of m0, m1
    uint32_t b0 = NONE, b1 = NONE, b2 = NONE, b3 = NONE;
    int nb = 0;
    // appends x if it is a first-level node not yet listed (selects, so the
    // list stays in registers)
    auto add_bot = [&](uint32_t x) {
        const bool add = x >= s0 && x != b0 && x != b1 && x != b2;
        b0 = add && nb == 0 ? x : b0;
        b1 = add && nb == 1 ? x : b1;
        b2 = add && nb == 2 ? x : b2;
        b3 = add && nb == 3 ? x : b3;
        nb += add ? 1 : 0;
    };
    if (v >= s2) {
        if (a >= s1) m0 = a;
        if (b >= s1) { if (m0 == NONE) m0 = b; else m1 = b; }
        if (m0 != NONE) { ml0 = f0[m0]; ml1 = f1[m0]; }
        if (m1 != NONE) { ml2 = f0[m1]; ml3 = f1[m1]; }
        if (a < s1) add_bot(a);
        if (b < s1) add_bot(b);
        if (m0 != NONE) { add_bot(LID(ml0)); add_bot(LID(ml1)); }
        if (m1 != NONE) { add_bot(LID(ml2)); add_bot(LID(ml3)); }
    } else {
        add_bot(a);
        add_bot(b);
    }
    // step 1: bottom nodes from the global records
    const uint32_t mine = w == 0 ? b0 : w == 1 ? b1 : w == 2 ? b2 : b3;
    if (w < nb) {
        const uint32_t g0 = f0[mine], g1 = f1[mine];
        cut_node<REC_PLAIN>((int)mine, lane, g0, g1, cuts + (size_t)LID(g0) * NCUT * 5,
                            cuts + (size_t)LID(g1) * NCUT * 5, s_rec[w], nRef, nullptr, nullptr, sigBits);
    }
    __syncthreads();
    // step 2: middle nodes
    if (v >= s2) {
        const uint32_t mm = w == 0 ? m0 : m1;
        if (w < 2 && mm != NONE) {
            const uint32_t g0 = w == 0 ? ml0 : ml2, g1 = w == 0 ? ml1 : ml3;
            cut_node<REC_PLAIN>((int)mm, lane, g0, g1, rec_or_lds(LID(g0), cuts, s_rec, b0, b1, b2, m0, m1, s0, s1),
                                rec_or_lds(LID(g1), cuts, s_rec, b0, b1, b2, m0, m1, s0, s1), s_rec[4 + w], nRef,
                                nullptr, nullptr, sigBits);
        }
        __syncthreads();
    }
    // step 3: the node itself
    if (w == 0)
        cut_node<REC_PLAIN>((int)v, lane, l0, l1, rec_or_lds(a, cuts, s_rec, b0, b1, b2, m0, m1, s0, s1),
                            rec_or_lds(b, cuts, s_rec, b0, b1, b2, m0, m1, s0, s1), cuts + (size_t)v * NCUT * 5, nRef,
                            nullptr, nullptr, sigBits);
}

// ---- planned schedule (GLS_RW_PLAN_CUTS): K levels per launch
// A launch covers K consecutive levels (positions 0..K-1).  The in-launch
// cone of a node (its transitive fanins inside the launch) is fixed by the
// graph alone, so the cones are listed once per pass before the launches:
//   - every node of the top position is a root; going down the positions, a
//     node that no higher root's cone contains becomes a root as well;
//   - a root's workgroup recomputes its cone position by position (one
//     wavefront per node, records in LDS, a barrier between positions), and
//     every cone node is stored to the global records by exactly one of the
//     workgroups that recompute it (the smallest root id), the root by its own;
//   - position-0 nodes that no cone contains are packed four to a workgroup.
// Each workgroup reads a header and its entries (node, fanin literals, where
// each fanin's record is: an LDS slot of this task or the global records)
// with scalar loads, so no fanin is looked up at run time.  Every record is
// computed by the deterministic cut_node, so the results are bit-identical to
// one launch per level.  On the 10M-AND workload with K = 3 a launch runs
// ~328 workgroups instead of k_cuts_triple's ~617.
// Header (uint4): x = first entry, y = entry count | top position << 16,
//   z, w = node count of positions 0..3 and 4..7 (8 bits each).
// Entry (uint4): x = node id | stored-globally << 31 | kept-in-LDS << 30,
//   y, z = fanin literals, w = fanin sources (8 bits each: an entry index of
//   this task, or PLAN_GLOBAL).
#include "cut_cone.h"

// Four levels in one launch (ids [s0, s1), [s1, s2), [s2, s3), [s3, e)), one
// workgroup of four wavefronts per node, as k_cuts_triple with one more
// level: a node recomputes its in-launch cone (at most 8, 4 and 2 nodes on
// the launch's three lower levels, listed by one thread into LDS) level by
// level, one wavefront per cone node (the lowest level's nodes beyond four in
// a second batch), records in LDS, a barrier between the levels; its own set
// goes to the global records.  One launch replaces four dependent ones at the
// price of larger cones.  (Eight wavefronts per workgroup, one per lowest-level
// node, put two of a workgroup's own wavefronts on every SIMD and measured
// 17.9 us per launch against 10.9 for three levels.)
constexpr int CUT4_BLOCK = 256;   // (cuts of the 10M AIG 133.5 ms, 111.6 with three levels)

// the record of fanin x for a cone node: its LDS slot if the cone lists it,
// else the global records (x below the launch)
__device__ __forceinline__ const uint32_t *cone4_rec(uint32_t x, const uint32_t *s, const Cone4 &c,
                                                     uint32_t (*s_rec)[NCUT * 5], const uint32_t *cuts) {
    const int p = cone4_level(x, s);
    if (p >= 0 && p <= 2) {
        const uint32_t base = p == 0 ? 0u : p == 1 ? 8u : 12u;
        for (uint32_t k = 0; k < c.n[p]; k++)
            if (c.id[p][k] == x) return s_rec[base + k];
    }
    return cuts + (size_t)x * NCUT * 5;
}

__global__ void __launch_bounds__(CUT4_BLOCK) k_cuts_quad(int32_t s0_, int32_t s1_, int32_t s2_, int32_t s3_,
                                                          const uint32_t *__restrict__ f0,
                                                          const uint32_t *__restrict__ f1,
                                                          const int32_t *__restrict__ nRef, uint32_t *cuts,
                                                          const uint8_t *__restrict__ sigBits) {
    __shared__ uint32_t s_rec[14][NCUT * 5];    // level 0: 0..7, level 1: 8..11, level 2: 12..13
    __shared__ Cone4 s_cone;
    const uint32_t s[4] = {(uint32_t)s0_, (uint32_t)s1_, (uint32_t)s2_, (uint32_t)s3_};
    const int lane = threadIdx.x & 63;
    const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t v = s[0] + blockIdx.x;
    const int pv = cone4_level(v, s);
    // issue priority by chain length: a top-level node's workgroup runs four
    // dependent steps and bounds the launch
    if (pv == 0) {                              // uniform per workgroup
        __builtin_amdgcn_s_setprio(0);
        if (w == 0) cut_node_global((int)v, lane, f0, f1, nRef, cuts, sigBits);
        return;
    }
    if (pv == 3) __builtin_amdgcn_s_setprio(3);
    else if (pv == 2) __builtin_amdgcn_s_setprio(2);
    else __builtin_amdgcn_s_setprio(1);
    if (threadIdx.x == 0) cone4_discover(v, s, f0, f1, s_cone);
    __syncthreads();
    const uint32_t n0 = s_cone.n[0], n1 = s_cone.n[1], n2 = s_cone.n[2];
    // level 0 of the cone: fanins below the launch; nodes 4..7 in a second batch
    if (w < n0) {
        const uint32_t x = s_cone.id[0][w], g0 = s_cone.l0[0][w], g1 = s_cone.l1[0][w];
        cut_node<REC_PLAIN>((int)x, lane, g0, g1, cuts + (size_t)LID(g0) * NCUT * 5,
                            cuts + (size_t)LID(g1) * NCUT * 5, s_rec[w], nRef, nullptr, nullptr, sigBits);
    }
    if (w + 4 < n0) {
        const uint32_t x = s_cone.id[0][w + 4], g0 = s_cone.l0[0][w + 4], g1 = s_cone.l1[0][w + 4];
        cut_node<REC_PLAIN>((int)x, lane, g0, g1, cuts + (size_t)LID(g0) * NCUT * 5,
                            cuts + (size_t)LID(g1) * NCUT * 5, s_rec[w + 4], nRef, nullptr, nullptr, sigBits);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __syncthreads();
    // level 1
    if (w < n1) {
        const uint32_t x = s_cone.id[1][w], g0 = s_cone.l0[1][w], g1 = s_cone.l1[1][w];
        cut_node<REC_PLAIN>((int)x, lane, g0, g1, cone4_rec(LID(g0), s, s_cone, s_rec, cuts),
                            cone4_rec(LID(g1), s, s_cone, s_rec, cuts), s_rec[8 + w], nRef, nullptr, nullptr,
                            sigBits);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __syncthreads();
    // level 2
    if (w < n2) {
        const uint32_t x = s_cone.id[2][w], g0 = s_cone.l0[2][w], g1 = s_cone.l1[2][w];
        cut_node<REC_PLAIN>((int)x, lane, g0, g1, cone4_rec(LID(g0), s, s_cone, s_rec, cuts),
                            cone4_rec(LID(g1), s, s_cone, s_rec, cuts), s_rec[12 + w], nRef, nullptr, nullptr,
                            sigBits);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __syncthreads();
    // the node itself
    if (w == 0) {
        const uint32_t l0 = f0[v], l1 = f1[v];
        cut_node<REC_PLAIN>((int)v, lane, l0, l1, cone4_rec(LID(l0), s, s_cone, s_rec, cuts),
                            cone4_rec(LID(l1), s, s_cone, s_rec, cuts), cuts + (size_t)v * NCUT * 5, nRef, nullptr,
                            nullptr, sigBits);
    }
}

#include "cut_plan.h"

// One planned task per workgroup (the launch's tasks start at `base`).
__global__ void __launch_bounds__(CUT3_BLOCK) k_cuts_plan(const uint4 *__restrict__ heads,
                                                          const uint4 *__restrict__ ents, int32_t base, int32_t K,
                                                          const int32_t *__restrict__ nRef, uint32_t *cuts,
                                                          const uint8_t *__restrict__ sigBits) {
    __shared__ uint32_t s_rec[PLAN_MAX_CONE][NCUT * 5];
    const int lane = threadIdx.x & 63;
    const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint4 h = heads[base + blockIdx.x];
    const uint32_t top = h.y >> 16;
    // issue priority by chain length: the roots of the top position bound the launch
    if (top + 1 >= (uint32_t)K && K > 1) __builtin_amdgcn_s_setprio(2);
    else if (top > 0) __builtin_amdgcn_s_setprio(1);
    else __builtin_amdgcn_s_setprio(0);
    uint32_t start = 0;
    bool first = true;
    for (int p = 0; p < K; p++) {
        const uint32_t cnt = (p < 4 ? h.z >> (8 * p) : h.w >> (8 * (p - 4))) & 0xFFu;
        if (cnt == 0) continue;                 // uniform per workgroup
        if (!first) {
            // this wavefront's LDS records are written before any wavefront
            // passes the barrier and reads them
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __syncthreads();
        }
        first = false;
        for (uint32_t k = w; k < cnt; k += CUT3_BLOCK / 64) {
            const uint4 e = ents[h.x + start + k];
            const uint32_t id = e.x & 0x3FFFFFFFu;
            const uint32_t s0 = e.w & 0xFFu, s1 = (e.w >> 8) & 0xFFu;
            const uint32_t *ra = s0 == PLAN_GLOBAL ? cuts + (size_t)LID(e.y) * NCUT * 5 : s_rec[s0];
            const uint32_t *rb = s1 == PLAN_GLOBAL ? cuts + (size_t)LID(e.z) * NCUT * 5 : s_rec[s1];
            uint32_t *glob = cuts + (size_t)id * NCUT * 5;
            const bool stored = (e.x >> 31) != 0u, kept = ((e.x >> 30) & 1u) != 0u;
            // separate call sites, so that the LDS record is written through an
            // LDS pointer (ds_write, which the barrier waits for; a pointer that
            // is LDS or global at run time would make it a flat store that the
            // barrier does not wait for)
            if (kept)
                cut_node<REC_PLAIN>((int)id, lane, e.y, e.z, ra, rb, s_rec[start + k], nRef, nullptr, nullptr, sigBits,
                                    stored ? glob : nullptr);
            else
                cut_node<REC_PLAIN>((int)id, lane, e.y, e.z, ra, rb, glob, nRef, nullptr, nullptr, sigBits);
        }
        start += cnt;
    }
}

// All levels in one cooperative launch: the wavefronts of the grid stride over
// each level's nodes, and a grid barrier separates the levels.
__global__ void __launch_bounds__(CUTW_BLOCK) k_cuts_levels(int32_t l0, int32_t l1, const int32_t *__restrict__ starts,
                                                            const uint32_t *__restrict__ f0,
                                                            const uint32_t *__restrict__ f1,
                                                            const int32_t *__restrict__ nRef, uint32_t *cuts,
                                                            const uint8_t *__restrict__ sigBits) {
    cooperative_groups::grid_group grid = cooperative_groups::this_grid();
    const int nw = gridDim.x * (CUTW_BLOCK / 64);
    const int gw = blockIdx.x * (CUTW_BLOCK / 64) + (threadIdx.x >> 6);
    for (int l = l0; l < l1; l++) {
        const int s = starts[l], e = starts[l + 1];
        for (int v = s + gw; v < e; v += nw)
            cut_node_global(v, threadIdx.x & 63, f0, f1, nRef, cuts, sigBits);
        grid.sync();
    }
}

// XCD-local schedule: one persistent kernel on the 32 CUs of one XCD.
// Workgroups are dispatched round-robin over the XCDs, so workgroups 0, 8, 16,
// ... share XCD 0 and its L2; the others return at once.  Between levels a
// counter barrier (device-scope atomics, about 1 us) replaces a kernel
// boundary (about 4.7 us on this path).  A CU's L1 is not coherent with the
// other CUs' stores: after each barrier one wavefront of the workgroup runs
// buffer_inv sc1, which drops the CU's L1 lines (buffer_inv sc0 does not in
// this mode), so the fanin records written by other CUs are read from L2.
// Every workgroup records its XCD; if they are not all on one, or a barrier
// wait exceeds its bound, ctl[2] is set, every workgroup stops, and the host
// recomputes the cut sets with one launch per level.
constexpr int XCD_WG = 1024;
constexpr int XCD_COUNT = 8;
constexpr uint32_t XCD_SPIN_LIMIT = 1u << 20;

__device__ __forceinline__ uint32_t xcc_id() {
    uint32_t v;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(v));
    return v & 0xFu;
}

// ctl[0] barrier arrivals, ctl[1] mask of XCDs seen, ctl[2] error
__device__ __forceinline__ bool xcd_barrier(uint32_t *ctl, uint32_t &epoch, uint32_t nwg, uint32_t *s_stop) {
    __builtin_amdgcn_s_waitcnt(0);          // this wavefront's stores have reached L2
    __syncthreads();
    ++epoch;
    if (threadIdx.x == 0) {
        __hip_atomic_fetch_add(&ctl[0], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint32_t target = epoch * nwg;
        uint32_t spins = 0;
        bool bad = false;
        while (__hip_atomic_load(&ctl[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < target) {
            if (++spins > XCD_SPIN_LIMIT || __hip_atomic_load(&ctl[2], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
                bad = true;
                break;
            }
            __builtin_amdgcn_s_sleep(1);
        }
        if (bad) __hip_atomic_fetch_or(&ctl[2], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("buffer_inv sc1\n\ts_waitcnt vmcnt(0)" ::: "memory");
        *s_stop = bad ? 1u : 0u;
    }
    __syncthreads();
    return *s_stop == 0;
}

__global__ void __launch_bounds__(XCD_WG) k_cuts_xcd(int32_t l0, int32_t l1, const int32_t *__restrict__ starts,
                                                     const uint32_t *__restrict__ f0, const uint32_t *__restrict__ f1,
                                                     const int32_t *__restrict__ nRef, uint32_t *cuts,
                                                     const uint8_t *__restrict__ sigBits, uint32_t nwg, uint32_t *ctl) {
    if (blockIdx.x % XCD_COUNT != 0) return;
    __shared__ uint32_t s_stop;
    const uint32_t wg = blockIdx.x / XCD_COUNT;
    if (wg >= nwg) return;
    const int lane = threadIdx.x & 63;
    // a level's nodes go round-robin over the workgroups (one per CU) first,
    // so a level of n nodes puts about n / nwg wavefronts on each CU
    const int gw = (int)(threadIdx.x >> 6) * (int)nwg + (int)wg;
    const int nw = (int)nwg * (XCD_WG / 64);
    uint32_t epoch = 0;
    if (threadIdx.x == 0) __hip_atomic_fetch_or(&ctl[1], 1u << xcc_id(), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (!xcd_barrier(ctl, epoch, nwg, &s_stop)) return;
    if (__popc(__hip_atomic_load(&ctl[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 1) {
        if (threadIdx.x == 0) __hip_atomic_fetch_or(&ctl[2], 2u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return;
    }
    for (int l = l0; l < l1; l++) {
        const int s = starts[l], e = starts[l + 1];
        for (int v = s + gw; v < e; v += nw)
            cut_node_global(v, lane, f0, f1, nRef, cuts, sigBits);
        if (!xcd_barrier(ctl, epoch, nwg, &s_stop)) return;
    }
}

// Dataflow schedule: persistent wavefronts take nodes in level-major id order
// from a ticket counter and wait only for their two fanins' cut sets, polled
// in the fence-free record format; no level waits for the whole previous
// level.  Progress: the smallest unfinished ticket has every fanin finished
// (fanin ids are smaller) and is held by a running wavefront.  Every wait is
// bounded; on overrun *err is set and all wavefronts stop.
__global__ void __launch_bounds__(CUTW_BLOCK) k_cuts_dataflow(int32_t first, int32_t last,
                                                              const uint32_t *__restrict__ f0,
                                                              const uint32_t *__restrict__ f1,
                                                              const int32_t *__restrict__ nRef,
                                                              unsigned long long *tcuts, uint32_t *ticket,
                                                              uint32_t *err, const uint8_t *__restrict__ sigBits) {
    const int lane = threadIdx.x & 63;
    for (;;) {
        if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) break;
        uint32_t t = 0;
        if (lane == 0) t = atomicAdd(ticket, 1u);
        t = (uint32_t)__shfl((int)t, 0);
        const int v = first + (int)t;
        if (v >= last) break;
        if (!cut_node<REC_TAGGED>(v, lane, f0[v], f1[v], nullptr, nullptr, nullptr, nRef, tcuts, err, sigBits)) break;
    }
}

// PI cut sets in the fence-free format (slot 0 trivial, others empty but valid).
__global__ void k_cuts_pi_tagged(int32_t nPIs, const int32_t *__restrict__ nRef, unsigned long long *tcuts) {
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= (int64_t)nPIs * NCUT) return;
    const int64_t v = 1 + i / NCUT;
    const int slot = (int)(i % NCUT);
    unsigned long long *q = tcuts + ((size_t)v * NCUT + slot) * 3;
    store_tagged(q + 0, slot == 0 ? (unsigned long long)v : 0ull);
    store_tagged(q + 1, 0ull);
    store_tagged(q + 2, slot == 0 ? 0xAAAAull | (1001ull << 16) | (1ull << 27) | (1ull << 30) : 0ull);
    (void)nRef;
}

// Fence-free records back to the plain 5-word records used by evaluation.
__global__ void k_untag_cuts(int64_t nslots, const unsigned long long *__restrict__ tcuts, uint32_t *cuts) {
    int64_t tid = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = tid; i < nslots; i += stride) {
        const unsigned long long w0 = tcuts[3 * i], w1 = tcuts[3 * i + 1], w2 = tcuts[3 * i + 2];
        uint32_t *o = cuts + 5 * i;
        if (!(w2 & TAG_V)) { o[0] = o[1] = o[2] = o[3] = o[4] = 0; continue; }
        o[0] = (uint32_t)(w0 & 0x7FFFFFFFull);
        o[1] = (uint32_t)((w0 >> 31) & 0x7FFFFFFFull);
        o[2] = (uint32_t)(w1 & 0x7FFFFFFFull);
        o[3] = (uint32_t)((w1 >> 31) & 0x7FFFFFFFull);
        o[4] = (uint32_t)w2;
    }
}

__global__ void k_nref(int32_t n, int32_t nPIs, const uint32_t *__restrict__ f0, const uint32_t *__restrict__ f1,
                       int32_t nPOs, const uint32_t *__restrict__ pos, int32_t *nRef) {
    int64_t tid = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t v = nPIs + 1 + tid; v < n; v += stride) {
        atomicAdd(&nRef[LID(f0[v])], 1);
        atomicAdd(&nRef[LID(f1[v])], 1);
    }
    for (int64_t i = tid; i < nPOs; i += stride) atomicAdd(&nRef[LID(pos[i])], 1);
}

// Structural table of the graph, indexed by fanin: bucket x holds the ANDs
// whose second fanin literal (the one of larger id) is on node x, as entries
// {first fanin literal, node | second literal's complement << 31}.  Buckets
// follow node ids, so the lookups of nearby nodes touch nearby memory (a hash
// table of the same keys spreads them over the whole table, which for the
// batched arena is far larger than the caches).
__global__ void k_table_count(int32_t n, int32_t nPIs, const uint32_t *__restrict__ f1, uint32_t *cnt) {
    int64_t tid = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t v = nPIs + 1 + tid; v < n; v += stride) atomicAdd(&cnt[LID(f1[v])], 1u);
}

__global__ void k_table_fill(int32_t n, int32_t nPIs, const uint32_t *__restrict__ f0,
                             const uint32_t *__restrict__ f1, const uint32_t *__restrict__ off, uint32_t *cur,
                             uint2 *ent) {
    int64_t tid = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t v = nPIs + 1 + tid; v < n; v += stride) {
        const uint32_t b = f1[v];
        const uint32_t k = off[LID(b)] + atomicAdd(&cur[LID(b)], 1u);
        ent[k] = make_uint2(f0[v], (uint32_t)v | (b & 1u) << 31);
    }
}

// ------------------------------------------------------------------------
// evaluation
// ------------------------------------------------------------------------
struct GraphView {
    const uint32_t *f0, *f1;
    const int32_t *nRef;
    const uint32_t *level;
    const uint32_t *tOff;       // structural table: bucket offsets (n + 1)
    const uint2 *tEnt;          // and entries (see k_table_fill)
    // batched: the members of the nodes, and their number of objects.  Members share
    // the constant; where a cone reaches it, member t's is object n + t, with
    // that member's references
    const uint32_t *tag = nullptr;
    int32_t n = 0;
};

// per-thread column of an LDS array laid out [j][lane]
struct Col {
    int32_t *p;
    __device__ __forceinline__ int32_t &operator[](int j) const { return p[j * EVAL_BLOCK]; }
};

struct Mffc {
    int size;
    int32_t id[MFFC_TAB], num[MFFC_TAB];
};

// The table and the DFS stack below are indexed by constants only (a write at
// a run-time position selects among the entries), so they live in registers
// instead of scratch memory.
__device__ __forceinline__ int mffc_decrease(const GraphView &g, int root, int x, const int *leaves, int nL, Mffc &t) {
#pragma unroll
    for (int i = 0; i < 4; i++)
        if (i < nL && x == leaves[i]) return 1;
    if (x == 0 && g.tag) x = g.n + (int)g.tag[root];
    int found = -1;
#pragma unroll
    for (int i = 0; i < MFFC_TAB; i++)
        if (found < 0 && i < t.size && t.id[i] == x) found = i;
    if (found >= 0) {
        int r = 0;
#pragma unroll
        for (int i = 0; i < MFFC_TAB; i++)
            if (i == found) r = --t.num[i];
        return r;
    }
    if (t.size == MFFC_TAB) return 1;
    const int r = g.nRef[x] - 1;
#pragma unroll
    for (int i = 0; i < MFFC_TAB; i++)
        if (i == t.size) { t.id[i] = x; t.num[i] = r; }
    t.size++;
    return r;
}

// CalcMFFC (rewrite.cu:319-326) without recursion: an explicit DFS stack that
// visits fanin0's subtree before decreasing fanin1, as the recursion does.
// At most MFFC_TAB nodes are pushed besides the root (a push needs a new
// table entry), so MFFC_TAB + 2 entries never overflow.  The stack's nodes go
// to the LDS column stk (the caller's match column, free until library
// matching fills it), one access each; their stages (0, 1: fanin to visit
// next, 2: done) are 2-bit fields of one register.
__device__ int calc_mffc(const GraphView &g, int root, const int *leaves, int nL, Mffc &t, Col stk) {
    stk[0] = root;
    uint32_t stg = 0;
    int sp = 1, ans = 1;
    t.size = 0;
#pragma unroll
    for (int i = 0; i < MFFC_TAB; i++) { t.id[i] = 0; t.num[i] = 0; }
    while (sp) {
        const int top = sp - 1;
        const int stage = (int)((stg >> (2 * top)) & 3u);
        if (stage < 2) {
            stg += 1u << (2 * top);
            const int cur = stk[top];
            const int x = (int)LID(stage == 0 ? g.f0[cur] : g.f1[cur]);
            if (mffc_decrease(g, root, x, leaves, nL, t) == 0) {
                stk[sp] = x;
                stg &= ~(3u << (2 * sp));
                sp++;
                ans++;
            }
        } else {
            sp--;
        }
    }
    return ans;
}

__device__ __forceinline__ int mffc_deleted(const Mffc &t, int x) {
    int r = 0;
    bool found = false;
#pragma unroll
    for (int i = 0; i < MFFC_TAB; i++)
        if (!found && i < t.size && t.id[i] == x) {
            found = true;
            r = t.num[i] == 0;
        }
    return r;
}

// The AND with fanins (in0, c0), (in1, c1) if the graph has one (the smallest
// such id), else -1: a scan of the bucket of the fanin of larger id.
__device__ __forceinline__ int table_lookup(const GraphView &g, int in0, int in1, int c0, int c1) {
    if (in0 > in1) { int x = in0; in0 = in1; in1 = x; x = c0; c0 = c1; c1 = x; }
    const uint32_t lo = 2u * (uint32_t)in0 + (uint32_t)c0, hc = (uint32_t)c1 << 31;
    const uint32_t e = g.tOff[in1 + 1];
    uint32_t best = 0xFFFFFFFFu;
    for (uint32_t k = g.tOff[in1]; k < e; k++) {
        const uint2 x = g.tEnt[k];
        if (x.x == lo && (x.y & 0x80000000u) == hc) best = min(best, x.y & 0x7FFFFFFFu);
    }
    return best == 0xFFFFFFFFu ? -1 : (int)best;
}

// library matching of one cut (rewrite.cu:391-418); returns the class
__device__ int match_cut(const GraphView &g, const Lib &L, int id, uint32_t tt, const int *leaves,
                         const Mffc &t, Col match, Col mlev, uint32_t &isC, uint64_t &matched) {
    uint32_t w = L.npn[tt];
    int uPhase = w & 31, perm = (w >> 5) & 31, cls = (w >> 10) & 255;
    const uint8_t *pp = L.perms4 + 4 * perm;
    // entries 0..3 (the inputs) and 4..nn+3 (the class's forest nodes) are all
    // written below before they are read; the library's roots and children
    // index only those, so the columns need no clearing.  matched: bit j set
    // when entry j holds an existing node (the inputs always do)
    isC = 0;
    matched = 0xFull;
    for (int j = 0; j < 4; j++) {
        const int q = pp[j];
        const int leaf = q == 0 ? leaves[0] : q == 1 ? leaves[1] : q == 2 ? leaves[2] : leaves[3];
        match[j] = leaf;
        mlev[j] = (int)g.level[leaf];
        if ((uPhase >> j) & 1) isC |= 1u << j;
    }
    const int nn = lib_nn(L, cls);
    for (int j = 0; j < nn; j++) {
        uint32_t wd = lib_word(L, cls, j);
        int a = wd & 63, b = (wd >> 6) & 63, ca = (wd >> 12) & 1, cb = (wd >> 13) & 1;
        int num = j + 4;
        const int la = mlev[a], lb = mlev[b];
        int lev = 1 + (la > lb ? la : lb);
        const int ma = match[a], mb = match[b];
        int found = -1;
        if (!(ma == -1 || mb == -1 || ma == id || mb == id)) {
            const int nid = table_lookup(g, ma, mb, (int)isc_bit(isC, a) ^ ca, (int)isc_bit(isC, b) ^ cb);
            if (nid != -1 && !mffc_deleted(t, nid)) {
                found = nid;
                lev = (int)g.level[nid];
            }
        }
        match[num] = found;
        mlev[num] = lev;
        if (found != -1) matched |= 1ull << num;
    }
    return cls;
}

// Forest nodes that replacing with root rt would create (Eval, rewrite.cu:369-374,
// counts them): from rt down, every unmatched node that a created node uses.  Children have
// lower indexes than their parents, so taking the highest unmatched used node
// each time visits exactly the nodes of a descending scan over all indexes,
// in the same order, with one step per created node instead of per index.
__device__ __forceinline__ uint64_t added_set(const Lib &L, int cls, int rt, uint64_t matched) {
    uint64_t used = 1ull << rt, add = 0;
    for (uint64_t cand = used & ~matched; cand; cand = used & ~matched & ~add) {
        const int j = 63 - __clzll((long long)cand);
        add |= 1ull << j;
        const uint32_t wd = lib_word(L, cls, j - 4);
        used |= 1ull << (wd & 63);
        used |= 1ull << ((wd >> 6) & 63);
    }
    return add;
}

__device__ __forceinline__ void cut_leaves4(const uint32_t *p, int *leaves, int &nL, uint32_t &tt) {
    uint32_t m = p[4];
    nL = (m >> 27) & 7;
    tt = m & 0xFFFF;
    for (int i = 0; i < 4; i++) leaves[i] = (int)p[i];
    if (nL == 3) { leaves[3] = 0; nL = 4; }
}

// Evaluation of every cut of a node (Eval, rewrite.cu:328-424): the gain of the
// best root, then its level, then the first cut and root decide.
// One wavefront takes NODES nodes.  First every lane computes the fanout-free
// cone of one of their cuts; then 16 lanes match one cut each time, four cuts
// side by side: a lane takes the class's forest nodes gl, gl + 16, .. and
// waits for a node's children (done: the forest nodes that are finished), and
// the set of nodes that a forest node would create is the union of its
// children's and itself unless it exists, so a root costs one popcount.
// What bounds it is the chain of lookups: a class has 15 forest nodes on
// average and 50 at most, but these need 3.5 rounds of 16 lanes.  State is per
// cut and not per lane, so 28 wavefronts fit a CU's LDS instead of 7.  With a
// node per lane, its cuts one after the other: 2k random ANDs 211 us (now 26),
// 200k windowed 575 (242), 4M windowed 6090 (1605), 10M in a batch of random
// AIGs 23500.
struct EvalCut {           // of one forest entry
    int32_t match, lev;    // the existing node or -1; its level, or that it would get
    uint64_t add;          // the entries it would create
};

constexpr int EG = 16, EGS = 64 / EG;      // lanes per cut, cuts side by side

template <int NODES>
__global__ void __launch_bounds__(64) k_eval(int32_t n, int32_t nPIs, GraphView g, Lib L,
                                             const uint32_t *__restrict__ cuts, int useZeros, int4 *best) {
    __shared__ EvalCut s_ent[EGS * NMATCH];            // first the cones' DFS stacks
    __shared__ int32_t s_del[MFFC_TAB * 64];           // the cones' nodes besides the root
    __shared__ unsigned long long s_best[NODES];
    __shared__ uint8_t s_list[64];
    static_assert(sizeof(EvalCut) * EGS * NMATCH >= 4 * (MFFC_TAB + 2) * EVAL_BLOCK, "stacks");
    static_assert(EVAL_BLOCK == 64 && NODES * NCUT <= 64 && NMATCH <= 64, "one wavefront");
    const int lane = threadIdx.x, grp = lane / EG, gl = lane % EG;
    const int64_t base = nPIs + 1 + blockIdx.x * (int64_t)NODES;
    if (lane < NODES) s_best[lane] = ~0ull;
    // ---- a cut per lane
    int leaves[4] = {}, nL = 0;
    uint32_t pack = 0, offs = 0;
    bool valid = false;
    if (lane < NODES * NCUT && base + lane / NCUT < n) {
        const uint32_t *p = cuts + ((size_t)(base + lane / NCUT) * NCUT + lane % NCUT) * 5;
        const uint32_t meta = p[4];
        valid = ((meta >> 30) & 1) && ((meta >> 27) & 7) >= 3;
        if (valid) {
            uint32_t tt;
            cut_leaves4(p, leaves, nL, tt);
            const uint32_t w = L.npn[tt];
            const int cls = (w >> 10) & 255;
            Mffc t;
            const int saved = calc_mffc(g, (int)(base + lane / NCUT), leaves, nL, t, Col{(int32_t *)s_ent + lane});
            int nd = 0;
#pragma unroll
            for (int i = 0; i < MFFC_TAB; i++)
                if (i < t.size && t.num[i] == 0) s_del[64 * nd++ + lane] = t.id[i];
            pack = (w & 0x3FFu) | (uint32_t)saved << 10 | (uint32_t)nd << 14 | (uint32_t)lib_nn(L, cls) << 18 |
                   (uint32_t)lib_nr(L, cls) << 24;
            offs = (uint32_t)L.nodeOff[cls] | (uint32_t)L.rootOff[cls] << 16;
        }
    }
    const uint64_t vm = __ballot(valid);
    const int count = __popcll(vm);
    if (valid) s_list[__popcll(vm & ((1ull << lane) - 1ull))] = (uint8_t)lane;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    // ---- a cut per 16 lanes
    EvalCut *ent = s_ent + grp * NMATCH;
    for (int c0 = 0; c0 < count; c0 += EGS) {
        const bool act = c0 + grp < count;
        const int src = s_list[act ? c0 + grp : 0];
        const uint32_t pk = (uint32_t)__shfl((int)pack, src), of = (uint32_t)__shfl((int)offs, src);
        const int l0 = __shfl(leaves[0], src), l1 = __shfl(leaves[1], src), l2 = __shfl(leaves[2], src),
                  l3 = __shfl(leaves[3], src);
        const int id = (int)(base + src / NCUT), saved = (int)((pk >> 10) & 15), nd = (int)((pk >> 14) & 15);
        const int nn = act ? (int)((pk >> 18) & 63) : 0, nr = act ? (int)(pk >> 24) : 0;
        const uint32_t isC = pk & 15u;
        const uint16_t *words = L.nodes + (of & 0xFFFFu);
        const int rt = gl < nr ? L.roots[(of >> 16) + gl] : 0;
        uint32_t wd = gl < nn ? words[gl] : 0u;
        if (act && gl < 4) {
            const int q = L.perms4[4 * ((pk >> 5) & 31) + gl];
            const int leaf = q == 0 ? l0 : q == 1 ? l1 : q == 2 ? l2 : l3;
            ent[gl] = EvalCut{leaf, (int32_t)g.level[leaf], 0ull};
        }
        uint64_t done = 0xFull;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        for (int j0 = 0; __ballot(j0 < nn) != 0; j0 += EG) {
            const int j = j0 + gl, a = wd & 63, b = (wd >> 6) & 63;
            const int ca = (wd >> 12) & 1, cb = (wd >> 13) & 1;
            bool pend = j < nn;
            wd = j + EG < nn ? words[j + EG] : 0u;
            while (__ballot(pend) != 0) {
                const bool ready = pend && ((done >> a) & (done >> b) & 1u);
                if (ready) {
                    const EvalCut x = ent[a], y = ent[b];
                    EvalCut e{-1, 1 + max(x.lev, y.lev), x.add | y.add | 1ull << (j + 4)};
                    if (x.match != -1 && y.match != -1 && x.match != id && y.match != id) {
                        const int nid = table_lookup(g, x.match, y.match, (int)isc_bit(isC, a) ^ ca,
                                                     (int)isc_bit(isC, b) ^ cb);
                        bool gone = nid == -1;
                        for (int i = 0; i < nd && !gone; i++) gone = s_del[64 * i + src] == nid;
                        if (!gone) e = EvalCut{nid, (int32_t)g.level[nid], 0ull};
                    }
                    ent[j + 4] = e;
                }
                const uint64_t m = __ballot(ready);
                done |= ((m >> (EG * grp)) & ((1ull << EG) - 1ull)) << (j0 + 4);
                pend = pend && !ready;
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            }
        }
        if (gl < nr) {
            const EvalCut e = ent[rt];
            const int gain = saved - __popcll(e.add);
            if (e.match != id && (gain > 0 || (gain == 0 && useZeros)))
                atomicMin(&s_best[src / NCUT], (unsigned long long)(255 - gain) << 48 |
                                                   (unsigned long long)(uint32_t)e.lev << 16 |
                                                   (unsigned long long)((src % NCUT) << 8 | gl));
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    if (lane < NODES && base + lane < n) {
        const unsigned long long k = s_best[lane];
        best[base + lane] = k == ~0ull ? make_int4(-1, 0, 0, 0)
                                       : make_int4((int)((k >> 8) & 255), (int)(k & 255), 255 - (int)(k >> 48),
                                                   (int)(uint32_t)(k >> 16));
    }
}

// ------------------------------------------------------------------------
// plans and selection
// ------------------------------------------------------------------------
struct Plan {
    int32_t id, gain;
    int32_t nW, nL, nM, nNew, valid, pad;
    int32_t W[MFFC_TAB + 1], L[4], M[PLAN_MAXM];
};

__device__ uint32_t lib_truth(const Lib &L, int cls, int rt, const uint8_t *pp, uint32_t isC) {
    const uint32_t ev[4] = {0xAAAA, 0xCCCC, 0xF0F0, 0xFF00};
    uint32_t tt[64];
    for (int j = 0; j < 4; j++) tt[j] = (ev[pp[j]] ^ (((isC >> j) & 1) ? 0xFFFFu : 0u)) & 0xFFFF;
    for (int j = 4; j <= rt; j++) {
        uint32_t wd = lib_word(L, cls, j - 4);
        uint32_t a = tt[wd & 63] ^ (((wd >> 12) & 1) ? 0xFFFFu : 0u);
        uint32_t b = tt[(wd >> 6) & 63] ^ (((wd >> 13) & 1) ? 0xFFFFu : 0u);
        tt[j] = a & b & 0xFFFF;
    }
    return tt[rt];
}

struct PlanCore {
    int cls, rt, compl_, valid;
    uint32_t isC;
    uint64_t addMask;
};

// Recomputes the chosen replacement of node `id` exactly as evaluated.
__device__ PlanCore plan_core(const GraphView &g, const Lib &L, int id, const uint32_t *p, int out, Mffc &t,
                              Col match, Col mlev) {
    int leaves[4], nL;
    uint32_t tt;
    cut_leaves4(p, leaves, nL, tt);
    calc_mffc(g, id, leaves, nL, t, match);
    PlanCore pc;
    uint64_t matched;
    pc.cls = match_cut(g, L, id, tt, leaves, t, match, mlev, pc.isC, matched);
    pc.rt = lib_root(L, pc.cls, out);
    pc.addMask = added_set(L, pc.cls, pc.rt, matched);
    pc.valid = 1;
    uint32_t w = L.npn[tt];
    uint32_t rtt = lib_truth(L, pc.cls, pc.rt, L.perms4 + 4 * ((w >> 5) & 31), pc.isC);
    if (rtt == tt) pc.compl_ = 0;
    else if (rtt == ((~tt) & 0xFFFF)) pc.compl_ = 1;
    else { pc.compl_ = 0; pc.valid = 0; }
    return pc;
}

// Candidates per wavefront of k_plan and k_build.  A lane replays its candidate's
// cone and forest, and a wavefront takes as long as the longest of its lanes'
// bucket scans, so few candidates are spread over more wavefronts, up to about
// eight on a CU.  k_plan and k_build of 2k ANDs 56 and 45 us with 64 to a
// wavefront, 36 and 29 with 4; of the 32-bit multiplier 73 and 58, 54 and 48.
constexpr int32_t PLAN_WAVES = 2048;
int plan_lanes(int32_t nCand) {
    int per = 4;
    while (per < EVAL_BLOCK && (int64_t)nCand > (int64_t)per * PLAN_WAVES) per *= 2;
    return per;
}

__global__ void __launch_bounds__(EVAL_BLOCK) k_plan(int32_t per, int32_t nCand, const uint32_t *__restrict__ candIds,
                                                      GraphView g, Lib L, const uint32_t *__restrict__ cuts,
                                                      const int4 *__restrict__ best, Plan *plans) {
    __shared__ int32_t s_match[NMATCH * EVAL_BLOCK], s_mlev[NMATCH * EVAL_BLOCK];
    int64_t c = blockIdx.x * (int64_t)per + threadIdx.x;
    if ((int32_t)threadIdx.x >= per || c >= nCand) return;
    Col match{s_match + threadIdx.x}, mlev{s_mlev + threadIdx.x};
    const int id = (int)candIds[c];
    const int4 b = best[id];
    const uint32_t *p = cuts + ((size_t)id * NCUT + b.x) * 5;
    Mffc t;
    PlanCore pc = plan_core(g, L, id, p, b.y, t, match, mlev);
    Plan pl;
    pl.id = id;
    pl.gain = b.z;
    pl.valid = pc.valid;
    pl.nNew = __popcll(pc.addMask);
    pl.pad = 0;
    pl.nW = 0;
    pl.W[pl.nW++] = id;
    for (int i = 0; i < MFFC_TAB; i++)
        if (i < t.size && t.num[i] == 0) pl.W[pl.nW++] = t.id[i];
    uint32_t meta = p[4];
    pl.nL = (meta >> 27) & 7;
    for (int i = 0; i < 4; i++) pl.L[i] = i < pl.nL ? (int32_t)p[i] : 0;
    uint64_t used = 1ull << pc.rt;
    for (int j = pc.rt; j >= 4; j--) {
        if (!((used >> j) & 1)) continue;
        uint32_t wd = lib_word(L, pc.cls, j - 4);
        used |= 1ull << (wd & 63);
        used |= 1ull << ((wd >> 6) & 63);
    }
    pl.nM = 0;
    for (int j = 4; j <= pc.rt; j++) {
        if (!((used >> j) & 1) || match[j] <= -1) continue;
        int m = match[j];
        int dup = 0;
        for (int q = 0; q < PLAN_MAXM; q++)
            if (q < pl.nM && pl.M[q] == m) dup = 1;
        if (m == id) pl.valid = 0;
        if (!dup) {
            if (pl.nM < PLAN_MAXM) pl.M[pl.nM++] = m;
            else pl.valid = 0;
        }
    }
    plans[c] = pl;
}

enum : uint32_t { MK_W = 1, MK_WNR = 2, MK_L = 4, MK_M = 8 };
enum : uint8_t { ST_ACTIVE = 0, ST_SELECTED = 1, ST_REJECTED = 2 };

__device__ __forceinline__ uint64_t stamp(uint32_t round, const Plan &p) {
    return (static_cast<uint64_t>(round) << 48) | (static_cast<uint64_t>(p.gain & 0xFFFF) << 32) |
           (0xFFFFFFFFu - static_cast<uint32_t>(p.id));
}

__global__ void k_sel_init(int32_t nCand, const Plan *__restrict__ plans, uint8_t *state) {
    int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (c < nCand) state[c] = plans[c].valid ? ST_ACTIVE : ST_REJECTED;
}

struct Claims {
    unsigned long long *W, *Wnr, *L, *M;
};

__global__ void k_sel_claim(uint32_t round, int32_t nCand, const Plan *__restrict__ plans,
                            const uint8_t *__restrict__ state, Claims cl, uint32_t *activeLeft) {
    int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (c == 0) *activeLeft = 0;             // counted by this round's k_sel_elim
    if (c >= nCand || state[c] != ST_ACTIVE) return;
    const Plan &p = plans[c];
    unsigned long long s = stamp(round, p);
    for (int i = 0; i < p.nW; i++) {
        atomicMax(&cl.W[p.W[i]], s);
        if (p.W[i] != p.id) atomicMax(&cl.Wnr[p.W[i]], s);
    }
    for (int i = 0; i < p.nL; i++) atomicMax(&cl.L[p.L[i]], s);
    for (int i = 0; i < p.nM; i++) atomicMax(&cl.M[p.M[i]], s);
}

__global__ void k_sel_decide(uint32_t round, int32_t nCand, const Plan *__restrict__ plans, uint8_t *state,
                             Claims cl, uint32_t *mk) {
    int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (c >= nCand || state[c] != ST_ACTIVE) return;
    const Plan &p = plans[c];
    unsigned long long s = stamp(round, p);
    bool win = true;
    for (int i = 0; i < p.nW && win; i++) {
        int x = p.W[i];
        if (cl.W[x] != s || cl.M[x] >= s) win = false;
        if (x != p.id && cl.L[x] >= s) win = false;
    }
    for (int i = 0; i < p.nL && win; i++)
        if (cl.Wnr[p.L[i]] >= s) win = false;
    for (int i = 0; i < p.nM && win; i++)
        if (cl.W[p.M[i]] >= s) win = false;
    if (!win) return;
    state[c] = ST_SELECTED;
    for (int i = 0; i < p.nW; i++) atomicOr(&mk[p.W[i]], MK_W | (p.W[i] != p.id ? MK_WNR : 0u));
    for (int i = 0; i < p.nL; i++) atomicOr(&mk[p.L[i]], MK_L);
    for (int i = 0; i < p.nM; i++) atomicOr(&mk[p.M[i]], MK_M);
}

// the first SEL_REST candidates still active also go to list, for k_sel_rest
constexpr uint32_t SEL_REST = 256, SEL_WG = 1024, SEL_LANES = 8;
constexpr uint32_t SEL_ROUNDS = 60000;         // stamps hold 16 bits of round

__global__ void k_sel_elim(int32_t nCand, const Plan *__restrict__ plans, uint8_t *state,
                           const uint32_t *__restrict__ mk, uint32_t *activeLeft, uint32_t *list) {
    int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (c >= nCand || state[c] != ST_ACTIVE) return;
    const Plan &p = plans[c];
    bool conf = false;
    for (int i = 0; i < p.nW && !conf; i++) {
        uint32_t m = mk[p.W[i]];
        if (m & (MK_W | MK_M)) conf = true;
        if (p.W[i] != p.id && (m & MK_L)) conf = true;
    }
    for (int i = 0; i < p.nL && !conf; i++)
        if (mk[p.L[i]] & MK_WNR) conf = true;
    for (int i = 0; i < p.nM && !conf; i++)
        if (mk[p.M[i]] & MK_W) conf = true;
    if (conf) { state[c] = ST_REJECTED; return; }
    const uint32_t k = atomicAdd(activeLeft, 1u);
    if (k < SEL_REST) list[k] = (uint32_t)c;
}

// All remaining rounds of the selection by one workgroup, once at most SEL_REST
// candidates are active (multipliers need 10 to 15 rounds, most of them for a
// few).  The candidates are in LDS, eight lanes share one's nodes.  Claims and
// marks are updated by atomics and read past the L1, which does not see them.
// What bounds it: a round is some trips to memory between three barriers, about
// 10 us; three kernels and the host's look at the count took 45.  With more
// candidates left the whole device is faster (at 2048 a burst of 32 requests
// lost 4 ms).
__global__ void __launch_bounds__(SEL_WG) k_sel_rest(uint32_t round, uint32_t n, const uint32_t *__restrict__ list,
                                                     const Plan *__restrict__ plans, uint8_t *state, Claims cl,
                                                     uint32_t *mk, uint32_t *out) {
    __shared__ uint32_t s_list[2][SEL_REST];
    __shared__ uint8_t s_won[SEL_REST];
    __shared__ uint32_t s_n;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, sub = tid % SEL_LANES;
    const uint64_t group = 0xFFull << (lane - lane % SEL_LANES);
    if (tid < n) s_list[0][tid] = list[tid];
    __syncthreads();
    auto ld = [](const unsigned long long *q) {
        return __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    auto ldm = [](const uint32_t *q) { return __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
    // a barrier that this wavefront's memory operations have passed
    auto settle = []() {
        __builtin_amdgcn_s_waitcnt(0x0070);     // vmcnt(0), lgkmcnt(0)
        __syncthreads();
    };
    for (uint32_t b = 0; n != 0 && round < SEL_ROUNDS; round++, b ^= 1u) {
        // node e of a plan: 0 of W, 1 of L, 2 of M
        auto node = [](const Plan &q, int e, int &kind) -> int {
            if (e < q.nW) { kind = 0; return q.W[e]; }
            e -= q.nW;
            if (e < q.nL) { kind = 1; return q.L[e]; }
            kind = 2;
            return q.M[e - q.nL];
        };
        for (uint32_t k = tid / SEL_LANES; k < n; k += SEL_WG / SEL_LANES) {
            const Plan &q = plans[s_list[b][k]];
            const unsigned long long st = stamp(round, q);
            for (int e = (int)sub, all = q.nW + q.nL + q.nM; e < all; e += (int)SEL_LANES) {
                int kind;
                const int x = node(q, e, kind);
                if (kind == 0) {
                    atomicMax(&cl.W[x], st);
                    if (x != q.id) atomicMax(&cl.Wnr[x], st);
                } else {
                    atomicMax(kind == 1 ? &cl.L[x] : &cl.M[x], st);
                }
            }
            if (sub == 0) s_won[k] = 0;
        }
        settle();
        for (uint32_t k0 = 0; k0 < n; k0 += SEL_WG / SEL_LANES) {
            const uint32_t k = k0 + tid / SEL_LANES;
            bool lost = k >= n;
            if (!lost) {
                const Plan &q = plans[s_list[b][k]];
                const unsigned long long st = stamp(round, q);
                for (int e = (int)sub, all = q.nW + q.nL + q.nM; e < all; e += (int)SEL_LANES) {
                    int kind;
                    const int x = node(q, e, kind);
                    if (kind == 0) lost |= ld(&cl.W[x]) != st || ld(&cl.M[x]) >= st || (x != q.id && ld(&cl.L[x]) >= st);
                    else lost |= ld(kind == 1 ? &cl.Wnr[x] : &cl.W[x]) >= st;
                }
            }
            const bool win = (__ballot(lost) & group) == 0;
            if (k < n && win) {
                const uint32_t c = s_list[b][k];
                const Plan &q = plans[c];
                if (sub == 0) { s_won[k] = 1; state[c] = ST_SELECTED; }
                for (int e = (int)sub, all = q.nW + q.nL + q.nM; e < all; e += (int)SEL_LANES) {
                    int kind;
                    const int x = node(q, e, kind);
                    atomicOr(&mk[x], kind == 0 ? MK_W | (x != q.id ? MK_WNR : 0u) : kind == 1 ? (uint32_t)MK_L : (uint32_t)MK_M);
                }
            }
        }
        if (tid == 0) s_n = 0;
        settle();
        for (uint32_t k0 = 0; k0 < n; k0 += SEL_WG / SEL_LANES) {
            const uint32_t k = k0 + tid / SEL_LANES;
            const bool open = k < n && !s_won[k];
            bool conf = false;
            if (open) {
                const Plan &q = plans[s_list[b][k]];
                for (int e = (int)sub, all = q.nW + q.nL + q.nM; e < all; e += (int)SEL_LANES) {
                    int kind;
                    const int x = node(q, e, kind);
                    const uint32_t m = ldm(&mk[x]);
                    conf |= (m & (kind == 0 ? MK_W | MK_M | (x != q.id ? MK_L : 0u) : kind == 1 ? (uint32_t)MK_WNR : (uint32_t)MK_W)) != 0;
                }
            }
            const bool out1 = (__ballot(conf) & group) != 0;
            if (open && sub == 0) {
                const uint32_t c = s_list[b][k];
                if (out1) state[c] = ST_REJECTED;
                else s_list[b ^ 1u][atomicAdd(&s_n, 1u)] = c;
            }
        }
        settle();
        n = s_n;
    }
    if (tid == 0) { out[0] = round; out[1] = n; }
}

// cnt: new nodes per candidate (0 past the last); sum: the selected ones' gain
// and number
__global__ void k_new_counts(int32_t nCand, const Plan *__restrict__ plans, const uint8_t *__restrict__ state,
                             uint32_t *cnt, unsigned long long *sum) {
    int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (c == nCand) cnt[c] = 0;
    const bool s = c < nCand && state[c] == ST_SELECTED;
    const uint64_t m = __ballot(s);
    if (m && (threadIdx.x & 63u) == 0) atomicAdd(&sum[1], (unsigned long long)__popcll(m));
    if (c >= nCand) return;
    cnt[c] = s ? (uint32_t)plans[c].nNew : 0u;
    if (s) atomicAdd(&sum[0], (unsigned long long)plans[c].gain);
}

__global__ void k_no_candidate(int32_t n, int4 *best) {
    const int32_t v = (int32_t)(blockIdx.x * blockDim.x + threadIdx.x);
    if (v < n) best[v] = make_int4(-1, 0, 0, 0);
}

__global__ void k_iota2(int32_t n, uint32_t *repl) {
    int64_t tid = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t v = tid; v < n; v += stride) repl[v] = 2u * (uint32_t)v;
}

// Creates the new nodes of each selected plan at ids n + off[c] + k, in
// ascending library index order, and records the replacement literal.
__global__ void __launch_bounds__(EVAL_BLOCK) k_build(int32_t per, int32_t n, int32_t nCand, const uint32_t *__restrict__ candIds,
                                                       GraphView g, Lib L, const uint32_t *__restrict__ cuts,
                                                       const int4 *__restrict__ best, const uint8_t *__restrict__ state,
                                                       const uint32_t *__restrict__ off, uint32_t *cf0, uint32_t *cf1,
                                                       uint32_t *repl, uint32_t *err, uint32_t *ctag) {
    __shared__ int32_t s_match[NMATCH * EVAL_BLOCK], s_mlev[NMATCH * EVAL_BLOCK];
    int64_t c = blockIdx.x * (int64_t)per + threadIdx.x;
    if ((int32_t)threadIdx.x >= per || c >= nCand || state[c] != ST_SELECTED) return;
    Col match{s_match + threadIdx.x}, mlev{s_mlev + threadIdx.x};
    const int id = (int)candIds[c];
    const int4 b = best[id];
    const uint32_t *p = cuts + ((size_t)id * NCUT + b.x) * 5;
    Mffc t;
    PlanCore pc = plan_core(g, L, id, p, b.y, t, match, mlev);
    uint32_t next = (uint32_t)n + off[c];
    for (int j = 4; j <= pc.rt; j++) {
        if (!((pc.addMask >> j) & 1)) continue;
        if (ctag) ctag[next] = ctag[id];   // a new node carries its root's tag
        uint32_t wd = lib_word(L, pc.cls, j - 4);
        int a = wd & 63, bb = (wd >> 6) & 63;
        if (match[a] < 0 || match[bb] < 0) {  // cannot happen for a consistent plan
            atomicOr(err, 2u);
            cf0[next] = 0;
            cf1[next] = 0;
            match[j] = (int32_t)next;
            next++;
            continue;
        }
        uint32_t la = 2u * (uint32_t)match[a] + (isc_bit(pc.isC, a) ^ ((wd >> 12) & 1u));
        uint32_t lb = 2u * (uint32_t)match[bb] + (isc_bit(pc.isC, bb) ^ ((wd >> 13) & 1u));
        cf0[next] = la;
        cf1[next] = lb;
        match[j] = (int32_t)next;
        next++;
    }
    repl[id] = 2u * (uint32_t)match[pc.rt] + (uint32_t)pc.compl_;
}

__global__ void k_compose(int32_t n, int32_t N, int32_t nPIs, const uint32_t *__restrict__ f0,
                          const uint32_t *__restrict__ f1, const uint32_t *__restrict__ repl, uint32_t *cf0,
                          uint32_t *cf1) {
    int64_t tid = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t v = tid; v < N; v += stride) {
        if (v <= nPIs) { cf0[v] = 0; cf1[v] = 0; continue; }
        uint32_t a = v < n ? f0[v] : cf0[v], b = v < n ? f1[v] : cf1[v];
        uint32_t ia = LID(a), ib = LID(b);
        cf0[v] = (ia < (uint32_t)n ? repl[ia] : 2u * ia) ^ LC(a);
        cf1[v] = (ib < (uint32_t)n ? repl[ib] : 2u * ib) ^ LC(b);
    }
}

__global__ void k_compose_pos(int32_t nPOs, const uint32_t *__restrict__ pos, const uint32_t *__restrict__ repl,
                              uint32_t *cpos) {
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i < nPOs) cpos[i] = repl[LID(pos[i])] ^ LC(pos[i]);
}

__global__ void k_flag_cand(int32_t n, const int4 *__restrict__ best, uint8_t *flag) {
    int64_t v = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (v < n) flag[v] = best[v].x >= 0;
}

// reorder: new position of every node, fanins remapped and sorted
__global__ void k_reorder_ids(int32_t m, const uint32_t *__restrict__ sortedIds, uint32_t *newId) {
    int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (p == 0) newId[0] = 0;
    if (p < m) newId[sortedIds[p]] = (uint32_t)(p + 1);
}

__global__ void k_reorder_emit(int32_t n, int32_t nPIs, const uint32_t *__restrict__ f0,
                               const uint32_t *__restrict__ f1, const uint32_t *__restrict__ level,
                               const uint32_t *__restrict__ newId, uint32_t *of0, uint32_t *of1, uint32_t *olevel,
                               const uint32_t *__restrict__ tagIn, uint32_t *tagOut) {
    int64_t v = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (v >= n) return;
    uint32_t nv = newId[v];
    olevel[nv] = level[v];
    if (tagOut) tagOut[nv] = tagIn[v];
    if (v <= nPIs) { of0[nv] = 0; of1[nv] = 0; return; }
    uint32_t a = 2u * newId[LID(f0[v])] | LC(f0[v]);
    uint32_t b = 2u * newId[LID(f1[v])] | LC(f1[v]);
    if (a > b) { uint32_t x = a; a = b; b = x; }
    of0[nv] = a;
    of1[nv] = b;
}

__global__ void k_reorder_pos(int32_t nPOs, const uint32_t *__restrict__ pos, const uint32_t *__restrict__ newId,
                              uint32_t *opos) {
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i < nPOs) opos[i] = 2u * newId[LID(pos[i])] | LC(pos[i]);
}

__global__ void k_level_starts(int32_t m, const uint32_t *__restrict__ keys, int32_t *starts) {
    int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (p >= m) return;
    if (p == 0 || keys[p] != keys[p - 1]) starts[keys[p]] = (int32_t)(p + 1);
}

__global__ void k_iota1(int32_t m, uint32_t *x) {
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i < m) x[i] = (uint32_t)(i + 1);
}

__global__ void k_gather_level(int32_t m, const uint32_t *__restrict__ level, uint32_t *keys) {
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i < m) keys[i] = level[i + 1];
}

struct Tmp {
    gls_ctx *ctx;
    std::vector<void *> ptrs;
    bool ok = true;
    template <class T> T *get(size_t n) {
        T *p = pool_get<T>(ctx, n);
        if (p) ptrs.push_back(p);
        else ok = false;
        return p;
    }
    ~Tmp() {
        for (void *p : ptrs) pool_put(ctx, p);
    }
};

// Owns a pool-backed graph until it is freed explicitly or the scope ends.
struct GraphGuard {
    gls_ctx *ctx;
    DevGraph *g;
    void free_now() {
        if (g) dev_graph_free(ctx, *g);
        g = nullptr;
    }
    ~GraphGuard() { free_now(); }
};

int blocks(int64_t n, int b) { return (int)((n + b - 1) / b > 0 ? (n + b - 1) / b : 1); }

uint32_t bits_for(uint32_t x) {
    uint32_t b = 1;
    while (b < 32 && (x >> b) != 0) ++b;
    return b;
}

Lib lib_of(gls_ctx *ctx) {
    return Lib{ctx->d_npn, ctx->d_perms4, ctx->d_lib_nodes, ctx->d_lib_node_off, ctx->d_lib_root_off, ctx->d_lib_roots};
}

// Stage timer of a pass (diagnostics only): an event call that fails makes
// every stage time read 0 instead of failing the pass.
struct Timer {
    gls_ctx *ctx;
    int next = 0;
    bool ok = true;
    void mark() {
        if (next < 16) {
            if (hipEventRecord(ctx->ev[next], ctx->stream) != hipSuccess) ok = false;
            ++next;
        }
    }
    double ms(int a, int b) {
        float x = 0;
        if (!ok || b >= next || hipEventElapsedTime(&x, ctx->ev[a], ctx->ev[b]) != hipSuccess) return 0.0;
        return x;
    }
};

} // namespace

// Signature bits of a batched pass: every node's id in its own AIG, & 31.
// Nodes 1..n-1 sorted stably by tag keep their id order inside each tag; in
// the reordered numbering an AIG's PIs come first, then its ANDs level-major
// (ties by id), exactly as its own reordered numbering, so the rank inside the
// tag group + 1 is that id.
__global__ void __launch_bounds__(kBlock) k_sig_keys(int32_t n, const uint32_t *__restrict__ tag, uint32_t *keys,
                                                     uint32_t *vals, uint32_t *hist) {
    __shared__ uint32_t s_bins[TAG_BINS];
    TagBins tb{s_bins};
    tb.init();
    int64_t b, e;
    tag_chunk(1, n, b, e);
    for (int64_t u = b + threadIdx.x; u < e; u += blockDim.x) {
        const uint32_t k = tag[u];
        keys[u - 1] = k;
        vals[u - 1] = (uint32_t)u;
        tb.add(hist, k, 1u);
    }
    tb.flush_add(hist, 0xFFFFFFFFu);
}

__global__ void k_sig_bits(int32_t m, const uint32_t *__restrict__ skeys, const uint32_t *__restrict__ svals,
                           const uint32_t *__restrict__ start, uint8_t *sigBits) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < m; q += stride)
        sigBits[svals[q]] = (uint8_t)((1u + (uint32_t)(q - start[skeys[q]])) & 31u);
    if (blockIdx.x == 0 && threadIdx.x == 0) sigBits[0] = 0;
}

static int sig_bits_for_tags(gls_ctx *ctx, int32_t n, const uint32_t *tag, uint8_t *sigBits) {
    hipStream_t st = ctx->stream;
    const int32_t m = n - 1;
    if (m <= 0) return GLS_OK;
    Tmp t{ctx};
    uint32_t *mx = t.get<uint32_t>(1);
    size_t tb = 0;
    GLS_HIP(ctx, rocprim::reduce(nullptr, tb, tag, mx, 0u, (size_t)n, rocprim::maximum<uint32_t>(), st));
    void *tmp = t.get<uint8_t>(tb);
    if (!mx || !tmp) return gls_fail(ctx, GLS_ERR_NOMEM, "signature bits: allocation");
    GLS_HIP(ctx, rocprim::reduce(tmp, tb, tag, mx, 0u, (size_t)n, rocprim::maximum<uint32_t>(), st));
    uint32_t maxTag = 0;
    GLS_TRY(stream_copy(ctx, &maxTag, mx, sizeof(uint32_t), hipMemcpyDeviceToHost));
    uint32_t *keys = t.get<uint32_t>(m), *vals = t.get<uint32_t>(m), *skeys = t.get<uint32_t>(m);
    uint32_t *svals = t.get<uint32_t>(m), *hist = t.get<uint32_t>(maxTag + 2), *start = t.get<uint32_t>(maxTag + 2);
    if (!t.ok) return gls_fail(ctx, GLS_ERR_NOMEM, "signature bits: allocation");
    GLS_TRY(Fills(ctx).add(hist, 0, sizeof(uint32_t) * (maxTag + 2)).run());
    k_sig_keys<<<tag_grid(m), kBlock, 0, st>>>(n, tag, keys, vals, hist);
    size_t tb2 = 0;
    const uint32_t eb = bits_for(maxTag + 1);
    GLS_HIP(ctx, rocprim::radix_sort_pairs(nullptr, tb2, keys, skeys, vals, svals, (size_t)m, 0u, eb, st));
    size_t tb3 = 0;
    GLS_HIP(ctx, rocprim::exclusive_scan(nullptr, tb3, hist, start, 0u, (size_t)maxTag + 1, rocprim::plus<uint32_t>(), st));
    void *tmp2 = t.get<uint8_t>(std::max(tb2, tb3));
    if (!tmp2) return gls_fail(ctx, GLS_ERR_NOMEM, "signature bits: sort storage");
    GLS_HIP(ctx, rocprim::radix_sort_pairs(tmp2, tb2, keys, skeys, vals, svals, (size_t)m, 0u, eb, st));
    GLS_HIP(ctx, rocprim::exclusive_scan(tmp2, tb3, hist, start, 0u, (size_t)maxTag + 1, rocprim::plus<uint32_t>(), st));
    k_sig_bits<<<grid_for(m), kBlock, 0, st>>>(m, skeys, svals, start, sigBits);
    GLS_HIP(ctx, hipGetLastError());
    GLS_HIP(ctx, hipStreamSynchronize(st));
    return GLS_OK;
}

int dev_reorder(gls_ctx *ctx, const DevGraph &in, DevGraph &out, std::vector<int32_t> &levelStart,
                const uint32_t *tagIn, uint32_t **tagOut) {
    const int32_t n = in.nObjs, m = n - 1;
    hipStream_t st = ctx->stream;
    Tmp t{ctx};
    uint32_t *keys = t.get<uint32_t>(m + 1), *keys2 = t.get<uint32_t>(m + 1), *ids = t.get<uint32_t>(m + 1);
    uint32_t *ids2 = t.get<uint32_t>(m + 1), *newId = t.get<uint32_t>(n);
    if (!t.ok) return gls_fail(ctx, GLS_ERR_NOMEM, "reorder: allocation");
    uint32_t maxLevel = 0;
    GLS_TRY(dev_graph_alloc(ctx, out, n, in.nPIs, in.nPOs));
    GraphGuard outGuard{ctx, &out};   // released to the caller on success
    uint32_t *tags = nullptr;
    if (tagIn && tagOut) {
        tags = pool_get<uint32_t>(ctx, (size_t)n);
        if (!tags) return gls_fail(ctx, GLS_ERR_NOMEM, "reorder: tags");
        *tagOut = tags;
    }
    if (m > 0) {
        k_gather_level<<<blocks(m, kBlock), kBlock, 0, st>>>(m, in.level, keys);
        k_iota1<<<blocks(m, kBlock), kBlock, 0, st>>>(m, ids);
        size_t tb = 0;
        GLS_HIP(ctx, rocprim::reduce(nullptr, tb, keys, keys2, 0u, (size_t)m, rocprim::maximum<uint32_t>(), st));
        void *tmp = t.get<uint8_t>(tb);
        if (!tmp) return gls_fail(ctx, GLS_ERR_NOMEM, "reorder: reduce storage");
        GLS_HIP(ctx, rocprim::reduce(tmp, tb, keys, keys2, 0u, (size_t)m, rocprim::maximum<uint32_t>(), st));
        GLS_TRY(stream_copy(ctx, &maxLevel, keys2, sizeof(uint32_t), hipMemcpyDeviceToHost));
        size_t tb2 = 0;
        uint32_t eb = bits_for(maxLevel);
        GLS_HIP(ctx, rocprim::radix_sort_pairs(nullptr, tb2, keys, keys2, ids, ids2, (size_t)m, 0u, eb, st));
        void *tmp2 = t.get<uint8_t>(tb2);
        if (!tmp2) return gls_fail(ctx, GLS_ERR_NOMEM, "reorder: sort storage");
        GLS_HIP(ctx, rocprim::radix_sort_pairs(tmp2, tb2, keys, keys2, ids, ids2, (size_t)m, 0u, eb, st));
        k_reorder_ids<<<blocks(m, kBlock), kBlock, 0, st>>>(m, ids2, newId);
        int32_t *d_starts = t.get<int32_t>(maxLevel + 2);
        if (!d_starts) return gls_fail(ctx, GLS_ERR_NOMEM, "reorder: starts");
        GLS_TRY(Fills(ctx).add(d_starts, 0, sizeof(int32_t) * (maxLevel + 2)).run());
        k_level_starts<<<blocks(m, kBlock), kBlock, 0, st>>>(m, keys2, d_starts);
        levelStart.assign(maxLevel + 2, 0);
        k_reorder_emit<<<blocks(n, kBlock), kBlock, 0, st>>>(n, in.nPIs, in.f0, in.f1, in.level, newId, out.f0,
                                                              out.f1, out.level, tagIn, tags);
        if (in.nPOs > 0)
            k_reorder_pos<<<blocks(in.nPOs, kBlock), kBlock, 0, st>>>(in.nPOs, in.pos, newId, out.pos);
        GLS_HIP(ctx, hipGetLastError());
        GLS_TRY(stream_copy(ctx, levelStart.data(), d_starts, sizeof(int32_t) * (maxLevel + 1), hipMemcpyDeviceToHost));
        levelStart[maxLevel + 1] = n;  // one past the last id
    } else {
        GLS_TRY(Fills(ctx)
                    .add(out.f0, 0, sizeof(uint32_t) * n)
                    .add(out.f1, 0, sizeof(uint32_t) * n)
                    .add(out.level, 0, sizeof(uint32_t) * n)
                    .run());
        if (in.nPOs > 0)
            GLS_HIP(ctx, hipMemcpyAsync(out.pos, in.pos, sizeof(uint32_t) * in.nPOs, hipMemcpyDeviceToDevice, st));
        if (tags) GLS_HIP(ctx, hipMemcpyAsync(tags, tagIn, sizeof(uint32_t) * n, hipMemcpyDeviceToDevice, st));
        GLS_HIP(ctx, hipStreamSynchronize(st));
        levelStart.assign(2, n);
    }
    outGuard.g = nullptr;
    return GLS_OK;
}

// per-level cut launches are timed in windows (see dev_enumerate_cuts)
// (GLS_KERNEL_SAMPLE=0 in the environment turns this off, e.g. under a
// profiler that collects counters per dispatch)
static constexpr int KSAMPLE_EVERY = 64;
static constexpr int KSAMPLE_WIN = 8;
static const bool kSampleLaunches = [] {
    const char *e = getenv("GLS_KERNEL_SAMPLE");
    return !(e && e[0] == '0');
}();

// Task lists of the planned schedule for nL launches of K levels each (lv:
// per launch the first ids of its K levels, then its end; K + 1 entries):
// heads / ents on the device, toff[j] = first task of launch j on the host
// (nL + 1 entries).  lv must stay alive until this returns (its upload is
// complete by then).
static int build_cut_plan(gls_ctx *ctx, Tmp &t, const DevGraph &g, int32_t K, const std::vector<int32_t> &lv,
                          uint4 *&heads, uint4 *&ents, std::vector<uint32_t> &toff) {
    hipStream_t st = ctx->stream;
    const int32_t n = g.nObjs, nL = (int32_t)(lv.size() / (size_t)(K + 1));
    int32_t *dlv = t.get<int32_t>(lv.size());
    int32_t *nodeLaunch = t.get<int32_t>((size_t)n);
    uint32_t *own = t.get<uint32_t>((size_t)n);
    uint8_t *coneSize = t.get<uint8_t>((size_t)n);
    unsigned long long *flag = t.get<unsigned long long>((size_t)n + 1);
    unsigned long long *S = t.get<unsigned long long>((size_t)n + 1);
    uint32_t *cnt = t.get<uint32_t>((size_t)nL + 1), *dOff = t.get<uint32_t>((size_t)nL + 1);
    if (!t.ok) return gls_fail(ctx, GLS_ERR_NOMEM, "cuts: plan storage");
    GLS_HIP(ctx, hipMemcpyAsync(dlv, lv.data(), sizeof(int32_t) * lv.size(), hipMemcpyHostToDevice, st));
    GLS_TRY(Fills(ctx)
                .add(nodeLaunch, 0xFF, sizeof(int32_t) * (size_t)n)
                .add(own, 0xFF, sizeof(uint32_t) * (size_t)n)
                .run());
    k_plan_fill<<<nL, kBlock, 0, st>>>(K, dlv, nodeLaunch);
    for (int p = K - 1; p >= 1; p--)
        k_plan_roots<<<grid_for(n), kBlock, 0, st>>>(n, g.nPIs, K, p, g.f0, g.f1, dlv, nodeLaunch, own, coneSize);
    k_plan_flags<<<grid_for((int64_t)n + 1), kBlock, 0, st>>>(n, K, dlv, nodeLaunch, own, flag);
    GLS_HIP(ctx, hipGetLastError());
    size_t tb = 0, tb2 = 0;
    GLS_HIP(ctx, rocprim::exclusive_scan(nullptr, tb, flag, S, 0ull, (size_t)n + 1,
                                         rocprim::plus<unsigned long long>(), st));
    GLS_HIP(ctx, rocprim::exclusive_scan(nullptr, tb2, cnt, dOff, 0u, (size_t)nL + 1, rocprim::plus<uint32_t>(), st));
    void *tmp = t.get<uint8_t>(std::max<size_t>(std::max(tb, tb2), 1));
    if (!tmp) return gls_fail(ctx, GLS_ERR_NOMEM, "cuts: plan scan storage");
    GLS_HIP(ctx, rocprim::exclusive_scan(tmp, tb, flag, S, 0ull, (size_t)n + 1, rocprim::plus<unsigned long long>(),
                                         st));
    k_plan_counts<<<blocks(nL + 1, kBlock), kBlock, 0, st>>>(nL, K, dlv, S, cnt);
    GLS_HIP(ctx, rocprim::exclusive_scan(tmp, tb2, cnt, dOff, 0u, (size_t)nL + 1, rocprim::plus<uint32_t>(), st));
    toff.assign((size_t)nL + 1, 0u);
    GLS_TRY(stream_copy(ctx, toff.data(), dOff, sizeof(uint32_t) * ((size_t)nL + 1), hipMemcpyDeviceToHost));
    const size_t nT = toff[nL];
    uint32_t *ecnt = t.get<uint32_t>(nT + 1), *eoff = t.get<uint32_t>(nT + 1);
    heads = t.get<uint4>(std::max<size_t>(nT, 1));
    size_t tb3 = 0;
    GLS_HIP(ctx, rocprim::exclusive_scan(nullptr, tb3, ecnt, eoff, 0u, nT + 1, rocprim::plus<uint32_t>(), st));
    void *tmp3 = t.get<uint8_t>(std::max<size_t>(tb3, 1));
    if (!ecnt || !eoff || !heads || !tmp3) return gls_fail(ctx, GLS_ERR_NOMEM, "cuts: plan tasks (%zu)", nT);
    GLS_TRY(Fills(ctx).add(ecnt, 0, sizeof(uint32_t) * (nT + 1)).run());
    k_plan_ecount<<<grid_for(n), kBlock, 0, st>>>(n, g.nPIs, K, dlv, nodeLaunch, own, S, dOff, coneSize, ecnt);
    GLS_HIP(ctx, rocprim::exclusive_scan(tmp3, tb3, ecnt, eoff, 0u, nT + 1, rocprim::plus<uint32_t>(), st));
    // entries: every node once as a root or packed node, plus the cone
    // members recomputed by other roots; bounded by the cone sizes' sum
    uint32_t nE = 0;
    GLS_TRY(stream_copy(ctx, &nE, eoff + nT, sizeof(uint32_t), hipMemcpyDeviceToHost));
    ents = t.get<uint4>(std::max<size_t>(nE, 1));
    if (!ents) return gls_fail(ctx, GLS_ERR_NOMEM, "cuts: plan entries (%u)", nE);
    k_plan_scatter<<<grid_for(n), kBlock, 0, st>>>(n, g.nPIs, K, g.f0, g.f1, dlv, nodeLaunch, own, S, dOff, eoff,
                                                   heads, ents);
    GLS_HIP(ctx, hipGetLastError());
    return GLS_OK;
}

int dev_enumerate_cuts(gls_ctx *ctx, const DevGraph &g, const std::vector<int32_t> &levelStart, uint32_t *d_cuts,
                       int32_t *d_nref, int mode, const uint8_t *sigBits, int *ranMode) {
    int ranDummy = 0;
    int &ran = ranMode ? *ranMode : ranDummy;
    ran = 0;
    hipStream_t st = ctx->stream;
    const int32_t n = g.nObjs;
    ctx->ksamp_n = 0;
    ctx->ksamp_units.clear();
    ctx->ksamp_launches.clear();
    ctx->cut_graph_ms = 0;
    ctx->cut_graph_nodes = 0;
    // The planned schedule is switched off: its kernel made an illegal memory
    // access on the GPU in the schedule tests, also after its LDS records were
    // written through LDS pointers with a wait before each barrier, and the
    // cause is not found (the task lists pass every bounds check in a host
    // build of the plan kernels).  It is refused before anything is launched.
    if (mode & GLS_RW_PLAN_CUTS)
        return gls_fail(ctx, GLS_ERR_ARG, "GLS_RW_PLAN_CUTS is disabled (its kernel faulted the GPU; cause not found)");
    const bool graphed = (mode & GLS_RW_GRAPH_CUTS) != 0;
    mode &= ~GLS_RW_GRAPH_CUTS;
    GLS_TRY(Fills(ctx)
                .add(d_nref, 0, sizeof(int32_t) * n)
                .add(d_cuts, 0, sizeof(uint32_t) * (size_t)n * NCUT * 5)
                .run());
    k_nref<<<grid_for(n), kBlock, 0, st>>>(n, g.nPIs, g.f0, g.f1, g.nPOs, g.pos, d_nref);
    if (g.nPIs > 0) k_cuts_pi<<<blocks(g.nPIs, kBlock), kBlock, 0, st>>>(g.nPIs, d_nref, d_cuts);
    // levelStart[l] = first id of level l (ids 1.. are level-major); the last
    // entry is one past the last id.
    const int L = (int)levelStart.size() - 1;
    if (L <= 1) return GLS_OK;
    if (mode == GLS_RW_DATAFLOW_CUTS && L > 16) {
        int perCU = 0, dev = 0, nCU = 0;
        GLS_HIP(ctx, hipGetDevice(&dev));
        GLS_HIP(ctx, hipDeviceGetAttribute(&nCU, hipDeviceAttributeMultiprocessorCount, dev));
        GLS_HIP(ctx, hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCU, k_cuts_dataflow, CUTW_BLOCK, 0));
        const int G = std::max(1, std::min(perCU, 2) * nCU);
        const size_t nslots = (size_t)n * NCUT;
        unsigned long long *tcuts = pool_get<unsigned long long>(ctx, nslots * 3);
        uint32_t *ctr = pool_get<uint32_t>(ctx, 4);
        if (!tcuts || !ctr) { pool_put(ctx, tcuts); pool_put(ctx, ctr); return gls_fail(ctx, GLS_ERR_NOMEM, "cuts: tagged records"); }
        GLS_TRY(Fills(ctx)
                    .add(tcuts, 0, sizeof(unsigned long long) * nslots * 3)
                    .add(ctr, 0, sizeof(uint32_t) * 4)
                    .run());
        if (g.nPIs > 0)
            k_cuts_pi_tagged<<<blocks((int64_t)g.nPIs * NCUT, kBlock), kBlock, 0, st>>>(g.nPIs, d_nref, tcuts);
        k_cuts_dataflow<<<G, CUTW_BLOCK, 0, st>>>(g.nPIs + 1, n, g.f0, g.f1, d_nref, tcuts, &ctr[0], &ctr[1],
                                                   sigBits);
        k_untag_cuts<<<grid_for((int64_t)nslots), kBlock, 0, st>>>((int64_t)nslots, tcuts, d_cuts);
        GLS_HIP(ctx, hipGetLastError());
        uint32_t hctr[2] = {0, 0};
        int rc = stream_copy(ctx, hctr, ctr, sizeof(hctr), hipMemcpyDeviceToHost);
        pool_put(ctx, tcuts);
        pool_put(ctx, ctr);
        if (rc != GLS_OK) return rc;
        if (hctr[1]) return gls_fail(ctx, GLS_ERR_INTERNAL, "cut enumeration: a wait exceeded its bound");
        // every node must have been taken (a wavefront stops once tickets pass the end)
        if (hctr[0] < (uint32_t)(n - g.nPIs - 1))
            return gls_fail(ctx, GLS_ERR_INTERNAL, "cut enumeration: %u of %d nodes processed", hctr[0],
                            n - g.nPIs - 1);
        ran = GLS_RW_DATAFLOW_CUTS;
        return GLS_OK;
    }
    if (mode == GLS_RW_XCD_CUTS && L > 16) {
        int dev = 0, nCU = 0;
        GLS_HIP(ctx, hipGetDevice(&dev));
        GLS_HIP(ctx, hipDeviceGetAttribute(&nCU, hipDeviceAttributeMultiprocessorCount, dev));
        const uint32_t nwg = (uint32_t)(nCU / XCD_COUNT);
        int32_t *d_starts = pool_get<int32_t>(ctx, levelStart.size());
        uint32_t *ctl = pool_get<uint32_t>(ctx, 4);
        if (!d_starts || !ctl) { pool_put(ctx, d_starts); pool_put(ctx, ctl); return gls_fail(ctx, GLS_ERR_NOMEM, "cuts: xcd control"); }
        GLS_HIP(ctx, hipMemcpyAsync(d_starts, levelStart.data(), sizeof(int32_t) * levelStart.size(),
                                    hipMemcpyHostToDevice, st));
        GLS_TRY(Fills(ctx).add(ctl, 0, sizeof(uint32_t) * 4).run());
        const dim3 grid((unsigned)(nwg * XCD_COUNT));
        if (kSampleLaunches) {
            const size_t k = 2 * (size_t)ctx->ksamp_n;
            while (ctx->kev.size() < k + 2) {
                hipEvent_t ev = nullptr;
                GLS_HIP(ctx, hipEventCreate(&ev));
                ctx->kev.push_back(ev);
            }
            hipExtLaunchKernelGGL(k_cuts_xcd, grid, dim3(XCD_WG), 0, st, ctx->kev[k], ctx->kev[k + 1], 0, 1, L,
                                  (const int32_t *)d_starts, (const uint32_t *)g.f0, (const uint32_t *)g.f1,
                                  (const int32_t *)d_nref, d_cuts, sigBits, nwg, ctl);
            ctx->ksamp_units.push_back(levelStart[L] - levelStart[1]);
            ctx->ksamp_launches.push_back(1);
            ctx->ksamp_n++;
        } else {
            k_cuts_xcd<<<grid, XCD_WG, 0, st>>>(1, L, d_starts, g.f0, g.f1, d_nref, d_cuts, sigBits, nwg, ctl);
        }
        GLS_HIP(ctx, hipGetLastError());
        uint32_t hctl[3] = {0, 0, 0};
        const int rc = stream_copy(ctx, hctl, ctl, sizeof(hctl), hipMemcpyDeviceToHost);
        pool_put(ctx, d_starts);
        pool_put(ctx, ctl);
        if (rc != GLS_OK) return rc;
        if (hctl[2] == 0) {
            ran = GLS_RW_XCD_CUTS;
            return GLS_OK;
        }
        // not all on one XCD, or a wait overran: redo with one launch per level
        ctx->ksamp_n = 0;
        ctx->ksamp_units.clear();
        ctx->ksamp_launches.clear();
        GLS_TRY(Fills(ctx).add(d_cuts, 0, sizeof(uint32_t) * (size_t)n * NCUT * 5).run());
        if (g.nPIs > 0) k_cuts_pi<<<blocks(g.nPIs, kBlock), kBlock, 0, st>>>(g.nPIs, d_nref, d_cuts);
        mode = 0;
    }
    bool coop = mode == GLS_RW_COOP_CUTS && L > 16;
    int G = 0;
    if (coop) {
        int perCU = 0, dev = 0, nCU = 0, coopOk = 0;
        GLS_HIP(ctx, hipGetDevice(&dev));
        GLS_HIP(ctx, hipDeviceGetAttribute(&nCU, hipDeviceAttributeMultiprocessorCount, dev));
        GLS_HIP(ctx, hipDeviceGetAttribute(&coopOk, hipDeviceAttributeCooperativeLaunch, dev));
        GLS_HIP(ctx, hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCU, k_cuts_levels, CUTW_BLOCK, 0));
        G = std::min(perCU * nCU, 64);
        coop = coopOk && G > 0;
    }
    if (coop) {
        int32_t *d_starts = pool_get<int32_t>(ctx, levelStart.size());
        if (!d_starts) return gls_fail(ctx, GLS_ERR_NOMEM, "cuts: level starts");
        GLS_HIP(ctx, hipMemcpyAsync(d_starts, levelStart.data(), sizeof(int32_t) * levelStart.size(),
                                    hipMemcpyHostToDevice, st));
        int32_t l0 = 1, l1 = L;
        const uint32_t *a0 = g.f0, *a1 = g.f1;
        const int32_t *ar = d_nref;
        uint32_t *ac = d_cuts;
        const uint8_t *sb = sigBits;
        void *args[] = {&l0, &l1, &d_starts, &a0, &a1, &ar, &ac, &sb};
        hipError_t e = hipLaunchCooperativeKernel((const void *)k_cuts_levels, dim3(G), dim3(CUTW_BLOCK), args, 0, st);
        // the pool block is reused only by later work on the same stream
        pool_put(ctx, d_starts);
        if (e != hipSuccess) return gls_fail(ctx, GLS_ERR_HIP, "cooperative cut launch: %s", hipGetErrorString(e));
        ran = GLS_RW_COOP_CUTS;
    } else {
        // default: three levels per launch (k_cuts_triple); GLS_RW_PAIR_CUTS:
        // two (k_cuts_pair); GLS_RW_LEVEL_CUTS: one (k_cuts_level).  A group
        // with a level wider than cut_wide nodes fills the GPU by itself: the
        // recomputed cones would only add work there, so its levels get one
        // launch each.
        // entries hold node ids in 30 bits
        const bool planned = mode == GLS_RW_PLAN_CUTS && n < (1 << 30);
        const int step = mode == GLS_RW_LEVEL_CUTS ? 1 : mode == GLS_RW_PAIR_CUTS ? 2 : mode == GLS_RW_QUAD_CUTS ? 4
                         : planned ? std::min(std::max(tuning_for(ctx, n).cut_levels, 1), PLAN_MAX_LEVELS) : 3;
        const int32_t cutWide = tuning_for(ctx, n).cut_wide;
        ran = planned ? GLS_RW_PLAN_CUTS : step == 1 ? GLS_RW_LEVEL_CUTS : step == 2 ? GLS_RW_PAIR_CUTS
              : step == 4 ? GLS_RW_QUAD_CUTS : 0;
        struct CutLaunch { int kind; int32_t s, m, m2, e, l; };
        std::vector<CutLaunch> plan;
        plan.reserve((size_t)L / step + 1);
        for (int l = 1; l < L; l += step) {
            const int32_t s = levelStart[l], m = levelStart[std::min(l + 1, L)];
            const int32_t m2 = levelStart[std::min(l + 2, L)];
            const int32_t e = levelStart[std::min(l + step, L)];
            if (e <= s) continue;
            int32_t widest = 0;
            for (int j = l; j < std::min(l + step, L); j++) widest = std::max(widest, levelStart[j + 1] - levelStart[j]);
            if (step > 1 && widest > cutWide) {
                for (int j = l; j < std::min(l + step, L); j++)
                    if (levelStart[j + 1] > levelStart[j])
                        plan.push_back({1, levelStart[j], levelStart[j + 1], levelStart[j + 1], levelStart[j + 1], j});
            } else {
                plan.push_back({step, s, m, m2, e, l});
            }
        }
        // sampled timing of the schedule's own kernel: a window of up to
        // KSAMPLE_WIN consecutive launches of it starts every KSAMPLE_EVERY
        // launches; its first dispatch carries the start event and its last the
        // stop event, so the elapsed time over the launches is the per-launch
        // kernel time a profiler reports, with the events' own cost spread over
        // the window
        // GLS_RW_GRAPH_CUTS: the same launches captured into a HIP graph (kernel
        // nodes only), instantiated and launched once; the host time of the
        // capture and the instantiation is reported apart
        // planned schedule: the task lists of the three-level launches, built
        // before any launch (and before a capture begins)
        Tmp pt{ctx};
        std::vector<int32_t> lv;
        std::vector<uint32_t> toff;
        uint4 *heads = nullptr, *ents = nullptr;
        if (planned && step > 1) {
            for (const CutLaunch &c : plan)
                if (c.kind == step)
                    for (int p = 0; p <= step; p++) lv.push_back(levelStart[std::min(c.l + p, L)]);
            if (!lv.empty()) GLS_TRY(build_cut_plan(ctx, pt, g, step, lv, heads, ents, toff));
        }
        size_t j3 = 0;
        hipGraph_t graph = nullptr;
        hipGraphExec_t exec = nullptr;
        const auto tg0 = std::chrono::steady_clock::now();
        if (graphed) GLS_HIP(ctx, hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
        int win = 0;
        for (size_t i = 0; i < plan.size(); i++) {
            const CutLaunch &c = plan[i];
            const bool pl = planned && step > 1 && c.kind == step;
            const uint32_t tbase = pl ? toff[j3] : 0u, tcount = pl ? toff[j3 + 1] - toff[j3] : 0u;
            if (pl) ++j3;
            const dim3 grid(pl ? tcount : c.kind > 1 ? (unsigned)(c.e - c.s) : blocks(c.e - c.s, CUTL_BLOCK / 64));
            hipEvent_t evStart = nullptr, evStop = nullptr;
            if (kSampleLaunches && !graphed && win == 0 && c.kind == step && i % KSAMPLE_EVERY == 0) {
                const size_t k = 2 * (size_t)ctx->ksamp_n;
                while (ctx->kev.size() < k + 2) {
                    hipEvent_t ev = nullptr;
                    GLS_HIP(ctx, hipEventCreate(&ev));
                    ctx->kev.push_back(ev);
                }
                evStart = ctx->kev[k];
                ctx->ksamp_units.push_back(0);
                ctx->ksamp_launches.push_back(0);
                ctx->ksamp_n++;
                win = KSAMPLE_WIN;
            }
            if (win > 0) {
                ctx->ksamp_units.back() += c.e - c.s;
                ctx->ksamp_launches.back() += 1;
                // the window ends at its last launch or before a launch of another kernel
                if (--win == 0 || i + 1 == plan.size() || plan[i + 1].kind != step) {
                    win = 0;
                    evStop = ctx->kev[2 * (size_t)ctx->ksamp_n - 1];
                }
                if (pl)
                    hipExtLaunchKernelGGL(k_cuts_plan, grid, dim3(CUT3_BLOCK), 0, st, evStart, evStop, 0,
                                          (const uint4 *)heads, (const uint4 *)ents, (int32_t)tbase, (int32_t)step,
                                          (const int32_t *)d_nref, d_cuts, sigBits);
                else if (c.kind == 4)
                    hipExtLaunchKernelGGL(k_cuts_quad, grid, dim3(CUT4_BLOCK), 0, st, evStart, evStop, 0, c.s, c.m,
                                          c.m2, levelStart[std::min(c.l + 3, L)], (const uint32_t *)g.f0,
                                          (const uint32_t *)g.f1, (const int32_t *)d_nref, d_cuts, sigBits);
                else if (c.kind == 3)
                    hipExtLaunchKernelGGL(k_cuts_triple, grid, dim3(CUT3_BLOCK), 0, st, evStart, evStop, 0, c.s, c.m,
                                          c.m2, (uint32_t)n, (const uint32_t *)g.f0, (const uint32_t *)g.f1,
                                          (const int32_t *)d_nref, d_cuts, sigBits);
                else if (c.kind == 2)
                    hipExtLaunchKernelGGL(k_cuts_pair, grid, dim3(CUTP_BLOCK), 0, st, evStart, evStop, 0, c.s,
                                          c.m - c.s, c.m, (const uint32_t *)g.f0, (const uint32_t *)g.f1,
                                          (const int32_t *)d_nref, d_cuts, sigBits);
                else
                    hipExtLaunchKernelGGL(k_cuts_level, grid, dim3(CUTL_BLOCK), 0, st, evStart, evStop, 0, c.s,
                                          c.e - c.s, (const uint32_t *)g.f0, (const uint32_t *)g.f1,
                                          (const int32_t *)d_nref, d_cuts, sigBits);
            } else if (pl) {
                k_cuts_plan<<<grid, CUT3_BLOCK, 0, st>>>(heads, ents, (int32_t)tbase, step, d_nref, d_cuts, sigBits);
            } else if (c.kind == 4) {
                k_cuts_quad<<<grid, CUT4_BLOCK, 0, st>>>(c.s, c.m, c.m2, levelStart[std::min(c.l + 3, L)], g.f0, g.f1,
                                                         d_nref, d_cuts, sigBits);
            } else if (c.kind == 3) {
                k_cuts_triple<<<grid, CUT3_BLOCK, 0, st>>>(c.s, c.m, c.m2, (uint32_t)n, g.f0, g.f1, d_nref, d_cuts, sigBits);
            } else if (c.kind == 2) {
                k_cuts_pair<<<grid, CUTP_BLOCK, 0, st>>>(c.s, c.m - c.s, c.m, g.f0, g.f1, d_nref, d_cuts, sigBits);
            } else {
                k_cuts_level<<<grid, CUTL_BLOCK, 0, st>>>(c.s, c.e - c.s, g.f0, g.f1, d_nref, d_cuts, sigBits);
            }
        }
        if (graphed) {
            const hipError_t ec = hipStreamEndCapture(st, &graph);
            if (ec != hipSuccess) return gls_fail(ctx, GLS_ERR_HIP, "cut graph capture: %s", hipGetErrorString(ec));
            const hipError_t ei = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
            if (ei != hipSuccess) {
                (void)hipGraphDestroy(graph);
                return gls_fail(ctx, GLS_ERR_HIP, "cut graph instantiation: %s", hipGetErrorString(ei));
            }
            ctx->cut_graph_ms =
                std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - tg0).count();
            ctx->cut_graph_nodes = (int64_t)plan.size();
            hipError_t el = hipGraphLaunch(exec, st);
            // the executable graph is released once its launch has run
            if (el == hipSuccess) el = hipStreamSynchronize(st);
            (void)hipGraphExecDestroy(exec);
            (void)hipGraphDestroy(graph);
            if (el != hipSuccess) return gls_fail(ctx, GLS_ERR_HIP, "cut graph launch: %s", hipGetErrorString(el));
            ran |= GLS_RW_GRAPH_CUTS;
        }
    }
    GLS_HIP(ctx, hipGetLastError());
    return GLS_OK;
}

// Few nodes: two per wavefront, so that more wavefronts share the chain of
// lookups; many: eight, so that the cones use every lane.  Two against eight,
// us: 2k random ANDs 26 / 56, 32k 53 / 69, a 50k windowed AIG 92 / 89, 64k
// random 95 / 91, 500k 638 / 512.
static void launch_eval(hipStream_t st, int32_t n, int32_t nPIs, const GraphView &g, const Lib &L, const uint32_t *cuts,
                        int useZeros, int4 *best) {
    const int32_t nAnd = n - nPIs - 1;
    if (nAnd <= 0) return;
    if (nAnd <= EVAL_FEW) k_eval<2><<<blocks(nAnd, 2), 64, 0, st>>>(n, nPIs, g, L, cuts, useZeros, best);
    else k_eval<8><<<blocks(nAnd, 8), 64, 0, st>>>(n, nPIs, g, L, cuts, useZeros, best);
}

static int build_table(gls_ctx *ctx, Tmp &t, const DevGraph &g, GraphView &gv) {
    hipStream_t st = ctx->stream;
    const int32_t n = g.nObjs;
    const size_t nAnd = n > g.nPIs + 1 ? (size_t)(n - g.nPIs - 1) : 0;
    uint32_t *cnt = t.get<uint32_t>((size_t)n + 1), *off = t.get<uint32_t>((size_t)n + 1);
    uint2 *ent = t.get<uint2>(std::max<size_t>(nAnd, 1));
    if (!cnt || !off || !ent) return gls_fail(ctx, GLS_ERR_NOMEM, "table allocation");
    GLS_TRY(Fills(ctx).add(cnt, 0, sizeof(uint32_t) * ((size_t)n + 1)).run());
    k_table_count<<<grid_for(n), kBlock, 0, st>>>(n, g.nPIs, g.f1, cnt);
    size_t tb = 0;
    GLS_HIP(ctx, rocprim::exclusive_scan(nullptr, tb, cnt, off, 0u, (size_t)n + 1, rocprim::plus<uint32_t>(), st));
    void *tmp = t.get<uint8_t>(std::max<size_t>(tb, 1));
    if (!tmp) return gls_fail(ctx, GLS_ERR_NOMEM, "table scan storage");
    GLS_HIP(ctx, rocprim::exclusive_scan(tmp, tb, cnt, off, 0u, (size_t)n + 1, rocprim::plus<uint32_t>(), st));
    GLS_TRY(Fills(ctx).add(cnt, 0, sizeof(uint32_t) * ((size_t)n + 1)).run());
    k_table_fill<<<grid_for(n), kBlock, 0, st>>>(n, g.nPIs, g.f0, g.f1, off, cnt, ent);
    GLS_HIP(ctx, hipGetLastError());
    gv.tOff = off;
    gv.tEnt = ent;
    return GLS_OK;
}

int dev_evaluate(gls_ctx *ctx, const DevGraph &g, const uint32_t *d_cuts, const int32_t *d_nref, int useZeros,
                 int32_t *d_best) {
    GLS_TRY(ctx_ensure_library(ctx));
    hipStream_t st = ctx->stream;
    Tmp t{ctx};
    GraphView gv{g.f0, g.f1, d_nref, g.level, nullptr, nullptr};
    GLS_TRY(build_table(ctx, t, g, gv));
    // PIs and the constant have no candidate
    k_no_candidate<<<blocks(g.nPIs + 1, kBlock), kBlock, 0, st>>>(g.nPIs + 1, reinterpret_cast<int4 *>(d_best));
    launch_eval(st, g.nObjs, g.nPIs, gv, lib_of(ctx), d_cuts, useZeros, reinterpret_cast<int4 *>(d_best));
    GLS_HIP(ctx, hipGetLastError());
    GLS_HIP(ctx, hipStreamSynchronize(st));
    return GLS_OK;
}

int dev_rewrite(gls_ctx *ctx, const DevGraph &in, int useZeros, int flags, DevGraph &out, int32_t *depth,
                gls_op_info *info, const uint32_t *tagIn, uint32_t **tagOut, uint32_t *tagDepth,
                const int32_t *constRef, int32_t nTags) {
    GLS_TRY(ctx_ensure_library(ctx));
    hipStream_t st = ctx->stream;
    Timer tm{ctx};
    tm.mark(); // 0
    DevGraph g;
    std::vector<int32_t> levelStart;
    const bool tagged = tagIn && tagOut;
    if (tagged && !constRef) return gls_fail(ctx, GLS_ERR_INTERNAL, "rewrite: tags without their constants' references");
    uint32_t *tagR = nullptr;   // tags in the reordered numbering (freed on every return)
    struct TagGuard {
        gls_ctx *c;
        uint32_t **p;
        ~TagGuard() { if (*p) pool_put(c, *p); }
    } tagGuard{ctx, &tagR};
    GLS_TRY(dev_reorder(ctx, in, g, levelStart, tagged ? tagIn : nullptr, tagged ? &tagR : nullptr));
    GraphGuard gGuard{ctx, &g};   // frees the reordered graph on every return path
    tm.mark(); // 1
    const int32_t n = g.nObjs, nPIs = g.nPIs, nPOs = g.nPOs;
    const size_t nRefs = (size_t)n + (tagged ? nTags : 0);     // objects and the members' constants
    int rc = GLS_OK;
    {
        Tmp t{ctx};
        uint32_t *cuts = t.get<uint32_t>((size_t)n * NCUT * 5);
        int32_t *nref = t.get<int32_t>(nRefs);
        int4 *best = t.get<int4>(n);
        uint8_t *flag = t.get<uint8_t>(n);
        uint32_t *candIds = t.get<uint32_t>(n), *d_cnt = t.get<uint32_t>(4), *d_err = t.get<uint32_t>(4);
        uint32_t *repl = t.get<uint32_t>(n);
        unsigned long long *d_gain = t.get<unsigned long long>(2);
        if (!t.ok) return gls_fail(ctx, GLS_ERR_NOMEM, "rewrite: allocation (n=%d)", n);
        GLS_TRY(Fills(ctx).add(d_err, 0, 16).run());
        uint8_t *sigBits = nullptr;
        if (tagged) {
            sigBits = t.get<uint8_t>(n);
            if (!sigBits) return gls_fail(ctx, GLS_ERR_NOMEM, "rewrite: signature bits");
            GLS_TRY(sig_bits_for_tags(ctx, n, tagR, sigBits));
        }
        int cutRan = 0;
        GLS_TRY(dev_enumerate_cuts(ctx, g, levelStart, cuts, nref,
                                   flags & (GLS_RW_COOP_CUTS | GLS_RW_DATAFLOW_CUTS | GLS_RW_XCD_CUTS |
                                            GLS_RW_LEVEL_CUTS | GLS_RW_PAIR_CUTS | GLS_RW_GRAPH_CUTS |
                                            GLS_RW_PLAN_CUTS | GLS_RW_QUAD_CUTS),
                                   sigBits, &cutRan));
        tm.mark(); // 2
        GraphView gv{g.f0, g.f1, nref, g.level, nullptr, nullptr};
        if (tagged) {
            gv.tag = tagR;
            gv.n = n;
            GLS_HIP(ctx, hipMemcpyAsync(nref + n, constRef, sizeof(int32_t) * nTags, hipMemcpyDeviceToDevice, st));
        }
        GLS_TRY(build_table(ctx, t, g, gv));
        tm.mark(); // 3
        k_no_candidate<<<blocks(nPIs + 1, kBlock), kBlock, 0, st>>>(nPIs + 1, best);
        const Lib L = lib_of(ctx);
        launch_eval(st, n, nPIs, gv, L, cuts, useZeros, best);
        GLS_HIP(ctx, hipGetLastError());
        tm.mark(); // 4
        // candidates in id order
        k_flag_cand<<<blocks(n, kBlock), kBlock, 0, st>>>(n, best, flag);
        size_t tb = 0;
        rocprim::counting_iterator<uint32_t> ids(0u);
        GLS_HIP(ctx, rocprim::select(nullptr, tb, ids, flag, candIds, d_cnt, (size_t)n, st));
        void *tmp = t.get<uint8_t>(tb);
        if (!tmp) return gls_fail(ctx, GLS_ERR_NOMEM, "rewrite: select storage");
        GLS_HIP(ctx, rocprim::select(tmp, tb, ids, flag, candIds, d_cnt, (size_t)n, st));
        uint32_t nCand = 0;
        GLS_TRY(stream_copy(ctx, &nCand, d_cnt, 4, hipMemcpyDeviceToHost));
        uint32_t herr = 0;
        uint32_t nSel = 0, rounds = 0, totalNew = 0;
        unsigned long long estGain = 0;
        k_iota2<<<grid_for(n), kBlock, 0, st>>>(n, repl);
        Plan *plans = nullptr;
        uint8_t *state = nullptr;
        uint32_t *newOff = nullptr;
        if (nCand > 0) {
            plans = t.get<Plan>(nCand);
            state = t.get<uint8_t>(nCand);
            uint32_t *mk = t.get<uint32_t>(nRefs), *newCnt = t.get<uint32_t>(nCand + 1);
            newOff = t.get<uint32_t>(nCand + 1);
            uint32_t *selList = t.get<uint32_t>(SEL_REST);
            Claims cl{t.get<unsigned long long>(nRefs), t.get<unsigned long long>(nRefs), t.get<unsigned long long>(nRefs),
                      t.get<unsigned long long>(nRefs)};
            if (!t.ok) return gls_fail(ctx, GLS_ERR_NOMEM, "rewrite: plan allocation");
            const int per = plan_lanes((int32_t)nCand);
            k_plan<<<blocks(nCand, per), EVAL_BLOCK, 0, st>>>(per, (int32_t)nCand, candIds, gv, L, cuts, best, plans);
            k_sel_init<<<blocks(nCand, kBlock), kBlock, 0, st>>>((int32_t)nCand, plans, state);
            GLS_TRY(Fills(ctx)
                        .add(mk, 0, sizeof(uint32_t) * nRefs)
                        .add(cl.W, 0, sizeof(unsigned long long) * nRefs)
                        .add(cl.Wnr, 0, sizeof(unsigned long long) * nRefs)
                        .add(cl.L, 0, sizeof(unsigned long long) * nRefs)
                        .add(cl.M, 0, sizeof(unsigned long long) * nRefs)
                        .run());
            for (uint32_t r = 1;; r++) {
                k_sel_claim<<<blocks(nCand, kBlock), kBlock, 0, st>>>(r, (int32_t)nCand, plans, state, cl, d_cnt);
                k_sel_decide<<<blocks(nCand, kBlock), kBlock, 0, st>>>(r, (int32_t)nCand, plans, state, cl, mk);
                k_sel_elim<<<blocks(nCand, kBlock), kBlock, 0, st>>>((int32_t)nCand, plans, state, mk, d_cnt, selList);
                GLS_HIP(ctx, hipGetLastError());
                uint32_t left = 0;
                GLS_TRY(stream_copy(ctx, &left, d_cnt, 4, hipMemcpyDeviceToHost));
                rounds = r;
                if (left == 0) break;
                if (r > SEL_ROUNDS) return gls_fail(ctx, GLS_ERR_INTERNAL, "selection did not converge");
                if (left > SEL_REST) continue;
                k_sel_rest<<<1, SEL_WG, 0, st>>>(r + 1, left, selList, plans, state, cl, mk, d_cnt);
                GLS_HIP(ctx, hipGetLastError());
                uint32_t rest[2] = {};
                GLS_TRY(stream_copy(ctx, rest, d_cnt, sizeof(rest), hipMemcpyDeviceToHost));
                if (rest[1]) return gls_fail(ctx, GLS_ERR_INTERNAL, "selection did not converge");
                rounds = rest[0] - 1;
                break;
            }
            GLS_TRY(Fills(ctx).add(d_gain, 0, 16).run());
            k_new_counts<<<blocks((int64_t)nCand + 1, kBlock), kBlock, 0, st>>>((int32_t)nCand, plans, state, newCnt, d_gain);
            size_t tb2 = 0;
            GLS_HIP(ctx, rocprim::exclusive_scan(nullptr, tb2, newCnt, newOff, 0u, (size_t)nCand + 1, rocprim::plus<uint32_t>(), st));
            void *tmp2 = t.get<uint8_t>(tb2);
            if (!tmp2) return gls_fail(ctx, GLS_ERR_NOMEM, "rewrite: scan storage");
            GLS_HIP(ctx, rocprim::exclusive_scan(tmp2, tb2, newCnt, newOff, 0u, (size_t)nCand + 1, rocprim::plus<uint32_t>(), st));
            unsigned long long sums[2] = {};
            GLS_TRY(fetch(ctx, {{&totalNew, newOff + nCand, 4}, {sums, d_gain, 16}}));
            estGain = sums[0];
            nSel = (uint32_t)sums[1];
        }
        tm.mark(); // 5
        const int32_t N = n + (int32_t)totalNew;
        DevGraph comb;
        GLS_TRY(dev_graph_alloc(ctx, comb, N, nPIs, nPOs));
        GraphGuard combGuard{ctx, &comb};
        uint32_t *tagC = nullptr;   // tags of the composed graph
        if (tagged) {
            tagC = t.get<uint32_t>(N);
            if (!tagC) return gls_fail(ctx, GLS_ERR_NOMEM, "rewrite: tags");
            GLS_HIP(ctx, hipMemcpyAsync(tagC, tagR, sizeof(uint32_t) * n, hipMemcpyDeviceToDevice, st));
        }
        const bool fullStrash = (flags & GLS_RW_FULL_STRASH) != 0;
        if (nCand > 0 && totalNew + nSel > 0) {
            const int per = plan_lanes((int32_t)nCand);
            k_build<<<blocks(nCand, per), EVAL_BLOCK, 0, st>>>(per, n, (int32_t)nCand, candIds, gv, L, cuts, best, state,
                                                               newOff, comb.f0, comb.f1, repl, d_err, tagC);
        }
        k_compose<<<grid_for(N), kBlock, 0, st>>>(n, N, nPIs, g.f0, g.f1, repl, comb.f0, comb.f1);
        if (nPOs > 0) k_compose_pos<<<blocks(nPOs, kBlock), kBlock, 0, st>>>(nPOs, g.pos, repl, comb.pos);
        GLS_HIP(ctx, hipGetLastError());
        GLS_TRY(stream_copy(ctx, &herr, d_err, 4, hipMemcpyDeviceToHost));
        if (herr) return gls_fail(ctx, GLS_ERR_INTERNAL, "rewrite: inconsistent plan (%u)", herr);
        tm.mark(); // 6
        gls_op_info stInfo = {};
        if (fullStrash) {
            gGuard.free_now();
            rc = dev_strash(ctx, comb, out, depth, &stInfo, tagC, tagged ? tagOut : nullptr,
                            tagged ? tagDepth : nullptr);
        } else {
            // the incremental strash reads the input graph's fanins: g is
            // released only after it
            const RwDelta delta{n, (int32_t)levelStart.size() - 2, g.f0, g.f1, g.level, gv.tOff, gv.tEnt};
            rc = dev_strash_rw(ctx, comb, delta, out, depth, &stInfo, tagC, tagged ? tagOut : nullptr,
                               tagged ? tagDepth : nullptr);
            gGuard.free_now();
        }
        combGuard.free_now();
        tm.mark(); // 7
        GLS_HIP(ctx, hipStreamSynchronize(st));
        if (info) {
            info->reorder_ms = tm.ms(0, 1);
            info->cuts_ms = tm.ms(1, 2);
            info->table_ms = tm.ms(2, 3);
            info->eval_ms = tm.ms(3, 4);
            info->select_ms = tm.ms(4, 5);
            info->build_ms = tm.ms(5, 6);
            info->strash_ms = tm.ms(6, 7);
            info->total_ms = tm.ms(0, 7);
            info->candidates = nCand;
            info->selected = nSel;
            info->new_nodes = totalNew;
            info->rounds = rounds;
            info->levels_enumerated = (int64_t)levelStart.size() - 2;
            info->est_gain = (int64_t)estGain;
            info->hash_probes = stInfo.hash_probes;
            info->final_strash = stInfo.final_strash;
            info->cut_schedule = cutRan;
            info->strash_rounds = stInfo.strash_rounds;
            info->strash_sweeps = stInfo.strash_sweeps;
            info->cut_graph_ms = ctx->cut_graph_ms;
            info->cut_graph_nodes = ctx->cut_graph_nodes;
            double kms = 0;
            int64_t kunits = 0, klaunches = 0;
            for (int i = 0; i < ctx->ksamp_n; i++) {
                float x = 0;
                if (hipEventElapsedTime(&x, ctx->kev[2 * i], ctx->kev[2 * i + 1]) != hipSuccess) continue;
                kms += x;
                kunits += ctx->ksamp_units[i];
                klaunches += ctx->ksamp_launches[i];
            }
            info->kernel_sample_ms = kms;
            info->kernel_samples = klaunches;
            info->kernel_sample_nodes = kunits;
        }
    }
    return rc;
}
