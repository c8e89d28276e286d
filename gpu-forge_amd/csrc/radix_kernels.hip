// radix_kernels.hip -- forge-sort's GpuSorter radix sort, written for gfx950
// (CDNA4, wave64).  Built into a code object with `hipcc --genco` and loaded by
// the host runtime through hipModuleLoad; every entry point is extern "C".
//
// Pipeline for one sort of n keys (8-bit digits, LSD order):
//   fs_upsweep      one read of the keys: histograms of every digit at once,
//                   key transform applied in registers.  Replaces
//                   sort_msd_histogram (sort.metal:64-142), which only counted
//                   the top byte.
//   (plan)          the upsweep block that finishes last: exclusive scans of
//                   the histograms into bin bases, detection of constant
//                   digits, and the device-side pass schedule (which digit
//                   passes run and which buffers they read and write).
//                   Replaces sort_msd_prep (sort.metal:153-181).
//   fs_onesweep_*   one launch per digit position; a digit that is constant
//                   over the whole input exits at once.  Each tile ranks its
//                   keys with wave64 ballot matching (stable: index order is
//                   (wave, item, lane)), gets its global offsets by decoupled
//                   look-back over the previous tiles, stages the tile in LDS
//                   in digit order and writes runs to HBM.  Replaces
//                   sort_msd_atomic_scatter (sort.metal:193-365) and
//                   sort_inner_fused (sort.metal:378-769), which are not
//                   stable.  Values (pairs) move with their keys; argsort
//                   indices are generated by the first pass, replacing
//                   sort_init_indices / sort_gather_values (sort.metal:777-800).
//   The copy of a single in-place pass through scratch, and argsort's index
//   fill when every digit is constant, run in the launch of a constant digit.
// Key transforms (sort.metal:812-868) are fused into the first and last pass.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fs_params.h"

#define DEV __device__ __forceinline__

// Global-address-space view of a device address held as an integer (the
// schedule stores addresses as u64): loads and stores through it compile to
// global_* instructions instead of flat_*.
#ifndef GLOBAL
#define GLOBAL __attribute__((address_space(1)))
#endif
// Constant-address-space view: wave-uniform loads through it are scalar loads
// (s_load, cached in the scalar cache).  Used only for data that a previous
// kernel wrote and no kernel running alongside writes: the acquire at every
// kernel start makes such data visible to plain loads.
#ifndef CONSTANT
#define CONSTANT __attribute__((address_space(4)))
#endif
template <typename T>
DEV GLOBAL T* gptr(uint64_t addr) {
    return (GLOBAL T*)(uintptr_t)addr;
}

// ---------------------------------------------------------------------------
// key traits
// ---------------------------------------------------------------------------

template <bool K64> struct KeyT;
template <> struct KeyT<false> {
    typedef uint32_t type;
    static constexpr uint32_t SIGN = 0x80000000u;
};
template <> struct KeyT<true> {
    typedef uint64_t type;
    static constexpr uint64_t SIGN = 0x8000000000000000ull;
};

// Forward transform: key order of i32/i64/f32/f64 -> unsigned order.
template <bool K64>
DEV typename KeyT<K64>::type xf_fwd(typename KeyT<K64>::type v, uint32_t xf) {
    typedef typename KeyT<K64>::type K;
    const K s = KeyT<K64>::SIGN;
    if (xf == FS_XF_SIGN) return v ^ s;
    if (xf == FS_XF_FLOAT) return (v & s) ? ~v : (v ^ s);
    return v;
}

// Both transforms branch-free from one pair of masks: (xa, xb) = (0, 0) none,
// (SIGN, 0) sign flip (i32/i64), (SIGN, ~0) FloatFlip / IFloatFlip (f32/f64).
// Forward: v ^ (xa | (xb & m)) with m all ones when the top bit of v is set
// (a negative float is inverted, any other value has its sign flipped).
// Inverse: the same with m all ones when the top bit of v is clear.
template <bool K64>
DEV void xf_inv_masks(uint32_t xf, typename KeyT<K64>::type& xa, typename KeyT<K64>::type& xb) {
    typedef typename KeyT<K64>::type K;
    xa = (xf == FS_XF_SIGN || xf == FS_XF_FLOAT) ? KeyT<K64>::SIGN : (K)0;
    xb = (xf == FS_XF_FLOAT) ? ~(K)0 : (K)0;
}
template <bool K64>
DEV typename KeyT<K64>::type xf_fwd_apply(typename KeyT<K64>::type v, typename KeyT<K64>::type xa,
                                          typename KeyT<K64>::type xb) {
    typedef typename KeyT<K64>::type K;
    return v ^ (xa | (xb & ((K)0 - (v >> (8 * sizeof(K) - 1)))));
}
template <bool K64>
DEV typename KeyT<K64>::type xf_inv_apply(typename KeyT<K64>::type v, typename KeyT<K64>::type xa,
                                          typename KeyT<K64>::type xb) {
    typedef typename KeyT<K64>::type K;
    return v ^ (xa | (xb & ((v >> (8 * sizeof(K) - 1)) - (K)1)));
}

// Returns v unchanged but hides its origin from the optimiser, so a digit is
// recomputed from the key (one bit-field extract) where it is needed instead
// of being kept live in a register across the phases of the pass.
template <typename T>
DEV T fresh(T v) {
    asm volatile("" : "+v"(v));
    return v;
}

template <bool K64>
DEV uint32_t digit_of(typename KeyT<K64>::type k, uint32_t shift) {
    return (uint32_t)(k >> shift) & 0xFFu;
}

// ---------------------------------------------------------------------------
// wave64 helpers
// ---------------------------------------------------------------------------

// Mask of the lanes whose 8-bit digit equals this lane's; all 64 lanes active.
// Per bit b: m = bit b of d replicated (0 or ~0), B = ballot of that bit, and
// the lanes that differ from this lane in bit b are (B ^ m); their union over
// the 8 bits is accumulated with one v_bitop3 per mask half (truth table 0xDE
// = b | (a ^ c) for operands (m, acc, B)); the last bit uses 0x21 = ~(b | (a ^ c))
// so the result is the peer mask itself.  4 VALU per bit.
// The digit is bits [shift, shift + 8) of the 32-bit word x (shift wave-uniform),
// so each bit is extracted from x directly.
// NB: digits of NB bits (the local sort's narrow stable passes).
template <int NB = FS_RADIX_BITS>
DEV uint64_t match_digit(uint32_t x, uint32_t shift) {
    uint32_t lo = 0u, hi = 0u;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const uint32_t m = (uint32_t)__builtin_amdgcn_sbfe((int32_t)x, shift + b, 1);
        const uint64_t bal = __builtin_amdgcn_uicmp(m, 0u, 33);   // ballot of (m != 0)
        if (b + 1 < NB) {
            lo = __builtin_amdgcn_bitop3_b32(m, lo, (uint32_t)bal, 0xDE);
            hi = __builtin_amdgcn_bitop3_b32(m, hi, (uint32_t)(bal >> 32), 0xDE);
        } else {
            lo = __builtin_amdgcn_bitop3_b32(m, lo, (uint32_t)bal, 0x21);
            hi = __builtin_amdgcn_bitop3_b32(m, hi, (uint32_t)(bal >> 32), 0x21);
        }
    }
    return ((uint64_t)hi << 32) | lo;
}

// base + number of set bits of `mask` below this lane.
DEV uint32_t lanes_below(uint64_t mask, uint32_t base) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                     __builtin_amdgcn_mbcnt_lo((uint32_t)mask, base));
}

DEV uint32_t ld_agent(const GLOBAL uint32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

DEV void st_agent(GLOBAL uint32_t* p, uint32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

DEV uint64_t ld_agent64(const GLOBAL uint64_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

DEV void st_agent64(GLOBAL uint64_t* p, uint64_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Look-back tile entries: [flag:2 | value:30] in 32 bits, or (WIDE) flag
// bits in the high and the value in the low half of 64 bits; one atomic
// access either way.
template <bool WIDE> struct LbEntry {
    typedef uint32_t type;
    static DEV uint32_t flags(uint32_t e) { return e & FS_LB_FLAGS; }
    static DEV uint32_t value(uint32_t e) { return e & FS_LB_VALUE; }
    static DEV uint32_t load(const GLOBAL uint32_t* lb, uint64_t i) { return ld_agent(lb + i); }
    static DEV void store(GLOBAL uint32_t* lb, uint64_t i, uint32_t flag, uint32_t v) { st_agent(lb + i, flag | v); }
};
template <> struct LbEntry<true> {
    typedef uint64_t type;
    static DEV uint32_t flags(uint64_t e) { return (uint32_t)(e >> 32) & FS_LB_FLAGS; }
    static DEV uint32_t value(uint64_t e) { return (uint32_t)e; }
    static DEV uint64_t load(const GLOBAL uint32_t* lb, uint64_t i) {
        return ld_agent64((const GLOBAL uint64_t*)lb + i);
    }
    static DEV void store(GLOBAL uint32_t* lb, uint64_t i, uint32_t flag, uint32_t v) {
        st_agent64((GLOBAL uint64_t*)lb + i, ((uint64_t)flag << 32) | v);
    }
};

// Device address of schedule buffer `id` (FS_BUF_*); 0 for an unknown id.
DEV uint64_t buf_addr(const FsArgs& a, uint32_t id) {
    switch (id) {
        case FS_BUF_KEYS: return a.keys;
        case FS_BUF_VALS: return a.vals;
        case FS_BUF_S1K: return a.s1k;
        case FS_BUF_S2K: return a.s2k;
        case FS_BUF_S1V: return a.s1v;
        case FS_BUF_S2V: return a.s2v;
        default: return 0;
    }
}

DEV void report(const FsArgs& a, uint32_t bit) {
    __hip_atomic_fetch_or((uint32_t*)a.status, bit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Inclusive scan across the 64 lanes of a wave.
DEV uint32_t wave_inclusive_scan(uint32_t v) {
    const uint32_t lane = threadIdx.x & 63u;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t t = __shfl_up(v, off, 64);
        if (lane >= (uint32_t)off) v += t;
    }
    return v;
}

// ---------------------------------------------------------------------------
// fs_upsweep: all-digit histograms in one read
// ---------------------------------------------------------------------------

template <bool CHOOSE>
DEV void plan_body(const FsArgs& a);
template <bool CHOOSE>
DEV void write_schedule(const FsArgs& a, uint32_t cmask, uint32_t D);

// Lanes of one LDS atomic that hit the same counter are serialised; on skewed
// keys (a dominant bin: small Zipf keys, concentrated float exponents) most
// lanes of a wave do.  skewed_digit: at least FS_PEEL_MIN active lanes share
// the first active lane's digit (a wave-uniform test, one compare).
// add_peeled: counts digit d of every active lane into hist[256], adding the
// lanes that share the first active lane's digit with one atomic.
DEV bool skewed_digit(bool same_as_first) {
    return __builtin_popcountll(__builtin_amdgcn_uicmp((uint32_t)same_as_first, 0u, 33)) >= FS_PEEL_MIN;
}
DEV void add_peeled(uint32_t* hist, uint32_t d, uint32_t lane) {
    const uint32_t f = __builtin_amdgcn_readfirstlane(d);
    const uint64_t grp = __builtin_amdgcn_uicmp((uint32_t)(d == f), 0u, 33);   // contains the first active lane
    const uint32_t leader = (uint32_t)__builtin_ctzll(grp);
    const uint32_t val = d == f ? (lane == leader ? (uint32_t)__builtin_popcountll(grp) : 0u) : 1u;
    if (val) atomicAdd(&hist[d], val);
}
// The same with every lane of the wave active and only the `valid` ones
// counting: a counted lane adds inc to word[idx]; the lanes that share the
// first counted lane's key (which fixes idx and inc) add theirs with one
// atomic.
DEV void add_peeled_valid(uint32_t* word, uint32_t key, uint32_t idx, uint32_t inc, uint32_t lane, bool valid) {
    const uint64_t vm = __builtin_amdgcn_uicmp((uint32_t)valid, 0u, 33);
    if (vm == 0u) return;                                       // (uniform)
    const uint32_t f = __builtin_amdgcn_readlane(key, (uint32_t)__builtin_ctzll(vm));
    const uint64_t grp = __builtin_amdgcn_uicmp((uint32_t)(valid && key == f), 0u, 33);
    const uint32_t leader = (uint32_t)__builtin_ctzll(grp);
    const uint32_t cnt = !valid ? 0u : key == f ? (lane == leader ? (uint32_t)__builtin_popcountll(grp) : 0u) : 1u;
    if (cnt) atomicAdd(&word[idx], cnt * inc);
}

// Slot of this lane's key among the keys of digit d counted into hist[256],
// in no particular order (one LDS atomic with return per lane); lanes with
// valid == false count nothing and get 0.  PEEL: the lanes that share the
// first active lane's digit take consecutive slots from one atomic of their
// leader (their count), each lane its offset in the group.  All lanes of the
// wave are active; the valid lanes are a prefix of them.
template <bool PEEL>
DEV uint32_t slot_in_digit(uint32_t* hist, uint32_t d, uint32_t lane, bool valid) {
    if (!PEEL) return valid ? atomicAdd(&hist[d], 1u) : 0u;
    const uint32_t f = __builtin_amdgcn_readfirstlane(d);
    const uint64_t grp = __builtin_amdgcn_uicmp((uint32_t)(valid && d == f), 0u, 33);
    if (grp == 0u) return 0u;                                  // no valid lane (uniform)
    const uint32_t leader = (uint32_t)__builtin_ctzll(grp);
    const bool in_grp = valid && d == f;
    const uint32_t val = !valid ? 0u : in_grp ? (lane == leader ? (uint32_t)__builtin_popcountll(grp) : 0u) : 1u;
    const uint32_t old = val ? atomicAdd(&hist[d], val) : 0u;
    const uint32_t gbase = __builtin_amdgcn_readlane(old, leader);
    return in_grp ? lanes_below(grp, gbase) : old;
}

// Position of sample s of 2^lm of n > 0 keys: hashed, within the s-th of as many parts.
DEV uint32_t sample_position(uint32_t s, uint32_t lm, uint32_t n) {
    const uint64_t p0 = ((uint64_t)s * n) >> lm, p1 = ((uint64_t)(s + 1u) * n) >> lm;
    const uint32_t h = (s * 0x9E3779B9u) ^ ((s * 0x85EBCA6Bu) >> 13);
    const uint64_t p = p0 + (((uint64_t)h * (p1 - p0)) >> 32);
    return p < n ? (uint32_t)p : n - 1u;
}

// Sorts that launch the digit passes and two levels of buckets
// (FS_BK2_FEW_DIGITS): the buckets do the sort.  (One thread writes this.)
DEV void leave_to_buckets(const FsArgs& a) {
    for (uint32_t i = 0; i < FS_PLAN_WORDS; ++i)
        if (i != FS_PLAN_TICKET) st_agent(gptr<uint32_t>(a.plan) + i, 0u);
    st_agent(gptr<uint32_t>(a.bk2_tab) + FS_BK2_MODE, 0u);
}

template <bool K64, bool CHOOSE>
DEV void upsweep_body(const FsArgs& a) {
    typedef typename KeyT<K64>::type K;
    constexpr int D = K64 ? 8 : 4;
    constexpr int P = D / 2;                          // digit pairs
    constexpr int R = K64 ? FS_UP_REPLICAS_K64 : FS_UP_REPLICAS_K32;
    constexpr int KPV = 16 / (int)sizeof(K);          // keys per 16-byte load
    constexpr uint32_t B = FS_HIST_BLOCK;
    // Replicated 16-bit counters: word h[p][v][r] counts value v of digit 2p
    // (low half) and of digit 2p+1 (high half) for the lanes with
    // lane % R == r.  With R = 32 the 32 lanes of each half of a wave's atomic
    // own 32 different banks whatever their digits (no bank conflicts, and
    // lanes with equal digits are not serialised); with R = 16 two lanes share
    // a pair of banks.  A chunk adds at most (B / R) * (FS_UP_CHUNK_STEPS * KPV + 1)
    // to a counter, and the replicas are folded into the histogram after every
    // chunk.
    static_assert(R == 16 || R == 32, "replicas");
    static_assert((B / R) * (FS_UP_CHUNK_STEPS * KPV + 1) <= 0xFFFFu, "16-bit counters");
    __shared__ uint32_t h[P][FS_RADIX][R];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;

    // Sorts that may go to the buckets: every block looks at the same sample
    // (the loads are in flight while the counters are cleared).
    K ref = 0, probe = 0;
    __shared__ uint32_t s_vary;
    if constexpr (CHOOSE) {
        constexpr uint32_t LB = __builtin_ctz(B);
        static_assert(B == 1u << LB, "a sample per thread");
        const GLOBAL K* keys = gptr<const K>(a.keys);
        ref = keys[sample_position(0u, LB, (uint32_t)a.n)];
        probe = keys[sample_position(tid, LB, (uint32_t)a.n)];
        if (tid == 0) s_vary = 0u;
    }
    for (uint32_t i = tid; i < P * FS_RADIX * R; i += B) (&h[0][0][0])[i] = 0u;

    // Clear the look-back array (tile and group entries) the first executed
    // pass will use.
    {
        GLOBAL uint32_t* lb = gptr<uint32_t>(a.lookback0);
        const uint64_t groups = (a.num_tiles + FS_LB_GROUP - 1) / FS_LB_GROUP;
        const uint64_t total = ((uint64_t)a.num_tiles * (a.wide ? 2u : 1u) + groups) * FS_RADIX;
        for (uint64_t i = (uint64_t)blockIdx.x * B + tid; i < total; i += (uint64_t)gridDim.x * B)
            st_agent(&lb[i], 0u);
    }
    __syncthreads();
    if constexpr (CHOOSE) {
        const K v = xf_fwd<K64>(probe, a.xform) ^ xf_fwd<K64>(ref, a.xform);
        uint32_t mine = 0;                               // digits that vary within the wave's samples
#pragma unroll
        for (uint32_t j = 0; j < 8u; ++j)
            mine |= __builtin_amdgcn_uicmp((uint32_t)((uint64_t)v >> (8u * j)) & 0xFFu, 0u, 33) ? 1u << j : 0u;
        if (lane == 0u) atomicOr(&s_vary, mine);
        __syncthreads();
        if ((uint32_t)__builtin_popcount(s_vary) > FS_BK2_FEW_DIGITS) {   // (uniform over the grid)
            if (blockIdx.x == 0 && tid == 0) leave_to_buckets(a);
            return;
        }
    }

    const GLOBAL K* src = gptr<const K>(a.keys);
    const GLOBAL uint4* src4 = (const GLOBAL uint4*)src;
    GLOBAL uint32_t* gh = gptr<uint32_t>(a.hist);
    uint32_t* hl = &h[0][0][lane % R];                   // this lane's replica

    K xa, xb;
    xf_inv_masks<K64>(a.xform, xa, xb);
    auto count_key = [&](K k) {
        k = xf_fwd_apply<K64>(k, xa, xb);
#pragma unroll
        for (int p = 0; p < P; ++p) {
            atomicAdd(&hl[(p * FS_RADIX + digit_of<K64>(k, 16u * p)) * R], 1u);
            atomicAdd(&hl[(p * FS_RADIX + digit_of<K64>(k, 16u * p + 8u)) * R], 0x10000u);
        }
    };
    auto count_vector = [&](const uint4 q) {
        if constexpr (K64) {
            count_key((K)(((uint64_t)q.y << 32) | q.x));
            count_key((K)(((uint64_t)q.w << 32) | q.z));
        } else {
            count_key(q.x);
            count_key(q.y);
            count_key(q.z);
            count_key(q.w);
        }
    };

    // The grid sweeps the keys front to back, so that all blocks read
    // neighbouring addresses at the same time: in step k, block b takes the
    // units [(k * grid + b) * U * B, +U * B), a unit being a 16-byte vector when
    // the key array is 16-byte aligned, else one key.  The counters are folded
    // every FS_UP_CHUNK_STEPS units per lane; the step ranges are the same for
    // every block.
    constexpr uint32_t U = FS_UPSWEEP_UNROLL;
    static_assert(FS_UP_CHUNK_STEPS % FS_UPSWEEP_UNROLL == 0, "whole steps per chunk");
    const bool vec = a.vec_ok != 0;
    const uint64_t units = vec ? a.n / KPV : a.n;
    const uint64_t span = (uint64_t)U * B;
    const uint64_t steps = (units + span * gridDim.x - 1) / (span * gridDim.x);
    // keys past the last whole vector (fewer than KPV): block 0, before its first fold
    if (vec && blockIdx.x == 0 && tid < a.n - units * KPV) count_key(src[units * KPV + tid]);
    bool first_chunk = true;
    for (uint64_t k0 = 0; k0 < steps || first_chunk; k0 += FS_UP_CHUNK_STEPS / U) {
        first_chunk = false;
        const uint64_t k1 = steps - k0 > FS_UP_CHUNK_STEPS / U ? k0 + FS_UP_CHUNK_STEPS / U : steps;
        for (uint64_t k = k0; k < k1; ++k) {
            const uint64_t u0 = (k * gridDim.x + blockIdx.x) * span + tid;   // this lane's first unit
            if (!vec) {
#pragma unroll
                for (uint32_t u = 0; u < U; ++u)
                    if (u0 + u * B < units) count_key(src[u0 + u * B]);
            } else if (u0 - lane + 63 + (U - 1) * B < units) {           // the wave's units all exist
                uint4 q[U];
#pragma unroll
                for (uint32_t u = 0; u < U; ++u) q[u] = src4[u0 + u * B];
#pragma unroll
                for (uint32_t u = 0; u < U; ++u) count_vector(q[u]);
            } else {
                for (uint32_t u = 0; u < U; ++u)
                    if (u0 + u * B < units) count_vector(src4[u0 + u * B]);
            }
        }
        __syncthreads();

        // Fold the replicas into the histogram and clear them; the threads of
        // a half-wave start on different banks.
        for (uint32_t t = tid; t < P * FS_RADIX; t += B) {
            // fresh(): the addresses are computed here, not hoisted out of the
            // chunk loop into registers
            const uint32_t tt = fresh(t);
            uint32_t* row = &h[0][0][0] + tt * R;        // h[p][v], p * 256 + v = t
            uint32_t lo = 0, hi = 0;
#pragma unroll
            for (uint32_t r = 0; r < (uint32_t)R; ++r) {
                const uint32_t j = (r + tt) % R;
                const uint32_t c = row[j];
                row[j] = 0u;
                lo += c & 0xFFFFu;
                hi += c >> 16;
            }
            const uint32_t p = t / FS_RADIX, val = t % FS_RADIX;
            if (lo) atomicAdd(&gh[(2u * p) * FS_RADIX + val], lo);
            if (hi) atomicAdd(&gh[(2u * p + 1u) * FS_RADIX + val], hi);
        }
        __syncthreads();
    }

    // The block that finishes last computes the schedule and resets the ticket
    // for the next sort.  The histogram is written only by device-coherent
    // atomics, so a block needs no cache write-back before taking its ticket,
    // only the completion of its own atomics: every wave waits for its memory
    // operations (s_waitcnt 0) before the barrier, then one relaxed atomic
    // takes the ticket.  (An agent-scope release fence per block, an L2
    // write-back and invalidate, made the upsweep 3x slower.)  The last block
    // alone fences before reading the histogram.
    __shared__ uint32_t s_last;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    GLOBAL uint32_t* ticket = gptr<uint32_t>(a.plan) + FS_PLAN_TICKET;
    if (tid == 0)
        s_last = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1u;
    __syncthreads();
    if (!s_last) return;
    __threadfence();
    plan_body<CHOOSE>(a);
    if (tid == 0) st_agent(ticket, 0u);
}

// two blocks per CU: at most 64 VGPRs at 1024 threads
#define FS_UP_OCC __attribute__((amdgpu_waves_per_eu(FS_HIST_BLOCK / 64 / 4 * 2)))
extern "C" __global__ void __launch_bounds__(FS_HIST_BLOCK) FS_UP_OCC fs_upsweep_k32(FsArgs a) {
    upsweep_body<false, false>(a);
}
extern "C" __global__ void __launch_bounds__(FS_HIST_BLOCK) FS_UP_OCC fs_upsweep_k64(FsArgs a) {
    upsweep_body<true, false>(a);
}
// ... of sorts that may go to two levels of buckets: a kernel of its own, since
// the choice within the kernels above, unused, cost the other sorts 0.3 to 2 us
// (u64 keys, 2.0M: 167.6 -> 165.8; u32, 2.5M: 94.0 -> 93.7)
extern "C" __global__ void __launch_bounds__(FS_HIST_BLOCK) FS_UP_OCC fs_upsweep_choose_k64(FsArgs a) {
    upsweep_body<true, true>(a);
}

// ---------------------------------------------------------------------------
// plan_body: bin bases, constant-digit detection, pass schedule; run by the
// last upsweep block to finish (its first 256 threads, one per bin; every
// thread of the block reaches the barriers)
// ---------------------------------------------------------------------------

template <bool CHOOSE>
DEV void plan_body(const FsArgs& a) {
    __shared__ uint32_t wsum[FS_MAX_DIGITS][FS_RADIX / 64];
    __shared__ uint32_t cmask;                 // bit j: digit j is constant
    const uint32_t d = threadIdx.x;           // one thread per bin
    const bool bin = d < FS_RADIX;
    const uint32_t lane = d & 63u, w = d >> 6;
    const uint32_t D = a.digits;
    // The histogram was built by other blocks' atomics; counters, histogram and
    // schedule are read and reset with agent-scope accesses, so no cache line
    // of an earlier kernel can be observed.
    GLOBAL uint32_t* hist = gptr<uint32_t>(a.hist);
    GLOBAL uint32_t* base = gptr<uint32_t>(a.binbase);
    if (D != (a.key64 ? 8u : 4u)) {          // the schedule holds FS_MAX_DIGITS passes (uniform)
        // Reported; the histogram is cleared for the next sort and the
        // schedule runs no pass, so the digit passes of this sort do nothing.
        if (d == 0) report(a, FS_DEVERR_BAD_DIGITS);
        if (bin)
            for (uint32_t j = 0; j < FS_MAX_DIGITS; ++j) st_agent(&hist[j * FS_RADIX + d], 0u);
        if (d < FS_PLAN_WORDS && d != FS_PLAN_TICKET) st_agent(&gptr<uint32_t>(a.plan)[d], 0u);   // all but the ticket
        return;
    }

    // All digits' totals in flight at once (the loads are the latency here).
    uint32_t totals[FS_MAX_DIGITS];
#pragma unroll
    for (uint32_t j = 0; j < FS_MAX_DIGITS; ++j) totals[j] = (bin && j < D) ? ld_agent(&hist[j * FS_RADIX + d]) : 0u;
    // Exclusive scans of every digit's totals over the 256 bins at once (the
    // scans are independent; digits beyond D scan zeros), and the constant
    // digits: digit j is constant when one bin holds every key.
    if (d == 0) cmask = 0u;
    __syncthreads();
    uint32_t inc[FS_MAX_DIGITS];
    uint32_t mine = 0;
#pragma unroll
    for (uint32_t j = 0; j < FS_MAX_DIGITS; ++j) {
        inc[j] = wave_inclusive_scan(totals[j]);
        if (bin && j < D && totals[j] == (uint32_t)a.n) mine |= 1u << j;
        if (bin && j < D && totals[j] > (uint32_t)(a.n / FS_SKEW_SHARE)) mine |= FS_SKEW_BIT << j;
    }
    if (bin && lane == 63) {
#pragma unroll
        for (uint32_t j = 0; j < FS_MAX_DIGITS; ++j) wsum[j][w] = inc[j];
    }
    if (mine) atomicOr(&cmask, mine);
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < FS_MAX_DIGITS; ++j) {
        if (j >= D || !bin) break;            // uniform per wave
        uint32_t excl = inc[j] - totals[j];
        for (uint32_t v = 0; v < w; ++v) excl += wsum[j][v];
        base[j * FS_RADIX + d] = excl;
        st_agent(&hist[j * FS_RADIX + d], 0u);        // ready for the next sort
    }

    if (d == 0) write_schedule<CHOOSE>(a, cmask, D);
}

// The standard schedule, written by one thread: which digit passes run (the
// digits whose bit in cmask is clear), their order of execution, flags and
// buffers.  Every pass reads the previous pass's output, the first the
// caller's keys.  CHOOSE: the sort may go to the buckets instead, and has
// FS_BK2_FEW_DIGITS launch slots.
template <bool CHOOSE>
DEV void write_schedule(const FsArgs& a, uint32_t cmask, uint32_t D) {
    {
        GLOBAL uint32_t* plan = gptr<uint32_t>(a.plan);
        uint32_t active[FS_MAX_DIGITS];
        for (uint32_t j = 0; j < FS_MAX_DIGITS; ++j) active[j] = (cmask >> j) & 1u ? 0u : 1u;
        uint32_t p = 0, mask = 0;
        for (uint32_t j = 0; j < D; ++j)
            if (active[j]) { ++p; mask |= 1u << j; }
        if (CHOOSE) {
            if (p > FS_BK2_FEW_DIGITS) {                 // more digits vary than the sample showed
                leave_to_buckets(a);
                return;
            }
            st_agent(gptr<uint32_t>(a.bk2_tab) + FS_BK2_MODE, 1u);
        }
        // Fewer launch slots than digits: the passes that run take slots in
        // order, after a copy if there is one.
        constexpr bool compact = CHOOSE;

        // Destination of executed pass e for keys (dk) and values (dv).
        uint32_t dk[FS_MAX_DIGITS], dv[FS_MAX_DIGITS];
        for (uint32_t e = 0; e < p; ++e) {
            if (a.op == FSK_OP_ARGSORT) {
                dk[e] = (e & 1u) ? FS_BUF_S2K : FS_BUF_S1K;                 // keys never go back
                dv[e] = ((p - 1u - e) & 1u) ? FS_BUF_S1V : FS_BUF_VALS;     // indices end in the output
            } else if (p == 1u) {
                dk[e] = FS_BUF_S1K;
                dv[e] = FS_BUF_S1V;
            } else if ((p & 1u) == 0u) {
                dk[e] = ((p - 1u - e) & 1u) ? FS_BUF_S1K : FS_BUF_KEYS;
                dv[e] = ((p - 1u - e) & 1u) ? FS_BUF_S1V : FS_BUF_VALS;
            } else {
                // odd p >= 3 in place: F -> S1 -> S2 -> F -> S2 -> F ...
                if (e == 0) { dk[e] = FS_BUF_S1K; dv[e] = FS_BUF_S1V; }
                else if (e == 1) { dk[e] = FS_BUF_S2K; dv[e] = FS_BUF_S2V; }
                else {
                    dk[e] = ((p - 1u - e) & 1u) ? FS_BUF_S2K : FS_BUF_KEYS;
                    dv[e] = ((p - 1u - e) & 1u) ? FS_BUF_S2V : FS_BUF_VALS;
                }
            }
        }
        // A single in-place pass cannot scatter into the buffer it reads, so its
        // keys (and values) go through scratch S1, copied by the launch of a
        // constant digit next to the pass: the one before it (the pass then
        // reads S1 and writes the caller's buffers) or, for a pass on digit 0,
        // the one after it (the pass writes S1).  Argsort with every digit
        // constant fills the indices in digit 0's launch.  No launch of its own.
        const bool single = p == 1u && a.op != FSK_OP_ARGSORT;
        uint32_t single_digit = 0;
        for (uint32_t j = D; j-- > 0;)
            if (active[j]) single_digit = j;
        const bool copy_before = single && (compact || single_digit > 0u);
        const bool pairs = a.op == FSK_OP_PAIRS;
        uint32_t duty_digit = FS_MAX_DIGITS, duty = FS_DUTY_NONE, duty_ids = 0;
        if (p == 0u && a.op == FSK_OP_ARGSORT) {
            duty_digit = 0;
            duty = FS_DUTY_IOTA;
            duty_ids = FS_BUF_VALS << 24;
        } else if (copy_before) {
            duty_digit = compact ? 0u : single_digit - 1u;
            duty = FS_DUTY_COPY;
            duty_ids = FS_BUF_KEYS | (FS_BUF_S1K << 8) | (pairs ? (FS_BUF_VALS << 16) | (FS_BUF_S1V << 24) : 0u);
        } else if (single) {
            duty_digit = 1;
            duty = FS_DUTY_COPY;
            duty_ids = FS_BUF_S1K | (FS_BUF_KEYS << 8) | (pairs ? (FS_BUF_S1V << 16) | (FS_BUF_VALS << 24) : 0u);
        }
        uint32_t e = 0;
        uint32_t slot = compact && duty != FS_DUTY_NONE ? 1u : 0u;
        if (slot) {
            st_agent(&plan[0], duty << 24);
            st_agent(&plan[1], duty_ids);
        }
        for (uint32_t j = 0; j < FS_MAX_DIGITS; ++j) {
            uint32_t w0 = 0, w1 = 0;
            if (compact && !(j < D && active[j])) continue;
            if (j < D && active[j]) {
                const uint32_t flags = (e == 0 ? FS_PASS_FIRST : 0u) | (e + 1 == p ? FS_PASS_LAST : 0u) |
                                       ((cmask >> j) & FS_SKEW_BIT ? FS_PASS_SKEWED : 0u);
                w0 = 1u | (j << 1) | (e << 8) | (flags << 16);
                uint32_t sk = (e == 0) ? FS_BUF_KEYS : dk[e - 1];
                uint32_t sv = (e == 0) ? FS_BUF_VALS : dv[e - 1];   // unused by argsort's first pass
                uint32_t tk = dk[e], tv = dv[e];
                if (copy_before) {
                    sk = FS_BUF_S1K; sv = FS_BUF_S1V;
                    tk = FS_BUF_KEYS; tv = FS_BUF_VALS;
                }
#ifdef FS_FAULT_INJECTION
                if (a.fault == FS_FAULT_BAD_BUFFER && e == 0) tk = FS_BUF_S2V + 1u;   // no such buffer
#endif
                w1 = sk | (tk << 8) | (sv << 16) | (tv << 24);
                ++e;
            } else if (j == duty_digit) {
                w0 = duty << 24;
                w1 = duty_ids;
            }
            const uint32_t at = (compact ? slot++ : j) * FS_PLAN_PASS_WORDS;
            st_agent(&plan[at], w0);
            st_agent(&plan[at + 1], w1);
        }
        for (; compact && slot < FS_BK2_FEW_DIGITS; ++slot) st_agent(&plan[slot * FS_PLAN_PASS_WORDS], 0u);
        st_agent(&plan[FS_PLAN_NPASSES], p);
        st_agent(&plan[FS_PLAN_MASK], mask);
        st_agent(&plan[FS_PLAN_LOCAL], 0u);
        st_agent(&plan[FS_PLAN_RESCATTER], 0u);
    }
}

// ---------------------------------------------------------------------------
// fs_onesweep: one stable digit pass
// ---------------------------------------------------------------------------

// f(i) for the items (rows of 64 keys) i < rows, rows wave-uniform.  When
// every row is taken (a wave inside its segment) the rows run unrolled with
// no branch between them, so that their memory and LDS operations stay
// pipelined (a branch per row makes each load or read wait for its data
// before the next row starts); otherwise each row is behind a scalar branch.
template <int ITEMS, typename F>
DEV void for_rows(uint32_t rows, F&& f) {
    if (rows >= (uint32_t)ITEMS) {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) f(i);
    } else {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i)
            if ((uint32_t)i < rows) f(i);
    }
}

// Compile-time tag of for_rows_v: whether every key of the rows lies in the
// segment, so that no lane needs a bounds test.
template <bool B>
struct AllValid {
    static constexpr bool value = B;
};

// As for_rows, the unrolled branch-free copy taken when `full` (every key of
// every row in the segment: f(i, AllValid<true>)), the copy with a branch
// per row otherwise (f(i, AllValid<false>) for the rows i < rows).
template <int ITEMS, typename F>
DEV void for_rows_v(uint32_t rows, bool full, F&& f) {
    if (full) {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) f(i, AllValid<true>{});
    } else {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i)
            if ((uint32_t)i < rows) f(i, AllValid<false>{});
    }
}

// Ranks of a thread's items, two 16-bit values per register (a rank is below
// 2^16: within a wave at most 64 * ITEMS, within a tile below TILE).  Items
// are set in increasing order: an even item starts its register, the odd one
// is or-ed into the high half.
template <int ITEMS>
struct Ranks {
    uint32_t r[(ITEMS + 1) / 2];
    DEV uint32_t get(int i) const { return (i & 1) ? (r[i >> 1] >> 16) : (r[i >> 1] & 0xFFFFu); }
    DEV void set_in_order(int i, uint32_t v) {
        if (i & 1) r[i >> 1] |= v << 16;
        else r[i >> 1] = v;
    }
};

// Stable rank of each key among the keys of its wave with the same digit,
// in (item, lane) order; wb holds the wave's running digit counts.  x[i] is a
// 32-bit word holding item i's digit at bit xshift; DIGITS: x[i] is the digit
// itself (xshift 0).  rows (wave-uniform): the items ranked, the first rows
// ones; the others are left unset.
template <bool DIGITS, int ITEMS, int NB = FS_RADIX_BITS>
DEV void rank_wave(const uint32_t (&x)[ITEMS], uint32_t xshift, uint16_t* wb, Ranks<ITEMS>& rank,
                   uint32_t rows = ITEMS) {
    for_rows<ITEMS>(rows, [&](int i) {
        // 32-bit keys: the digit through the bit-field-extract intrinsic, a form
        // no other phase uses, so the compiler cannot keep one digit live across
        // phases
        const uint32_t d = DIGITS ? x[i] : __builtin_amdgcn_ubfe(x[i], xshift, NB);
        const uint64_t peers = match_digit<NB>(x[i], xshift);
        const uint32_t before = wb[d];
        // fresh(): the rank is computed here, not sunk into the staging loop
        // (which would keep the peer mask and count live per item instead)
        rank.set_in_order(i, fresh(lanes_below(peers, before)));
        // Every lane of a digit group reads the running count before any lane
        // stores the new one.  A wave executes in lockstep, so program order
        // gives this; the wave barrier keeps the compiler from moving the read
        // past the store and states the dependency.  All lanes of the group
        // store the same value, so no leader has to be chosen.
        __builtin_amdgcn_wave_barrier();
        // two v_bcnt_u32_b32 with accumulator; fresh() keeps the compiler from
        // reassociating the sum into two counts and an add3
        wb[d] = (uint16_t)((uint32_t)__builtin_popcount((uint32_t)(peers >> 32)) +
                           fresh((uint32_t)__builtin_popcount((uint32_t)peers) + before));
    });
}

// Decoupled look-back for digit d of `tile`, in two levels, over one chain of
// all tiles.  Every tile publishes its count (AGG) in its own entry, later
// replaced by its inclusive prefix (INC), and adds the count to its group's
// entry: FS_LB_GROUP consecutive tiles share one word per digit holding
// (tiles added << 24) | sum, complete once all the group's tiles have added.
// The look-back first reads the tile's own group back to the group start,
// FS_LB_WINDOW entries per round trip, then whole groups, FS_LB_GWIN per round
// trip, taking a group's sum when it is complete and its last tile's INC when
// that is published; it stops at the first INC or at tile 0 (which publishes
// INC).  Then it publishes this tile's INC.  Every wait is bounded
// (FS_SPIN_LIMIT).  WIDE selects the 64-bit tile entries.
template <bool WIDE>
DEV uint32_t lookback(GLOBAL uint32_t* lb, const GLOBAL uint32_t* grp, uint32_t tile, uint32_t d,
                      uint32_t valid, uint64_t status, uint32_t& rounds, uint32_t& stalls, uint32_t& entries,
                      uint32_t radix = FS_RADIX) {
    typedef LbEntry<WIDE> E;
    uint32_t excl = 0;
    uint32_t spins = 0;
    bool done = false;
    bool timed_out = false;
    auto stall = [&]() {
        ++stalls;
        if (++spins > FS_SPIN_LIMIT) {
            __hip_atomic_fetch_or((uint32_t*)status, FS_DEVERR_LOOKBACK_TIMEOUT,
                                  __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);   // reported, then bounded
            timed_out = true;
        } else {
            __builtin_amdgcn_s_sleep(1);
        }
    };

    // Level 1: the tiles of this tile's group below it.
    const uint32_t gstart = tile & ~(uint32_t)(FS_LB_GROUP - 1);
    uint32_t t = tile;              // entries below t are still to be read
    while (!done && !timed_out && t > gstart) {
        const uint32_t avail = min(t - gstart, (uint32_t)FS_LB_WINDOW);
        typename E::type e[FS_LB_WINDOW];
#pragma unroll
        for (int j = 0; j < FS_LB_WINDOW; ++j)
            e[j] = (j < (int)avail) ? E::load(lb, (uint64_t)(t - 1 - j) * radix + d) : 0u;
        uint32_t used = 0;
        bool stalled = false;
#pragma unroll
        for (int j = 0; j < FS_LB_WINDOW; ++j) {
            if (done || stalled || j >= (int)avail) continue;
            const uint32_t f = E::flags(e[j]);
            if (f == 0u) { stalled = true; continue; }
            excl += E::value(e[j]);
            ++used;
            // tile 0 always publishes INC; the bound keeps t in range regardless
            if (f == FS_LB_INC || t - 1 - j == 0u) done = true;
        }
        t -= used;
        ++rounds;
        entries += used;
        if (!done && stalled) stall();
    }

    // Level 2: whole groups below this tile's group, newest first.
    uint32_t g = gstart / FS_LB_GROUP;   // groups below g are still to be added
    while (!done && !timed_out && g > 0u) {
        const uint32_t avail = min(g, (uint32_t)FS_LB_GWIN);
        typename E::type ei[FS_LB_GWIN];
        uint32_t eg[FS_LB_GWIN];
#pragma unroll
        for (int j = 0; j < FS_LB_GWIN; ++j) {
            const uint64_t gg = g - 1 - j;
            ei[j] = (j < (int)avail) ? E::load(lb, (gg * FS_LB_GROUP + FS_LB_GROUP - 1) * radix + d) : 0u;
            eg[j] = (j < (int)avail) ? ld_agent(&grp[gg * radix + d]) : 0u;
        }
        uint32_t used = 0;
        bool stalled = false;
#pragma unroll
        for (int j = 0; j < FS_LB_GWIN; ++j) {
            if (done || stalled || j >= (int)avail) continue;
            if (E::flags(ei[j]) == FS_LB_INC) {
                excl += E::value(ei[j]);             // inclusive prefix through the end of the group
                done = true;
            } else if ((eg[j] >> FS_LB_GCOUNT_SHIFT) == FS_LB_GROUP) {
                excl += eg[j] & FS_LB_GSUM;          // the whole group
                ++used;
                if (g - 1 - j == 0u) done = true;
            } else {
                stalled = true;
            }
        }
        g -= used;
        ++rounds;
        entries += used;
        if (!done && stalled) stall();
    }
    E::store(lb, (uint64_t)tile * radix + d, FS_LB_INC, excl + valid);
    return excl;
}

// Tile processed by block b of a digit pass (grid: one block per tile).
// Blocks go to the XCDs round-robin (block b to XCD b % FS_XCDS) and each XCD
// starts its blocks in increasing order.  FS_XCD_TILES consecutive tiles go to
// one XCD: neighbouring tiles write the two halves of the same cache lines at
// every digit-run boundary, and on one XCD those writes merge in its L2
// instead of reaching HBM as two partial lines.  The last, partial round of
// groups keeps tile = block.
// Progress: on every XCD, blocks in start order take increasing tiles, and a
// tile only waits (look-back) on smaller tiles; the smallest unfinished tile
// therefore starts as soon as its XCD's earlier blocks - smaller tiles, all
// finished - leave, whatever the relative speed of the XCDs.  Should blocks
// be spread over the XCDs in another way, a block still waits on at most the
// next FS_XCDS * FS_XCD_TILES blocks, far fewer than the blocks a CU group
// holds; and every wait is bounded (FS_SPIN_LIMIT).
DEV uint32_t tile_of_block(uint32_t b, uint32_t num_tiles) {
    constexpr uint32_t R = FS_XCDS * FS_XCD_TILES;
    const uint32_t q = b / R, r = b % R;
    if ((uint64_t)q * R + R > num_tiles) return b;
    return FS_XCD_TILES * (FS_XCDS * q + r % FS_XCDS) + r / FS_XCDS;
}

// A lane's walk over the fused pass's region layout: region k holds the
// virtual positions [lo, hi) (region start table entries k and k + 1).
struct RegionWalk {
    uint32_t k, lo, hi;
    DEV void start(const FsArgs& a, uint32_t k0) {
        const GLOBAL uint32_t* rs = gptr<const uint32_t>(a.rstart);
        k = k0 < FS_REGIONS ? k0 : FS_REGIONS - 1u;
        lo = rs[k];
        hi = rs[k + 1];
    }
    // Index in S1 of virtual position p (p < n, p >= lo, positions of one lane
    // only grow): the walk moves forward to the region holding p, reading the
    // start table only when it crosses a region end.
    DEV uint64_t index(const FsArgs& a, uint32_t p) {
        const GLOBAL uint32_t* rs = gptr<const uint32_t>(a.rstart);
        while (p >= hi && k + 1u < FS_REGIONS) {
            ++k;
            lo = hi;
            hi = rs[k + 1];
        }
        return (uint64_t)gptr<const uint32_t>(a.rtable)[k] + (p - lo);
    }
};

// The descriptor of tile `tile` (two scalar loads; the table holds num_tiles
// descriptors on the fused path).
DEV void tile_desc(const FsArgs& a, uint32_t tile, uint64_t& d0, uint64_t& d1) {
    const CONSTANT uint64_t* dp = (const CONSTANT uint64_t*)(uintptr_t)a.tilemap + 2u * (uint64_t)tile;
    d0 = dp[0];
    d1 = dp[1];
}

// The value of the regions' digit that every key of a tile shares, from the
// second half of its descriptor, or FS_RADIX when the tile's regions hold
// several values.
DEV uint32_t tile_seg_w(uint64_t d1) {
    const uint32_t w = (uint32_t)(d1 >> 32);
    return (w & FS_TILE_ONE_DIGIT) ? (w & ~(FS_TILE_MULTI | FS_TILE_ONE_DIGIT)) / FS_SUBS : FS_RADIX;
}

// S1 indices of the positions first + i * STRIDE (i < N) of a tile in the
// fused pass's region layout; positions at or past n get an index that is
// never dereferenced.  The tile's descriptor d0, d1 (written by the fused
// pass's schedule step) gives, for a tile within at most two regions, the offset
// from position to index on either side of the region boundary, so that no
// memory access stands between the descriptor and the key loads; a tile over
// more regions copies its slice of the region start table into `table`
// (LDS, table_words words) once, or walks the table in memory when the slice
// does not fit.  Every thread of the block calls it (the descriptor is the
// block's, so the branch is uniform).
template <int N, uint32_t STRIDE, int BLOCK>
DEV void region_indices(const FsArgs& a, uint64_t d0, uint64_t d1, uint32_t first, uint32_t* table,
                        uint32_t table_words, uint32_t (&idx)[N]) {
    const uint32_t dx = (uint32_t)d0, dy = (uint32_t)(d0 >> 32), dz = (uint32_t)d1, dw = (uint32_t)(d1 >> 32);
    if (!(dw & FS_TILE_MULTI)) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const uint32_t p = first + (uint32_t)i * STRIDE;
            idx[i] = p + (p < dy ? dx : dz);
        }
        return;
    }
    const uint32_t k0 = dw & ~(FS_TILE_MULTI | FS_TILE_ONE_DIGIT), k1 = dx;
    const uint32_t cnt = (k0 <= k1 && k1 < FS_REGIONS) ? k1 - k0 + 2u : 0u;   // starts of regions k0 .. k1 + 1
    if (cnt != 0u && 2u * cnt <= table_words) {
        // the regions' starts, then their S1 bases
        const GLOBAL uint32_t* rs = gptr<const uint32_t>(a.rstart);
        const GLOBAL uint32_t* rb = gptr<const uint32_t>(a.rtable);
        for (uint32_t j = threadIdx.x; j < cnt; j += BLOCK) {
            table[j] = rs[k0 + j];
            table[cnt + j] = rb[k0 + j];
        }
        __syncthreads();
        uint32_t j = 0;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const uint32_t p = first + (uint32_t)i * STRIDE;
            while (j + 2u < cnt && p >= table[j + 1]) ++j;
            idx[i] = table[cnt + j] + (p - table[j]);
        }
        __syncthreads();                              // the table's area is the caller's again
        return;
    }
    RegionWalk rw;
    rw.start(a, k0);
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const uint32_t p = first + (uint32_t)i * STRIDE;
        idx[i] = p < (uint32_t)a.n ? (uint32_t)rw.index(a, p) : 0u;
    }
}

// Side duty of a constant digit's launch, one block per tile range: the copy
// that takes a single in-place pass through scratch, or argsort's index fill
// when every digit is constant (the schedule step assigns it).
template <bool K64, bool VALS, uint32_t TILE, int BLOCK>
DEV void pass_duty(const FsArgs& a, uint32_t duty, uint32_t ids, uint32_t unit, uint32_t* table,
                   uint32_t table_words) {
    typedef typename KeyT<K64>::type K;
    const uint64_t begin = (uint64_t)unit * TILE;
    const uint64_t end = begin + TILE < a.n ? begin + TILE : a.n;
    const uint64_t dst_v = VALS ? buf_addr(a, ids >> 24) : 0;
    if (duty == FS_DUTY_IOTA && VALS && dst_v) {
        GLOBAL uint32_t* out = gptr<uint32_t>(dst_v);
        for (uint64_t i = begin + threadIdx.x; i < end; i += BLOCK) out[i] = (uint32_t)i;
        return;
    }
    if (duty == FS_DUTY_UNREGION && !VALS) {
        // keys-only, only digit 0 varies: the fused pass's regions, in order,
        // to the caller's keys with the inverse transform
        const uint64_t src = buf_addr(a, ids & 0xFFu), dst = buf_addr(a, (ids >> 8) & 0xFFu);
        if (!src || !dst || !a.fused) {
            if (threadIdx.x == 0) report(a, FS_DEVERR_BAD_PLAN);
            return;
        }
        K xa, xb;
        xf_inv_masks<K64>(a.xform, xa, xb);
        const GLOBAL K* sk = gptr<const K>(src);
        GLOBAL K* dk = gptr<K>(dst);
        if (begin >= end) return;                    // (uniform) a block past the tiles
        constexpr int N = (int)((TILE + BLOCK - 1) / BLOCK);
        uint32_t idx[N];
        uint64_t d0, d1;
        tile_desc(a, unit, d0, d1);
        region_indices<N, (uint32_t)BLOCK, BLOCK>(a, d0, d1, (uint32_t)begin + threadIdx.x, table, table_words, idx);
        K v[N];
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const uint64_t i = begin + threadIdx.x + (uint64_t)j * BLOCK;
            v[j] = i < end ? sk[idx[j]] : (K)0;
        }
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const uint64_t i = begin + threadIdx.x + (uint64_t)j * BLOCK;
            if (i < end) dk[i] = xf_inv_apply<K64>(v[j], xa, xb);
        }
        return;
    }
    const bool with_vals = VALS && a.op == FSK_OP_PAIRS;
    const uint64_t src_k = buf_addr(a, ids & 0xFFu), dst_k = buf_addr(a, (ids >> 8) & 0xFFu);
    const uint64_t src_v = with_vals ? buf_addr(a, (ids >> 16) & 0xFFu) : 0;
    if (duty != FS_DUTY_COPY || !src_k || !dst_k || (with_vals && (!src_v || !dst_v))) {
        if (threadIdx.x == 0) report(a, FS_DEVERR_BAD_PLAN);
        return;
    }
    const GLOBAL K* sk = gptr<const K>(src_k);
    GLOBAL K* dk = gptr<K>(dst_k);
    for (uint64_t i = begin + threadIdx.x; i < end; i += BLOCK) dk[i] = sk[i];
    if (with_vals) {
        const GLOBAL uint32_t* sv = gptr<const uint32_t>(src_v);
        GLOBAL uint32_t* dv = gptr<uint32_t>(dst_v);
        for (uint64_t i = begin + threadIdx.x; i < end; i += BLOCK) dv[i] = sv[i];
    }
}

// ANY_ORDER: the first pass of a keys-only sort (digit 0), which needs no
// stability (below); otherwise a stable pass.
// unit: the block's tile in a launch of one block per tile (mapped to the
// XCDs by tile_of_block), or (PERSISTENT) the tile a block of a small grid
// takes in its loop over the tiles in increasing order.
template <bool K64, bool VALS, int BLOCK, int ITEMS, bool ANY_ORDER = false, bool PERSISTENT = false>
DEV void onesweep_body(const FsArgs& a, const uint32_t slot, const uint32_t unit) {
    typedef typename KeyT<K64>::type K;
    constexpr int WAVES = BLOCK / 64;
    constexpr uint32_t TILE = BLOCK * ITEMS;
    static_assert(BLOCK >= FS_RADIX && BLOCK % 64 == 0, "one thread per digit needed");
    static_assert((uint64_t)FS_LB_GROUP * TILE < (1ull << FS_LB_GCOUNT_SHIFT), "group sums must fit their field");

    __shared__ union {
        K keys[TILE];
        uint32_t vals[TILE];
    } stage;
    // per-wave digit counts, then tile-local bases: 16 bits hold both (a
    // wave counts at most 64 * ITEMS keys, a tile-local base is below TILE)
    __shared__ uint16_t wbase[WAVES][FS_RADIX];
    static_assert(TILE <= 0xFFFFu, "tile-local bases must fit 16 bits");
    __shared__ uint32_t gbase[FS_RADIX];          // global index of tile position 0 of each digit
    __shared__ uint32_t thist[FS_RADIX];          // tile digit counts (padding included)
    __shared__ uint32_t sstat[FS_STAT_COUNT];
    __shared__ uint32_t wsum[FS_RADIX / 64];

    if (slot >= a.digits || a.digits > FS_MAX_DIGITS) {      // the schedule holds FS_MAX_DIGITS passes
        if (threadIdx.x == 0) report(a, FS_DEVERR_BAD_DIGITS);
        return;
    }
    // The schedule was written by the upsweep, an earlier kernel, and is read-only
    // here: both words of this launch slot in one scalar load.
    static_assert(FS_PLAN_PASS_WORDS == 2, "one 64-bit schedule entry per slot");
    const uint64_t pw = ((const CONSTANT uint64_t*)(uintptr_t)a.plan)[slot];
    const uint32_t pw0 = (uint32_t)pw, pw1 = (uint32_t)(pw >> 32);
    const uint32_t digit = (pw0 >> 1) & 7u;       // the digit this slot sorts (< digits: checked below)
    if (slot == 0u && unit == 0u && ((const CONSTANT uint32_t*)(uintptr_t)a.plan)[FS_PLAN_RESCATTER]) {
        // the fused pass's re-scatter launch left its region fills in the
        // cursors, which start the next sort at zero
        GLOBAL uint32_t* cursors = gptr<uint32_t>(a.cursors);
        for (uint32_t i = threadIdx.x; i < FS_REGIONS; i += BLOCK) st_agent(&cursors[i], 0u);
    }
    if (!(pw0 & 1u)) {                             // no pass in this slot (a constant digit)
        if (pw0 >> 24)
            pass_duty<K64, VALS, BLOCK * ITEMS, BLOCK>(a, pw0 >> 24, pw1, unit, reinterpret_cast<uint32_t*>(&stage),
                                                      (uint32_t)(sizeof(stage) / 4));
        return;
    }
    if (digit >= a.digits) {
        if (threadIdx.x == 0) report(a, FS_DEVERR_BAD_DIGITS);
        return;
    }
    const uint32_t exec_index = (pw0 >> 8) & 0xFFu;
    const uint32_t pflags = (pw0 >> 16) & 0xFFu;
    const uint64_t src_k_addr = buf_addr(a, pw1 & 0xFFu), dst_k_addr = buf_addr(a, (pw1 >> 8) & 0xFFu);
    const uint64_t src_v_addr = VALS ? buf_addr(a, (pw1 >> 16) & 0xFFu) : 0;
    const uint64_t dst_v_addr = VALS ? buf_addr(a, pw1 >> 24) : 0;
    const bool argsort_first = VALS && (pflags & FS_PASS_FIRST) && a.op == FSK_OP_ARGSORT;
    if (src_k_addr == 0 || dst_k_addr == 0 ||
        (VALS && (dst_v_addr == 0 || (src_v_addr == 0 && !argsort_first)))) {
        if (threadIdx.x == 0) report(a, FS_DEVERR_BAD_PLAN);
        return;
    }

    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u;
    const uint32_t w = tid >> 6;
    const uint32_t shift = 8u * digit;
    const bool first = (pflags & FS_PASS_FIRST) != 0;
    const bool last = (pflags & FS_PASS_LAST) != 0;
    static_assert(!(ANY_ORDER && VALS), "argsort and pairs need a stable first pass");
    if (ANY_ORDER && !first) {                     // digit 0, when it has a pass, is the first
        if (tid == 0) report(a, FS_DEVERR_BAD_PLAN);
        return;
    }
    const uint32_t n32 = (uint32_t)a.n;

    const uint32_t tile = PERSISTENT ? unit : tile_of_block(unit, a.num_tiles);
    if (tile >= a.num_tiles) {                     // never, for a grid of one block per tile
        if (tid == 0) report(a, FS_DEVERR_BAD_TILE);
        return;
    }

    // Look-back arrays: [num_tiles][256] tile entries (u32, or u64 when wide),
    // then u32 [groups][256] group entries; the two arrays alternate between
    // executed passes.
    const bool wide = a.wide != 0;
    GLOBAL uint32_t* lb = gptr<uint32_t>((exec_index & 1u) ? a.lookback1 : a.lookback0);
    GLOBAL uint32_t* lb_next = gptr<uint32_t>((exec_index & 1u) ? a.lookback0 : a.lookback1);
    const uint64_t tile_words = (uint64_t)a.num_tiles * FS_RADIX * (wide ? 2u : 1u);
    GLOBAL uint32_t* grp = lb + tile_words;
    GLOBAL uint32_t* grp_next = lb_next + tile_words;
    // This tile's entries of the other array (and its group's, by the group's
    // first tile) are dead (their pass is over) and must read "not ready" and
    // "empty" for the next executed pass.
    if (tid < FS_RADIX) {
        if (wide) LbEntry<true>::store(lb_next, (uint64_t)tile * FS_RADIX + tid, 0u, 0u);
        else LbEntry<false>::store(lb_next, (uint64_t)tile * FS_RADIX + tid, 0u, 0u);
        if (tile % FS_LB_GROUP == 0) st_agent(&grp_next[(uint64_t)(tile / FS_LB_GROUP) * FS_RADIX + tid], 0u);
    }

    // ---- load (wave-striped: item i of lane l is tile key w*64*ITEMS + i*64 + l)
    const uint32_t tile_begin = tile * TILE;               // < n < 2^32
    // Key indices of the last tile's upper waves can pass 2^32 when n is
    // within a tile of it: index arithmetic and bounds tests in 64 bits.
    const uint64_t wave_begin = (uint64_t)tile_begin + w * 64u * ITEMS;
    const bool full_tile = (uint64_t)tile_begin + TILE <= a.n;
    const GLOBAL K* src_k = gptr<const K>(src_k_addr) + wave_begin + lane;
    K k[ITEMS];
    // A tile may take its keys' slots in any order within a digit when no two
    // of its keys need an order: in the first pass (ANY_ORDER), and in the pass
    // over the fused pass's regions for a tile inside one region (its keys
    // share digit 0; the look-back's tile order keeps the regions' order).
    bool unstable = ANY_ORDER;
    // top-16 path: the value of the regions' digit (the one below the top
    // byte) every key of the tile shares (a tile inside one value's regions),
    // or FS_RADIX
    uint32_t seg_w = FS_RADIX;
    const bool segcount = !VALS && (pflags & FS_PASS_SEGCOUNT) != 0u;
    bool seg_first = true, seg_last = true;             // (a one-value tile: first / last of its value's tiles)
    if (!VALS && (pflags & FS_PASS_REGIONED)) {
        // the first pass after a fused first pass: the keys in digit-0 order
        // are the regions of S1 in order (a region change inside a tile is
        // rare: each lane walks the region start table forward)
        if (!a.fused) {
            if (tid == 0) report(a, FS_DEVERR_BAD_PLAN);
            return;
        }
        const GLOBAL K* base = gptr<const K>(src_k_addr);
        uint64_t d0, d1;
        tile_desc(a, tile, d0, d1);
        // A wave whose positions all lie on one side of the tile's region
        // boundary (all but at most one wave of a tile; a tile inside one
        // region has no boundary) reads them at one offset: one base address
        // and the same loads as an ordinary pass.  (uint32 index arithmetic as
        // in region_indices; the index of a position below n fits 32 bits.)
        const uint32_t dx = (uint32_t)d0, dy = (uint32_t)(d0 >> 32), dz = (uint32_t)d1;
        const uint32_t wf = (uint32_t)wave_begin, wl = wf + (uint32_t)(ITEMS - 1) * 64u + 63u;
        const bool multi = ((uint32_t)(d1 >> 32) & FS_TILE_MULTI) != 0u;         // block-uniform
        if ((uint32_t)(d1 >> 32) & FS_TILE_ONE_DIGIT) {                         // one value of the regions' digit
            unstable = true;
            seg_w = tile_seg_w(d1);
            if (segcount) {
                uint64_t e0, e1;
                if (tile > 0u) {
                    tile_desc(a, tile - 1u, e0, e1);
                    seg_first = tile_seg_w(e1) != seg_w;
                }
                if (tile + 1u < a.num_tiles) {
                    tile_desc(a, tile + 1u, e0, e1);
                    seg_last = tile_seg_w(e1) != seg_w;
                }
            }
        }
        if (!multi && (wl < dy || wf >= dy)) {                                    // wave-uniform
            const GLOBAL K* src_r = base + (uint32_t)(wf + (wl < dy ? dx : dz)) + lane;
            if (full_tile) {
#pragma unroll
                for (int i = 0; i < ITEMS; ++i) k[i] = src_r[i * 64];
            } else {
#pragma unroll
                for (int i = 0; i < ITEMS; ++i) k[i] = (wave_begin + i * 64 + lane < a.n) ? src_r[i * 64] : (K)0;
            }
        } else {
            // (the multi-region path synchronises the block: every wave of a
            // multi-region tile takes it)
            uint32_t idx[ITEMS];
            region_indices<ITEMS, 64u, BLOCK>(a, d0, d1, (uint32_t)wave_begin + lane,
                                              reinterpret_cast<uint32_t*>(&stage), (uint32_t)(sizeof(stage) / 4), idx);
            if (full_tile) {
#pragma unroll
                for (int i = 0; i < ITEMS; ++i) k[i] = base[idx[i]];
            } else {
#pragma unroll
                for (int i = 0; i < ITEMS; ++i) k[i] = (wave_begin + i * 64 + lane < a.n) ? base[idx[i]] : (K)0;
            }
        }
    } else if (full_tile) {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) k[i] = src_k[i * 64];
    } else {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) k[i] = (wave_begin + i * 64 + lane < a.n) ? src_k[i * 64] : (K)0;
    }
    // The tile histogram of a skewed digit (FS_PASS_SKEWED) in replicated
    // counters: word [d][lane % HR] counts digit d for the lanes of that
    // residue, so that the lanes of a half-wave hit different banks whatever
    // their digits; they live in the staging area, free until the tile is
    // staged.  Other digits count into thist[], a wave with a dominant digit
    // adding that digit's lanes with one atomic (add_peeled): cheaper when no
    // bin dominates, as the replicas cost a clear and a 32-way sum per digit.
    // (32 replicas; fewer where a small test tile's staging area holds fewer)
    constexpr uint32_t HW = (uint32_t)(sizeof(stage) / (FS_RADIX * 4u));
    constexpr uint32_t HR = HW >= 32u ? 32u : HW >= 16u ? 16u : HW >= 8u ? 8u : HW >= 4u ? 4u : HW >= 2u ? 2u : 1u;
    static_assert(HW >= 1u && sizeof(stage) >= FS_RADIX * HR * 4u, "replicated histogram fits the staging area");
    uint32_t* thr = reinterpret_cast<uint32_t*>(&stage);
    // LDS clears and the barrier overlap the loads above.
    for (uint32_t i = tid; i < WAVES * FS_RADIX / 2; i += BLOCK) ((uint32_t*)&wbase[0][0])[i] = 0u;
    // (32-bit keys only: measured neutral on skewed 64-bit keys, and the
    // extra path cost the 64-bit pass 1% on uniform keys)
    const bool rep_hist = !K64 && (pflags & FS_PASS_SKEWED) != 0u;     // uniform
    if (rep_hist) {
        for (uint32_t i = tid; i < FS_RADIX * HR / 4u; i += BLOCK) reinterpret_cast<uint4*>(thr)[i] = uint4{0u, 0u, 0u, 0u};
    } else if (tid < FS_RADIX) {
        thist[tid] = 0u;
    }
    if (tid < FS_STAT_COUNT) sstat[tid] = 0u;
    __syncthreads();
    if (first) {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) k[i] = xf_fwd<K64>(k[i], a.xform);
    }
    if (!full_tile) {
        // Padding keys rank last in digit 255 and are never stored.
#pragma unroll
        for (int i = 0; i < ITEMS; ++i)
            if (wave_begin + i * 64 + lane >= a.n) k[i] = ~(K)0;
    }

    const bool chain_head = tile == 0u;
    const GLOBAL uint32_t* bb = gptr<const uint32_t>(a.binbase) + (uint64_t)digit * FS_RADIX;
    Ranks<ITEMS> rank;
    uint32_t lb_rounds = 0, lb_stalls = 0, lb_entries = 0;

    // Histogram, publish, look back and publish the inclusive prefix before
    // ranking: the inclusive frontier then trails the newest tiles closely and
    // successors walk short chains.
    // Digits of the register-held keys.  64-bit keys: one byte permute of the
    // key's halves (selector: byte shift/8 of the 64-bit key into byte 0, zero
    // bytes above), computed once and kept (8 items leave room in the register
    // budget).  32-bit keys: recomputed in each phase from the key, in a form of
    // the phase's own (16 items leave no room for 16 digits).
    const uint32_t psel = 0x0C0C0C00u | (shift >> 3);
    uint32_t dg[K64 ? ITEMS : 1];
    if constexpr (K64) {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) dg[i] = __builtin_amdgcn_perm((uint32_t)(k[i] >> 32), (uint32_t)k[i], psel);
    }
    auto hist_digit = [&](int i) -> uint32_t {
        if constexpr (K64) return dg[i];
        else return digit_of<K64>(k[i], shift);
    };
    constexpr int SB = (FS_STAGE_BATCH > 0 && FS_STAGE_BATCH < ITEMS) ? FS_STAGE_BATCH : ITEMS;
    Ranks<VALS ? ITEMS : 1> pos;                   // tile positions, kept for the values
    // ---- tile histogram (the skew test on the wave's first item is for the
    // first pass's slots below)
    const uint32_t d0 = hist_digit(0);
    const bool skew = skewed_digit(d0 == __builtin_amdgcn_readfirstlane(d0));
    if (rep_hist) {
        uint32_t* hc = thr + (lane % HR);
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) atomicAdd(&hc[hist_digit(i) * HR], 1u);
    } else if (skew) {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) add_peeled(thist, hist_digit(i), lane);
    } else {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) atomicAdd(&thist[hist_digit(i)], 1u);
    }
    __syncthreads();
    if (tid < FS_RADIX) {
        const uint32_t d = tid;
        uint32_t count = 0;
        if (rep_hist) {
#pragma unroll
            for (uint32_t r = 0; r < HR; ++r) count += thr[d * HR + (r + d) % HR];   // rotated: no bank conflicts
        } else {
            count = thist[d];
        }
        uint32_t valid = count;
        if (d == FS_RADIX - 1 && !full_tile) valid -= tile_begin + TILE - n32;
#ifdef FS_FAULT_INJECTION
        const bool publish = !(a.fault == FS_FAULT_STALL_TILE && exec_index == 0 && tile == 1u);
#else
        constexpr bool publish = true;
#endif
        if (publish) {
            if (wide) LbEntry<true>::store(lb, (uint64_t)tile * FS_RADIX + d, chain_head ? FS_LB_INC : FS_LB_AGG, valid);
            else LbEntry<false>::store(lb, (uint64_t)tile * FS_RADIX + d, chain_head ? FS_LB_INC : FS_LB_AGG, valid);
            __hip_atomic_fetch_add(&grp[(uint64_t)(tile / FS_LB_GROUP) * FS_RADIX + d],
                                   (1u << FS_LB_GCOUNT_SHIFT) | valid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        const uint32_t inc = wave_inclusive_scan(count);
        if (lane == 63) wsum[w] = inc;
        thist[d] = inc - count;
        gbase[d] = valid;
    }
    __syncthreads();
    if (tid < FS_RADIX) {
        const uint32_t d = tid;
        uint32_t local_excl = thist[d];
        for (uint32_t ww = 0; ww < w; ++ww) local_excl += wsum[ww];
        const uint32_t valid = gbase[d];
#ifdef FS_FAULT_INJECTION
        const bool stalled = a.fault == FS_FAULT_STALL_TILE && exec_index == 0 && tile == 1u;   // publishes nothing
#else
        constexpr bool stalled = false;
#endif
        const uint32_t excl = (chain_head || stalled) ? 0u
            : wide ? lookback<true>(lb, grp, tile, d, valid, a.status, lb_rounds, lb_stalls, lb_entries)
                   : lookback<false>(lb, grp, tile, d, valid, a.status, lb_rounds, lb_stalls, lb_entries);
        gbase[d] = bb[d] + excl - local_excl;     // modulo 2^32; exact for every stored key
        thist[d] = local_excl;                    // tile-local base of digit d
        // top-16 path, a tile of one value w of the regions' digit: its keys
        // of top-digit value d all belong to segment (d, w).  The tiles of
        // one value are consecutive in the chain, so the segment's keys in
        // them number the inclusive prefix at the last such tile less the
        // exclusive prefix at the first: the first tile subtracts excl, the
        // last adds excl + valid, the ones between add nothing (one
        // counter atomic per digit for about two tiles per value, not for
        // every tile).  Tiles of several values count their runs below.
        if (segcount && seg_w < FS_RADIX) {
            const uint32_t add = (seg_first ? 0u - excl : 0u) + (seg_last ? excl + valid : 0u);
            if (add != 0u)
                __hip_atomic_fetch_add(gptr<uint32_t>(a.segc) + d * FS_RADIX + seg_w, add, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    if (unstable) {
        // The first pass of a keys-only sort, or a one-region tile of the pass
        // over the regions (above).  An LSD sort needs no stability in its
        // first pass (the order of equal digits is undone by the later
        // passes, and equal keys are indistinguishable), so instead of a
        // ballot ranking each key takes any free slot of its digit's run in
        // the tile: one LDS atomic with return on a second set of counters
        // (the per-wave counter area, zeroed above, which this tile does not
        // otherwise use).  Padding keys take no slot.
        uint32_t* slots = reinterpret_cast<uint32_t*>(&wbase[0][0]);
        static_assert(sizeof(wbase) >= FS_RADIX * sizeof(uint32_t), "slot counters fit the per-wave counter area");
        if (!skew && full_tile) {
#pragma unroll
            for (int i = 0; i < ITEMS; ++i) rank.set_in_order(i, atomicAdd(&slots[hist_digit(i)], 1u));
        } else if (!skew) {
#pragma unroll
            for (int i = 0; i < ITEMS; ++i)
                rank.set_in_order(i, slot_in_digit<false>(slots, hist_digit(i), lane, wave_begin + i * 64 + lane < a.n));
        } else {
#pragma unroll
            for (int i = 0; i < ITEMS; ++i)
                rank.set_in_order(i, slot_in_digit<true>(slots, hist_digit(i), lane,
                                                         full_tile || wave_begin + i * 64 + lane < a.n));
        }
    } else {
        if constexpr (K64) rank_wave<true, ITEMS>(dg, 0u, wbase[w], rank);
        else rank_wave<false, ITEMS>(k, shift, wbase[w], rank);
    }
    __syncthreads();
    if (!unstable && tid < FS_RADIX) {
        const uint32_t d = tid;
        uint32_t run = thist[d];
#pragma unroll
        for (int ww = 0; ww < WAVES; ++ww) {
            const uint32_t c = wbase[ww][d];
            wbase[ww][d] = (uint16_t)run;    // tile-local base of (wave, digit)
            run += c;
        }
    }
    if (a.stats && tid < FS_RADIX) {
        const uint32_t r = wave_inclusive_scan(lb_rounds), sl = wave_inclusive_scan(lb_stalls),
                       en = wave_inclusive_scan(lb_entries);
        if (lane == 63) {
            atomicAdd(&sstat[FS_STAT_ROUNDS], r);
            atomicAdd(&sstat[FS_STAT_STALLS], sl);
            atomicAdd(&sstat[FS_STAT_ENTRIES], en);
        }
    }
    __syncthreads();
    if (a.stats && tid == 0 && !chain_head) {
        // 64 slots keep the atomics of concurrent tiles apart
        GLOBAL unsigned long long* st = gptr<unsigned long long>(a.stats) + (tile & 63u) * FS_STAT_COUNT;
        atomicAdd(&st[FS_STAT_TILES], 1ull);
        atomicAdd(&st[FS_STAT_ROUNDS], (unsigned long long)sstat[FS_STAT_ROUNDS]);
        atomicAdd(&st[FS_STAT_STALLS], (unsigned long long)sstat[FS_STAT_STALLS]);
        atomicAdd(&st[FS_STAT_ENTRIES], (unsigned long long)sstat[FS_STAT_ENTRIES]);
    }

    // ---- stage the tile in digit order (all base reads issued first)
    if (unstable) {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            if (!(full_tile || wave_begin + i * 64 + lane < a.n)) continue;
            uint32_t r = thist[hist_digit(i)] + rank.get(i);
            r = r < TILE ? r : TILE - 1;           // a permutation of the valid positions; bound kept explicit
            stage.keys[r] = k[i];
        }
    } else {
        // 32-bit keys: the digit by a byte permute, again a form of its own
        // (FS_STAGE_BATCH items' base reads in flight at once)
#pragma unroll
        for (int c = 0; c < ITEMS; c += SB) {
            uint32_t wofs[SB];
#pragma unroll
            for (int i = 0; i < SB; ++i) {
                if (c + i >= ITEMS) continue;
                if constexpr (K64) wofs[i] = wbase[w][dg[c + i]];
                else wofs[i] = wbase[w][__builtin_amdgcn_perm(0u, (uint32_t)k[c + i], psel)];
            }
#pragma unroll
            for (int i = 0; i < SB; ++i) {
                if (c + i >= ITEMS) continue;
                uint32_t r = rank.get(c + i) + wofs[i];
                r = r < TILE ? r : TILE - 1;                 // a permutation of [0, TILE); bound kept explicit
                if (VALS) pos.set_in_order(c + i, r);
                stage.keys[r] = k[c + i];
            }
        }
    }
    __syncthreads();
    if constexpr (!VALS) {
        if (segcount && seg_w == FS_RADIX) {
            // top-16 path, a tile of several values of the regions' digit (in
            // their order, ranked stably): the staged tile is ordered by the
            // top 16 bits, so each run of one top-16 value [s, e) is one
            // segment's share; it adds e - s to that segment's counter, as -s
            // at the run's first position and +e at its last
            constexpr uint32_t TOPSH = 8u * sizeof(K) - 16u;
            GLOBAL uint32_t* segc = gptr<uint32_t>(a.segc);
            const uint32_t tv = full_tile ? TILE : n32 - tile_begin;
            for (uint32_t p = tid; p < tv; p += BLOCK) {
                const uint32_t sg = (uint32_t)(stage.keys[p] >> TOPSH);
                const uint32_t sp = p ? (uint32_t)(stage.keys[p - 1] >> TOPSH) : 0xFFFFFFFFu;
                const uint32_t sn = p + 1u < tv ? (uint32_t)(stage.keys[p + 1] >> TOPSH) : 0xFFFFFFFFu;
                if (sg != sp) __hip_atomic_fetch_add(&segc[sg], 0u - p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (sg != sn) __hip_atomic_fetch_add(&segc[sg], p + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    }

    // Values are loaded only now, so their registers are not live during the
    // ranking (the key stores below hide the load latency); argsort's first
    // pass generates them.
    uint32_t v[VALS ? ITEMS : 1];
    if (VALS) {
        if (first && a.op == FSK_OP_ARGSORT) {
#pragma unroll
            for (int i = 0; i < ITEMS; ++i) v[i] = (uint32_t)(wave_begin + i * 64 + lane);   // padding lanes: unused
        } else {
            const GLOBAL uint32_t* src_v = gptr<const uint32_t>(src_v_addr) + wave_begin + lane;
#pragma unroll
            for (int i = 0; i < ITEMS; ++i)
                v[i] = (full_tile || wave_begin + i * 64 + lane < a.n) ? src_v[i * 64] : 0u;
        }
    }

    // ---- write runs to HBM: every stage and base read of a thread is issued
    // before its stores, and the inverse transform is branch-free
    const uint32_t tile_valid = full_tile ? TILE : n32 - tile_begin;
    const bool store_keys = !(last && a.op == FSK_OP_ARGSORT);
    K xa, xb;
    xf_inv_masks<K64>(last ? a.xform : FS_XF_NONE, xa, xb);
    // Byte offsets of every key (and value) fit 32 bits: stores then address
    // from the buffer base with one 32-bit offset per lane.
    const bool off32 = a.n * sizeof(K) <= (1ull << 32);
    GLOBAL K* dst_k = gptr<K>(dst_k_addr);
    const bool fast_store = full_tile && off32 && xa == (K)0;
    uint32_t gpos[VALS ? ITEMS : 1];                  // kept for the values
#pragma unroll
    for (int c = 0; c < ITEMS; c += SB) {
        K sk[SB];
        uint32_t gp[SB];
#pragma unroll
        for (int j = 0; j < SB; ++j)
            if (c + j < ITEMS) sk[j] = stage.keys[(c + j) * BLOCK + tid];
#pragma unroll
        for (int j = 0; j < SB; ++j) {
            if (c + j >= ITEMS) continue;
            const uint32_t d = K64 ? __builtin_amdgcn_perm((uint32_t)((uint64_t)sk[j] >> 32), (uint32_t)sk[j], psel)
                                   : digit_of<K64>(sk[j], shift);
            gp[j] = gbase[d] + ((c + j) * BLOCK + tid);
            if (VALS) gpos[c + j] = gp[j];
        }
        // g < n holds for every valid position; the tests on g only keep a
        // wrong offset from turning into an out-of-bounds store
        if (store_keys) {
            if (fast_store) {
                GLOBAL char* dk = gptr<char>(dst_k_addr);
#pragma unroll
                for (int j = 0; j < SB; ++j)
                    if (c + j < ITEMS && gp[j] < n32) *(GLOBAL K*)(dk + gp[j] * (uint32_t)sizeof(K)) = sk[j];
            } else {
#pragma unroll
                for (int j = 0; j < SB; ++j)
                    if (c + j < ITEMS && (c + j) * BLOCK + tid < tile_valid && gp[j] < n32)
                        dst_k[gp[j]] = xf_inv_apply<K64>(sk[j], xa, xb);
            }
        }
    }
    if (VALS) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) stage.vals[pos.get(i)] = v[i];
        __syncthreads();
        GLOBAL uint32_t* dst_v = gptr<uint32_t>(dst_v_addr);
#pragma unroll
        for (int c = 0; c < ITEMS; c += SB) {
            uint32_t sv[SB];
#pragma unroll
            for (int j = 0; j < SB; ++j)
                if (c + j < ITEMS) sv[j] = stage.vals[(c + j) * BLOCK + tid];
            if (full_tile && off32) {
                GLOBAL char* dv = gptr<char>(dst_v_addr);
#pragma unroll
                for (int j = 0; j < SB; ++j)
                    if (c + j < ITEMS && gpos[c + j] < n32) *(GLOBAL uint32_t*)(dv + gpos[c + j] * 4u) = sv[j];
            } else {
#pragma unroll
                for (int j = 0; j < SB; ++j)
                    if (c + j < ITEMS && (c + j) * BLOCK + tid < tile_valid && gpos[c + j] < n32)
                        dst_v[gpos[c + j]] = sv[j];
            }
        }
    }
}

// ---------------------------------------------------------------------------
// fs_first_*: the fused first pass of keys-only sorts (region layout in
// fs_params.h).  One read of the caller's keys replaces the histogram read
// and the first digit pass: each tile counts digits 1.. for the later passes
// (folded into histogram copy tile % FS_HIST_SLOTS), ranks digit 0 in any
// order (LDS atomics with return, which also give the tile's digit-0
// histogram), takes the space of each digit run in its region with one atomic
// on the region's cursor, and writes the runs from LDS.  No look-back.  The
// tile that finishes last writes the schedule (fused_plan).
// ---------------------------------------------------------------------------

template <int BLOCK> DEV void fused_plan(const FsArgs& a, uint32_t* lds);
// Words of LDS the schedule step of the fused pass uses: region fills,
// region starts, digit totals.
#define FS_FUSED_PLAN_WORDS (2 * FS_REGIONS + 1 + FS_MAX_DIGITS * FS_RADIX)

// byte j of a key
template <bool K64>
DEV uint32_t key_byte(typename KeyT<K64>::type k, uint32_t j) {
    return (uint32_t)(k >> (8u * j)) & 0xFFu;
}

// LDS of the fused pass, declared once per kernel (its body is instantiated
// per scatter digit, which must not double the block's LDS).  Tile counts of
// the other digits (all but the scatter digit sd, in increasing order
// o_0 < o_1 < ...) live in replicated 16-bit counters in the staging area,
// which is free until the tile is staged: word [p][v][lane % R] counts value v
// of digit o_2p (low half) and of digit o_2p+1 (high half), so that the lanes
// of a half-wave that count the same plane hit different banks whatever their
// digits (R = 32; 8 for 64-bit keys, whose tile leaves room for fewer).
template <bool K64, int BLOCK, int ITEMS>
struct FirstPassLds {
    typedef typename KeyT<K64>::type K;
    static constexpr uint32_t TILE = BLOCK * ITEMS;
    static constexpr uint32_t OTHER = K64 ? 7u : 3u;   // digits counted for the later passes
    static constexpr uint32_t R = K64 ? 8u : 32u;
    static constexpr uint32_t PLANES = (OTHER + 1u) / 2u;
    static constexpr uint32_t HC_WORDS = PLANES * FS_RADIX * R;
    // the staging area; the tile's counters before staging, the last tile's
    // schedule step after it (16-byte aligned: the counters are cleared as uint4)
    union alignas(16) {
        K keys[TILE];
        uint32_t plan[FS_FUSED_PLAN_WORDS];
        uint32_t hc[HC_WORDS];
    } stage;
    uint32_t slots[FS_RADIX];                          // scatter-digit slot counters, then tile-local bases
    uint32_t gbase[FS_RADIX];                          // S1 index of tile position 0 of each digit run
    uint32_t wsum[FS_RADIX / 64];
    uint32_t s_last;
};

// SD: the scatter digit (the region sample's choice, read by the kernel
// entry; sd_table its raw value, checked here); 2 (32-bit keys) or 6 (64-bit
// keys) only on the top-16 path.
// A compile-time digit keeps the pass free of register spills (a digit read
// at run time spilled 100 bytes per lane, and that build gave wrong regions
// on the GPU while the CPU emulator's run of the same source was exact).
// unit: the block's tile in the one-block-per-tile launch (mapped to the
// XCDs by tile_of_block); PERSISTENT: the tile itself (the re-scatter launch's
// small grid loops over the tiles).
template <bool K64, int BLOCK, int ITEMS, uint32_t SD, bool PERSISTENT = false>
DEV void first_pass_body(const FsArgs& a, const uint32_t launch, const uint32_t sd_table, const uint32_t unit,
                         FirstPassLds<K64, BLOCK, ITEMS>& L) {
    typedef typename KeyT<K64>::type K;
    typedef FirstPassLds<K64, BLOCK, ITEMS> Lds;
    constexpr uint32_t TILE = Lds::TILE;
    constexpr uint32_t OTHER = Lds::OTHER;
    constexpr uint32_t DROP = 0xFFFFFFFFu;              // run dropped: its region is full
    static_assert(BLOCK >= FS_RADIX && BLOCK % 64 == 0, "a digit per thread");
    static_assert(SD == 0u || SD == (K64 ? 6u : 2u), "scatter digit 0, or the one below the top byte on the top-16 path");
    // threads that fold the other digits' counts: those past the first
    // FS_RADIX, or (blocks of FS_RADIX threads) all of them, after reserving
    constexpr bool SPLIT = BLOCK >= 2 * FS_RADIX;
    constexpr uint32_t FOLDERS = SPLIT ? BLOCK - FS_RADIX : BLOCK;
    constexpr uint32_t R = Lds::R;
    constexpr uint32_t PLANES = Lds::PLANES;
    // every wave of the block adds to word [p][v][lane % R]: one half counts at
    // most TILE / R keys
    static_assert((uint64_t)TILE / R <= 0xFFFFu, "a replica's count must fit 16 bits");
    auto& stage = L.stage;
    uint32_t* slots = L.slots;
    uint32_t* gbase = L.gbase;
    uint32_t* wsum = L.wsum;
    uint32_t& s_last = L.s_last;

    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    // launch 0 (fs_first_*) counts, scatters and writes the schedule; launch
    // 1 (fs_rescatter_*) re-scatters into the exact regions the schedule step
    // wrote after an overflow, or does nothing
    const bool rescatter = launch != 0u;
    if (rescatter && ((const CONSTANT uint32_t*)(uintptr_t)a.plan)[FS_PLAN_RESCATTER] == 0u) return;
    if (a.digits != (K64 ? 8u : 4u) || sd_table != SD) {   // the schedule step reports it
        if (tid == 0) report(a, FS_DEVERR_BAD_DIGITS);
    }
    constexpr uint32_t sd = SD;
    constexpr uint32_t sshift = 8u * sd;
    // the top-16 path needs the top digit's counts only (the bin bases of
    // the pass on the top digit); the LSD passes need every other digit's
    constexpr bool top16 = SD != 0u;
    constexpr uint32_t ncount = top16 ? 1u : OTHER;
    auto counted = [](uint32_t m) -> uint32_t { return top16 ? sd + 1u : (m < sd ? m : m + 1u); };   // digit o_m
    const uint32_t tile = PERSISTENT ? unit : tile_of_block(unit, a.num_tiles);
    if (tile >= a.num_tiles) {                         // never, for a grid of one block per tile
        if (tid == 0) report(a, FS_DEVERR_BAD_TILE);
        return;
    }
    // The region group of the tile: the XCD its block runs on when blocks are
    // dealt to the XCDs round-robin (tile_of_block), so that neighbouring runs
    // of a region are written through one L2.  Any value is correct.
    const uint32_t sub = (tile / FS_XCD_TILES) % FS_SUBS;
    const GLOBAL uint32_t* rtab = gptr<const uint32_t>(a.rtable);   // written by fs_region_sample_*

    if (!rescatter) {
        // The first stable pass after this one uses look-back array 0: this
        // tile's entries (and its group's, by the group's first tile) start
        // "not ready".
        GLOBAL uint32_t* lb0 = gptr<uint32_t>(a.lookback0);
        GLOBAL uint32_t* grp0 = lb0 + (uint64_t)a.num_tiles * FS_RADIX * (a.wide ? 2u : 1u);
        if (tid < FS_RADIX) {
            if (a.wide) LbEntry<true>::store(lb0, (uint64_t)tile * FS_RADIX + tid, 0u, 0u);
            else LbEntry<false>::store(lb0, (uint64_t)tile * FS_RADIX + tid, 0u, 0u);
            if (tile % FS_LB_GROUP == 0) st_agent(&grp0[(uint64_t)(tile / FS_LB_GROUP) * FS_RADIX + tid], 0u);
        }
        // top-16 path: the segment counters of the top digit's pass, and the
        // local sort's count of deferred segments, start at zero (the tiles
        // clear them between them)
        if (a.seg_bits) {
            GLOBAL uint32_t* segc = gptr<uint32_t>(a.segc);
            for (uint32_t i = tile * BLOCK + tid; i <= FS_SEGS; i += a.num_tiles * BLOCK) st_agent(&segc[i], 0u);
        }
    }

    // ---- load the caller's keys (wave-striped), apply the key transform
    const uint32_t n32 = (uint32_t)a.n;
    const uint32_t tile_begin = tile * TILE;
    const uint64_t wave_begin = (uint64_t)tile_begin + w * 64u * ITEMS;
    const bool full_tile = (uint64_t)tile_begin + TILE <= a.n;
    const GLOBAL K* src_k = gptr<const K>(a.keys) + wave_begin + lane;
    K k[ITEMS];
    if (full_tile) {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) k[i] = src_k[i * 64];
    } else {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) k[i] = (wave_begin + i * 64 + lane < a.n) ? src_k[i * 64] : (K)0;
    }
    static_assert(Lds::HC_WORDS % 4u == 0u, "counters cleared 16 bytes at a time");
    if (!rescatter)
        for (uint32_t i = tid; i < Lds::HC_WORDS / 4u; i += BLOCK) reinterpret_cast<uint4*>(stage.hc)[i] = uint4{0u, 0u, 0u, 0u};
    if (tid < FS_RADIX) slots[tid] = 0u;
    __syncthreads();
    {
        K xa, xb;
        xf_inv_masks<K64>(a.xform, xa, xb);
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) k[i] = xf_fwd_apply<K64>(k[i], xa, xb);
    }
    auto valid = [&](int i) -> bool { return full_tile || wave_begin + i * 64 + lane < a.n; };
    auto sdig = [&](K key) -> uint32_t { return digit_of<K64>(key, sshift); };

    // ---- the scatter digit: slots in any order (the counters end as the
    // tile histogram; a wave whose first item shares a digit over many lanes
    // takes those lanes' slots with one atomic); the other digits: the
    // replicated counts.
    Ranks<ITEMS> rank;
    {
        const uint32_t d0 = sdig(k[0]);
        const bool skew = skewed_digit(d0 == __builtin_amdgcn_readfirstlane(d0));
        if (!skew && full_tile) {
#pragma unroll
            for (int i = 0; i < ITEMS; ++i) rank.set_in_order(i, atomicAdd(&slots[sdig(k[i])], 1u));
        } else if (!skew) {
#pragma unroll
            for (int i = 0; i < ITEMS; ++i) rank.set_in_order(i, slot_in_digit<false>(slots, sdig(k[i]), lane, valid(i)));
        } else {
#pragma unroll
            for (int i = 0; i < ITEMS; ++i) rank.set_in_order(i, slot_in_digit<true>(slots, sdig(k[i]), lane, valid(i)));
        }
    }
    if (!rescatter) {
        uint32_t* hc = stage.hc + (lane % R);
#pragma unroll
        for (uint32_t m = 0; m < OTHER; ++m) {
            if (m >= ncount) break;                                  // (uniform)
            const uint32_t j = counted(m);
            const uint32_t plane = m / 2u, inc = m % 2u ? 0x10000u : 1u;
#pragma unroll
            for (int i = 0; i < ITEMS; ++i)
                if (valid(i)) atomicAdd(&hc[(plane * FS_RADIX + key_byte<K64>(k[i], j)) * R], inc);
        }
    }
    __syncthreads();

    // ---- runs: the first FS_RADIX threads take each digit run's space in its
    // region (one atomic with return); the folding threads add the counts of
    // the other digits to the histogram copy and wait until the folds are
    // done, so that the tile counts as finished only with its folds complete.
    GLOBAL uint32_t* cursors = gptr<uint32_t>(a.cursors);
    if (tid < FS_RADIX) {
        const uint32_t d = tid;
        const uint32_t count = slots[d];
        const uint32_t inc = wave_inclusive_scan(count);
        if (lane == 63) wsum[w] = inc;
        uint32_t g = DROP;
        if (count) {
            const uint32_t kreg = d * FS_SUBS + sub;
            const uint32_t cap = rtab[FS_RTABLE_CAPS + d], rbase = rtab[kreg];
            const uint32_t at = __hip_atomic_fetch_add(&cursors[kreg], count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (at <= cap && count <= cap - at) g = rbase + at;   // the run fits its region
        }
        slots[d] = inc - count;                       // wave-local exclusive
        gbase[d] = g;
    }
    if (!rescatter && (!SPLIT || tid >= FS_RADIX)) {
        // each row [p][v]: its replicas summed (read in a rotated order, so
        // that a half-wave's reads fall in different banks), both halves
        GLOBAL uint32_t* hist = gptr<uint32_t>(a.hist) + (uint64_t)(tile % FS_HIST_SLOTS) * FS_MAX_DIGITS * FS_RADIX;
        for (uint32_t row = SPLIT ? tid - FS_RADIX : tid; row < (ncount + 1u) / 2u * FS_RADIX; row += FOLDERS) {
            const uint32_t* rw = stage.hc + row * R;
            uint32_t lo = 0, hi = 0;
#pragma unroll
            for (uint32_t r = 0; r < R; ++r) {
                const uint32_t wv = rw[(r + row) % R];
                lo += wv & 0xFFFFu;
                hi += wv >> 16;
            }
            const uint32_t plane = row / FS_RADIX, v = row % FS_RADIX;
            const uint32_t m1 = 2u * plane, m2 = m1 + 1u;              // o_m of the low and high halves
            const uint32_t j1 = counted(m1), j2 = counted(m2);
            if (lo) __hip_atomic_fetch_add(&hist[j1 * FS_RADIX + v], lo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (hi && m2 < ncount)
                __hip_atomic_fetch_add(&hist[j2 * FS_RADIX + v], hi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __builtin_amdgcn_s_waitcnt(0);
    }
    __syncthreads();
    // this tile's reservations and folds are complete: take the ticket
    GLOBAL uint32_t* ticket = gptr<uint32_t>(a.plan) + FS_PLAN_TICKET;
    if (tid == 0)
        s_last = !rescatter &&
                 __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == a.num_tiles - 1u;
    if (tid < FS_RADIX) {
        const uint32_t d = tid;
        uint32_t local_excl = slots[d];
        for (uint32_t ww = 0; ww < w; ++ww) local_excl += wsum[ww];
        if (gbase[d] != DROP) gbase[d] -= local_excl;   // modulo 2^32; exact for every stored key
        slots[d] = local_excl;                          // tile-local base of digit d
    }
    __syncthreads();

    // ---- stage the tile in scatter-digit order, then write each run to its region
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        if (!valid(i)) continue;
        uint32_t r = slots[sdig(k[i])] + rank.get(i);
        r = r < TILE ? r : TILE - 1;                  // a permutation of the valid positions; bound kept explicit
        stage.keys[r] = k[i];
    }
    __syncthreads();
    const uint32_t tile_valid = full_tile ? TILE : n32 - tile_begin;
    const uint32_t bound = rtab[FS_REGIONS];          // the regions' total (at most FsArgs.s1_keys < 2^32)
    GLOBAL K* dst = gptr<K>(a.s1k);
    constexpr int SB = (FS_STAGE_BATCH > 0 && FS_STAGE_BATCH < ITEMS) ? FS_STAGE_BATCH : ITEMS;
#pragma unroll
    for (int c = 0; c < ITEMS; c += SB) {
        K sk[SB];
        uint32_t gb[SB];
#pragma unroll
        for (int j = 0; j < SB; ++j)
            if (c + j < ITEMS) sk[j] = stage.keys[(c + j) * BLOCK + tid];
#pragma unroll
        for (int j = 0; j < SB; ++j)
            if (c + j < ITEMS) gb[j] = gbase[sdig(sk[j])];
#pragma unroll
        for (int j = 0; j < SB; ++j) {
            if (c + j >= ITEMS) continue;
            const uint32_t pos = (c + j) * BLOCK + tid;
            const uint32_t gp = gb[j] + pos;
            if (pos < tile_valid && gb[j] != DROP && gp < bound) dst[gp] = sk[j];
        }
    }
    if (s_last) {                                      // uniform
        __threadfence();
        __syncthreads();                               // the staging area is free
        fused_plan<BLOCK>(a, stage.plan);
        if (tid == 0) st_agent(ticket, 0u);
    }
}

// Scan helper: exclusive prefix over the first FS_RADIX threads (one value
// each), with every thread of the block at the barriers.
DEV uint32_t radix_exclusive_scan(uint32_t v, uint32_t* wsum) {
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    uint32_t inc = 0;
    if (tid < FS_RADIX) {
        inc = wave_inclusive_scan(v);
        if (lane == 63) wsum[w] = inc;
    }
    __syncthreads();
    uint32_t excl = inc - v;
    if (tid < FS_RADIX)
        for (uint32_t ww = 0; ww < w; ++ww) excl += wsum[ww];
    __syncthreads();
    return excl;
}

DEV void write_fused_schedule(const FsArgs& a, uint32_t cmask, uint32_t D, bool exact);
DEV void write_top16_schedule(const FsArgs& a, uint32_t cmask, bool exact);

// fs_region_sample_*: the fused pass's region table (fs_params.h), one block
// of FS_HIST_BLOCK threads, before the pass.  The digit the pass scatters by
// (after the key transform; see below for how it is chosen) is counted over FS_SAMPLE_CHUNKS runs of FS_SAMPLE_CHUNK
// consecutive keys spread evenly over the input (every key when there are
// fewer); digit value d gets regions of cap[d] = 1.5 x max(share_d, 1/1024)
// of the fullest region group's keys (FsArgs.sub_keys), plus 64, and the
// regions are laid out in order.  Their total stays within FS_FUSED_S1_KEYS
// (the S1 the host sized); should it not (a bug), every region gets an equal
// part of S1 instead - still correct, a full region only costs the
// re-scatter into exact regions.
template <bool K64>
DEV void region_sample_body(const FsArgs& a) {
    typedef typename KeyT<K64>::type K;
    // the scatter digit of the top-16 path: the one below the top byte
    constexpr uint32_t TSD = K64 ? 6u : 2u, KBITS = 8u * sizeof(K);
    __shared__ uint32_t h[2][FS_RADIX];               // the sample's counts of digit 0 and digit TSD
    // top-16 launch sequence: 16-bit counts of the sample's top TB =
    // min(seg_bits, 15) bits, two per word (at most 2^15 samples each; 64 KiB,
    // within a block's LDS; with 16 segment bits a count covers two segments,
    // so the estimate errs high)
    __shared__ uint32_t seg[FS_SEGS / 4];
    __shared__ uint32_t wsum[FS_RADIX / 64];
    __shared__ uint32_t s_total, s_max;
    static_assert((uint64_t)FS_SAMPLE_CHUNKS * FS_SAMPLE_CHUNK <= 0xFFFFu, "16-bit segment counts");
    const uint32_t tid = threadIdx.x;
    const uint32_t S = a.seg_bits;
    const bool top = S >= 8u && S <= 16u;             // (uniform)
    const uint32_t TB = S < 15u ? S : 15u;
    for (uint32_t i = tid; i < 2 * FS_RADIX; i += FS_HIST_BLOCK) (&h[0][0])[i] = 0u;   // (blocks of 256 threads too)
    if (top)
        for (uint32_t i = tid; i < (1u << TB) / 2u; i += FS_HIST_BLOCK) seg[i] = 0u;
    if (tid == 0) s_max = 0u;
    __syncthreads();
    const uint64_t n = a.n;
    constexpr uint64_t SMP = (uint64_t)FS_SAMPLE_CHUNKS * FS_SAMPLE_CHUNK;
    const uint64_t taken = n < SMP ? n : SMP;
    const GLOBAL K* src = gptr<const K>(a.keys);
    K xa, xb;
    xf_inv_masks<K64>(a.xform, xa, xb);
    // wave w reads chunks [w * CPW, (w + 1) * CPW), 64 consecutive keys per
    // load; chunk c starts at c * step (<= n - FS_SAMPLE_CHUNK), or at
    // c * FS_SAMPLE_CHUNK when every key is taken.  The loads of a batch are
    // issued together: one round trip per batch, no division per key.
    constexpr uint32_t WAVES = FS_HIST_BLOCK / 64, CPW = FS_SAMPLE_CHUNKS / WAVES;
    constexpr uint32_t LPC = FS_SAMPLE_CHUNK / 64, PER = CPW * LPC, BATCH = K64 ? 16 : 32;   // (64-bit keys: registers)
    static_assert(FS_SAMPLE_CHUNKS % WAVES == 0 && FS_SAMPLE_CHUNK % 64 == 0 && PER % BATCH == 0, "sample layout");
    const uint32_t lane = tid & 63u, w = tid >> 6;
    const uint64_t step = n <= SMP ? (uint64_t)FS_SAMPLE_CHUNK : (n - FS_SAMPLE_CHUNK) / (FS_SAMPLE_CHUNKS - 1);
    for (uint32_t b0 = 0; b0 < PER; b0 += BATCH) {
        K k[BATCH];
        bool ok[BATCH];
#pragma unroll
        for (uint32_t j = 0; j < BATCH; ++j) {
            const uint32_t e = b0 + j, c = w * CPW + e / LPC;
            const uint64_t pos = (uint64_t)c * step + (e % LPC) * 64u + lane;
            ok[j] = pos < n;                           // (false only when every key is taken)
            k[j] = src[ok[j] ? pos : 0u];
        }
#pragma unroll
        for (uint32_t j = 0; j < BATCH; ++j) {
            // (every lane takes part, the keys past n counting nothing; where
            // many lanes share the first lane's value - a skewed or constant
            // digit or segment, which would serialise their atomics - the
            // lanes that share the first counted lane's value add with one)
            const K kt = xf_fwd_apply<K64>(k[j], xa, xb);
            const bool v = ok[j];
            const uint32_t d0 = digit_of<K64>(kt, 0u);
            if (skewed_digit(d0 == __builtin_amdgcn_readfirstlane(d0))) add_peeled_valid(h[0], d0, d0, 1u, lane, v);
            else if (v) atomicAdd(&h[0][d0], 1u);
            if (top) {
                const uint32_t t = (uint32_t)(kt >> (KBITS - TB)), dt = digit_of<K64>(kt, 8u * TSD);
                if (skewed_digit(dt == __builtin_amdgcn_readfirstlane(dt))) add_peeled_valid(h[1], dt, dt, 1u, lane, v);
                else if (v) atomicAdd(&h[1][dt], 1u);
                // two 16-bit segment counts per word: segment t adds to half t & 1
                if (skewed_digit(t == __builtin_amdgcn_readfirstlane(t)))
                    add_peeled_valid(seg, t, t >> 1, 1u << (16u * (t & 1u)), lane, v);
                else if (v)
                    atomicAdd(&seg[t >> 1], 1u << (16u * (t & 1u)));
            }
        }
    }
    __syncthreads();
    // The scatter digit: TSD (the top-16 path) unless the sample's largest
    // segment, scaled to the input, exceeds FsArgs.seg_limit (a count of at
    // least FS_SEG_MIN_SAMPLES, so that a uniform input's few sampled keys per
    // segment never decide); otherwise 0 (the LSD passes).
    uint32_t sd = 0;
    if (top) {
        uint32_t m = 0;
        for (uint32_t i = tid; i < (1u << TB) / 2u; i += FS_HIST_BLOCK) {
            const uint32_t v = seg[i];
            m = max(m, max(v & 0xFFFFu, v >> 16));
        }
        if (m) atomicMax(&s_max, m);
        __syncthreads();
        const uint32_t mx = s_max;
        sd = (mx < FS_SEG_MIN_SAMPLES || (uint64_t)mx * n <= (uint64_t)a.seg_limit * taken) ? TSD : 0u;
    }
    GLOBAL uint32_t* rt = gptr<uint32_t>(a.rtable);
    uint32_t cap = 0;
    if (tid < FS_RADIX) {
        // share_d * 1024 * taken, at least taken (1/1024); < 2^27, times
        // sub_keys < 2^32: fits 64 bits
        const uint32_t hc = h[sd == TSD ? 1 : 0][tid];
        const uint64_t num = (uint64_t)hc * 1024u > taken ? (uint64_t)hc * 1024u : taken;
        cap = (uint32_t)((3u * num * (uint64_t)a.sub_keys) / (2048u * taken)) + 64u;
    }
    const uint32_t dbase = radix_exclusive_scan(cap * FS_SUBS, wsum);   // every thread at the barriers
    if (tid == FS_RADIX - 1) s_total = dbase + cap * FS_SUBS;
    __syncthreads();
    const bool fits = s_total <= a.s1_keys && s_total >= dbase;        // (no wrap either)
    if (tid < FS_RADIX) {
        const uint32_t even = a.s1_keys / FS_REGIONS;
        const uint32_t c = fits ? cap : even, b = fits ? dbase : tid * FS_SUBS * even;
        for (uint32_t sb = 0; sb < FS_SUBS; ++sb) rt[tid * FS_SUBS + sb] = b + sb * c;
        rt[FS_RTABLE_CAPS + tid] = c;
        if (tid == 0) {
            rt[FS_REGIONS] = fits ? s_total : FS_REGIONS * even;
            rt[FS_RTABLE_SDIGIT] = sd;
        }
    }
}

extern "C" __global__ void __launch_bounds__(FS_HIST_BLOCK) fs_region_sample_k32(FsArgs a) {
    region_sample_body<false>(a);
}
extern "C" __global__ void __launch_bounds__(FS_HIST_BLOCK) fs_region_sample_k64(FsArgs a) {
    region_sample_body<true>(a);
}

// Region of position x in a region start table rs[0..FS_REGIONS] (LDS): the
// largest r with rs[r] <= x, which for x < n is the non-empty region holding x.
DEV uint32_t region_at(const uint32_t* rs, uint32_t x) {
    uint32_t lo = 0, len = FS_REGIONS;            // rs[lo] <= x (rs[0] = 0)
    while (len > 1u) {
        const uint32_t half = len >> 1;
        if (rs[lo + half] <= x) {
            lo += half;
            len -= half;
        } else {
            len = half;
        }
    }
    return lo;
}

// Schedule step of the fused pass, run by its last tile (every thread of the
// block; lds: FS_FUSED_PLAN_WORDS words).  Region fills from the cursors and
// the other digits' totals from the histogram copies, every load in flight at
// once (both cleared for the next sort, also when the digit count is wrong);
// bin bases of every digit and the constant digits; region starts; then the
// schedule: without an overflowing region (and unless every digit is
// constant) the digit-0 pass is done, the tile descriptors of the region
// layout are written, and the passes of the other digits follow, the first
// reading the regions; otherwise the standard schedule over the caller's
// untouched keys.
template <int BLOCK>
DEV void fused_plan(const FsArgs& a, uint32_t* lds) {
    __shared__ uint32_t f_wsum[FS_MAX_DIGITS][FS_RADIX / 64];
    __shared__ uint32_t f_cmask, f_over;
    uint32_t* fill = lds;                                   // [FS_REGIONS]
    uint32_t* rsl = lds + FS_REGIONS;                       // [FS_REGIONS + 1]
    uint32_t* tot = lds + 2 * FS_REGIONS + 1;               // [FS_MAX_DIGITS][FS_RADIX]
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    const uint32_t D = a.digits, Dk = a.key64 ? 8u : 4u;
    const uint32_t n32 = (uint32_t)a.n;
    const GLOBAL uint32_t* rtab = gptr<const uint32_t>(a.rtable);
    GLOBAL uint32_t* hist = gptr<uint32_t>(a.hist);
    GLOBAL uint32_t* base = gptr<uint32_t>(a.binbase);
    GLOBAL uint32_t* cursors = gptr<uint32_t>(a.cursors);
    GLOBAL uint32_t* rstart = gptr<uint32_t>(a.rstart);
    GLOBAL uint32_t* plan = gptr<uint32_t>(a.plan);
    if (tid == 0) {
        f_cmask = 0u;
        f_over = 0u;
    }
    constexpr uint32_t RPT = (FS_REGIONS + BLOCK - 1) / BLOCK;
    uint32_t fv[RPT];
#pragma unroll
    for (uint32_t r = 0; r < RPT; ++r) {
        const uint32_t i = tid + r * BLOCK;
        fv[r] = i < FS_REGIONS ? ld_agent(&cursors[i]) : 0u;
    }
#pragma unroll
    for (uint32_t r = 0; r < RPT; ++r) {
        const uint32_t i = tid + r * BLOCK;
        if (i < FS_REGIONS) {
            fill[i] = fv[r];
            st_agent(&cursors[i], 0u);
        }
    }
    const uint32_t sd = rtab[FS_RTABLE_SDIGIT] < Dk ? rtab[FS_RTABLE_SDIGIT] : 0u;   // the digit of the regions
    const bool top16 = a.seg_bits != 0u && sd == Dk - 2u;   // regions by the digit below the top byte
    for (uint32_t e = tid; e < (Dk - 1u) * FS_RADIX; e += BLOCK) {   // digit o_(e / 256), bin e % 256
        const uint32_t m = e / FS_RADIX, j = m < sd ? m : m + 1u, d = e % FS_RADIX;
        uint32_t v[FS_HIST_SLOTS];
#pragma unroll
        for (uint32_t sl = 0; sl < FS_HIST_SLOTS; ++sl) v[sl] = ld_agent(&hist[(sl * FS_MAX_DIGITS + j) * FS_RADIX + d]);
        uint32_t t = 0;
#pragma unroll
        for (uint32_t sl = 0; sl < FS_HIST_SLOTS; ++sl) t += v[sl];
#pragma unroll
        for (uint32_t sl = 0; sl < FS_HIST_SLOTS; ++sl) st_agent(&hist[(sl * FS_MAX_DIGITS + j) * FS_RADIX + d], 0u);
        tot[j * FS_RADIX + d] = t;
    }
    __syncthreads();
    if (D != Dk) {                                          // reported by the tiles; no pass runs (uniform)
        if (tid < FS_PLAN_WORDS && tid != FS_PLAN_TICKET) st_agent(&plan[tid], 0u);
        return;
    }
    const bool bin = tid < FS_RADIX;
    const uint32_t d = tid;
    if (bin) {                                              // digit sd: the region fills
        uint32_t t = 0, over = 0;
        const uint32_t cap = rtab[FS_RTABLE_CAPS + d];
#pragma unroll
        for (uint32_t s = 0; s < FS_SUBS; ++s) {
            const uint32_t f = fill[d * FS_SUBS + s];
            t += f;
            over |= f > cap ? 1u : 0u;
        }
        tot[sd * FS_RADIX + d] = t;
        if (over) atomicOr(&f_over, 1u);
    }
    __syncthreads();
    // exclusive scans of every digit's totals over the bins at once; digit j
    // is constant when one bin holds every key
    uint32_t totals[FS_MAX_DIGITS], inc[FS_MAX_DIGITS];
    uint32_t mine = 0;
#pragma unroll
    for (uint32_t j = 0; j < FS_MAX_DIGITS; ++j) {
        totals[j] = (bin && j < Dk) ? tot[j * FS_RADIX + d] : 0u;
        inc[j] = wave_inclusive_scan(totals[j]);
        if (bin && j < Dk && totals[j] == n32) mine |= 1u << j;
        if (bin && j < Dk && totals[j] > n32 / FS_SKEW_SHARE) mine |= FS_SKEW_BIT << j;
    }
    if (bin && lane == 63) {
#pragma unroll
        for (uint32_t j = 0; j < FS_MAX_DIGITS; ++j) f_wsum[j][w] = inc[j];
    }
    if (mine) atomicOr(&f_cmask, mine);
    __syncthreads();
    if (bin) {
#pragma unroll
        for (uint32_t j = 0; j < FS_MAX_DIGITS; ++j) {
            if (j >= Dk) break;
            uint32_t excl = inc[j] - totals[j];
            for (uint32_t v = 0; v < w; ++v) excl += f_wsum[j][v];
            base[j * FS_RADIX + d] = excl;
            if (j == sd) {                                  // region starts: regions in order
                uint32_t at = excl;
#pragma unroll
                for (uint32_t s = 0; s < FS_SUBS; ++s) {
                    rsl[d * FS_SUBS + s] = at;
                    rstart[d * FS_SUBS + s] = at;
                    at += fill[d * FS_SUBS + s];
                }
            }
        }
        if (d == 0) {
            rsl[FS_REGIONS] = n32;
            rstart[FS_REGIONS] = n32;
        }
    }
    __syncthreads();
    const uint32_t all = (1u << D) - 1u;
    const bool every_constant = (f_cmask & all) == all;
    // After an overflow the second launch of the fused pass re-scatters the
    // keys into exact regions - region k at S1 + its start in digit order,
    // holding exactly its fill (the second launch's tiles add the same counts
    // to the same regions) - and the schedule goes on as without one.
    const bool exact = f_over != 0u && !every_constant;
    if (exact) {
        GLOBAL uint32_t* rt = gptr<uint32_t>(a.rtable);
        for (uint32_t k = tid; k < FS_REGIONS; k += BLOCK) rt[k] = rsl[k];
        if (tid < FS_RADIX) rt[FS_RTABLE_CAPS + tid] = 0xFFFFFFFFu;
        if (tid == 0) rt[FS_REGIONS] = n32;
    }
    const bool fast = !every_constant;
    if (fast) {
        // the descriptor of every tile of the next pass: each non-empty region
        // writes those of the tiles whose first key it holds
        GLOBAL uint32_t* desc = gptr<uint32_t>(a.tilemap);
        const uint32_t T = a.tile;
        // S1 index of region k's first key: its base in the sampled layout, or
        // its start in the exact one
        auto rbase = [&](uint32_t k) -> uint32_t { return exact ? rsl[k] : rtab[k]; };
        for (uint32_t k = tid; k < FS_REGIONS; k += BLOCK) {
            const uint32_t lo = rsl[k], hi = rsl[k + 1];
            if (lo == hi) continue;
            const uint32_t phys0 = rbase(k) - lo;           // index - position in region k
            // first tile whose first key lies in the region (in 64 bits, so
            // that lo + T cannot wrap whatever n)
            for (uint32_t t = (uint32_t)(((uint64_t)lo + T - 1u) / T); (uint64_t)t * T < hi; ++t) {
                const uint32_t p0 = t * T;
                const uint32_t pend = n32 - p0 < T ? n32 : p0 + T;
                uint32_t x = phys0, y = 0xFFFFFFFFu, z = phys0, wd = k, last = k;
                if (pend > hi) {                            // the tile runs past region k
                    const uint32_t k1 = region_at(rsl, hi);
                    if (pend <= rsl[k1 + 1]) {
                        y = hi;
                        z = rbase(k1) - hi;
                        last = k1;
                    } else {
                        x = last = region_at(rsl, pend - 1u);
                        y = z = 0u;
                        wd = k | FS_TILE_MULTI;
                    }
                }
                // regions in order: the tile's keys share digit 0 when its
                // first and last regions do
                if (k / FS_SUBS == last / FS_SUBS) wd |= FS_TILE_ONE_DIGIT;
                GLOBAL uint32_t* q = desc + (uint64_t)t * FS_TILE_DESC_WORDS;
                q[0] = x;
                q[1] = y;
                q[2] = z;
                q[3] = wd;
            }
        }
    }
    if (tid == 0) {
        if (fast && top16) write_top16_schedule(a, f_cmask, exact);
        else if (fast) write_fused_schedule(a, f_cmask, D, exact);
        else write_schedule<false>(a, f_cmask, D);
    }
}

// Schedule after a fused first pass on digit 0 (its regions sampled, or
// exact when `exact`, which the fused pass's second launch then fills):
// digit 0 needs no pass; the passes of the other non-constant digits take the
// digit-pass launch slots 0, 1, ... in order, with execution indices from 0
// (look-back array 0, cleared by the fused pass), the first reading the
// regions of S1 (no key transform: the fused pass applied it), the last
// writing the caller's keys with the inverse transform.  Their destinations
// alternate S2, S1, ... and end in the caller's keys.  With no other digit
// varying, slot 0's launch copies the regions to the caller's keys instead
// (FS_DUTY_UNREGION).
DEV void write_fused_schedule(const FsArgs& a, uint32_t cmask, uint32_t D, bool exact) {
    GLOBAL uint32_t* plan = gptr<uint32_t>(a.plan);
    uint32_t r = 0, mask = 1u;                          // digit 0 was sorted by the fused pass
    for (uint32_t j = 1; j < D; ++j)
        if (!((cmask >> j) & 1u)) { ++r; mask |= 1u << j; }
    uint32_t w0s[FS_MAX_DIGITS], w1s[FS_MAX_DIGITS];
    for (uint32_t e = 0; e < FS_MAX_DIGITS; ++e) w0s[e] = w1s[e] = 0u;
    if (r == 0) {
        w0s[0] = FS_DUTY_UNREGION << 24;
        w1s[0] = FS_BUF_S1K | (FS_BUF_KEYS << 8);
    }
    uint32_t e = 0;
    for (uint32_t j = 1; j < D && j < FS_MAX_DIGITS; ++j) {
        if ((cmask >> j) & 1u) continue;
        const uint32_t flags = (e == 0 ? FS_PASS_REGIONED : 0u) | (e + 1 == r ? FS_PASS_LAST : 0u) |
                               ((cmask >> j) & FS_SKEW_BIT ? FS_PASS_SKEWED : 0u);
        w0s[e] = 1u | (j << 1) | (e << 8) | (flags << 16);
        const uint32_t sk = e == 0 ? FS_BUF_S1K : ((e - 1) % 2 == 0 ? FS_BUF_S2K : FS_BUF_S1K);
        uint32_t tk = e + 1 == r ? FS_BUF_KEYS : (e % 2 == 0 ? FS_BUF_S2K : FS_BUF_S1K);
#ifdef FS_FAULT_INJECTION
        if (a.fault == FS_FAULT_BAD_BUFFER && e == 0) tk = FS_BUF_S2V + 1u;   // no such buffer
#endif
        w1s[e] = sk | (tk << 8);
        ++e;
    }
    for (uint32_t sl = 0; sl < FS_MAX_DIGITS; ++sl) {
        st_agent(&plan[sl * FS_PLAN_PASS_WORDS], w0s[sl]);
        st_agent(&plan[sl * FS_PLAN_PASS_WORDS + 1], w1s[sl]);
    }
    st_agent(&plan[FS_PLAN_NPASSES], r + 1u);             // the fused pass counts as digit 0's
    st_agent(&plan[FS_PLAN_MASK], mask | FS_MASK_FUSED);
    st_agent(&plan[FS_PLAN_LOCAL], 0u);
    st_agent(&plan[FS_PLAN_RESCATTER], exact ? 1u : 0u);
}

// Schedule of the top-16 path after its fused pass (regions by the digit
// below the top byte - digit 2 of 32-bit keys, 6 of 64-bit keys - in exact
// regions when `exact`, which its second launch then fills): launch slot 0
// is the stable pass on the top digit, reading the regions in order and
// writing S2 ordered by the top 16 bits while it counts the segments; the
// local sort of every segment reads S2 and writes the caller's keys with the
// inverse transform.
DEV void write_top16_schedule(const FsArgs& a, uint32_t cmask, bool exact) {
    GLOBAL uint32_t* plan = gptr<uint32_t>(a.plan);
    const uint32_t top = a.digits - 1u;                 // the top digit (a.digits is 4 or 8 here)
    uint32_t mask = 0;
    for (uint32_t j = 0; j < a.digits; ++j)
        if (!((cmask >> j) & 1u)) mask |= 1u << j;
    const uint32_t flags = FS_PASS_REGIONED | FS_PASS_SEGCOUNT | ((cmask >> top) & FS_SKEW_BIT ? FS_PASS_SKEWED : 0u);
    for (uint32_t j = 0; j < FS_MAX_DIGITS; ++j) {
        uint32_t w0 = 0, w1 = 0;
        if (j == 0) {
            w0 = 1u | (top << 1) | (flags << 16);         // the top digit, execution index 0
            uint32_t tk = FS_BUF_S2K;
#ifdef FS_FAULT_INJECTION
            if (a.fault == FS_FAULT_BAD_BUFFER) tk = FS_BUF_S2V + 1u;   // no such buffer
#endif
            w1 = FS_BUF_S1K | (tk << 8);
        }
        st_agent(&plan[j * FS_PLAN_PASS_WORDS], w0);
        st_agent(&plan[j * FS_PLAN_PASS_WORDS + 1], w1);
    }
    st_agent(&plan[FS_PLAN_NPASSES], 3u);                 // fused pass, top-digit pass, local sort
    st_agent(&plan[FS_PLAN_MASK], mask | FS_MASK_FUSED | FS_MASK_TOP16);
    st_agent(&plan[FS_PLAN_LOCAL], 1u | (a.seg_bits << 8) | (FS_PASS_LAST << 16));
    st_agent(&plan[FS_PLAN_LOCAL + 1], FS_BUF_S2K | (FS_BUF_KEYS << 8));
    st_agent(&plan[FS_PLAN_RESCATTER], exact ? 1u : 0u);
}

// ---------------------------------------------------------------------------
// fs_local_*: the local sort that ends the top-16 path.  After the pass on
// the top digit (digit 3 of 32-bit keys, 7 of 64-bit keys), S2 holds the
// keys ordered by their top 16 bits, and the keys of each segment - the keys
// that share their top seg_bits bits - are one contiguous range: its start
// is the top digit's bin base plus the counts of the smaller values of the
// digit below (segment counters), its length the counts of its own values.
// Block b sorts segment tile_of_block(b) by the bits below its top seg_bits:
// a segment of at most BLOCK * ITEMS keys is read once, sorted in LDS and
// written once, in place of the two (32-bit keys) or six (64-bit keys)
// device-wide passes an LSD sort would still need; a larger one (skewed
// keys) is sorted by the same block a digit at a time through scratch S1
// (big_segment).  32-bit keys: LSD in LDS (8-bit digits, the first in any
// order, the others stable by wave64 ballot ranking).  64-bit keys: the keys
// grouped by the next FS_L64_GBITS bits (LDS atomics, any order), then each
// key's rank within its group by comparing it with the group's keys (LSD in
// LDS when a group is too large for that).  Replaces sort_inner_fused
// (sort.metal:378-769), whose threadgroup per top-byte bucket runs three LSD
// passes through device memory.
// ---------------------------------------------------------------------------

// Segment (start, length) by the first FS_RADIX threads (every thread of the
// block at the barriers): seg is (top-digit value v) << (S - 8) | the top
// S - 8 bits of the value of the digit below it.
template <int BLOCK>
DEV void segment_range(const FsArgs& a, uint32_t seg, uint32_t S, uint32_t* wsum, uint32_t* s_seg,
                       uint32_t& start, uint32_t& len) {
    const uint32_t tid = threadIdx.x;
    const uint32_t v = seg >> (S - 8u);
    const uint32_t wlo = (seg & ((1u << (S - 8u)) - 1u)) << (16u - S), whi = wlo + (1u << (16u - S));
    const uint32_t c = tid < FS_RADIX ? gptr<const uint32_t>(a.segc)[v * FS_RADIX + tid] : 0u;
    const uint32_t ex = radix_exclusive_scan(c, wsum);
    if (tid == wlo) s_seg[0] = ex;
    if (tid == whi - 1u) s_seg[1] = ex + c;
    __syncthreads();
    start = ((const CONSTANT uint32_t*)(uintptr_t)a.binbase)[(a.digits - 1u) * FS_RADIX + v] + s_seg[0];
    len = s_seg[1] - s_seg[0];
}

// Per-digit bases of a stably ranked chunk: wcnt[w][d] (the wave's count of
// digit d) becomes the number of the chunk's keys of digit d in earlier
// waves; returns, to thread d < FS_RADIX, the chunk's count of digit d.
// Every thread of the block calls it (barrier inside is the caller's).
template <int WAVES>
DEV uint32_t wave_bases(uint16_t (*wcnt)[FS_RADIX]) {
    const uint32_t d = threadIdx.x;
    uint32_t run = 0;
    if (d < FS_RADIX) {
#pragma unroll
        for (int ww = 0; ww < WAVES; ++ww) {
            const uint32_t c = wcnt[ww][d];
            wcnt[ww][d] = (uint16_t)run;
            run += c;
        }
    }
    return run;
}

// A segment larger than the block's LDS holds: per digit, a histogram read of
// the segment, then its chunks of CAP keys in order, each ranked stably and
// written to its digit's running base (device memory in, device memory out:
// S2 -> S1 -> S2 ... -> the destination, within the segment's range).
template <bool K64, int BLOCK, int ITEMS>
DEV void big_segment(const FsArgs& a, uint64_t src_addr, uint64_t dst_addr, uint32_t start, uint32_t len,
                     uint32_t npass, bool last, uint16_t (*wcnt)[FS_RADIX], uint32_t* bins, uint32_t* wsum) {
    typedef typename KeyT<K64>::type K;
    constexpr int WAVES = BLOCK / 64;
    constexpr uint32_t CAP = BLOCK * ITEMS;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    const uint32_t wb = w * 64u * ITEMS;
    K xa, xb;
    xf_inv_masks<K64>(last ? a.xform : FS_XF_NONE, xa, xb);
    for (uint32_t q = 0; q < npass; ++q) {
        const uint32_t shift = 8u * q;
        const bool final_pass = q + 1u == npass;
        const uint64_t in_addr = q == 0u ? src_addr : (q & 1u) ? a.s1k : a.s2k;
        const uint64_t out_addr = final_pass ? dst_addr : (q & 1u) ? a.s2k : a.s1k;
        const GLOBAL K* in = gptr<const K>(in_addr) + start;
        GLOBAL K* out = gptr<K>(out_addr) + start;
        if (tid < FS_RADIX) bins[tid] = 0u;
        __syncthreads();
        // (every lane in every step, so that a wave whose lanes share the
        // first lane's digit - a segment of few distinct keys - adds them
        // with one atomic instead of one each on the same counter)
        for (uint32_t p0 = 0; p0 < len; p0 += BLOCK) {
            const uint32_t p = p0 + tid;
            const bool v = p < len;
            const uint32_t d = digit_of<K64>(in[v ? p : 0u], shift);
            if (skewed_digit(d == __builtin_amdgcn_readfirstlane(d))) add_peeled_valid(bins, d, d, 1u, lane, v);
            else if (v) atomicAdd(&bins[d], 1u);
        }
        __syncthreads();
        const uint32_t ex = radix_exclusive_scan(tid < FS_RADIX ? bins[tid] : 0u, wsum);
        if (tid < FS_RADIX) bins[tid] = ex;                    // running base of each digit
        for (uint32_t c0 = 0; c0 < len; c0 += CAP) {
            const uint32_t clen = len - c0 < CAP ? len - c0 : CAP;
            K k[ITEMS];
            uint32_t x[ITEMS];                                 // the 32 bits from the digit up
#pragma unroll
            for (int i = 0; i < ITEMS; ++i) {
                const uint32_t p = wb + (uint32_t)i * 64u + lane;
                k[i] = p < clen ? in[c0 + p] : ~(K)0;         // padding: digit 255, ranked last
                x[i] = (uint32_t)(k[i] >> shift);
            }
            for (uint32_t i = tid; i < WAVES * FS_RADIX / 2u; i += BLOCK) reinterpret_cast<uint32_t*>(&wcnt[0][0])[i] = 0u;
            __syncthreads();
            Ranks<ITEMS> rank;
            rank_wave<false, ITEMS>(x, 0u, wcnt[w], rank);
            __syncthreads();
            uint32_t tot = wave_bases<WAVES>(wcnt);
            if (tid == FS_RADIX - 1u) tot -= CAP - clen;       // the padding's
            __syncthreads();
#pragma unroll
            for (int i = 0; i < ITEMS; ++i) {
                const uint32_t p = wb + (uint32_t)i * 64u + lane;
                if (p >= clen) continue;
                const uint32_t d = x[i] & 0xFFu;
                const uint32_t pos = bins[d] + wcnt[w][d] + rank.get(i);
                if (pos < len) out[pos] = final_pass ? xf_inv_apply<K64>(k[i], xa, xb) : k[i];
            }
            __syncthreads();
            if (tid < FS_RADIX) bins[tid] += tot;
        }
        __syncthreads();                                       // this pass's writes before the next reads
    }
}

// Exclusive prefix of one value per thread over the whole block (every
// thread at the barriers; wsum holds BLOCK / 64 words).
template <int BLOCK>
DEV uint32_t block_exclusive_scan(uint32_t v, uint32_t* wsum) {
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    const uint32_t inc = wave_inclusive_scan(v);
    if (lane == 63) wsum[w] = inc;
    __syncthreads();
    uint32_t excl = inc - v;
    for (uint32_t ww = 0; ww < w; ++ww) excl += wsum[ww];
    __syncthreads();
    return excl;
}

// Rows of 64 keys (wave-striped items) of the wave whose first key is key
// wb that hold a key below len: wave-uniform, so that whole rows past the
// segment are skipped by a scalar branch.
template <int ITEMS>
DEV uint32_t wave_rows(uint32_t len, uint32_t wb) {
    const uint32_t l = __builtin_amdgcn_readfirstlane(len), f = __builtin_amdgcn_readfirstlane(wb);
    return l <= f ? 0u : min((uint32_t)ITEMS, (l - f + 63u) / 64u);
}

// Whether every key of the wave's ITEMS rows (from key wb) is below len:
// wave-uniform.
template <int ITEMS>
DEV bool wave_full(uint32_t len, uint32_t wb) {
    return __builtin_amdgcn_readfirstlane(wb) + (uint32_t)ITEMS * 64u <= __builtin_amdgcn_readfirstlane(len);
}

// Rows of BLOCK keys (thread-striped items: item i of thread t is key
// i * BLOCK + t) that hold a key below len: block-uniform.
template <int BLOCK, int ITEMS>
DEV uint32_t block_rows(uint32_t len) {
    return min((uint32_t)ITEMS, (__builtin_amdgcn_readfirstlane(len) + (uint32_t)BLOCK - 1u) / (uint32_t)BLOCK);
}

// One stable pass of the local sort on the NB-bit digit at bit `pos`: the
// keys of the previous pass's result, read wave-striped, ranked in (wave,
// item, lane) order and staged at their new positions.  wcnt (per-wave digit
// counts) is zero on entry and on return, with the block past a barrier.
template <int BLOCK, int ITEMS, int NB>
DEV void local_stable_pass(uint32_t (&k)[ITEMS], uint32_t pos, uint32_t len, uint32_t* stage,
                           uint16_t (*wcnt)[FS_RADIX], uint32_t* wsum) {
    constexpr int WAVES = BLOCK / 64;
    constexpr uint32_t CAP = BLOCK * ITEMS;             // stage[CAP]: a spare word for padding writes
    constexpr uint32_t NBINS = 1u << NB;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    const uint32_t wb = w * 64u * ITEMS;
    const uint32_t rows = wave_rows<ITEMS>(len, wb);    // ranked and staged; the rows past them skipped
    // (no branch per item: every read is within the stage, padding selected
    // after; a wave wholly inside the segment selects nothing)
    if (wave_full<ITEMS>(len, wb)) {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) k[i] = stage[wb + (uint32_t)i * 64u + lane];
    } else {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            const uint32_t p = wb + (uint32_t)i * 64u + lane;
            const uint32_t v = stage[p];
            k[i] = p < len ? v : 0xFFFFFFFFu;           // padding: the largest digit, ranked last
        }
    }
    Ranks<ITEMS> rank;
    rank_wave<false, ITEMS, NB>(k, pos, wcnt[w], rank, rows);
    __syncthreads();
    uint32_t tot = 0;
    if (tid < NBINS) {
#pragma unroll
        for (int ww = 0; ww < WAVES; ++ww) {
            const uint32_t c = wcnt[ww][tid];
            wcnt[ww][tid] = (uint16_t)tot;
            tot += c;
        }
    }
    const uint32_t ex = radix_exclusive_scan(tot, wsum);   // digit bases (barriers inside)
    if (tid < NBINS) {
#pragma unroll
        for (int ww = 0; ww < WAVES; ++ww) wcnt[ww][tid] = (uint16_t)(wcnt[ww][tid] + ex);
    }
    __syncthreads();
    for_rows<ITEMS>(rows, [&](int i) {
        const uint32_t r = wcnt[w][__builtin_amdgcn_ubfe(k[i], pos, NB)] + rank.get(i);
        stage[r < len ? r : CAP] = k[i];                 // padding ranks last (r >= len): the spare word
    });
    __syncthreads();
    // the counters zero for the next pass, before any wave of it ranks (a
    // wave's counters are cleared by threads of every wave)
    for (uint32_t i = tid; i < WAVES * NBINS; i += BLOCK) wcnt[i / NBINS][i % NBINS] = 0u;
    __syncthreads();
}

// Counters of the local sort's unordered pass (2^FS_LOCAL_UBITS: its low
// bits).  Its LDS and the stage's set the blocks per CU.
#ifndef FS_LOCAL_UBITS
#define FS_LOCAL_UBITS 10
#endif
#define FS_LOCAL_UBINS (1u << FS_LOCAL_UBITS)

// The sort of one segment of len <= BLOCK * ITEMS keys (src -> dst, both at
// the segment's start): the low ub bits in any order (an LDS atomic per key
// gives its slot among the keys of its value), then NSTABLE stable passes of
// NB bits each above them.  Every item of every lane takes part in each LDS
// step: padding lanes count into the spare counter ucnt[2^ub] and write the
// spare word stage[CAP], so that no branch per item separates the LDS
// operations (a branch makes each atomic wait for its return before the next).
template <int BLOCK, int ITEMS, int NB, int NSTABLE>
DEV void local_sort_segment(const FsArgs& a, const GLOBAL uint32_t* src, GLOBAL uint32_t* dst, uint32_t len,
                            uint32_t ub, bool last, uint32_t* stage, uint32_t* ucnt, uint16_t (*wcnt)[FS_RADIX],
                            uint32_t* wsum) {
    typedef uint32_t K;
    constexpr int WAVES = BLOCK / 64;
    constexpr uint32_t CAP = BLOCK * ITEMS;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    const uint32_t nb = 1u << ub, umask = nb - 1u;

    // ---- load the segment (wave-striped: item i of lane l is key w*64*ITEMS + i*64 + l)
    const uint32_t wb = w * 64u * ITEMS;
    const uint32_t rows = wave_rows<ITEMS>(len, wb);    // the wave's rows holding keys: the rest skipped
    const bool full = wave_full<ITEMS>(len, wb);        // every key of the wave's rows in the segment
    K k[ITEMS];
    if (full) {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) k[i] = src[wb + (uint32_t)i * 64u + lane];
    } else {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            const uint32_t p = wb + (uint32_t)i * 64u + lane;
            const K v = src[p < len ? p : len - 1u];    // in bounds for every lane: no branch
            k[i] = p < len ? v : 0xFFFFFFFFu;           // padding, never stored
        }
    }
    for (uint32_t i = tid; i <= nb; i += BLOCK) ucnt[i] = 0u;
    __syncthreads();

    // ---- the low ub bits, in any order: a slot per key from an LDS atomic
    Ranks<ITEMS> rank;
    {
        const uint32_t d0 = k[0] & umask;
        const bool skew = skewed_digit(d0 == __builtin_amdgcn_readfirstlane(d0));
        if (!skew) {
            for_rows_v<ITEMS>(rows, full, [&](int i, auto all) {
                const bool valid = decltype(all)::value || wb + (uint32_t)i * 64u + lane < len;
                rank.set_in_order(i, atomicAdd(&ucnt[valid ? k[i] & umask : nb], 1u));
            });
        } else {
            for_rows_v<ITEMS>(rows, full, [&](int i, auto all) {
                const bool valid = decltype(all)::value || wb + (uint32_t)i * 64u + lane < len;
                rank.set_in_order(i, slot_in_digit<true>(ucnt, k[i] & umask, lane, valid));
            });
        }
    }
    __syncthreads();
    {
        // bases: thread t owns counters [t * per, (t + 1) * per)
        const uint32_t per = nb >= (uint32_t)BLOCK ? nb / BLOCK : 1u;
        constexpr uint32_t PER_MAX = FS_LOCAL_UBINS / BLOCK;
        uint32_t c[PER_MAX];
        uint32_t sum = 0;
#pragma unroll
        for (uint32_t j = 0; j < PER_MAX; ++j) {
            const uint32_t idx = tid * per + j;
            c[j] = (j < per && idx < nb) ? ucnt[idx] : 0u;
            sum += c[j];
        }
        uint32_t ex = block_exclusive_scan<BLOCK>(sum, wsum);
#pragma unroll
        for (uint32_t j = 0; j < PER_MAX; ++j) {
            const uint32_t idx = tid * per + j;
            if (j < per && idx < nb) ucnt[idx] = ex;
            ex += c[j];
        }
    }
    __syncthreads();
    for_rows_v<ITEMS>(rows, full, [&](int i, auto all) {
        const bool valid = decltype(all)::value || wb + (uint32_t)i * 64u + lane < len;
        uint32_t r = ucnt[valid ? k[i] & umask : nb] + rank.get(i);
        r = r < CAP ? r : CAP - 1u;                     // a permutation of [0, len); bound kept explicit
        stage[valid ? r : CAP] = k[i];
    });
    __syncthreads();
    // the stable passes' per-wave counters zero (they may share ucnt's words,
    // whose last use was the staging above)
    for (uint32_t i = tid; i < WAVES * FS_RADIX / 2u; i += BLOCK) reinterpret_cast<uint32_t*>(&wcnt[0][0])[i] = 0u;
    __syncthreads();

    // ---- the bits above, stable
#pragma unroll
    for (int q = 0; q < NSTABLE; ++q) local_stable_pass<BLOCK, ITEMS, NB>(k, ub + (uint32_t)(q * NB), len, stage, wcnt, wsum);

    // ---- write the sorted segment (consecutive positions per thread index)
    K xa, xb;
    xf_inv_masks<false>(last ? a.xform : FS_XF_NONE, xa, xb);
    const uint32_t out_rows = block_rows<BLOCK, ITEMS>(len);
    for_rows<ITEMS>(out_rows, [&](int i) { k[i] = stage[(uint32_t)i * BLOCK + tid]; });
    if (xa != 0u) {                                      // (uniform) i32 / f32 keys
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) k[i] = xf_inv_apply<false>(k[i], xa, xb);
    }
    for_rows<ITEMS>(out_rows, [&](int i) {
        const uint32_t p = (uint32_t)i * BLOCK + tid;
        if ((uint32_t)(i + 1) * BLOCK <= len || p < len) dst[p] = k[i];   // (the first test is block-uniform)
    });
}

// The local sort's plan word, checked, and segment b's range; false when the
// block has nothing to do (no local sort in the schedule, an empty segment,
// or a reported error).
template <int BLOCK, uint32_t DIGITS>
DEV bool local_segment(const FsArgs& a, uint32_t b, uint32_t* wsum, uint32_t* s_seg, uint32_t& S, bool& last,
                       uint64_t& src_addr, uint64_t& dst_addr, uint32_t& start, uint32_t& len) {
    const uint32_t tid = threadIdx.x;
    static_assert(FS_PLAN_LOCAL % 2 == 0, "one 64-bit load");
    const uint64_t lw = ((const CONSTANT uint64_t*)(uintptr_t)a.plan)[FS_PLAN_LOCAL / 2];
    const uint32_t lw0 = (uint32_t)lw, lw1 = (uint32_t)(lw >> 32);
    if (!(lw0 & 1u)) return false;                      // no local sort in this schedule (uniform)
    S = (lw0 >> 8) & 0xFFu;
    last = ((lw0 >> 16) & FS_PASS_LAST) != 0u;
    src_addr = buf_addr(a, lw1 & 0xFFu);
    dst_addr = buf_addr(a, (lw1 >> 8) & 0xFFu);
    if (S < 8u || S > 16u || S != a.seg_bits || !src_addr || !dst_addr || !a.segc || a.digits != DIGITS ||
        b >= (1u << S)) {
        if (tid == 0) report(a, FS_DEVERR_BAD_PLAN);
        return false;
    }
    segment_range<BLOCK>(a, b, S, wsum, s_seg, start, len);
    if (len == 0u) return false;                        // (uniform)
    if (start > (uint32_t)a.n || len > (uint32_t)a.n - start) {   // counters out of step with the input
        if (tid == 0) report(a, FS_DEVERR_BAD_PLAN);
        return false;
    }
    return true;
}

// A segment the first launch of the local sort leaves to the second: appended
// to the list after the segment counters.
DEV void defer_segment(const FsArgs& a, uint32_t seg) {
    GLOBAL uint32_t* list = gptr<uint32_t>(a.segc) + FS_SEGS;
    const uint32_t at = __hip_atomic_fetch_add(list, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (at < FS_SEGS) list[1u + at] = seg;              // (at most one entry per segment)
}

// First launch (32-bit keys): block b sorts segment tile_of_block(b) when it
// fits the block and its bits below the segment's fit one stable pass (at
// most FS_LOCAL_UBITS + 8: segments of at least 14 bits, which the host
// always names unless a test forces fewer); it defers the others (larger
// segments, fewer segment bits) to the second launch, whose paths need more
// registers than seven blocks per CU allow.
template <int BLOCK, int ITEMS>
DEV void local_body(const FsArgs& a) {
    typedef uint32_t K;
    constexpr int WAVES = BLOCK / 64;
    constexpr uint32_t CAP = BLOCK * ITEMS;
    static_assert(BLOCK >= FS_RADIX && BLOCK % 64 == 0, "a digit per thread");
    static_assert(CAP <= 0xFFFFu, "16-bit chunk-local bases");
    static_assert(FS_LOCAL_UBINS % BLOCK == 0 && FS_LOCAL_UBINS / BLOCK <= 16, "counters per thread");
    __shared__ K stage[CAP + 1];                        // stage[CAP]: the spare word padding lanes write
    // the unordered pass's counters, then bases; after its staging, the
    // stable pass's per-wave counters in the same words (2 KiB less LDS per
    // block: seven blocks per CU instead of six)
    constexpr uint32_t CNT_WORDS = FS_LOCAL_UBINS + 1u > WAVES * FS_RADIX / 2u ? FS_LOCAL_UBINS + 1u : WAVES * FS_RADIX / 2u;
    __shared__ uint32_t cnt_area[CNT_WORDS];
    uint32_t* ucnt = cnt_area;
    uint16_t (*wcnt)[FS_RADIX] = reinterpret_cast<uint16_t (*)[FS_RADIX]>(cnt_area);
    __shared__ uint32_t wsum[BLOCK / 64];
    __shared__ uint32_t s_seg[2];

    const uint32_t tid = threadIdx.x;
    if (gridDim.x != (1u << a.seg_bits)) {
        if (tid == 0) report(a, FS_DEVERR_BAD_PLAN);
        return;
    }
    const uint32_t seg = tile_of_block(blockIdx.x, gridDim.x);
    uint32_t S, start, len;
    bool last;
    uint64_t src_addr, dst_addr;
    if (!local_segment<BLOCK, 4u>(a, seg, wsum, s_seg, S, last, src_addr, dst_addr, start, len)) return;
    const uint32_t nbits = 32u - S;                     // bits below the segment's
    // The low bits go in any order (one LDS atomic per key), the rest through
    // one stable pass (ballot matching, 4 VALU per bit): 16 bits = 10 + 6 (10 +
    // 6 measured faster than 8 + 8, 9 + 7, 11 + 5 and 12 + 4 at 2^28 keys);
    // up to FS_LOCAL_UBITS + 8 bits = the rest + 8.  Each plan is a body of
    // its own, so that no register stays live across alternatives.
    if (len > CAP || nbits > FS_LOCAL_UBITS + 8u) {   // (uniform)
        if (tid == 0) defer_segment(a, seg);
        return;
    }
    const GLOBAL K* src = gptr<const K>(src_addr) + start;
    GLOBAL K* dst = gptr<K>(dst_addr) + start;
    static_assert(FS_LOCAL_UBITS >= 10, "16 bits = 10 + 6");
    if (nbits <= 16u)
        local_sort_segment<BLOCK, ITEMS, 6, 1>(a, src, dst, len, nbits - 6u, last, stage, ucnt, wcnt, wsum);
    else
        local_sort_segment<BLOCK, ITEMS, 8, 1>(a, src, dst, len, nbits - 8u, last, stage, ucnt, wcnt, wsum);
}

// Second launch (32-bit keys): a small grid takes the deferred segments in
// turn: larger than a block, a digit at a time through scratch
// (big_segment); else the low bits in any order and two stable 8-bit passes.
template <int BLOCK, int ITEMS>
DEV void local_deferred_body(const FsArgs& a) {
    typedef uint32_t K;
    constexpr int WAVES = BLOCK / 64;
    constexpr uint32_t CAP = BLOCK * ITEMS;
    __shared__ K stage[CAP + 1];
    __shared__ uint32_t ucnt[FS_LOCAL_UBINS + 1];
    __shared__ uint16_t wcnt[WAVES][FS_RADIX];
    __shared__ uint32_t wsum[BLOCK / 64];
    __shared__ uint32_t s_seg[2];
    if (!a.segc) return;
    const GLOBAL uint32_t* list = gptr<const uint32_t>(a.segc) + FS_SEGS;
    const uint32_t count = min(ld_agent(list), FS_SEGS);
    for (uint32_t e = blockIdx.x; e < count; e += gridDim.x) {
        const uint32_t seg = ld_agent(&list[1u + e]);
        uint32_t S, start, len;
        bool last;
        uint64_t src_addr, dst_addr;
        if (!local_segment<BLOCK, 4u>(a, seg, wsum, s_seg, S, last, src_addr, dst_addr, start, len)) return;
        const uint32_t nbits = 32u - S;
        static_assert(FS_LOCAL_UBITS + 16 >= 24, "segments of at least 8 bits: the rest + 8 + 8");
        if (len > CAP)
            big_segment<false, BLOCK, 4>(a, src_addr, dst_addr, start, len, (nbits + 7u) / 8u, last, wcnt, ucnt, wsum);
        else
            local_sort_segment<BLOCK, ITEMS, 8, 2>(a, gptr<const K>(src_addr) + start, gptr<K>(dst_addr) + start, len,
                                                   nbits - 16u, last, stage, ucnt, wcnt, wsum);
        __syncthreads();                                // the segment's LDS is the next one's
    }
}

// ---- the local sort of 64-bit keys

// rank_wave for 64-bit keys: the NB-bit digit at bit pos (any pos below
// 64 - NB), taken from the key's 32 bits from pos up as each item is ranked.
template <int ITEMS, int NB>
DEV void rank_wave64(const uint64_t (&k)[ITEMS], uint32_t pos, uint16_t* wb, Ranks<ITEMS>& rank,
                     uint32_t rows = ITEMS) {
    for_rows<ITEMS>(rows, [&](int i) {
        const uint32_t x = (uint32_t)(k[i] >> pos);
        const uint32_t d = x & ((1u << NB) - 1u);
        const uint64_t peers = match_digit<NB>(x, 0u);
        const uint32_t before = wb[d];
        rank.set_in_order(i, fresh(lanes_below(peers, before)));
        __builtin_amdgcn_wave_barrier();                 // (as rank_wave: reads before the store)
        wb[d] = (uint16_t)((uint32_t)__builtin_popcount((uint32_t)(peers >> 32)) +
                           fresh((uint32_t)__builtin_popcount((uint32_t)peers) + before));
    });
}

// One stable pass of the 64-bit local sort on the NB-bit digit at bit `pos`,
// as local_stable_pass.
template <int BLOCK, int ITEMS, int NB, bool SKIP = true>
DEV void local_stable_pass64(uint64_t (&k)[ITEMS], uint32_t pos, uint32_t len, uint64_t* stage,
                             uint16_t (*wcnt)[FS_RADIX], uint32_t* wsum) {
    constexpr int WAVES = BLOCK / 64;
    constexpr uint32_t CAP = BLOCK * ITEMS;             // stage[CAP]: a spare word for padding writes
    constexpr uint32_t NBINS = 1u << NB;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    const uint32_t wb = w * 64u * ITEMS;
    const uint32_t rows = SKIP ? wave_rows<ITEMS>(len, wb) : ITEMS;   // ranked and staged; the rows past them skipped
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const uint32_t p = wb + (uint32_t)i * 64u + lane;
        const uint64_t v = stage[p];
        k[i] = p < len ? v : ~0ull;                     // padding: the largest digit, ranked last
    }
    Ranks<ITEMS> rank;
    rank_wave64<ITEMS, NB>(k, pos, wcnt[w], rank, rows);
    __syncthreads();
    uint32_t tot = 0;
    if (tid < NBINS) {
#pragma unroll
        for (int ww = 0; ww < WAVES; ++ww) {
            const uint32_t c = wcnt[ww][tid];
            wcnt[ww][tid] = (uint16_t)tot;
            tot += c;
        }
    }
    const uint32_t ex = radix_exclusive_scan(tot, wsum);   // digit bases (barriers inside)
    if (tid < NBINS) {
#pragma unroll
        for (int ww = 0; ww < WAVES; ++ww) wcnt[ww][tid] = (uint16_t)(wcnt[ww][tid] + ex);
    }
    __syncthreads();
    for_rows<ITEMS>(rows, [&](int i) {
        const uint32_t r = wcnt[w][(uint32_t)(k[i] >> pos) & (NBINS - 1u)] + rank.get(i);
        stage[r < len ? r : CAP] = k[i];                 // padding ranks last (r >= len): the spare word
    });
    __syncthreads();
    // the counters zero for the next pass, before any wave of it ranks (a
    // wave's counters are cleared by threads of every wave)
    for (uint32_t i = tid; i < WAVES * NBINS; i += BLOCK) wcnt[i / NBINS][i % NBINS] = 0u;
    __syncthreads();
}

// Slots in any order by the ub bits at bit `shift` of each key (an LDS atomic
// per key, padding lanes on the spare counter cnt[2^ub]), then the counters'
// exclusive prefix in starts (16 or 32 bits each, ST; each thread owns
// 2^ub / BLOCK consecutive counters).  Returns, block-uniform, whether any
// counter exceeded `limit`.  cnt holds at least 2^ub + 1 words, starts 2^ub
// + 1 entries (it may be cnt itself); ub <= FS_L64_GBITS.  When starts is not
// cnt, cnt is dead on return (it may share the stage's words: the block is
// past a barrier after its last read).
template <int BLOCK, int ITEMS, bool SKIP = true, typename ST>
DEV bool group_slots64(const uint64_t (&k)[ITEMS], uint32_t len, uint32_t shift, uint32_t ub, uint32_t limit,
                       uint32_t* cnt, ST* starts, uint32_t* wsum, uint32_t* s_flag, Ranks<ITEMS>& slot) {
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    const uint32_t wb = w * 64u * ITEMS;
    const uint32_t rows = SKIP ? wave_rows<ITEMS>(len, wb) : ITEMS;   // slotted; the rows past them skipped
    const uint32_t nb = 1u << ub, umask = nb - 1u;
    for (uint32_t i = tid; i <= nb; i += BLOCK) cnt[i] = 0u;
    if (tid == 0) *s_flag = 0u;
    __syncthreads();
    {
        const uint32_t d0 = (uint32_t)(k[0] >> shift) & umask;
        const bool skew = skewed_digit(d0 == __builtin_amdgcn_readfirstlane(d0));
        if (!skew) {
            for_rows<ITEMS>(rows, [&](int i) {
                const bool valid = wb + (uint32_t)i * 64u + lane < len;
                slot.set_in_order(i, atomicAdd(&cnt[valid ? (uint32_t)(k[i] >> shift) & umask : nb], 1u));
            });
        } else {
            for_rows<ITEMS>(rows, [&](int i) {
                slot.set_in_order(i, slot_in_digit<true>(cnt, (uint32_t)(k[i] >> shift) & umask, lane,
                                                         wb + (uint32_t)i * 64u + lane < len));
            });
        }
    }
    __syncthreads();
    constexpr uint32_t PER_MAX = (1u << FS_L64_GBITS) / BLOCK;
    static_assert(PER_MAX >= 1u && (1u << FS_L64_GBITS) % BLOCK == 0u, "counters per thread");
    const uint32_t per = nb >= (uint32_t)BLOCK ? nb / BLOCK : 1u;
    uint32_t c[PER_MAX];
    uint32_t sum = 0;
    bool over = false;
#pragma unroll
    for (uint32_t j = 0; j < PER_MAX; ++j) {
        const uint32_t idx = tid * per + j;
        c[j] = (j < per && idx < nb) ? cnt[idx] : 0u;
        sum += c[j];
        over |= c[j] > limit;
    }
    if (__builtin_amdgcn_uicmp((uint32_t)over, 0u, 33) != 0u && lane == 0) *s_flag = 1u;
    uint32_t ex = block_exclusive_scan<BLOCK>(sum, wsum);   // (barriers inside: s_flag is complete after)
#pragma unroll
    for (uint32_t j = 0; j < PER_MAX; ++j) {
        const uint32_t idx = tid * per + j;
        if (j < per && idx < nb) starts[idx] = (ST)ex;
        ex += c[j];
    }
    const bool any_over = *s_flag != 0u;
    __syncthreads();
    return any_over;
}

// 64-bit keys, a segment of len <= BLOCK * ITEMS keys with nbits bits below
// its top bits (k: the segment's keys, wave-striped, padding ~0): LSD in LDS,
// the low ub bits in any order, then 8-bit stable passes up to nbits (a
// pass's bits above nbits are the segment's own, equal in all its keys).
template <int BLOCK, int ITEMS, bool SKIP = true, typename ST>
DEV void local_lsd64(const FsArgs& a, uint64_t (&k)[ITEMS], GLOBAL uint64_t* dst, uint32_t len, uint32_t nbits,
                     bool last, uint64_t* stage, uint32_t* cnt, ST* starts, uint16_t (*wcnt)[FS_RADIX],
                     uint32_t* wsum, uint32_t* s_flag) {
    constexpr uint32_t CAP = BLOCK * ITEMS;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    const uint32_t wb = w * 64u * ITEMS;
    // fewest stable passes with at most FS_L64_GBITS bits in any order
    const uint32_t npass = nbits > FS_L64_GBITS ? (nbits - FS_L64_GBITS + 7u) / 8u : 0u;
    const uint32_t ub = nbits - 8u * npass;
    for (uint32_t i = tid; i < (BLOCK / 64) * FS_RADIX / 2u; i += BLOCK) reinterpret_cast<uint32_t*>(&wcnt[0][0])[i] = 0u;
    Ranks<ITEMS> slot;
    group_slots64<BLOCK, ITEMS, SKIP>(k, len, 0u, ub, 0xFFFFFFFFu, cnt, starts, wsum, s_flag, slot);
    const uint32_t umask = (1u << ub) - 1u;
    for_rows<ITEMS>(SKIP ? wave_rows<ITEMS>(len, wb) : ITEMS, [&](int i) {
        const bool valid = wb + (uint32_t)i * 64u + lane < len;
        uint32_t r = starts[valid ? (uint32_t)k[i] & umask : 0u] + slot.get(i);
        r = r < CAP ? r : CAP - 1u;                     // a permutation of [0, len); bound kept explicit
        stage[valid ? r : CAP] = k[i];
    });
    __syncthreads();
    for (uint32_t q = 0; q < npass; ++q) local_stable_pass64<BLOCK, ITEMS, 8, SKIP>(k, ub + 8u * q, len, stage, wcnt, wsum);
    uint64_t xa, xb;
    xf_inv_masks<true>(last ? a.xform : FS_XF_NONE, xa, xb);
    for_rows<ITEMS>(SKIP ? block_rows<BLOCK, ITEMS>(len) : ITEMS, [&](int i) {
        const uint32_t p = (uint32_t)i * BLOCK + tid;
        if (p < len) dst[p] = xf_inv_apply<true>(stage[p], xa, xb);
    });
}

// First launch: block b sorts segment tile_of_block(b) when it fits the
// block and no group of it holds more than FS_L64_GLIM keys; it defers the
// others (larger segments, many equal keys) to the second launch, whose
// paths need more registers than this one may use at seven blocks per CU.
// The sort of one 64-bit segment of len <= BLOCK * ITEMS keys (k: its keys,
// wave-striped, padding ~0) with nbits bits below its top bits, into dst:
// groups by the FS_L64_GBITS bits below the segment's (2^11 LDS counters:
// about one key per group), each key then ranked within its group by
// comparison; a group of more than FS_L64_GLIM keys that are all equal takes
// its slots as ranks.  Returns false, having written nothing, when a larger
// group holds different keys (the caller sorts the segment otherwise).
template <int BLOCK, int ITEMS, bool SKIP = true, typename ST>
DEV bool group_sort64(const FsArgs& a, const uint64_t (&k)[ITEMS], GLOBAL uint64_t* dst, uint32_t len,
                      uint32_t nbits, bool last, uint64_t* stage, uint32_t* cnt, ST* starts, uint32_t* wsum,
                      uint32_t* s_flag) {
    typedef uint64_t K;
    constexpr uint32_t CAP = BLOCK * ITEMS;
    constexpr uint32_t NG = 1u << FS_L64_GBITS;
    static_assert(CAP <= 0xFFFFu && FS_L64_GLIM < 0x8000u, "16-bit group starts and lengths");
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    const uint32_t wb = w * 64u * ITEMS;
    // ---- groups: the FS_L64_GBITS bits below the segment's, slots in any order
    const uint32_t gshift = nbits - FS_L64_GBITS;
    Ranks<ITEMS> slot;
    const bool big = group_slots64<BLOCK, ITEMS, SKIP>(k, len, gshift, FS_L64_GBITS, FS_L64_GLIM, cnt, starts, wsum,
                                                       s_flag, slot);
    if (tid == 0) starts[NG] = (ST)len;                 // the last group's end
    __syncthreads();
    // each key at its group's start + slot; gsl: the group's start | its length << 16
    // (rows past the segment: gsl 0, a group of no keys)
    const uint32_t rows = SKIP ? wave_rows<ITEMS>(len, wb) : ITEMS;
    uint32_t gsl[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) gsl[i] = 0u;
    for_rows<ITEMS>(rows, [&](int i) {
        const bool valid = wb + (uint32_t)i * 64u + lane < len;
        const uint32_t g = valid ? (uint32_t)(k[i] >> gshift) & (NG - 1u) : NG - 1u;
        const uint32_t gs = starts[g], ge = starts[g + 1u];
        gsl[i] = valid ? gs | ((ge - gs) << 16) : 0u;
        uint32_t r = gs + slot.get(i);
        r = r < CAP ? r : CAP - 1u;                     // a permutation of [0, len); bound kept explicit
        stage[valid ? r : CAP] = k[i];
    });
    __syncthreads();
    if (big) {                                          // (uniform)
        // A group of more than FS_L64_GLIM keys: when all its keys are equal
        // (a key that occurs many times), they take their slots as their
        // ranks, in any order (a keys-only sort), with no comparisons; any
        // other such group: false, nothing written.
        bool mixed = false;
#pragma unroll
        for (int i = 0; i < ITEMS; ++i)
            mixed |= (gsl[i] >> 16) > FS_L64_GLIM && stage[gsl[i] & 0xFFFFu] != k[i];
        if (tid == 0) *s_flag = 0u;
        __syncthreads();
        if (__builtin_amdgcn_uicmp((uint32_t)mixed, 0u, 33) != 0u && lane == 0) *s_flag = 1u;
        __syncthreads();
        const bool any_mixed = *s_flag != 0u;
        __syncthreads();                                // (every thread has read the flag: the LDS is the caller's)
        if (any_mixed) return false;                    // (uniform)
#pragma unroll
        for (int i = 0; i < ITEMS; ++i)
            if ((gsl[i] >> 16) > FS_L64_GLIM) gsl[i] = ((gsl[i] & 0xFFFFu) + slot.get(i)) | (1u << 16);
    }
    // ---- rank within the group: the group's other keys below this one, and
    // its equal keys at smaller slots (each group holds at most FS_L64_GLIM
    // keys, so the loop ends within that many rounds; a key alone in its
    // group reads nothing)
    uint32_t rk[ITEMS];
    uint32_t lmax = 0;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        rk[i] = gsl[i] & 0xFFFFu;
        lmax = max(lmax, gsl[i] >> 16);
    }
    for (uint32_t o = 0; o + 1u < FS_L64_GLIM; ++o) {
        if (__builtin_amdgcn_uicmp((uint32_t)(o + 1u < lmax), 0u, 33) == 0u) break;   // (wave-uniform)
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            if (o + 1u < (gsl[i] >> 16)) {
                const uint32_t me = slot.get(i);               // this key's slot in its group
                const uint32_t oo = o + (o >= me ? 1u : 0u);   // the o-th other slot
                const K kj = stage[(gsl[i] & 0xFFFFu) + oo];
                rk[i] += (kj < k[i] || (kj == k[i] && oo < me)) ? 1u : 0u;
            }
        }
    }
    __syncthreads();
    for_rows<ITEMS>(rows, [&](int i) {
        const uint32_t r = rk[i] < CAP ? rk[i] : CAP - 1u;   // a permutation of [0, len); bound kept explicit
        stage[(gsl[i] >> 16) ? r : CAP] = k[i];          // (a valid key's group has at least itself)
    });
    __syncthreads();
    K xa, xb;
    xf_inv_masks<true>(last ? a.xform : FS_XF_NONE, xa, xb);
    for_rows<ITEMS>(SKIP ? block_rows<BLOCK, ITEMS>(len) : ITEMS, [&](int i) {
        const uint32_t p = (uint32_t)i * BLOCK + tid;
        if (p < len) dst[p] = xf_inv_apply<true>(stage[p], xa, xb);
    });
    return true;
}

template <int BLOCK, int ITEMS>
DEV void local64_body(const FsArgs& a) {
    typedef uint64_t K;
    constexpr int WAVES = BLOCK / 64;
    constexpr uint32_t CAP = BLOCK * ITEMS;
    constexpr uint32_t NG = 1u << FS_L64_GBITS;
    static_assert(BLOCK >= FS_RADIX && BLOCK % 64 == 0, "a digit per thread");
    static_assert(CAP <= 0xFFFFu && FS_L64_GLIM < 0x8000u, "16-bit group starts and lengths");
    __shared__ K stage[CAP + 1];                        // stage[CAP]: the spare word padding lanes write
    // the group counters in the stage's words (the stage is written only
    // after their last read), the group starts in 16 bits (starts[NG] = len):
    // 22 KiB per block, seven blocks per CU
    // (blocks of few keys, as test builds use, keep the counters apart)
    constexpr bool CNT_IN_STAGE = (NG + 1u) * sizeof(uint32_t) <= sizeof(stage);
    __shared__ uint32_t cnt_apart[CNT_IN_STAGE ? 1u : NG + 1u];
    uint32_t* cnt = CNT_IN_STAGE ? reinterpret_cast<uint32_t*>(stage) : cnt_apart;
    __shared__ uint16_t starts[NG + 2];
    __shared__ uint32_t wsum[BLOCK / 64];
    __shared__ uint32_t s_seg[2];
    __shared__ uint32_t s_flag;

    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    uint32_t S, start, len;
    bool last;
    uint64_t src_addr, dst_addr;
    if (gridDim.x != (1u << a.seg_bits)) {
        if (tid == 0) report(a, FS_DEVERR_BAD_PLAN);
        return;
    }
    const uint32_t seg = tile_of_block(blockIdx.x, gridDim.x);
    if (!local_segment<BLOCK, 8u>(a, seg, wsum, s_seg, S, last, src_addr, dst_addr, start, len)) return;
    const uint32_t nbits = 64u - S;                     // bits below the segment's (48 to 56)
    if (len > CAP) {                                    // (uniform)
        if (tid == 0) defer_segment(a, seg);
        return;
    }
    const GLOBAL K* src = gptr<const K>(src_addr) + start;
    GLOBAL K* dst = gptr<K>(dst_addr) + start;
    const uint32_t wb = w * 64u * ITEMS;
    K k[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const uint32_t p = wb + (uint32_t)i * 64u + lane;
        const K v = src[p < len ? p : len - 1u];        // in bounds for every lane: no branch
        k[i] = p < len ? v : ~0ull;                     // padding, never stored
    }

    if (!group_sort64<BLOCK, ITEMS>(a, k, dst, len, nbits, last, stage, cnt, starts, wsum, &s_flag))
        if (tid == 0) defer_segment(a, seg);           // (uniform)
}

// Waves per SIMD each digit-pass kernel is compiled for (0: compiler's choice).
// Two 12-wave (768-thread) blocks per CU need 6, i.e. at most 80 VGPRs.
#ifndef FS_K32_WAVES_PER_EU
#define FS_K32_WAVES_PER_EU 6
#endif
#ifndef FS_K32V_WAVES_PER_EU
#define FS_K32V_WAVES_PER_EU 6
#endif
#ifndef FS_K64_WAVES_PER_EU
#define FS_K64_WAVES_PER_EU 6
#endif
#ifndef FS_K64V_WAVES_PER_EU
#define FS_K64V_WAVES_PER_EU 6
#endif
#define FS_OCC(w) __attribute__((amdgpu_waves_per_eu((w) ? (w) : 1)))

extern "C" __global__ void __launch_bounds__(FS_K32_BLOCK) FS_OCC(FS_K32_WAVES_PER_EU) fs_onesweep_k32(FsArgs a, uint32_t slot) {
    onesweep_body<false, false, FS_K32_BLOCK, FS_K32_ITEMS>(a, slot, blockIdx.x);
}
extern "C" __global__ void __launch_bounds__(FS_K32V_BLOCK) FS_OCC(FS_K32V_WAVES_PER_EU) fs_onesweep_k32_v(FsArgs a, uint32_t slot) {
    onesweep_body<false, true, FS_K32V_BLOCK, FS_K32V_ITEMS>(a, slot, blockIdx.x);
}
extern "C" __global__ void __launch_bounds__(FS_K64_BLOCK) FS_OCC(FS_K64_WAVES_PER_EU) fs_onesweep_k64(FsArgs a, uint32_t slot) {
    onesweep_body<true, false, FS_K64_BLOCK, FS_K64_ITEMS>(a, slot, blockIdx.x);
}
extern "C" __global__ void __launch_bounds__(FS_K64V_BLOCK) FS_OCC(FS_K64V_WAVES_PER_EU) fs_onesweep_k64_v(FsArgs a, uint32_t slot) {
    onesweep_body<true, true, FS_K64V_BLOCK, FS_K64V_ITEMS>(a, slot, blockIdx.x);
}
// Fused first pass of keys-only sorts (tiles of the stable kernels' size).
// (the scatter digit, chosen by the region sample, an earlier kernel, picks
// the body)
extern "C" __global__ void __launch_bounds__(FS_K32_BLOCK) FS_OCC(FS_K32_WAVES_PER_EU) fs_first_k32(FsArgs a) {
    constexpr uint32_t launch = 0;
    __shared__ FirstPassLds<false, FS_K32_BLOCK, FS_K32_ITEMS> lds;
    const uint32_t sd = ((const CONSTANT uint32_t*)(uintptr_t)a.rtable)[FS_RTABLE_SDIGIT];
    if (sd == 2u) first_pass_body<false, FS_K32_BLOCK, FS_K32_ITEMS, 2u>(a, launch, sd, blockIdx.x, lds);
    else first_pass_body<false, FS_K32_BLOCK, FS_K32_ITEMS, 0u>(a, launch, sd, blockIdx.x, lds);
}
extern "C" __global__ void __launch_bounds__(FS_K64_BLOCK) FS_OCC(FS_K64_WAVES_PER_EU) fs_first_k64(FsArgs a) {
    constexpr uint32_t launch = 0;
    __shared__ FirstPassLds<true, FS_K64_BLOCK, FS_K64_ITEMS> lds;
    const uint32_t sd = ((const CONSTANT uint32_t*)(uintptr_t)a.rtable)[FS_RTABLE_SDIGIT];
    if (sd == 6u) first_pass_body<true, FS_K64_BLOCK, FS_K64_ITEMS, 6u>(a, launch, sd, blockIdx.x, lds);
    else first_pass_body<true, FS_K64_BLOCK, FS_K64_ITEMS, 0u>(a, launch, sd, blockIdx.x, lds);
}
// The fused pass's re-scatter after a region overflow (its launch 1): a small
// grid looping over the tiles, so that the launch costs a few blocks when
// there was no overflow (the tiles only take atomic region space: no order
// among them is needed).  One block per CU, as the digit-pass loop kernel.
extern "C" __global__ void __launch_bounds__(FS_K32_BLOCK) FS_OCC(FS_K32_BLOCK / 64 / 4) fs_rescatter_k32(FsArgs a) {
    if (((const CONSTANT uint32_t*)(uintptr_t)a.plan)[FS_PLAN_RESCATTER] == 0u) return;   // (uniform)
    __shared__ FirstPassLds<false, FS_K32_BLOCK, FS_K32_ITEMS> lds;
    const uint32_t sd = ((const CONSTANT uint32_t*)(uintptr_t)a.rtable)[FS_RTABLE_SDIGIT];
    for (uint32_t t = blockIdx.x; t < a.num_tiles; t += gridDim.x) {
        if (sd == 2u) first_pass_body<false, FS_K32_BLOCK, FS_K32_ITEMS, 2u, true>(a, 1u, sd, t, lds);
        else first_pass_body<false, FS_K32_BLOCK, FS_K32_ITEMS, 0u, true>(a, 1u, sd, t, lds);
        __syncthreads();                                    // the tile's LDS is the next tile's
    }
}
extern "C" __global__ void __launch_bounds__(FS_K64_BLOCK) FS_OCC(FS_K64_BLOCK / 64 / 4) fs_rescatter_k64(FsArgs a) {
    if (((const CONSTANT uint32_t*)(uintptr_t)a.plan)[FS_PLAN_RESCATTER] == 0u) return;   // (uniform)
    __shared__ FirstPassLds<true, FS_K64_BLOCK, FS_K64_ITEMS> lds;
    const uint32_t sd = ((const CONSTANT uint32_t*)(uintptr_t)a.rtable)[FS_RTABLE_SDIGIT];
    for (uint32_t t = blockIdx.x; t < a.num_tiles; t += gridDim.x) {
        if (sd == 6u) first_pass_body<true, FS_K64_BLOCK, FS_K64_ITEMS, 6u, true>(a, 1u, sd, t, lds);
        else first_pass_body<true, FS_K64_BLOCK, FS_K64_ITEMS, 0u, true>(a, 1u, sd, t, lds);
        __syncthreads();
    }
}
// Digit 0 of keys-only sorts (the first pass, in any order within a digit);
// same tiles as the stable kernels of the same key width.
extern "C" __global__ void __launch_bounds__(FS_K32_BLOCK) FS_OCC(FS_K32_WAVES_PER_EU) fs_onesweep_any_k32(FsArgs a, uint32_t slot) {
    onesweep_body<false, false, FS_K32_BLOCK, FS_K32_ITEMS, true>(a, slot, blockIdx.x);
}
extern "C" __global__ void __launch_bounds__(FS_K64_BLOCK) FS_OCC(FS_K64_WAVES_PER_EU) fs_onesweep_any_k64(FsArgs a, uint32_t slot) {
    onesweep_body<true, false, FS_K64_BLOCK, FS_K64_ITEMS, true>(a, slot, blockIdx.x);
}
// The small tiles of small sorts (FS_VAR_K32S, FS_VAR_K32VS, FS_VAR_K64VS): the stable
// passes, and for keys-only sorts digit 0's pass in any order.
#ifndef FS_KS_WAVES_PER_EU
#define FS_KS_WAVES_PER_EU 6
#endif
extern "C" __global__ void __launch_bounds__(FS_K32S_BLOCK) FS_OCC(FS_KS_WAVES_PER_EU) fs_onesweep_k32_s(FsArgs a, uint32_t slot) {
    onesweep_body<false, false, FS_K32S_BLOCK, FS_K32S_ITEMS>(a, slot, blockIdx.x);
}
extern "C" __global__ void __launch_bounds__(FS_K32S_BLOCK) FS_OCC(FS_KS_WAVES_PER_EU) fs_onesweep_any_k32_s(FsArgs a, uint32_t slot) {
    onesweep_body<false, false, FS_K32S_BLOCK, FS_K32S_ITEMS, true>(a, slot, blockIdx.x);
}
extern "C" __global__ void __launch_bounds__(FS_KS_BLOCK) FS_OCC(FS_KS_WAVES_PER_EU) fs_onesweep_k32_vs(FsArgs a, uint32_t slot) {
    onesweep_body<false, true, FS_KS_BLOCK, FS_K32VS_ITEMS>(a, slot, blockIdx.x);
}
extern "C" __global__ void __launch_bounds__(FS_KS_BLOCK) FS_OCC(FS_KS_WAVES_PER_EU) fs_onesweep_k64_vs(FsArgs a, uint32_t slot) {
    onesweep_body<true, true, FS_KS_BLOCK, FS_K64VS_ITEMS>(a, slot, blockIdx.x);
}

// Local sort of the top-16 path: one block per segment.  Seven 256-thread
// blocks per CU (22 KiB of LDS and at most 72 VGPRs each) measured 5% faster
// than six at u32 256M; the wide blocks' LDS allows three per CU.
#ifndef FS_L32_WAVES_PER_EU
#define FS_L32_WAVES_PER_EU 7
#endif
#ifndef FS_LW_WAVES_PER_EU
#define FS_LW_WAVES_PER_EU 6
#endif
extern "C" __global__ void __launch_bounds__(FS_L32_BLOCK) FS_OCC(FS_L32_WAVES_PER_EU) fs_local_k32(FsArgs a) {
    local_body<FS_L32_BLOCK, FS_L32_ITEMS>(a);
}
extern "C" __global__ void __launch_bounds__(FS_LD32_BLOCK) FS_OCC(1) fs_local_deferred_k32(FsArgs a) {
    local_deferred_body<FS_LD32_BLOCK, FS_L32_ITEMS>(a);
}
// Wide blocks (FS_LW_BLOCK threads, twice the keys): the sizes whose
// segments outgrow the blocks above.
extern "C" __global__ void __launch_bounds__(FS_LW_BLOCK) FS_OCC(FS_LW_WAVES_PER_EU) fs_local_k32_w(FsArgs a) {
    local_body<FS_LW_BLOCK, FS_L32_ITEMS>(a);
}
extern "C" __global__ void __launch_bounds__(FS_LD32_BLOCK) FS_OCC(1) fs_local_deferred_k32_w(FsArgs a) {
    local_deferred_body<FS_LD32_BLOCK, FS_L32_ITEMS>(a);
}

// Second launch: a small grid takes the deferred segments in turn; a segment
// larger than a block holds goes a digit at a time through scratch
// (big_segment), the others by the LSD passes in LDS.
template <int BLOCK, int ITEMS>
DEV void local64_deferred_body(const FsArgs& a) {
    typedef uint64_t K;
    constexpr int WAVES = BLOCK / 64;
    constexpr uint32_t CAP = BLOCK * ITEMS;
    constexpr uint32_t NG = 1u << FS_L64_GBITS;
    __shared__ K stage[CAP + 1];
    __shared__ uint32_t cnt[NG + 1];                    // group counters, then group starts (cnt[NG] = len)
    __shared__ uint16_t wcnt[WAVES][FS_RADIX];
    __shared__ uint32_t wsum[BLOCK / 64];
    __shared__ uint32_t s_seg[2];
    __shared__ uint32_t s_flag;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    if (!a.segc) return;
    const GLOBAL uint32_t* list = gptr<const uint32_t>(a.segc) + FS_SEGS;
    const uint32_t count = min(ld_agent(list), FS_SEGS);
    for (uint32_t e = blockIdx.x; e < count; e += gridDim.x) {
        const uint32_t seg = ld_agent(&list[1u + e]);
        uint32_t S, start, len;
        bool last;
        uint64_t src_addr, dst_addr;
        if (!local_segment<BLOCK, 8u>(a, seg, wsum, s_seg, S, last, src_addr, dst_addr, start, len)) return;
        const uint32_t nbits = 64u - S;
        if (len > CAP) {
            big_segment<true, BLOCK, 4>(a, src_addr, dst_addr, start, len, (nbits + 7u) / 8u, last, wcnt, cnt, wsum);
        } else {
            const uint32_t wb = w * 64u * ITEMS;
            const GLOBAL K* src = gptr<const K>(src_addr) + start;
            K k[ITEMS];
#pragma unroll
            for (int i = 0; i < ITEMS; ++i) {
                const uint32_t p = wb + (uint32_t)i * 64u + lane;
                const K v = src[p < len ? p : len - 1u];
                k[i] = p < len ? v : ~0ull;
            }
            // the group sort when the segment's large groups hold equal keys
            // (keys that occur many times), else LSD in LDS
            // (every row taken: this kernel's registers leave no room for
            // the branch-free and the row-skipping copy of each step)
            if (!group_sort64<BLOCK, ITEMS, false>(a, k, gptr<K>(dst_addr) + start, len, nbits, last, stage, cnt,
                                                   cnt, wsum, &s_flag))
                local_lsd64<BLOCK, ITEMS, false>(a, k, gptr<K>(dst_addr) + start, len, nbits, last, stage, cnt,
                                                 cnt, wcnt, wsum, &s_flag);
        }
        __syncthreads();                                // the segment's LDS is the next one's
    }
}

// Seven 256-thread blocks per CU, as the 32-bit local sort (22 KiB of LDS
// each: the group counters in the stage's words, the group starts in 16
// bits; at most 72 VGPRs).
#ifndef FS_L64_WAVES_PER_EU
#define FS_L64_WAVES_PER_EU 7
#endif
extern "C" __global__ void __launch_bounds__(FS_L64_BLOCK) FS_OCC(FS_L64_WAVES_PER_EU) fs_local_k64(FsArgs a) {
    local64_body<FS_L64_BLOCK, FS_L64_ITEMS>(a);
}
extern "C" __global__ void __launch_bounds__(FS_LD64_BLOCK) FS_OCC(1) fs_local_deferred_k64(FsArgs a) {
    local64_deferred_body<FS_LD64_BLOCK, FS_L64_ITEMS>(a);
}
extern "C" __global__ void __launch_bounds__(FS_LW_BLOCK) FS_OCC(FS_LW_WAVES_PER_EU) fs_local_k64_w(FsArgs a) {
    local64_body<FS_LW_BLOCK, FS_L64_ITEMS>(a);
}
extern "C" __global__ void __launch_bounds__(FS_LD64_BLOCK) FS_OCC(1) fs_local_deferred_k64_w(FsArgs a) {
    local64_deferred_body<FS_LD64_BLOCK, FS_L64_ITEMS>(a);
}

// Late digit-pass slots of 64-bit keys (FS_LOOP_SLOT64 on), which run only
// when the region sample chose the LSD passes on the top-16 launch sequence
// and more than five digits vary (else they have nothing to do): a small
// grid of blocks, each taking tiles blockIdx, blockIdx + grid, ... in
// increasing order, so that an idle launch costs a few blocks, not one per
// tile.  Progress as for one block per tile: blocks start in increasing
// order and a tile waits only on smaller tiles, which blocks that started
// earlier hold (every block of the grid fits on the device at once: one
// block per CU, compiled for that occupancy so that the loop spills no
// registers; at two blocks per CU it spilled, and a working launch at one
// block per CU takes about 1.5 times a pass of one block per tile).
extern "C" __global__ void __launch_bounds__(FS_K64_BLOCK) FS_OCC(FS_K64_BLOCK / 64 / 4) fs_onesweep_loop_k64(FsArgs a, uint32_t slot) {
    const uint64_t pw = ((const CONSTANT uint64_t*)(uintptr_t)a.plan)[slot < FS_MAX_DIGITS ? slot : 0u];
    if (!(pw & 1u) && !((uint32_t)pw >> 24)) return;       // no pass and no duty in this slot (uniform)
    for (uint32_t t = blockIdx.x; t < a.num_tiles; t += gridDim.x) {
        onesweep_body<true, false, FS_K64_BLOCK, FS_K64_ITEMS, false, true>(a, slot, t);
        __syncthreads();                                    // the tile's LDS is the next tile's
    }
}

#include "bucket_sort.h"

// Tile sizes of the digit-pass variants (FS_VAR_*), read by the host runtime.
extern "C" __constant__ __attribute__((used)) uint32_t fs_kernel_tile_keys[FS_VARIANTS] = {
    FS_K32_BLOCK * FS_K32_ITEMS, FS_K32V_BLOCK * FS_K32V_ITEMS,
    FS_K64_BLOCK * FS_K64_ITEMS, FS_K64V_BLOCK * FS_K64V_ITEMS, FS_K32S_BLOCK * FS_K32S_ITEMS,
    FS_KS_BLOCK * FS_K32VS_ITEMS, FS_KS_BLOCK * FS_K64VS_ITEMS};
// Keys a block of the local sort holds, and its threads per block (32-bit
// keys, then 64-bit keys); then the fewest segment bits whose 32-bit
// segments the first launch sorts itself; then the same two pairs for the
// wide blocks.
extern "C" __constant__ __attribute__((used)) uint32_t fs_kernel_local_geometry[9] = {
    FS_L32_BLOCK * FS_L32_ITEMS, FS_L32_BLOCK, FS_L64_BLOCK * FS_L64_ITEMS, FS_L64_BLOCK, 32u - (FS_LOCAL_UBITS + 8u),
    FS_LW_BLOCK * FS_L32_ITEMS, FS_LW_BLOCK, FS_LW_BLOCK * FS_L64_ITEMS, FS_LW_BLOCK};
// Bucket path: threads per block of the bucket kernels, the partition, the
// sample and a child; most samples of the input and of a bucket; most buckets;
// then keys of a bucket's block and of the partition's tile, each for 32-bit
// keys, with values, 64-bit, with values; then keys of a child's block and of
// the tiles of two levels, for 64-bit keys and with values.
extern "C" __constant__ __attribute__((used)) uint32_t fs_kernel_bucket_geometry[FS_BG_WORDS] = {
    FS_BK_BLOCK, FS_BP_BLOCK, FS_BS_BLOCK, FS_BC_BLOCK, FS_BS_BLOCK * FS_BS_ITEMS, FS_BS_BLOCK * FS_BS2_ITEMS, FS_BK_NB,
    FS_BK_BLOCK * FS_BK32_ITEMS, FS_BK_BLOCK * FS_BK32V_ITEMS, FS_BK_BLOCK * FS_BK64_ITEMS, FS_BK_BLOCK * FS_BK64V_ITEMS,
    FS_BP_BLOCK * FS_BP32_ITEMS, FS_BP_BLOCK * FS_BP32_ITEMS, FS_BP_BLOCK * FS_BP64_ITEMS, FS_BP_BLOCK * FS_BP64_ITEMS,
    FS_BC_BLOCK * FS_BC64_ITEMS, FS_BC_BLOCK * FS_BC64V_ITEMS, FS_BP_BLOCK * FS_BP2_64_ITEMS, FS_BP_BLOCK * FS_BP2_64V_ITEMS};
// Threads per block of the same variants.
extern "C" __constant__ __attribute__((used)) uint32_t fs_kernel_block_threads[FS_VARIANTS] = {
    FS_K32_BLOCK, FS_K32V_BLOCK, FS_K64_BLOCK, FS_K64V_BLOCK, FS_K32S_BLOCK, FS_KS_BLOCK, FS_KS_BLOCK};

// ---------------------------------------------------------------------------
// fs_gather_elems: output[i] = source[indices[i]] for 4- or 8-byte elements
// (forge-runtime shaders/gather.metal:5-27).  An index at or past src_len is
// reported through the status word and yields 0 instead of a read.
// ---------------------------------------------------------------------------

extern "C" __global__ void __launch_bounds__(256) fs_gather_elems(uint64_t src, uint64_t src_len, uint64_t idx,
                                                                  uint64_t dst, uint64_t count, uint32_t is64,
                                                                  uint64_t status) {
    const GLOBAL uint32_t* ix = gptr<const uint32_t>(idx);
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    bool bad = false;
    if (is64) {
        const GLOBAL uint64_t* s = gptr<const uint64_t>(src);
        GLOBAL uint64_t* d = gptr<uint64_t>(dst);
        for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride) {
            const uint32_t j = ix[i];
            const bool ok = j < src_len;
            bad |= !ok;
            d[i] = ok ? s[j] : 0ull;
        }
    } else {
        const GLOBAL uint32_t* s = gptr<const uint32_t>(src);
        GLOBAL uint32_t* d = gptr<uint32_t>(dst);
        for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride) {
            const uint32_t j = ix[i];
            const bool ok = j < src_len;
            bad |= !ok;
            d[i] = ok ? s[j] : 0u;
        }
    }
    if (bad)
        __hip_atomic_fetch_or((uint32_t*)status, FS_DEVERR_GATHER_INDEX, __ATOMIC_RELAXED,
                              __HIP_MEMORY_SCOPE_SYSTEM);
}

// ---------------------------------------------------------------------------
// Scratch of fs_encode_no_alloc: one static array per loaded code object,
// laid out by the FS_NA_* offsets (fs_params.h).  The host never names it: at
// set-up it runs fs_scratch_address once and keeps the device address that
// kernel reports (a module-scope static has no symbol the module API can look
// up).
// ---------------------------------------------------------------------------
static __device__ __align__(256) uint8_t scratch[FS_NA_SCRATCH_BYTES];

// out[0] = device address of `scratch`, out[1] = its size in bytes.
extern "C" __global__ void __launch_bounds__(64) fs_scratch_address(uint64_t* out) {
    if (threadIdx.x == 0) {
        out[0] = (uint64_t)(uintptr_t)&scratch[0];
        out[1] = (uint64_t)sizeof(scratch);
    }
}

// Index fill for argsort of a single key (lib.rs:1680-1682 returns [0]); a
// kernel rather than a memset so that captured graphs stay memset-free.
extern "C" __global__ void __launch_bounds__(64) fs_iota(uint32_t* out, uint64_t n) {
    for (uint64_t i = threadIdx.x; i < n; i += blockDim.x) out[i] = (uint32_t)i;
}
