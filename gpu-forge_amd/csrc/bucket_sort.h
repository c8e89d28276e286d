// bucket_sort.h -- kernels of the bucket path (included by radix_kernels.hip):
// sorts too small for device-wide digit passes to pay, whose cost is the
// number of dependent launches rather than the bytes they move.
//
//   one block (n <= a block's keys)
//     fs_bucket_*   reads the caller's keys, sorts them in LDS and writes them
//                   back: one launch.
//   buckets (up to FS_BK_MAX_* keys)
//     fs_split_*    one block sorts a sample of the keys and takes its
//                   quantiles as splitters of at most FS_BK_NB buckets; a
//                   value that several quantiles share gets a bucket of its
//                   own, so that copies of one key never crowd a bucket with
//                   other keys
//     fs_part_*     every key to its bucket's region of scratch S1: the bucket
//                   by binary search in the splitters (LDS), its place by one
//                   atomic per tile and bucket (keys only) or, for values,
//                   whose order among equal keys must hold, by the decoupled
//                   look-back of the digit passes
//     fs_bucket_*   one block per bucket: read once, sorted in LDS, written
//                   once to its place in the output
//
// The block sort groups the keys by the top bits of their range and ranks each
// within its group by comparison; blocks with large groups (many copies of a
// key) fall back to stable passes over the bits of the range, 8 at a time,
// ranked by wave64 ballots.  With values each key carries its position in the
// block (16 bits) and the values follow by one gather at the end.
//
// Buckets are sized by the sample, so a bucket can outgrow its region or a
// block's LDS (16 samples a bucket and regions of FS_BK_ROOM times the
// estimate: not once in 10^6 sorts).  Such a sort stays exact: the block of an
// oversized bucket, or block 0 for every key after an overflowed region, sorts
// it alone through device memory (slow_sort).

// Elements of the LDS block sort of WAVES waves: rows of 64 keys, `per` rows
// to each wave (wave w: rows w * per ...), so that a small segment still uses
// every wave.
template <bool K64, bool VALS, int BLOCK, int ITEMS>
struct BlockSortLds {
    typedef typename KeyT<K64>::type K;
    static constexpr uint32_t CAP = BLOCK * ITEMS;
    static constexpr int WAVES = BLOCK / 64;
    alignas(16) K keys[CAP];
    uint16_t pos[VALS ? CAP : 1];                // with values: each key's position in the block
    alignas(16) uint16_t wcnt[WAVES][FS_RADIX];  // per-wave digit counts, then bases
    uint32_t dbase[FS_RADIX];
    uint16_t starts[(1u << FS_BK_GBITS) + 2u];   // group starts
    uint32_t wsum[WAVES];
    uint32_t flag;
    K red[2][WAVES];
};

template <typename K>
DEV K shfl_up_key(K v, int off) {
    if constexpr (sizeof(K) == 4) {
        return __shfl_up(v, off, 64);
    } else {
        const uint32_t lo = __shfl_up((uint32_t)v, off, 64), hi = __shfl_up((uint32_t)((uint64_t)v >> 32), off, 64);
        return (K)(((uint64_t)hi << 32) | lo);
    }
}

// f folded over the whole wave, in lane 63.
template <typename K, typename F>
DEV K wave_fold(K v, F&& f) {
    const uint32_t lane = threadIdx.x & 63u;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const K t = shfl_up_key<K>(v, off);
        if (lane >= (uint32_t)off) v = f(v, t);
    }
    return v;
}

// One stable pass of the block sort on the 8 bits at `shift`: k (and p, the
// positions) in row order in, the sorted rows in L.keys (L.pos) on return,
// the block past a barrier.
template <bool K64, bool VALS, int BLOCK, int ITEMS>
DEV void block_sort_pass(typename KeyT<K64>::type (&k)[ITEMS], Ranks<VALS ? ITEMS : 1>& p, uint32_t shift, uint32_t per,
                         BlockSortLds<K64, VALS, BLOCK, ITEMS>& L) {
    constexpr int WAVES = BLOCK / 64;
    constexpr uint32_t CAP = BLOCK * ITEMS;
    const uint32_t tid = threadIdx.x, w = tid >> 6;
    for (uint32_t i = tid; i < WAVES * FS_RADIX / 2u; i += BLOCK) reinterpret_cast<uint32_t*>(&L.wcnt[0][0])[i] = 0u;
    __syncthreads();
    Ranks<ITEMS> rank;
    uint16_t* wb = L.wcnt[w];
    for_rows<ITEMS>(per, [&](int i) __attribute__((always_inline)) {
        const uint32_t x = (uint32_t)(k[i] >> shift);
        const uint64_t peers = match_digit(x, 0u);
        const uint32_t before = wb[x & 0xFFu];
        rank.set_in_order(i, fresh(lanes_below(peers, before)));
        __builtin_amdgcn_wave_barrier();                 // (as rank_wave: reads before the store)
        wb[x & 0xFFu] = (uint16_t)((uint32_t)__builtin_popcount((uint32_t)(peers >> 32)) +
                                   fresh((uint32_t)__builtin_popcount((uint32_t)peers) + before));
    });
    __syncthreads();
    uint32_t tot = 0;
    if (tid < FS_RADIX) {
        uint32_t c[WAVES];
#pragma unroll
        for (int ww = 0; ww < WAVES; ++ww) c[ww] = L.wcnt[ww][tid];
#pragma unroll
        for (int ww = 0; ww < WAVES; ++ww) {
            L.wcnt[ww][tid] = (uint16_t)tot;
            tot += c[ww];
        }
    }
    const uint32_t ex = radix_exclusive_scan(tot, L.wsum);
    if (tid < FS_RADIX) L.dbase[tid] = ex;
    __syncthreads();
    for_rows<ITEMS>(per, [&](int i) __attribute__((always_inline)) {
        const uint32_t d = (uint32_t)(k[i] >> shift) & 0xFFu;
        uint32_t r = L.dbase[d] + L.wcnt[w][d] + rank.get(i);
        r = r < CAP ? r : CAP - 1u;                     // a permutation of the block's rows; bound kept explicit
        L.keys[r] = k[i];
        if constexpr (VALS) L.pos[r] = (uint16_t)p.get(i);
    });
    __syncthreads();
}

// Monotone map of a block's keys (k: key less `base`, in the sort's unsigned
// order) to 2^FS_BK_GBITS groups: by the top bits of k, or (floats) by value,
// linear between the least and greatest finite values of the block; keys
// beyond those, the infinities and NaNs among them, fall into the outer groups.
template <bool K64>
struct GroupMap {
    typedef typename KeyT<K64>::type K;
    bool by_value;
    uint32_t shift;
    K base, span;                                        // the least key, and the greatest less it
    double low, scale;
    static DEV double value(K u) {                       // of the key u (FloatFlip's inverse)
        const K f = xf_inv_apply<K64>(u, KeyT<K64>::SIGN, ~(K)0);
        if constexpr (K64) return __builtin_bit_cast(double, f);
        else return (double)__builtin_bit_cast(float, f);
    }
    static constexpr K FINITE = K64 ? (K)0xFFEFFFFFFFFFFFFFull : (K)0xFF7FFFFFu;   // the greatest finite key
    DEV bool exact() const { return !by_value && shift == 0u; }
    // A key in group g, `part` of the way through it; in key order over (g, part).
    DEV K inside(uint32_t g, float part) const {
        if (!by_value) {
            const K t = ((K)g << shift) + (K)((double)part * (double)((K)1 << shift));
            return base + (t < span ? t : span);
        }
        const double v = low + ((double)g + (double)part) / scale;
        K f;
        if constexpr (K64) f = __builtin_bit_cast(uint64_t, v);
        else f = __builtin_bit_cast(uint32_t, (float)v);
        return xf_fwd<K64>(f, FS_XF_FLOAT);
    }
    DEV uint32_t operator()(K k) const {
        if (!by_value) return (uint32_t)(k >> shift) & ((1u << FS_BK_GBITS) - 1u);
        K u = k + base;
        u = u > FINITE ? FINITE : u < ~FINITE ? ~FINITE : u;
        const double t = (value(u) - low) * scale;
        const double top = (double)((1u << FS_BK_GBITS) - 1u);
        return (uint32_t)(t > top ? top : t > 0.0 ? t : 0.0);
    }
};

// The block sort of keys of `bits` bits by groups: the keys grouped by `map`
// (an LDS atomic each, in any order), then each key's rank in its group by
// comparing it with the others.  A key of a group of a few costs about half
// the VALU of one stable 8-bit pass per byte of a 32-bit range, a quarter at
// 64 bits.  False, the rows untouched in registers, when a group holds more
// than FS_BK_GLIM keys (keys crowded in a small part of the range, or, with
// values, many copies of a key).
template <bool K64, bool VALS, int BLOCK, int ITEMS>
DEV bool group_sort(const typename KeyT<K64>::type (&k)[ITEMS], uint32_t len, const GroupMap<K64>& map, uint32_t per,
                    BlockSortLds<K64, VALS, BLOCK, ITEMS>& L) {
    typedef typename KeyT<K64>::type K;
    constexpr uint32_t CAP = BLOCK * ITEMS, NG = 1u << FS_BK_GBITS;
    constexpr uint32_t GPT = NG / BLOCK, GLIM = FS_BK_GLIM(K64, VALS);
    static_assert(NG % BLOCK == 0 && sizeof(L.keys) >= (NG + 1u) * 4u, "group counters in the keys' words");
    const uint32_t tid = threadIdx.x;
    const uint32_t row0 = (tid >> 6) * per * 64u + (tid & 63u);
    uint32_t* cnt = reinterpret_cast<uint32_t*>(L.keys);
    for (uint32_t i = tid; i < NG; i += BLOCK) cnt[i] = 0u;
    if (tid == 0) L.flag = 0u;
    __syncthreads();
    Ranks<ITEMS> slot;
#pragma unroll
    for (int g = 0; g < ITEMS; g += 4) {                // (four rows' atomics in flight)
        if ((uint32_t)g >= per) continue;
        uint32_t got[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            got[j] = 0u;
            if (g + j < ITEMS && (uint32_t)(g + j) < per && row0 + (uint32_t)(g + j) * 64u < len)
                got[j] = atomicAdd(&cnt[map(k[g + j < ITEMS ? g + j : 0])], 1u);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (g + j < ITEMS) slot.set_in_order(g + j, got[j]);
    }
    __syncthreads();
    uint32_t c[GPT], sum = 0;
    bool over = false;
#pragma unroll
    for (uint32_t j = 0; j < GPT; ++j) {
        c[j] = cnt[tid * GPT + j];
        sum += c[j];
        over |= c[j] > GLIM;
    }
    if (over) L.flag = 1u;
    uint32_t ex = block_exclusive_scan<BLOCK>(sum, L.wsum);
    const bool big = L.flag != 0u;                      // (uniform)
    if (VALS && big) {
        __syncthreads();
        return false;
    }
#pragma unroll
    for (uint32_t j = 0; j < GPT; ++j) {
        L.starts[tid * GPT + j] = (uint16_t)ex;
        ex += c[j];
    }
    if (tid == BLOCK - 1) L.starts[NG] = (uint16_t)ex;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        if ((uint32_t)i >= per || row0 + (uint32_t)i * 64u >= len) continue;
        uint32_t r = L.starts[map(k[i])] + slot.get(i);
        r = r < CAP ? r : CAP - 1u;
        L.keys[r] = k[i];
        if constexpr (VALS) L.pos[r] = (uint16_t)(row0 + (uint32_t)i * 64u);
    }
    __syncthreads();
    if (!VALS && map.exact()) return true;              // (uniform) a group's keys are equal
    if (!VALS && big) {
        // (uniform) keys only: a large group of equal keys is sorted as it
        // is; one of different keys ends the attempt
        if (tid == 0) L.flag = 0u;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            if ((uint32_t)i >= per || row0 + (uint32_t)i * 64u >= len) continue;
            const uint32_t g = map(k[i]);
            const uint32_t s0 = L.starts[g];
            if (L.starts[g + 1u] - s0 > GLIM && L.keys[s0] != k[i]) L.flag = 1u;
        }
        __syncthreads();
        const bool mixed = L.flag != 0u;
        __syncthreads();
        if (mixed) return false;
    }
    // the key at every position, one after the other (a group's keys are read
    // four at a time; holding every row's group at once took 250 registers)
    K kk[ITEMS];
    Ranks<ITEMS> rank;
    Ranks<VALS ? ITEMS : 1> kp;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const uint32_t x = (uint32_t)i * BLOCK + tid;
        kk[i] = 0;
        uint32_t r = 0, px = 0;
        if (x < len) {
            const K key = L.keys[x];
            kk[i] = key;
            if constexpr (VALS) px = L.pos[x];
            const uint32_t g = map(key);
            const uint32_t s0 = L.starts[g], s1 = L.starts[g + 1u];
            r = !VALS && s1 - s0 > GLIM ? x : s0;
            if (s1 - s0 > 1u && (VALS || s1 - s0 <= GLIM)) {
                for (uint32_t y = s0; y < s1; y += 4u) {
                    K o[4];
#pragma unroll
                    for (uint32_t j = 0; j < 4u; ++j) o[j] = L.keys[min(y + j, CAP - 1u)];
#pragma unroll
                    for (uint32_t j = 0; j < 4u; ++j) {
                        // before this key: smaller ones, and equal ones that come first
                        bool before = o[j] < key;
                        if constexpr (VALS) before |= o[j] == key && L.pos[min(y + j, CAP - 1u)] < px;
                        else before |= o[j] == key && y + j < x;
                        r += before && y + j < s1 ? 1u : 0u;
                    }
                }
            }
        }
        rank.set_in_order(i, r);
        if constexpr (VALS) kp.set_in_order(i, px);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        if ((uint32_t)i * BLOCK + tid >= len) continue;
        const uint32_t r = rank.get(i) < CAP ? rank.get(i) : CAP - 1u;
        L.keys[r] = kk[i];
        if constexpr (VALS) L.pos[r] = (uint16_t)kp.get(i);
    }
    __syncthreads();
    return true;
}

// Sorts the block's rows (k, p: `per` rows to a wave, padding ~0 at the end)
// by bits [lo, hi) of the keys, stably, leaving them in L.keys (L.pos).
// varying: the bits that differ between some keys; digits without any are
// skipped (with none at all the rows are copied as they are).
template <bool K64, bool VALS, int BLOCK, int ITEMS>
DEV void block_sort(typename KeyT<K64>::type (&k)[ITEMS], Ranks<VALS ? ITEMS : 1>& p, uint32_t lo, uint32_t hi,
                    typename KeyT<K64>::type varying, uint32_t per, BlockSortLds<K64, VALS, BLOCK, ITEMS>& L) {
    const uint32_t row0 = (threadIdx.x >> 6) * per * 64u + (threadIdx.x & 63u);
    bool staged = false;
    for (uint32_t shift = lo; shift < hi; shift += FS_RADIX_BITS) {
        if (!((uint32_t)(varying >> shift) & 0xFFu)) continue;          // (uniform)
        if (staged) {
            // (four rows behind one branch, so that their reads overlap; a
            // row past the wave's is within L.keys and never used)
#pragma unroll
            for (int g = 0; g < ITEMS; g += 4) {
                if ((uint32_t)g >= per) continue;
#pragma unroll
                for (int i = g; i < g + 4 && i < ITEMS; ++i) {
                    k[i] = L.keys[row0 + (uint32_t)i * 64u];
                    if constexpr (VALS) p.set_in_order(i, L.pos[row0 + (uint32_t)i * 64u]);
                }
            }
            __syncthreads();                            // every row read before the pass writes
        }
        block_sort_pass<K64, VALS, BLOCK, ITEMS>(k, p, shift, per, L);
        staged = true;
    }
    if (!staged) {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            if ((uint32_t)i >= per) continue;
            L.keys[row0 + (uint32_t)i * 64u] = k[i];
            if constexpr (VALS) L.pos[row0 + (uint32_t)i * 64u] = (uint16_t)p.get(i);
        }
        __syncthreads();
    }
}

// Two folds of the block's valid keys, to every thread: the least and the
// greatest (BITS false), or the bits set in some key and those clear in some
// key.
template <bool K64, bool VALS, int BLOCK, int ITEMS, bool BITS>
DEV void block_fold(const typename KeyT<K64>::type (&k)[ITEMS], uint32_t len, uint32_t per,
                    BlockSortLds<K64, VALS, BLOCK, ITEMS>& L, typename KeyT<K64>::type& r0,
                    typename KeyT<K64>::type& r1) {
    typedef typename KeyT<K64>::type K;
    constexpr int WAVES = BLOCK / 64;
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
    const uint32_t row0 = w * per * 64u + lane;
    auto f0 = [](K a, K b) -> K { return BITS ? (K)(a | b) : a < b ? a : b; };
    auto f1 = [](K a, K b) -> K { return BITS ? (K)(a | b) : a > b ? a : b; };
    const K id0 = BITS ? (K)0 : ~(K)0;
    K x0 = id0, x1 = 0;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        if ((uint32_t)i < per && row0 + (uint32_t)i * 64u < len) {
            x0 = f0(x0, k[i]);
            x1 = f1(x1, BITS ? (K)~k[i] : k[i]);
        }
    }
    x0 = wave_fold<K>(x0, f0);
    x1 = wave_fold<K>(x1, f1);
    if (lane == 63u) {
        L.red[0][w] = x0;
        L.red[1][w] = x1;
    }
    __syncthreads();
    K y0 = id0, y1 = 0;
#pragma unroll
    for (int ww = 0; ww < WAVES; ++ww) {
        y0 = f0(y0, L.red[0][ww]);
        y1 = f1(y1, L.red[1][ww]);
    }
    __syncthreads();
    r0 = y0;
    r1 = y1;
}

template <typename K>
DEV uint32_t bit_length(K v) {
    if constexpr (sizeof(K) == 4) return v ? 32u - (uint32_t)__builtin_clz(v) : 0u;
    else return v ? 64u - (uint32_t)__builtin_clzll((unsigned long long)v) : 0u;
}

// The map of a block whose keys run from `least` to `most`: by value (floats),
// or by the top bits of the range.
template <bool K64>
DEV GroupMap<K64> group_map(typename KeyT<K64>::type least, typename KeyT<K64>::type most, bool by_value) {
    typedef typename KeyT<K64>::type K;
    typedef GroupMap<K64> Map;
    const uint32_t bits = bit_length<K>(most - least);
    Map map{by_value, bits > FS_BK_GBITS ? bits - FS_BK_GBITS : 0u, least, (K)(most - least), 0.0, 0.0};
    if (by_value) {
        const K lo = least < (K)~Map::FINITE ? (K)~Map::FINITE : least > Map::FINITE ? Map::FINITE : least;
        const K hi = most > Map::FINITE ? Map::FINITE : most < (K)~Map::FINITE ? (K)~Map::FINITE : most;
        map.low = Map::value(lo);
        const double span = Map::value(hi) - map.low;
        map.scale = span > 0.0 ? (double)(1u << FS_BK_GBITS) / span : 0.0;
    }
    return map;
}

// The block sort: the block's len keys (rows of k, which are less `base` on
// return; p: their positions) into L.keys (L.pos), in stable order.
template <bool K64, bool VALS, int BLOCK, int ITEMS>
DEV void sort_rows(typename KeyT<K64>::type (&k)[ITEMS], Ranks<VALS ? ITEMS : 1>& p, uint32_t len, uint32_t per,
                   bool floats, BlockSortLds<K64, VALS, BLOCK, ITEMS>& L, typename KeyT<K64>::type& base) {
    typedef typename KeyT<K64>::type K;
    const uint32_t row0 = (threadIdx.x >> 6) * per * 64u + (threadIdx.x & 63u);
    K least = 0, most = 0;
    block_fold<K64, VALS, BLOCK, ITEMS, false>(k, len, per, L, least, most);
    base = least;
    const uint32_t bits = bit_length<K>(most - least);
#pragma unroll
    for (int i = 0; i < ITEMS; ++i)
        if ((uint32_t)i < per && row0 + (uint32_t)i * 64u < len) k[i] -= least;
    // (values: a range of two digits takes two stable passes at most, fewer
    // than the groups' steps)
    if (!VALS || bits > 2u * FS_RADIX_BITS) {
        // floats: by value where that spreads them (most data), then by bits
        if (floats && bits > FS_BK_GBITS &&
            group_sort<K64, VALS, BLOCK, ITEMS>(k, len, group_map<K64>(least, most, true), per, L))
            return;
        if (group_sort<K64, VALS, BLOCK, ITEMS>(k, len, group_map<K64>(least, most, false), per, L)) return;
    }
    K on = 0, off = 0;
    block_fold<K64, VALS, BLOCK, ITEMS, true>(k, len, per, L, on, off);
    block_sort<K64, VALS, BLOCK, ITEMS>(k, p, 0u, bits, on & off, per, L);
}

// Counts the block's keys by group (k less the map's base) and leaves the
// groups' starts in L.starts; true when no group holds more than `limit`.
template <bool K64, bool VALS, int BLOCK, int ITEMS>
DEV bool count_groups(const typename KeyT<K64>::type (&k)[ITEMS], uint32_t len, const GroupMap<K64>& map, uint32_t per,
                      uint32_t limit, BlockSortLds<K64, VALS, BLOCK, ITEMS>& L) {
    constexpr uint32_t NG = 1u << FS_BK_GBITS, GPT = NG / BLOCK;
    const uint32_t tid = threadIdx.x;
    const uint32_t row0 = (tid >> 6) * per * 64u + (tid & 63u);
    uint32_t* cnt = reinterpret_cast<uint32_t*>(L.keys);
    for (uint32_t i = tid; i < NG; i += BLOCK) cnt[i] = 0u;
    if (tid == 0) L.flag = 0u;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i)
        if ((uint32_t)i < per && row0 + (uint32_t)i * 64u < len) atomicAdd(&cnt[map(k[i])], 1u);
    __syncthreads();
    uint32_t c[GPT], sum = 0;
    bool over = false;
#pragma unroll
    for (uint32_t j = 0; j < GPT; ++j) {
        c[j] = cnt[tid * GPT + j];
        sum += c[j];
        over |= c[j] > limit;
    }
    if (over) L.flag = 1u;
    uint32_t ex = block_exclusive_scan<BLOCK>(sum, L.wsum);
#pragma unroll
    for (uint32_t j = 0; j < GPT; ++j) {
        L.starts[tid * GPT + j] = (uint16_t)ex;
        ex += c[j];
    }
    if (tid == BLOCK - 1) L.starts[NG] = (uint16_t)ex;
    const bool fine = L.flag == 0u;
    __syncthreads();
    return fine;
}

// The schedule words fs_last_pass_info reads: a digit counts as sorted when
// some key has a bit of it set that another has clear.
template <bool K64>
DEV void bucket_pass_info(const FsArgs& a, uint64_t varying) {
    uint32_t mask = 0, p = 0;
    for (uint32_t j = 0; j < (K64 ? 8u : 4u); ++j)
        if ((varying >> (8u * j)) & 0xFFu) {
            mask |= 1u << j;
            ++p;
        }
    GLOBAL uint32_t* plan = gptr<uint32_t>(a.plan);
    st_agent(&plan[FS_PLAN_NPASSES], p);
    st_agent(&plan[FS_PLAN_MASK], mask | FS_MASK_FUSED);
    st_agent(&plan[FS_PLAN_RESCATTER], 0u);
}

// ---------------------------------------------------------------------------
// fs_split_*: the splitters
// ---------------------------------------------------------------------------

template <bool K64, int BLOCK, int ITEMS>
DEV void split_body(const FsArgs& a) {
    typedef typename KeyT<K64>::type K;
    constexpr uint32_t CAP = BLOCK * ITEMS;
    __shared__ BlockSortLds<K64, false, BLOCK, ITEMS> L;
    __shared__ K lbs[FS_BK_NB];
    static_assert(BLOCK >= FS_BK_NB, "a bucket per thread");
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    const uint32_t nb = 1u << a.bk_lnb, m = 1u << a.bk_lm;
    if (nb > FS_BK_NB || m > CAP || m < nb) {
        if (tid == 0) report(a, FS_DEVERR_BAD_PLAN);
        return;
    }
    GLOBAL uint32_t* tab = gptr<uint32_t>(a.bk_tab);

    // samples 4i .. 4i + 3: consecutive keys (one line of memory) at a hashed
    // position within the i-th of m / 4 equal parts of the input
    const GLOBAL K* src = gptr<const K>(a.keys);
    const uint32_t per = (m + BLOCK - 1u) / BLOCK;
    const uint32_t row0 = w * per * 64u + lane;
    K k[ITEMS];
    Ranks<1> none;
    none.r[0] = 0u;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const uint32_t s = row0 + (uint32_t)i * 64u;
        k[i] = ~(K)0;
        if ((uint32_t)i < per && s < m) {
            const uint32_t c = s >> 2;
            const uint64_t p0 = ((uint64_t)c * a.n) >> (a.bk_lm - 2u), p1 = ((uint64_t)(c + 1u) * a.n) >> (a.bk_lm - 2u);
            const uint32_t h = (c * 0x9E3779B9u) ^ ((c * 0x85EBCA6Bu) >> 13);
            const uint64_t p = p0 + (((uint64_t)h * (p1 > p0 + 4u ? p1 - p0 - 4u : 1u)) >> 32) + (s & 3u);
            k[i] = xf_fwd<K64>(src[p < a.n ? p : a.n - 1u], a.xform);
        }
    }
    // counters of the partition and (values) its look-back entries start at zero
    for (uint32_t i = tid; i < FS_BK_NB; i += BLOCK) st_agent(&tab[FS_BK_CNT + i], 0u);
    for (uint32_t i = tid; i < 4u * FS_BK_BIT_SLOTS; i += BLOCK) st_agent(&tab[FS_BK_BITS + i], 0u);
    if (a.op != FSK_OP_KEYS) {
        GLOBAL uint4* lb = gptr<uint4>(a.lookback0);
        const uint32_t words = (a.num_tiles + (a.num_tiles + FS_LB_GROUP - 1u) / FS_LB_GROUP) * FS_BK_NB;
        for (uint32_t i = tid; i < words / 4u; i += BLOCK) lb[i] = uint4{0u, 0u, 0u, 0u};
    }

    const uint32_t stride = m / nb;
    K least = 0, most = 0;
    block_fold<K64, false, BLOCK, ITEMS, false>(k, m, per, L, least, most);
    const K base = least;
    const uint32_t bits = bit_length<K>(most - least);
#pragma unroll
    for (int i = 0; i < ITEMS; ++i)
        if ((uint32_t)i < per && row0 + (uint32_t)i * 64u < m) k[i] -= base;
    // Where the groups of the block sort spread the sample (none holds more
    // than two quantiles' share), their counts alone give the splitters: the
    // key a quantile's share of the way through its group.
    GroupMap<K64> map = group_map<K64>(least, most, a.xform == FS_XF_FLOAT);
    uint32_t s0 = 0, s1 = 0;                             // samples below this thread's bucket, and below the next
    bool spread = count_groups<K64, false, BLOCK, ITEMS>(k, m, map, per, 2u * stride, L);   // (uniform)
    if (!spread && map.by_value) {
        map = group_map<K64>(least, most, false);
        spread = count_groups<K64, false, BLOCK, ITEMS>(k, m, map, per, 2u * stride, L);
    }
    if (spread) {
        for (uint32_t i = tid; i < FS_BK_NB; i += BLOCK) lbs[i] = i ? ~(K)0 : (K)0;
        __syncthreads();
        s0 = tid * stride;
        s1 = s0 + stride;
        if (tid >= 1u && tid < nb) {
            uint32_t g = 0;                              // the group holding sample s0 (in order)
#pragma unroll
            for (uint32_t step = 1u << (FS_BK_GBITS - 1); step; step >>= 1)
                if (L.starts[g + step] <= s0) g += step;
            const uint32_t g0 = L.starts[g], gn = L.starts[g + 1u] - g0;
            lbs[tid] = map.inside(g, gn ? (float)(s0 - g0) / (float)gn : 0.0f);
        }
        __syncthreads();
    } else {
        // Keys crowded in parts of the range, or many copies of some: the
        // sample sorted, by groups where those hold copies of one key each,
        // else by stable passes.  64-bit keys take the top FS_BK_SAMPLE_BITS
        // bits of their range first (enough to order most samples), all of
        // them when two neighbours are then out of order.
        bool done = a.xform == FS_XF_FLOAT &&
                    group_sort<K64, false, BLOCK, ITEMS>(k, m, group_map<K64>(least, most, true), per, L);
        if (!done) done = group_sort<K64, false, BLOCK, ITEMS>(k, m, group_map<K64>(least, most, false), per, L);
        if (!done) {
            const uint32_t lo = bits > FS_BK_SAMPLE_BITS ? bits - FS_BK_SAMPLE_BITS : 0u;
            K on = 0, off = 0;
            block_fold<K64, false, BLOCK, ITEMS, true>(k, m, per, L, on, off);
            block_sort<K64, false, BLOCK, ITEMS>(k, none, lo, bits, on & off, per, L);
            if (lo) {
                bool bad = false;
                for (uint32_t i = tid; i + 1u < m; i += BLOCK) bad |= L.keys[i] > L.keys[i + 1u];
                if (tid == 0) L.flag = 0u;
                __syncthreads();
                if (bad) L.flag = 1u;
                __syncthreads();
                const bool again = L.flag != 0u;
                __syncthreads();
                if (again) {
#pragma unroll
                    for (int i = 0; i < ITEMS; ++i)
                        if ((uint32_t)i < per) k[i] = L.keys[row0 + (uint32_t)i * 64u];
                    __syncthreads();
                    block_sort<K64, false, BLOCK, ITEMS>(k, none, 0u, bits, on & off, per, L);
                }
            }
        }
        // Splitters: quantile v, and v + 1 after a value that the next
        // quantile repeats (its copies fill the bucket [v, v + 1) alone).  At
        // most one splitter per quantile, since a repeated quantile adds none
        // of its own.
        K q = 0;
        uint32_t emit = 0;
        if (tid >= 1u && tid < nb) {
            q = L.keys[tid * stride];
            const bool rep = tid > 1u && q == L.keys[(tid - 1u) * stride];
            const bool dup = tid + 1u < nb && q == L.keys[(tid + 1u) * stride] && (K)(q + base) != ~(K)0;
            emit = rep ? 0u : dup ? 2u : 1u;
        }
        for (uint32_t i = tid; i < FS_BK_NB; i += BLOCK) lbs[i] = i ? ~(K)0 : (K)0;
        const uint32_t at = block_exclusive_scan<BLOCK>(emit, L.wsum) + 1u;
        if (emit && at < nb) lbs[at] = q + base;
        if (emit == 2u && at + 1u < nb) lbs[at + 1u] = q + base + 1u;
        __syncthreads();
        auto below = [&](K v) -> uint32_t {              // samples less than v
            if (v <= base) return 0u;
            const K t = v - base;
            uint32_t x = 0;
            for (uint32_t step = m >> 1; step; step >>= 1)
                if (L.keys[x + step - 1u] < t) x += step;
            return x + ((x < m && L.keys[x] < t) ? 1u : 0u);
        };
        if (tid < nb) {
            s0 = tid ? below(lbs[tid]) : 0u;
            s1 = tid + 1u < nb ? below(lbs[tid + 1u]) : m;
        }
    }

    // Region of bucket j: room for its share of the sample plus six standard
    // deviations, scaled to n.
    uint32_t cap = 0;
    if (tid < nb) {
        const float c = (float)(s1 > s0 ? s1 - s0 : 0u);
        const float room = c + 6.0f * __builtin_sqrtf(c) + FS_BK_ROOM;
        cap = ((uint32_t)(room * ((float)a.n / (float)m)) + 16u) & ~15u;
        if (cap > (uint32_t)a.n) cap = ((uint32_t)a.n + 15u) & ~15u;
    }
#ifdef FS_FAULT_INJECTION
    if (a.fault == FS_FAULT_SMALL_REGIONS && tid == 1u) cap = 64u;
#endif
    const uint32_t rbase = block_exclusive_scan<BLOCK>(cap, L.wsum);
    if (tid < nb) {
        // (a layout beyond S1 cannot be: the host sized it for the largest)
        const bool fits = (uint64_t)rbase + cap <= a.s1_keys;
        if (!fits) report(a, FS_DEVERR_BAD_PLAN);
        tab[FS_BK_BASE + tid] = fits ? rbase : 0u;
        tab[FS_BK_CAPS + tid] = fits ? cap : 0u;
        reinterpret_cast<GLOBAL K*>(tab + FS_BK_LB)[tid] = lbs[tid];
    }
}

// ---------------------------------------------------------------------------
// fs_part_*: keys (and values) to their buckets' regions
// ---------------------------------------------------------------------------

template <bool K64, bool VALS, int BLOCK, int ITEMS>
DEV void part_body(const FsArgs& a) {
    typedef typename KeyT<K64>::type K;
    constexpr int WAVES = BLOCK / 64;
    constexpr uint32_t TILE = BLOCK * ITEMS;
    constexpr uint32_t NB = FS_BK_NB;
    constexpr uint32_t DROP = 0xFFFFFFFFu;
    static_assert(BLOCK >= FS_BK_NB && TILE <= 0xFFFFu, "a bucket per thread, 16-bit tile positions");
    static_assert((uint64_t)FS_LB_GROUP * TILE < (1ull << FS_LB_GCOUNT_SHIFT), "group sums must fit their field");
    __shared__ union {
        K keys[TILE];
        uint32_t vals[TILE];
    } stage;
    __shared__ uint16_t bid[TILE];                     // bucket of every staged position
    __shared__ uint16_t wcnt[VALS ? WAVES : 1][NB];    // values: per-wave bucket counts, then bases
    __shared__ K lbs[NB];
    __shared__ uint32_t cnt[NB];                       // the tile's bucket counts, then starts
    __shared__ uint32_t gbase[NB];
    __shared__ uint32_t wsum[WAVES];
    __shared__ uint32_t bits[4];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    const uint32_t lnb = a.bk_lnb, nb = 1u << lnb;
    const uint32_t tile = blockIdx.x, n32 = (uint32_t)a.n;
    const uint32_t rows = a.tile / BLOCK;               // keys per thread of this sort's tiles (at most ITEMS)
    if (tile >= a.num_tiles || nb > NB || rows > (uint32_t)ITEMS || rows == 0u) {
        if (tid == 0) report(a, FS_DEVERR_BAD_TILE);
        return;
    }
    GLOBAL uint32_t* tab = gptr<uint32_t>(a.bk_tab);
    const uint32_t begin = tile * a.tile, wbegin = begin + w * 64u * rows + lane;
    const uint32_t tv = n32 - begin < a.tile ? n32 - begin : a.tile;  // the tile's keys
    const GLOBAL K* src = gptr<const K>(a.keys);
    auto valid = [&](int i) -> bool { return (uint32_t)i < rows && wbegin + (uint32_t)i * 64u < n32; };
    K k[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) k[i] = valid(i) ? src[wbegin + (uint32_t)i * 64u] : (K)0;
    for (uint32_t i = tid; i < NB; i += BLOCK) {
        lbs[i] = i < nb ? reinterpret_cast<const GLOBAL K*>(tab + FS_BK_LB)[i] : ~(K)0;
        cnt[i] = 0u;
    }
    if (tid < 4u) bits[tid] = 0u;
    if (VALS)
        for (uint32_t i = tid; i < WAVES * NB / 2u; i += BLOCK) reinterpret_cast<uint32_t*>(&wcnt[0][0])[i] = 0u;
    __syncthreads();
    K on = 0, off = 0;
    uint32_t b[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        k[i] = xf_fwd<K64>(k[i], a.xform);
        if (valid(i)) {
            on |= k[i];
            off |= ~k[i];
        }
        b[i] = 0u;
    }
    // bucket: the number of splitters at or below the key (every item's
    // search advances together: the reads of a step are independent)
    for (uint32_t step = nb >> 1; step; step >>= 1) {
#pragma unroll
        for (int g = 0; g < ITEMS; g += 4) {
            if ((uint32_t)g >= rows) continue;
#pragma unroll
            for (int i = g; i < g + 4 && i < ITEMS; ++i) b[i] += lbs[b[i] + step] <= k[i] ? step : 0u;
        }
    }
    // the tile's bits to one of several slots (every tile on one word would
    // queue there)
    on = wave_fold<K>(on, [](K x, K y) { return (K)(x | y); });
    off = wave_fold<K>(off, [](K x, K y) { return (K)(x | y); });
    if (lane == 63u) {
        atomicOr(&bits[0], (uint32_t)on);
        atomicOr(&bits[2], (uint32_t)off);
        if (K64) {
            atomicOr(&bits[1], (uint32_t)((uint64_t)on >> 32));
            atomicOr(&bits[3], (uint32_t)((uint64_t)off >> 32));
        }
    }
    // (every lane takes part in the counting; the lanes past n count nothing)
    Ranks<ITEMS> rank;
    {
        const bool skew = skewed_digit(b[0] == __builtin_amdgcn_readfirstlane(b[0]));
        if (VALS) {
#pragma unroll
            for (int i = 0; i < ITEMS; ++i) {
                if (skew) add_peeled_valid(cnt, b[i], b[i], 1u, lane, valid(i));
                else if (valid(i)) atomicAdd(&cnt[b[i]], 1u);
            }
        } else if (!skew) {
#pragma unroll
            for (int i = 0; i < ITEMS; ++i)
                rank.set_in_order(i, slot_in_digit<false>(cnt, b[i], lane, valid(i)));
        } else {
#pragma unroll
            for (int i = 0; i < ITEMS; ++i)
                rank.set_in_order(i, slot_in_digit<true>(cnt, b[i], lane, valid(i)));
        }
    }
    __syncthreads();
    if (tid < 4u && bits[tid])
        __hip_atomic_fetch_or(&tab[FS_BK_BITS + 4u * (tile % FS_BK_BIT_SLOTS) + tid], bits[tid], __ATOMIC_RELAXED,
                              __HIP_MEMORY_SCOPE_AGENT);
    GLOBAL uint32_t* lb = gptr<uint32_t>(a.lookback0);
    GLOBAL uint32_t* grp = lb + (uint64_t)a.num_tiles * NB;
    const uint32_t count = tid < nb ? cnt[tid] : 0u;
    if (VALS && tid < nb) {
        LbEntry<false>::store(lb, (uint64_t)tile * NB + tid, tile == 0u ? FS_LB_INC : FS_LB_AGG, count);
        __hip_atomic_fetch_add(&grp[(uint64_t)(tile / FS_LB_GROUP) * NB + tid], (1u << FS_LB_GCOUNT_SHIFT) | count,
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    const uint32_t ex = block_exclusive_scan<BLOCK>(count, wsum);
    if (tid < nb) {
        uint32_t at = 0;
        if (VALS) {
            uint32_t r0 = 0, r1 = 0, r2 = 0;
            at = tile == 0u ? 0u : lookback<false, NB>(lb, grp, tile, tid, count, a.status, r0, r1, r2);
            if (tile + 1u == a.num_tiles) st_agent(&tab[FS_BK_CNT + tid], at + count);
        } else if (count) {
            at = __hip_atomic_fetch_add(&tab[FS_BK_CNT + tid], count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        const uint32_t cap = tab[FS_BK_CAPS + tid];
        // (a run that does not fit is dropped: the bucket launch sees the count)
        gbase[tid] = (at <= cap && count <= cap - at) ? tab[FS_BK_BASE + tid] + at - ex : DROP;
        cnt[tid] = ex;
    }
    if (VALS) rank_wave<true, ITEMS, FS_BK_LNB>(b, 0u, wcnt[w], rank, rows);
    __syncthreads();
    if (VALS) {
        if (tid < nb) {
            uint32_t run = cnt[tid];
#pragma unroll
            for (int ww = 0; ww < WAVES; ++ww) {
                const uint32_t c = wcnt[ww][tid];
                wcnt[ww][tid] = (uint16_t)run;           // tile position of (wave, bucket)
                run += c;
            }
        }
        __syncthreads();
    }
    // With values the lanes past n rank too (bucket of the key 0 they hold,
    // after the wave's keys): the last tile's last waves' counts hold them, so
    // those lanes' positions are taken out again below by writing nothing.
    Ranks<VALS ? ITEMS : 1> pos;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        uint32_t r = (VALS ? wcnt[VALS ? w : 0][b[i]] : cnt[b[i]]) + rank.get(i);
        r = r < TILE ? r : TILE - 1u;
        if (VALS) pos.set_in_order(i, r);
        if (valid(i)) {
            stage.keys[r] = k[i];
            bid[r] = (uint16_t)b[i];
        }
    }
    __syncthreads();
    GLOBAL K* dst = gptr<K>(a.s1k);
    uint32_t gp[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const uint32_t p = (uint32_t)i * BLOCK + tid;
        gp[i] = DROP;
        if (p < tv) {
            const uint32_t g = gbase[bid[p] & (NB - 1u)];
            if (g != DROP && g + p < a.s1_keys) {
                gp[i] = g + p;
                dst[g + p] = stage.keys[p];
            }
        }
    }
    if (VALS) {
        uint32_t v[ITEMS];
        const GLOBAL uint32_t* sv = gptr<const uint32_t>(a.vals);
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            const uint32_t p = wbegin + (uint32_t)i * 64u;
            v[i] = a.op == FSK_OP_ARGSORT ? p : valid(i) ? sv[p] : 0u;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < ITEMS; ++i)
            if (valid(i)) stage.vals[pos.get(i)] = v[i];
        __syncthreads();
        GLOBAL uint32_t* dv = gptr<uint32_t>(a.s1v);
#pragma unroll
        for (int i = 0; i < ITEMS; ++i)
            if (gp[i] != DROP) dv[gp[i]] = stage.vals[(uint32_t)i * BLOCK + tid];
    }
}

// ---------------------------------------------------------------------------
// fs_bucket_*: one block sorts one bucket (or the whole of a small input)
// ---------------------------------------------------------------------------

// Keys (and values) of one range sorted by one block through device memory, a
// digit at a time: src -> A -> B -> A ... -> dst.  For ranges that LDS cannot
// hold (see above: hardly ever).  fwd: the source holds the caller's keys; a
// source without values takes their positions (argsort).
template <bool K64, bool VALS, int BLOCK, int ITEMS>
DEV void slow_sort(const FsArgs& a, uint64_t src_k, uint64_t src_v, bool fwd, uint64_t ak, uint64_t av, uint64_t bk,
                   uint64_t bv, uint64_t dst_k, uint64_t dst_v, uint32_t len,
                   BlockSortLds<K64, VALS, BLOCK, ITEMS>& L) {
    typedef typename KeyT<K64>::type K;
    constexpr int WAVES = BLOCK / 64, IT = 4;
    constexpr uint32_t CH = BLOCK * IT, D = sizeof(K);
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    const uint32_t wb = w * 64u * IT + lane;
    uint32_t* bins = L.dbase;
    for (uint32_t q = 0; q < D; ++q) {
        const uint32_t shift = 8u * q;
        const bool final_pass = q + 1u == D, from_a = (q & 1u) != 0u;
        const GLOBAL K* in = gptr<const K>(q == 0u ? src_k : from_a ? ak : bk);
        const uint64_t in_v = q == 0u ? src_v : from_a ? av : bv;
        GLOBAL K* out = gptr<K>(final_pass ? dst_k : from_a ? bk : ak);
        GLOBAL uint32_t* out_v = gptr<uint32_t>(final_pass ? dst_v : from_a ? bv : av);
        const uint32_t xf = q == 0u && fwd ? a.xform : FS_XF_NONE;
        K xa, xb;
        xf_inv_masks<K64>(final_pass ? a.xform : FS_XF_NONE, xa, xb);
        if (tid < FS_RADIX) bins[tid] = 0u;
        __syncthreads();
        for (uint32_t p0 = 0; p0 < len; p0 += BLOCK) {
            const uint32_t p = p0 + tid;
            const bool v = p < len;
            const uint32_t d = digit_of<K64>(xf_fwd<K64>(in[v ? p : 0u], xf), shift);
            if (skewed_digit(d == __builtin_amdgcn_readfirstlane(d))) add_peeled_valid(bins, d, d, 1u, lane, v);
            else if (v) atomicAdd(&bins[d], 1u);
        }
        __syncthreads();
        const uint32_t ex = radix_exclusive_scan(tid < FS_RADIX ? bins[tid] : 0u, L.wsum);
        if (tid < FS_RADIX) bins[tid] = ex;
        for (uint32_t c0 = 0; c0 < len; c0 += CH) {
            const uint32_t clen = len - c0 < CH ? len - c0 : CH;
            K k[IT];
            uint32_t x[IT];
#pragma unroll
            for (int i = 0; i < IT; ++i) {
                const uint32_t p = wb + (uint32_t)i * 64u;
                k[i] = p < clen ? xf_fwd<K64>(in[c0 + p], xf) : ~(K)0;   // padding: digit 255, ranked last
                x[i] = (uint32_t)(k[i] >> shift);
            }
            for (uint32_t i = tid; i < WAVES * FS_RADIX / 2u; i += BLOCK) reinterpret_cast<uint32_t*>(&L.wcnt[0][0])[i] = 0u;
            __syncthreads();
            Ranks<IT> rank;
            rank_wave<false, IT>(x, 0u, L.wcnt[w], rank);
            __syncthreads();
            uint32_t tot = wave_bases<WAVES>(L.wcnt);
            if (tid == FS_RADIX - 1u) tot -= CH - clen;
            __syncthreads();
#pragma unroll
            for (int i = 0; i < IT; ++i) {
                const uint32_t p = wb + (uint32_t)i * 64u;
                if (p >= clen) continue;
                const uint32_t d = x[i] & 0xFFu;
                const uint32_t pos = bins[d] + L.wcnt[w][d] + rank.get(i);
                if (pos >= len) continue;
                if (!(final_pass && a.op == FSK_OP_ARGSORT)) out[pos] = xf_inv_apply<K64>(k[i], xa, xb);
                if (VALS) out_v[pos] = in_v ? gptr<const uint32_t>(in_v)[c0 + p] : c0 + p;
            }
            __syncthreads();
            if (tid < FS_RADIX) bins[tid] += tot;
        }
        __syncthreads();                               // this pass's writes before the next reads
    }
}

template <bool K64, bool VALS, int BLOCK, int ITEMS>
DEV void bucket_body(const FsArgs& a) {
    typedef typename KeyT<K64>::type K;
    typedef BlockSortLds<K64, VALS, BLOCK, ITEMS> Lds;
    constexpr uint32_t CAP = Lds::CAP;
    __shared__ Lds L;
    __shared__ uint32_t s_seg[2];
    __shared__ uint32_t s_over, s_giants;
    __shared__ uint16_t giant[FS_BK_NB];
    static_assert(CAP <= 0x10000u, "16-bit positions");
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    const uint32_t lnb = a.bk_lnb, nb = 1u << lnb;
    const bool whole = lnb == 0u;                       // (uniform) one block, the caller's keys
    const GLOBAL uint32_t* tab = gptr<const uint32_t>(a.bk_tab);
    uint32_t start = 0, len = (uint32_t)a.n;
    uint64_t src_k = a.keys, src_v = a.op == FSK_OP_PAIRS ? a.vals : 0u;
    const bool put_keys = a.op != FSK_OP_ARGSORT;
    K xa, xb;
    xf_inv_masks<K64>(a.xform, xa, xb);
    GLOBAL K* dk = gptr<K>(a.keys);
    GLOBAL uint32_t* dv = gptr<uint32_t>(a.vals);
    if (!whole) {
        if (nb > FS_BK_NB || gridDim.x != nb) {
            if (tid == 0) report(a, FS_DEVERR_BAD_PLAN);
            return;
        }
        // the bucket's place: the keys of the buckets before it
        if (tid == 0) s_over = s_giants = 0u;
        const uint32_t c = tid < nb ? tab[FS_BK_CNT + tid] : 0u;
        const uint32_t cap = tid < nb ? tab[FS_BK_CAPS + tid] : 0u, rb = tid < nb ? tab[FS_BK_BASE + tid] : 0u;
        const GLOBAL K* lbs = reinterpret_cast<const GLOBAL K*>(tab + FS_BK_LB);
        const uint32_t ex = block_exclusive_scan<BLOCK>(c, L.wsum);
        if (tid < nb) {
            if (c > cap) s_over = 1u;
            // buckets of one value that outgrow a block: copied by every block
            // in turn, a block's keys at a time
            if (c > CAP && (tid + 1u < nb ? lbs[tid + 1u] - lbs[tid] == (K)1 : lbs[tid] == ~(K)0))
                giant[atomicAdd(&s_giants, 1u)] = (uint16_t)tid;
            if (tid == blockIdx.x) {
                s_seg[0] = ex;
                s_seg[1] = c;
            }
            reinterpret_cast<uint32_t*>(L.keys)[tid] = ex;
            reinterpret_cast<uint32_t*>(L.keys)[FS_BK_NB + tid] = c;
        }
        static_assert(sizeof(L.keys) >= 8u * FS_BK_NB, "bucket starts and counts in the sort's words");
        __syncthreads();
        start = s_seg[0];
        len = s_seg[1];
        if (blockIdx.x == 0 && tid == 0) {
            uint32_t b[4] = {0u, 0u, 0u, 0u};
#pragma unroll
            for (uint32_t i = 0; i < 4u * FS_BK_BIT_SLOTS; ++i) b[i % 4u] |= tab[FS_BK_BITS + i];
            bucket_pass_info<K64>(a, ((uint64_t)(b[1] & b[3]) << 32) | (b[0] & b[2]));
        }
        if (s_over) {                                   // (uniform) a region overflowed: block 0 sorts the caller's keys
            __syncthreads();
            if (blockIdx.x == 0)
                slow_sort<K64, VALS, BLOCK, ITEMS>(a, a.keys, src_v, true, a.s2k, a.s2v, a.s1k, a.s1v, a.keys, a.vals,
                                                   (uint32_t)a.n, L);
            return;
        }
        const uint32_t giants = s_giants;
        bool mine = false;
        for (uint32_t g = 0; g < giants; ++g) {
            const uint32_t j = giant[g];
            mine |= j == blockIdx.x;
            const uint32_t gs = reinterpret_cast<const uint32_t*>(L.keys)[j];
            const uint32_t gc = reinterpret_cast<const uint32_t*>(L.keys)[FS_BK_NB + j];
            const K v = xf_inv_apply<K64>(lbs[j], xa, xb);
            const GLOBAL uint32_t* sv = gptr<const uint32_t>(a.s1v) + tab[FS_BK_BASE + j];
            for (uint32_t p = blockIdx.x * BLOCK + tid; p < gc; p += nb * BLOCK) {
                if (put_keys) dk[gs + p] = v;
                if (VALS) dv[gs + p] = sv[p];
            }
        }
        __syncthreads();                                // the starts' words are the sort's again
        if (mine || len == 0u) return;                  // (uniform)
        const uint64_t r = tab[FS_BK_BASE + blockIdx.x];
        src_k = a.s1k + r * sizeof(K);
        src_v = VALS ? a.s1v + r * 4u : 0u;
        if (len > CAP) {                                // (uniform) larger than LDS holds
            slow_sort<K64, VALS, BLOCK, ITEMS>(a, src_k, src_v, false, a.s2k + (uint64_t)start * sizeof(K),
                                               a.s2v + (uint64_t)start * 4u, src_k, src_v,
                                               a.keys + (uint64_t)start * sizeof(K), a.vals + (uint64_t)start * 4u, len, L);
            return;
        }
    } else if (len > CAP) {
        if (tid == 0) report(a, FS_DEVERR_BAD_PLAN);
        return;
    }

    const uint32_t per = (len + BLOCK - 1u) / BLOCK;     // rows per wave
    const uint32_t row0 = w * per * 64u + lane;
    const GLOBAL K* src = gptr<const K>(src_k);
    K k[ITEMS];
    Ranks<VALS ? ITEMS : 1> p;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const uint32_t x = row0 + (uint32_t)i * 64u;
        k[i] = (uint32_t)i < per && x < len ? src[x] : ~(K)0;
        if (VALS) p.set_in_order(i, x & 0xFFFFu);
    }
    if (whole) {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i)
            if (row0 + (uint32_t)i * 64u < len) k[i] = xf_fwd<K64>(k[i], a.xform);
    }
    if (whole) {
        K on = 0, off = 0;
        block_fold<K64, VALS, BLOCK, ITEMS, true>(k, len, per, L, on, off);
        if (tid == 0) bucket_pass_info<K64>(a, (uint64_t)(on & off));
    }
    K base = 0;
    sort_rows<K64, VALS, BLOCK, ITEMS>(k, p, len, per, a.xform == FS_XF_FLOAT, L, base);

    // consecutive positions per thread index; values by the position their key had
    if constexpr (VALS) {
        uint32_t v[ITEMS];
        const GLOBAL uint32_t* sv = gptr<const uint32_t>(src_v);
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            const uint32_t x = (uint32_t)i * BLOCK + tid;
            v[i] = x < len ? (src_v ? sv[L.pos[x]] : L.pos[x]) : 0u;
        }
        if (whole) __syncthreads();                     // in place: every value read before any is written
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            const uint32_t x = (uint32_t)i * BLOCK + tid;
            if (x < len) dv[start + x] = v[i];
        }
    }
    if (put_keys) {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            const uint32_t x = (uint32_t)i * BLOCK + tid;
            if (x < len) dk[start + x] = xf_inv_apply<K64>((K)(L.keys[x] + base), xa, xb);
        }
    }
}

// Blocks per CU by LDS: the bucket kernels' registers leave room for them.
#define FS_BK_KERNELS(sfx, K64, VALS, PITEMS, BITEMS, WAVES)                                                      \
    extern "C" __global__ void __launch_bounds__(FS_BP_BLOCK) fs_part_##sfx(FsArgs a) {                           \
        part_body<K64, VALS, FS_BP_BLOCK, PITEMS>(a);                                                             \
    }                                                                                                             \
    extern "C" __global__ void __launch_bounds__(FS_BK_BLOCK) FS_OCC(WAVES) fs_bucket_##sfx(FsArgs a) {           \
        bucket_body<K64, VALS, FS_BK_BLOCK, BITEMS>(a);                                                           \
    }
FS_BK_KERNELS(k32, false, false, FS_BP32_ITEMS, FS_BK32_ITEMS, FS_BK32_WAVES)
FS_BK_KERNELS(k32_v, false, true, FS_BP32_ITEMS, FS_BK32V_ITEMS, FS_BK32V_WAVES)
FS_BK_KERNELS(k64, true, false, FS_BP64_ITEMS, FS_BK64_ITEMS, FS_BK64_WAVES)
FS_BK_KERNELS(k64_v, true, true, FS_BP64_ITEMS, FS_BK64V_ITEMS, FS_BK64V_WAVES)

extern "C" __global__ void __launch_bounds__(FS_BS_BLOCK) fs_split_k32(FsArgs a) {
    split_body<false, FS_BS_BLOCK, FS_BS_ITEMS>(a);
}
extern "C" __global__ void __launch_bounds__(FS_BS_BLOCK) fs_split_k64(FsArgs a) {
    split_body<true, FS_BS_BLOCK, FS_BS_ITEMS>(a);
}
