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
//                   from a table of the keys' groups or by binary search in
//                   the splitters (LDS), its place by one atomic per tile and
//                   bucket (keys only) or, for values, whose order among
//                   equal keys must hold, by the decoupled look-back of the
//                   digit passes
//     fs_bucket_*   one block per bucket: read once, sorted in LDS, written
//                   once to its place in the output
//   two levels (larger sorts of 64-bit keys: three passes over them instead
//   of eight digits')
//     fs_split_*, fs_part1_*   as above, 256 buckets
//     fs_split2_*   one block per bucket samples it, in S1, for its children
//     fs_part2_*    every bucket's keys to its children's regions of S2
//     fs_child_*    one block per child, as fs_bucket_*
//     fs_rest_*     children larger than a block and buckets of an overflowed
//                   child, from a list, on a small grid
//   The digit passes run before these and sort keys of few varying digits
//   (FS_BK2_FEW_DIGITS); f64, 128M keys in place: 4,319 -> 2,227 us (part1 659,
//   part2 574, child 677, rest 156), u64 pairs, 16M: 830 -> 471 (146, 106, 149,
//   18).  The partitions move 1 GB of reads and 1 GB of scattered writes of
//   f64 128M at 3.3 and 3.7 TB/s (a copy here: 4.75), the children's blocks
//   are bound by their LDS passes.
//
// The block sort groups the keys by the top bits of their range and ranks each
// within its group by comparison; blocks with large groups (many copies of a
// key) fall back to stable passes over the bits of the range, 8 at a time,
// ranked by wave64 ballots.  With values each key carries its position in the
// block (16 bits) and the values follow by one gather at the end.
//
// Buckets are sized by the sample, so a bucket can outgrow its region or a
// block's LDS.  A region has room for the samples c that fell in its bucket,
// six standard deviations of them and FS_BK_ROOM more: with as many keys, a
// sample would show c or fewer of them below once in 10^9 (none at all: 10^7;
// c not counted but bounded, see split_body: 10^5).  Such a sort stays exact:
// the block of an oversized bucket sorts it alone through device memory
// (slow_sort); after an overflowed region every bucket's block gathers its keys
// from the caller's first (sort_overflowed; of two levels, fs_split2_*), and a
// bucket with an overflowed child is sorted from S1 by one block (fs_rest_*).

// Elements of the LDS block sort of WAVES waves: rows of 64 keys, `per` rows
// to each wave (wave w: rows w * per ...), so that a small segment still uses
// every wave.
template <bool K64, bool VALS, int BLOCK, int ITEMS, int GB = FS_BK_GBITS>
struct BlockSortLds {
    typedef typename KeyT<K64>::type K;
    static constexpr uint32_t CAP = BLOCK * ITEMS;
    static constexpr int WAVES = BLOCK / 64;
    alignas(16) K keys[CAP];
    uint16_t pos[VALS ? CAP : 1];                // with values: each key's position in the block
    // stable passes (not in the children's blocks, which leave those to fs_rest_*):
    // per-wave digit counts, then bases
    static constexpr bool LSD = GB == FS_BK_GBITS;
    alignas(16) uint16_t wcnt[LSD ? WAVES : 1][LSD ? FS_RADIX : 2];
    uint32_t dbase[LSD ? FS_RADIX : 1];
    uint16_t starts[(1u << GB) + 2u];   // group starts
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
template <bool K64, int GB = FS_BK_GBITS>
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
    // The group of any key of the input (not less `base`), also one outside the
    // range the map was made for.
    DEV uint32_t of_key(K u) const {
        if (by_value) return (*this)(u - base);
        const K t = u < base ? (K)0 : u - base;
        return (uint32_t)((t < span ? t : span) >> shift) & ((1u << GB) - 1u);
    }
    DEV uint32_t operator()(K k) const {
        if (!by_value) return (uint32_t)(k >> shift) & ((1u << GB) - 1u);
        K u = k + base;
        u = u > FINITE ? FINITE : u < ~FINITE ? ~FINITE : u;
        const double t = (value(u) - low) * scale;
        const double top = (double)((1u << GB) - 1u);
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
template <bool K64, bool VALS, int BLOCK, int ITEMS, int GB>
DEV bool group_sort(const typename KeyT<K64>::type (&k)[ITEMS], uint32_t len, const GroupMap<K64, GB>& map, uint32_t per,
                    BlockSortLds<K64, VALS, BLOCK, ITEMS, GB>& L) {
    typedef typename KeyT<K64>::type K;
    constexpr uint32_t CAP = BLOCK * ITEMS, NG = 1u << GB;
    constexpr uint32_t GPT = NG / BLOCK, GLIM = FS_BK_GLIM(K64, VALS);
    static_assert(NG % BLOCK == 0 && sizeof(L.keys) >= NG * 4u, "group counters in the keys' words");
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
template <bool K64, bool VALS, int BLOCK, int ITEMS, bool BITS, int GB>
DEV void block_fold(const typename KeyT<K64>::type (&k)[ITEMS], uint32_t len, uint32_t per,
                    BlockSortLds<K64, VALS, BLOCK, ITEMS, GB>& L, typename KeyT<K64>::type& r0,
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
template <bool K64, int GB = FS_BK_GBITS>
DEV GroupMap<K64, GB> group_map(typename KeyT<K64>::type least, typename KeyT<K64>::type most, bool by_value) {
    typedef typename KeyT<K64>::type K;
    typedef GroupMap<K64, GB> Map;
    const uint32_t bits = bit_length<K>(most - least);
    Map map{by_value, bits > GB ? bits - GB : 0u, least, (K)(most - least), 0.0, 0.0};
    if (by_value) {
        const K lo = least < (K)~Map::FINITE ? (K)~Map::FINITE : least > Map::FINITE ? Map::FINITE : least;
        const K hi = most > Map::FINITE ? Map::FINITE : most < (K)~Map::FINITE ? (K)~Map::FINITE : most;
        map.low = Map::value(lo);
        const double span = Map::value(hi) - map.low;
        map.scale = span > 0.0 ? (double)(1u << GB) / span : 0.0;
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

// The schedule words fs_last_pass_info and fs_last_bucket_info read: a digit
// counts as sorted when some key has a bit of it set that another has clear;
// overs: regions (second level: buckets with such a region) that overflowed.
template <bool K64>
DEV void bucket_pass_info(const FsArgs& a, uint64_t varying, uint32_t overs) {
    uint32_t mask = 0, p = 0;
    for (uint32_t j = 0; j < (K64 ? 8u : 4u); ++j)
        if ((varying >> (8u * j)) & 0xFFu) {
            mask |= 1u << j;
            ++p;
        }
    GLOBAL uint32_t* plan = gptr<uint32_t>(a.plan);
    st_agent(&plan[FS_PLAN_NPASSES], p);
    st_agent(&plan[FS_PLAN_MASK], mask | FS_MASK_BUCKETS);
    st_agent(&plan[FS_PLAN_RESCATTER], overs);
}

// The keys of one bucket (lo <= key, and key < hi unless it is the last), in
// order, from the len keys at src_k to dst_k, with their values (dst_v 0: none;
// src_v 0: their positions, argsort).  fwd: the source holds the caller's keys.
// ws: 2 * BLOCK / 64 words of LDS.  Every block reads the whole source, which
// bounds it: 3 TB/s of a grid of 256 (8 keys per thread in flight: a tenth
// faster).  With one region too small, us, against a sort without: u32, 1M keys
// 1,530 / 54; f64, two levels, 2M 1,260 / 170, 16M 10,100 / 380, 128M 91,800 / 2,120.
template <bool K64, int BLOCK>
DEV void gather_bucket(const FsArgs& a, uint64_t src_k, uint64_t src_v, bool fwd, uint32_t len, typename KeyT<K64>::type lo,
                       typename KeyT<K64>::type hi, bool last, uint64_t dst_k, uint64_t dst_v, uint32_t count, uint32_t* ws) {
    typedef typename KeyT<K64>::type K;
    constexpr int WAVES = BLOCK / 64, IT = 4;
    constexpr uint32_t CH = BLOCK * IT;
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6, wb = w * 64u * IT + lane;
    const uint32_t xf = fwd ? a.xform : FS_XF_NONE;
    const GLOBAL K* in = gptr<const K>(src_k);
    GLOBAL K* out = gptr<K>(dst_k);
    uint32_t done = 0, half = 0;                         // (the waves' counts alternate between two halves of ws)
    for (uint32_t c0 = 0; c0 < len; c0 += CH, half ^= 1u) {
        K k[IT];
        uint64_t in_bucket[IT];
        uint32_t mine = 0;
#pragma unroll
        for (int i = 0; i < IT; ++i) {
            const uint32_t p = c0 + wb + (uint32_t)i * 64u;
            k[i] = p < len ? xf_fwd<K64>(in[p], xf) : (K)0;
        }
#pragma unroll
        for (int i = 0; i < IT; ++i) {
            const bool is = c0 + wb + (uint32_t)i * 64u < len && k[i] >= lo && (last || k[i] < hi);
            in_bucket[i] = __builtin_amdgcn_uicmp((uint32_t)is, 0u, 33);
            mine += (uint32_t)__builtin_popcountll(in_bucket[i]);
        }
        if (lane == 0u) ws[half * WAVES + w] = mine;
        __syncthreads();
        uint32_t at = done;
#pragma unroll
        for (uint32_t ww = 0; ww < (uint32_t)WAVES; ++ww) {
            const uint32_t c = ws[half * WAVES + ww];
            at += ww < w ? c : 0u;
            done += c;
        }
#pragma unroll
        for (int i = 0; i < IT; ++i) {
            const uint32_t p = c0 + wb + (uint32_t)i * 64u, r = lanes_below(in_bucket[i], at);
            if (((in_bucket[i] >> lane) & 1u) && r < count) {
                out[r] = k[i];
                if (dst_v) gptr<uint32_t>(dst_v)[r] = src_v ? gptr<const uint32_t>(src_v)[p] : p;
            }
            at += (uint32_t)__builtin_popcountll(in_bucket[i]);
        }
    }
    __syncthreads();
}

// ---------------------------------------------------------------------------
// fs_split_*: the splitters
// ---------------------------------------------------------------------------

// L2 false: one block, the caller's keys (further blocks only clear look-back
// entries); L2 true: block p samples bucket p of the first level, in S1, for
// its children in S2, and writes the bucket's description (FS_BK2_*).
// What bounds it: one block's chain of loads, counts and scans (8,192 single
// keys of 1.5M: 23 us, of which the loads of as many cache lines are 6; taking
// neighbours together was that much faster, but runs of equal keys then made
// regions overflow).

// (two levels) whether the digit passes have done the sort
DEV bool digits_sort(const FsArgs& a) {
    return a.bk2_tab && ((const CONSTANT uint32_t*)(uintptr_t)a.bk2_tab)[FS_BK2_MODE] != 0u;
}

template <bool K64, int BLOCK, int ITEMS, bool L2>
DEV void split_body(const FsArgs& a) {
    typedef typename KeyT<K64>::type K;
    constexpr uint32_t CAP = BLOCK * ITEMS, NB = L2 ? FS_BK2_NB : FS_BK_NB;
    __shared__ BlockSortLds<K64, false, BLOCK, ITEMS> L;
    __shared__ K lbs[NB];
    __shared__ uint32_t s_par[4];
    static_assert(BLOCK >= FS_BK_NB && FS_BK_NB >= FS_BK2_NB, "a bucket per thread");
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    const uint32_t nb = 1u << (L2 ? a.bk2_lnb : a.bk_lnb), lm = L2 ? a.bk2_lm : a.bk_lm, m = 1u << lm;
    const uint32_t par = L2 ? blockIdx.x : 0u;
    if (nb > NB || m > CAP || m < nb || (L2 && gridDim.x != 1u << a.bk_lnb)) {
        if (tid == 0) report(a, FS_DEVERR_BAD_PLAN);
        return;
    }
    if (digits_sort(a)) return;                          // (uniform)
    GLOBAL uint32_t* tab1 = gptr<uint32_t>(a.bk_tab);
    GLOBAL uint32_t* tab2 = gptr<uint32_t>(a.bk2_tab);
    GLOBAL uint32_t* cnt = L2 ? tab2 + FS_BK2_CNT + par * NB : tab1 + FS_BK_CNT;
    GLOBAL uint32_t* bases = L2 ? tab2 + FS_BK2_BASE + par * NB : tab1 + FS_BK_BASE;
    GLOBAL uint32_t* caps = L2 ? tab2 + FS_BK2_CAPS + par * NB : tab1 + FS_BK_CAPS;
    GLOBAL K* glb = L2 ? reinterpret_cast<GLOBAL K*>(tab2 + FS_BK2_LB) + par * NB : reinterpret_cast<GLOBAL K*>(tab1 + FS_BK_LB);
    GLOBAL uint32_t* gmap = L2 ? tab2 + FS_BK2_MAP + par * FS_BK_MAP_WORDS : tab1 + FS_BK_MAP;
    uint32_t n = (uint32_t)a.n, origin = 0;              // keys sampled; first S2 key of the children's regions
    const GLOBAL K* src = gptr<const K>(a.keys);
    if constexpr (L2) {
        const uint32_t nb1 = 1u << a.bk_lnb;
        const uint32_t c = tid < nb1 ? tab1[FS_BK_CNT + tid] : 0u, t = (c + a.tile - 1u) / a.tile;
        const GLOBAL K* lb1 = reinterpret_cast<const GLOBAL K*>(tab1 + FS_BK_LB);
        // a bucket of one value has no children: its tiles copy it to its place
        const bool one = tid < nb1 && (tid + 1u < nb1 ? lb1[tid + 1u] - lb1[tid] == (K)1 : lb1[tid] == ~(K)0);
        if (tid == 0) L.flag = 0u;
        const uint32_t start = block_exclusive_scan<BLOCK>(c, L.wsum), tstart = block_exclusive_scan<BLOCK>(t, L.wsum);
        if (tid < nb1 && c > tab1[FS_BK_CAPS + tid]) atomicAdd(&L.flag, 1u);
        if (tid == par) {
            s_par[0] = c;
            s_par[1] = start;
            s_par[2] = tstart;
            s_par[3] = one ? 1u : 0u;
        }
        __syncthreads();
        n = s_par[0];
        origin = (uint32_t)(((uint64_t)s_par[1] * a.bk2_room) >> 8) + par * (32u * nb + 64u);
        origin = (origin + 15u) & ~15u;
        uint32_t rbase = tab1[FS_BK_BASE + par];
        const uint32_t ts = s_par[2], tn = (n + a.tile - 1u) / a.tile;
        if (L.flag) {
            // (uniform over the grid) a region overflowed: every block gathers
            // its bucket's keys from the caller's, which are still whole, to
            // their place in the output within S1
            if (tid == 0 && par == 0u) st_agent(&tab2[FS_BK2_OVER], L.flag);
            rbase = s_par[1];
            const bool last = par + 1u == nb1;
            gather_bucket<K64, BLOCK>(a, a.keys, a.op == FSK_OP_PAIRS ? a.vals : 0u, true, (uint32_t)a.n, lb1[par],
                                      last ? (K)0 : lb1[par + 1u], last, a.s1k + (uint64_t)rbase * sizeof(K),
                                      a.op != FSK_OP_KEYS ? a.s1v + (uint64_t)rbase * 4u : 0u, n,
                                      reinterpret_cast<uint32_t*>(&L.red[0][0]));
        }
        if (tid < FS_BK2_INFO_WORDS) {
            const uint32_t v = tid == 0u ? n : tid == 1u ? rbase : tid == 2u ? s_par[1] : tid == 3u ? ts : tid == 4u ? s_par[3] : 0u;
            tab2[FS_BK2_INFO + par * FS_BK2_INFO_WORDS + tid] = v;
        }
        GLOBAL uint32_t* tmap = gptr<uint32_t>(a.tilemap);
        for (uint32_t i = tid; i < tn; i += BLOCK)
            if (ts + i < a.tiles2) tmap[ts + i] = par;
        if (par + 1u == nb1)                             // (tiles the grid has to spare)
            for (uint32_t i = ts + tn + tid; i < a.tiles2; i += BLOCK) tmap[i] = 0xFFFFFFFFu;
        for (uint32_t i = tid; i < nb; i += BLOCK) st_agent(&cnt[i], 0u);
        if (a.op != FSK_OP_KEYS) {
            GLOBAL uint32_t* lb = gptr<uint32_t>(a.lookback0);
            for (uint32_t i = tid; i < tn * nb; i += BLOCK) lb[(uint64_t)ts * nb + i] = 0u;
            GLOBAL uint32_t* grp = lb + (uint64_t)a.tiles2 * nb + (uint64_t)(ts / FS_LB_GROUP + par) * nb;
            for (uint32_t i = tid; i < (tn + FS_LB_GROUP - 1u) / FS_LB_GROUP * nb; i += BLOCK) grp[i] = 0u;
        }
        if (n == 0u || s_par[3]) return;                 // (uniform)
        src = gptr<const K>(a.s1k) + rbase;
    } else {
        // counters of the partition and (values) its look-back entries start at zero
        if (a.op != FSK_OP_KEYS) {
            GLOBAL uint32_t* lb = gptr<uint32_t>(a.lookback0);
            const uint32_t words = (a.num_tiles + (a.num_tiles + FS_LB_GROUP - 1u) / FS_LB_GROUP) * nb;
            const uint32_t from = gridDim.x > 1u ? blockIdx.x - 1u : 0u, by = gridDim.x > 1u ? gridDim.x - 1u : 1u;
            if (gridDim.x == 1u || blockIdx.x)
                for (uint32_t i = from * BLOCK + tid; i < words; i += by * BLOCK) lb[i] = 0u;
        }
        if (blockIdx.x) return;                          // (uniform)
        for (uint32_t i = tid; i < nb; i += BLOCK) st_agent(&cnt[i], 0u);
        for (uint32_t i = tid; i < 4u * FS_BK_BIT_SLOTS; i += BLOCK) st_agent(&tab1[FS_BK_BITS + i], 0u);
        if (tid == 0) st_agent(&tab1[FS_BK_DONE], 0u);
        if (a.bk2_tab && tid < FS_BK2_INFO && tid != FS_BK2_MODE) st_agent(&tab2[tid], 0u);
    }

    // sample i: the key at a hashed position within the i-th of m equal parts
    // of the input.  (Single keys: neighbours often belong together, in runs of
    // one value or one file's records, and tell little more than one of them.)
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
            k[i] = src[sample_position(s, lm, n)];
            if (!L2) k[i] = xf_fwd<K64>(k[i], a.xform);
        }
    }

    const uint32_t stride = m / nb;
    // Region of a bucket: room for its share of the samples plus six standard
    // deviations, scaled to n.  budget: the keys that all of them can take.
    auto region_keys = [&](uint32_t c) -> uint32_t {
        const float room = (float)c + 6.0f * __builtin_sqrtf((float)c) + FS_BK_ROOM;
        const uint32_t keys = ((uint32_t)(room * ((float)n / (float)m)) + 16u) & ~15u;
        return keys > n ? (n + 15u) & ~15u : keys;
    };
    const uint32_t budget = L2 ? (uint32_t)(((uint64_t)n * a.bk2_room) >> 8) + 32u * nb : a.s1_keys;
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
    uint32_t share = 0;                                  // samples in this thread's bucket
    bool spread = count_groups<K64, false, BLOCK, ITEMS>(k, m, map, per, 2u * stride, L);   // (uniform)
    if (!spread && map.by_value) {
        map = group_map<K64>(least, most, false);
        spread = count_groups<K64, false, BLOCK, ITEMS>(k, m, map, per, 2u * stride, L);
    }
    if (spread) {
        for (uint32_t i = tid; i < NB; i += BLOCK) lbs[i] = i ? ~(K)0 : (K)0;
        uint32_t* const gi = reinterpret_cast<uint32_t*>(&L.wcnt[0][0]);   // each splitter's group
        static_assert(sizeof(L.wcnt) >= 4u * NB, "the splitters' groups, then the shares, in the stable passes' words");
        if (tid == 0) L.flag = 0u;
        __syncthreads();
        uint32_t g = 0;                                  // the group holding sample s0 (in order)
        if (tid >= 1u && tid < nb) {
            const uint32_t s0 = tid * stride;
#pragma unroll
            for (uint32_t step = 1u << (FS_BK_GBITS - 1); step; step >>= 1)
                if (L.starts[g + step] <= s0) g += step;
            const uint32_t g0 = L.starts[g], gn = L.starts[g + 1u] - g0;
            lbs[tid] = map.inside(g, gn ? (float)(s0 - g0) / (float)gn : 0.0f);
            gi[tid] = g;
        }
        __syncthreads();
        // A bucket's share of the samples: a quantile's where keys spread
        // within the splitters' groups, but up to all of both its splitters'
        // groups where those are of a value each.  A bucket for which that is
        // more than a quantile's room holds, but for once in 10^5, is given
        // all of it, and where the regions then take more than there is room
        // for the samples are counted instead.  (Counted always: u32, 1M keys,
        // 44.1 -> 45.8 us; wherever there was such a bucket: f64 pairs, normal,
        // 1M keys, 72.1 -> 75.2.)
        if (tid < nb) {
            const uint32_t to = tid + 1u < nb ? L.starts[gi[tid + 1u] + 1u] : m;
            share = to - L.starts[g];
            if ((float)share > (float)stride + 2.0f * __builtin_sqrtf((float)stride) + 4.0f) L.flag = 1u;
            else share = stride;
        }
        // The partition finds a key's bucket from its group: the splitters in
        // smaller groups, all below the key, then the few in its own.
        constexpr uint32_t TG = 1u << (FS_BK_GBITS - 1), TPT = (TG + BLOCK - 1) / BLOCK;
        uint32_t* tc = reinterpret_cast<uint32_t*>(L.keys);
        for (uint32_t i = tid; i < TG; i += BLOCK) tc[i] = 0u;
        __syncthreads();
        if (tid >= 1u && tid < nb) atomicAdd(&tc[map.of_key(lbs[tid]) >> 1], 1u);
        __syncthreads();
        uint32_t tsum = 0;
#pragma unroll
        for (uint32_t j = 0; j < TPT; ++j) tsum += tid * TPT + j < TG ? tc[tid * TPT + j] : 0u;
        uint32_t tx = block_exclusive_scan<BLOCK>(tsum, L.wsum);
        GLOBAL uint16_t* gt = reinterpret_cast<GLOBAL uint16_t*>(gmap + FS_BK_MAP_HEAD);
#pragma unroll
        for (uint32_t j = 0; j < TPT; ++j) {
            if (tid * TPT + j >= TG) continue;
            const uint32_t here = tc[tid * TPT + j];
            gt[tid * TPT + j] = (uint16_t)tx;
            tc[tid * TPT + j] = tx;
            tx += here;
        }
        bool count = L.flag != 0u;                       // (uniform)
        if (count) {
            const uint32_t c16 = tid < nb ? region_keys(share) >> 4 : 0u;
            const uint32_t before = block_exclusive_scan<BLOCK>(c16, L.wsum);
            if (tid == nb - 1u) s_par[0] = before + c16;
            __syncthreads();
            count = s_par[0] > budget >> 4;
        }
        if (count) {                                     // found as the partition finds its keys'
            uint32_t* const sc = reinterpret_cast<uint32_t*>(&L.wcnt[0][0]);
            for (uint32_t i = tid; i < NB; i += BLOCK) sc[i] = 0u;
            __syncthreads();
#pragma unroll
            for (int i = 0; i < ITEMS; ++i) {
                if ((uint32_t)i >= per || row0 + (uint32_t)i * 64u >= m) continue;
                const K key = k[i] + base;
                uint32_t b = tc[map.of_key(key) >> 1];
                while (b + 1u < nb && lbs[b + 1u] <= key) ++b;
                atomicAdd(&sc[b], 1u);
            }
            __syncthreads();
            if (tid < nb) share = sc[tid];
        }
        if (tid == 0) {
            const uint64_t w64[4] = {(uint64_t)map.base, (uint64_t)map.span, __builtin_bit_cast(uint64_t, map.low),
                                     __builtin_bit_cast(uint64_t, map.scale)};
            gmap[0] = 1u;
            gmap[1] = map.by_value ? 1u : 0u;
            gmap[2] = map.shift;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                gmap[4 + 2 * i] = (uint32_t)w64[i];
                gmap[5 + 2 * i] = (uint32_t)(w64[i] >> 32);
            }
        }
    } else {
        if (tid == 0) gmap[0] = 0u;
        // Keys crowded in parts of the range, or many copies of some: the
        // sample sorted, by groups where those hold copies of one key each,
        // else by stable passes.  64-bit keys take the top FS_BK_SAMPLE_BITS
        // bits of their range first.  Where two neighbours are then out of
        // order, the quantiles' top bits alone are the splitters (in order, and
        // below them exactly the samples of smaller top bits), unless two
        // quantiles share them: then the rest is sorted too.  (u64 argsort,
        // 995,000 keys, file and offset, most in few files: sorted twice, the
        // sample took 93 of 146 us.)
        K down = ~(K)0;                                  // the bits of a quantile that make a splitter
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
                const bool shared = tid >= 1u && tid < nb &&
                                    L.keys[tid * stride] >> lo == L.keys[(tid - 1u) * stride] >> lo;
                if (tid < 2u) s_par[tid] = 0u;
                __syncthreads();
                if (bad) s_par[0] = 1u;
                if (shared) s_par[1] = 1u;
                __syncthreads();
                const bool again = s_par[0] && s_par[1];
                if (s_par[0] && !again) down <<= lo;
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
            q = L.keys[tid * stride] & down;
            const bool rep = tid > 1u && q == (L.keys[(tid - 1u) * stride] & down);
            const bool dup = tid + 1u < nb && q == (L.keys[(tid + 1u) * stride] & down) && (K)(q + base) != ~(K)0;
            emit = rep ? 0u : dup ? 2u : 1u;
        }
        for (uint32_t i = tid; i < NB; i += BLOCK) lbs[i] = i ? ~(K)0 : (K)0;
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
            const uint32_t s0 = tid ? below(lbs[tid]) : 0u, s1 = tid + 1u < nb ? below(lbs[tid + 1u]) : m;
            share = s1 > s0 ? s1 - s0 : 0u;
        }
    }

    uint32_t cap = tid < nb ? region_keys(share) : 0u;
#ifdef FS_FAULT_INJECTION
    if (a.fault == (L2 ? FS_FAULT_SMALL_REGIONS2 : FS_FAULT_SMALL_REGIONS) && tid == 1u) cap = 16u;
#endif
    // (Should the regions not fit what the host sized for them, a bug, their
    // buckets overflow: the sort stays exact.)
    const uint32_t rbase = block_exclusive_scan<BLOCK>(cap, L.wsum);
    if (tid < nb) {
        const bool fits = rbase + cap <= budget;
        bases[tid] = fits ? origin + rbase : 0u;
        caps[tid] = fits ? cap : 0u;
        glb[tid] = lbs[tid];
    }
}

// ---------------------------------------------------------------------------
// fs_part_*: keys (and values) to their buckets' regions
// ---------------------------------------------------------------------------

// LEVEL 0: one level; 1, 2: the levels of two.  2: tiles of the first level's buckets, in S1, to their children's regions in
// S2; a tile of a bucket of one value goes to its place in the output.
template <bool K64, bool VALS, int BLOCK, int ITEMS, int LEVEL>
DEV void part_body(const FsArgs& a) {
    typedef typename KeyT<K64>::type K;
    constexpr bool L2 = LEVEL == 2;
    constexpr int WAVES = BLOCK / 64;
    constexpr uint32_t TILE = BLOCK * ITEMS;
    constexpr uint32_t NB = LEVEL ? FS_BK2_NB : FS_BK_NB;
    constexpr uint32_t DROP = 0xFFFFFFFFu;
    static_assert(BLOCK >= NB && TILE <= 0xFFFFu, "a bucket per thread, 16-bit tile positions");
    static_assert((uint64_t)FS_LB_GROUP * TILE < (1ull << FS_LB_GCOUNT_SHIFT), "group sums must fit their field");
    __shared__ union {
        K keys[TILE];
        uint32_t vals[TILE];
    } stage;
    __shared__ uint16_t bid[TILE];                     // bucket of every staged position
    __shared__ uint32_t table[VALS ? 1 : FS_BK_MAP_WORDS - FS_BK_MAP_HEAD];   // two pairs of groups to a word
    __shared__ uint16_t wcnt[VALS ? WAVES : 1][NB];    // values: per-wave bucket counts, then bases
    __shared__ K lbs[NB];
    __shared__ uint32_t cnt[NB];                       // the tile's bucket counts, then starts
    __shared__ uint32_t gbase[NB];
    __shared__ uint32_t wsum[WAVES];
    __shared__ uint32_t bits[4];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    const uint32_t nb = 1u << (L2 ? a.bk2_lnb : a.bk_lnb);
    const uint32_t rows = a.tile / BLOCK;               // keys per thread of this sort's tiles (at most ITEMS)
    if (blockIdx.x >= (L2 ? a.tiles2 : a.num_tiles) || nb > NB || rows > (uint32_t)ITEMS || rows == 0u) {
        if (tid == 0) report(a, FS_DEVERR_BAD_TILE);
        return;
    }
    if (LEVEL && digits_sort(a)) return;                 // (uniform)
    GLOBAL uint32_t* tab1 = gptr<uint32_t>(a.bk_tab);
    GLOBAL uint32_t* tab2 = gptr<uint32_t>(a.bk2_tab);
    uint32_t par = 0, tile = blockIdx.x, n32 = (uint32_t)a.n;   // the bucket, the tile of it, its keys
    uint64_t src_k = a.keys, src_v = a.vals;
    uint64_t lb_at = 0, grp_at = (uint64_t)a.num_tiles * nb;
    if constexpr (L2) {
        par = ((const CONSTANT uint32_t*)(uintptr_t)a.tilemap)[blockIdx.x];
        if (par >= 1u << a.bk_lnb) return;              // no tile for this block
        const CONSTANT uint32_t* info = (const CONSTANT uint32_t*)(uintptr_t)a.bk2_tab + FS_BK2_INFO + par * FS_BK2_INFO_WORDS;
        n32 = info[0];
        const uint32_t rbase = info[1], start = info[2], ts = info[3];
        tile = blockIdx.x - ts;
        if (tile * a.tile >= n32) return;
        src_k = a.s1k + (uint64_t)rbase * sizeof(K);
        src_v = a.s1v + (uint64_t)rbase * 4u;
        lb_at = (uint64_t)ts * nb;
        grp_at = (uint64_t)a.tiles2 * nb + (uint64_t)(ts / FS_LB_GROUP + par) * nb;
        if (info[4]) {                                   // one value
            const uint32_t t0 = tile * a.tile, t1 = min(t0 + a.tile, n32);
            K xa, xb;
            xf_inv_masks<K64>(a.xform, xa, xb);
            const K v = xf_inv_apply<K64>(reinterpret_cast<const GLOBAL K*>(tab1 + FS_BK_LB)[par], xa, xb);
            const GLOBAL uint32_t* sv = gptr<const uint32_t>(src_v);
            for (uint32_t i = t0 + tid; i < t1; i += BLOCK) {
                if (a.op != FSK_OP_ARGSORT) gptr<K>(a.keys)[start + i] = v;
                if (VALS) gptr<uint32_t>(a.vals)[start + i] = sv[i];
            }
            return;
        }
    }
    GLOBAL uint32_t* counts = L2 ? tab2 + FS_BK2_CNT + par * NB : tab1 + FS_BK_CNT;
    const GLOBAL uint32_t* bases = L2 ? tab2 + FS_BK2_BASE + par * NB : tab1 + FS_BK_BASE;
    const GLOBAL uint32_t* caps = L2 ? tab2 + FS_BK2_CAPS + par * NB : tab1 + FS_BK_CAPS;
    const GLOBAL K* glb = L2 ? reinterpret_cast<const GLOBAL K*>(tab2 + FS_BK2_LB) + par * NB
                             : reinterpret_cast<const GLOBAL K*>(tab1 + FS_BK_LB);
    const uint32_t tiles = L2 ? (n32 + a.tile - 1u) / a.tile : a.num_tiles;
    const uint32_t dst_keys = L2 ? a.s2_keys : a.s1_keys;
    const uint32_t begin = tile * a.tile, wbegin = begin + w * 64u * rows + lane;
    const uint32_t tv = n32 - begin < a.tile ? n32 - begin : a.tile;  // the tile's keys
    const GLOBAL K* src = gptr<const K>(src_k);
    auto valid = [&](int i) -> bool { return (uint32_t)i < rows && wbegin + (uint32_t)i * 64u < n32; };
    K k[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) k[i] = valid(i) ? src[wbegin + (uint32_t)i * 64u] : (K)0;
    for (uint32_t i = tid; i < NB; i += BLOCK) {
        lbs[i] = i < nb ? glb[i] : ~(K)0;
        cnt[i] = 0u;
    }
    const CONSTANT uint32_t* gmap = L2 ? (const CONSTANT uint32_t*)(uintptr_t)a.bk2_tab + FS_BK2_MAP + par * FS_BK_MAP_WORDS
                                       : (const CONSTANT uint32_t*)(uintptr_t)a.bk_tab + FS_BK_MAP;
    // (the stable partition waits on its look-back, not on the search: it
    // measured 4% faster without the table)
    const bool mapped = !VALS && gmap[0] != 0u;         // (uniform)
    if (mapped) {
        const GLOBAL uint32_t* gt = (L2 ? tab2 + FS_BK2_MAP + par * FS_BK_MAP_WORDS : tab1 + FS_BK_MAP) + FS_BK_MAP_HEAD;
        for (uint32_t i = tid; i < (uint32_t)(sizeof(table) / 4u); i += BLOCK) table[i] = gt[i];
    }
    const uint32_t my_cap = tid < nb ? caps[tid] : 0u, my_base = tid < nb ? bases[tid] : 0u;
    if (tid < 4u) bits[tid] = 0u;
    if (VALS)
        for (uint32_t i = tid; i < WAVES * NB / 2u; i += BLOCK) reinterpret_cast<uint32_t*>(&wcnt[0][0])[i] = 0u;
    __syncthreads();
    K on = 0, off = 0;
    uint32_t b[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        if (!L2) k[i] = xf_fwd<K64>(k[i], a.xform);
        if (!L2 && valid(i)) {
            on |= k[i];
            off |= ~k[i];
        }
        b[i] = 0u;
    }
    // bucket: the number of splitters at or below the key.  Where the sample
    // spread over its groups: those in smaller groups from the table, then the
    // few of the key's own (1.1 LDS reads a key more, where a binary search
    // takes 8 or 9); else by search (every item's search advances together:
    // the reads of a step are independent).
    if (mapped) {
        GroupMap<K64> map;
        map.by_value = gmap[1] != 0u;
        map.shift = gmap[2];
        uint64_t w64[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) w64[i] = ((uint64_t)gmap[5 + 2 * i] << 32) | gmap[4 + 2 * i];
        map.base = (K)w64[0];
        map.span = (K)w64[1];
        map.low = __builtin_bit_cast(double, w64[2]);
        map.scale = __builtin_bit_cast(double, w64[3]);
        const uint16_t* tb = reinterpret_cast<const uint16_t*>(table);
#pragma unroll
        for (int g = 0; g < ITEMS; g += 4) {
            if ((uint32_t)g >= rows) continue;
#pragma unroll
            for (int i = g; i < g + 4 && i < ITEMS; ++i) b[i] = tb[map.of_key(k[i]) >> 1];
#pragma unroll
            for (int i = g; i < g + 4 && i < ITEMS; ++i)
                while (b[i] + 1u < nb && lbs[b[i] + 1u] <= k[i]) ++b[i];
        }
    } else {
        for (uint32_t step = nb >> 1; step; step >>= 1) {
#pragma unroll
            for (int g = 0; g < ITEMS; g += 4) {
                if ((uint32_t)g >= rows) continue;
#pragma unroll
                for (int i = g; i < g + 4 && i < ITEMS; ++i) b[i] += lbs[b[i] + step] <= k[i] ? step : 0u;
            }
        }
    }
    // the tile's bits to one of several slots (every tile on one word would
    // queue there)
    if constexpr (!L2) {
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
    if (!L2 && tid < 4u && bits[tid])
        __hip_atomic_fetch_or(&tab1[FS_BK_BITS + 4u * (tile % FS_BK_BIT_SLOTS) + tid], bits[tid], __ATOMIC_RELAXED,
                              __HIP_MEMORY_SCOPE_AGENT);
    GLOBAL uint32_t* lb = gptr<uint32_t>(a.lookback0) + lb_at;
    GLOBAL uint32_t* grp = gptr<uint32_t>(a.lookback0) + grp_at;
    const uint32_t count = tid < nb ? cnt[tid] : 0u;
    if (VALS && tid < nb) {
        LbEntry<false>::store(lb, (uint64_t)tile * nb + tid, tile == 0u ? FS_LB_INC : FS_LB_AGG, count);
        __hip_atomic_fetch_add(&grp[(uint64_t)(tile / FS_LB_GROUP) * nb + tid], (1u << FS_LB_GCOUNT_SHIFT) | count,
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    const uint32_t ex = block_exclusive_scan<BLOCK>(count, wsum);
    if (tid < nb) {
        uint32_t at = 0;
        if (VALS) {
            uint32_t r0 = 0, r1 = 0, r2 = 0;
            at = tile == 0u ? 0u : lookback<false>(lb, grp, tile, tid, count, a.status, r0, r1, r2, nb);
            if (tile + 1u == tiles) st_agent(&counts[tid], at + count);
        } else if (count) {
            at = __hip_atomic_fetch_add(&counts[tid], count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        // (a run that does not fit is dropped: the bucket launch sees the count)
        gbase[tid] = (at <= my_cap && count <= my_cap - at) ? my_base + at - ex : DROP;
        cnt[tid] = ex;
    }
    if (VALS) rank_wave<true, ITEMS, LEVEL ? FS_BK2_LNB : FS_BK_LNB>(b, 0u, wcnt[w], rank, rows);
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
    GLOBAL K* dst = gptr<K>(L2 ? a.s2k : a.s1k);
    uint32_t gp[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const uint32_t p = (uint32_t)i * BLOCK + tid;
        gp[i] = DROP;
        if (p < tv) {
            const uint32_t g = gbase[bid[p] & (NB - 1u)];
            if (g != DROP && g + p < dst_keys) {
                gp[i] = g + p;
                dst[g + p] = stage.keys[p];
            }
        }
    }
    if (VALS) {
        uint32_t v[ITEMS];
        const GLOBAL uint32_t* sv = gptr<const uint32_t>(src_v);
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            const uint32_t p = wbegin + (uint32_t)i * 64u;
            v[i] = !L2 && a.op == FSK_OP_ARGSORT ? p : valid(i) ? sv[p] : 0u;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < ITEMS; ++i)
            if (valid(i)) stage.vals[pos.get(i)] = v[i];
        __syncthreads();
        GLOBAL uint32_t* dv = gptr<uint32_t>(L2 ? a.s2v : a.s1v);
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

// One block sorts len keys (at most its LDS's) at src_k, with their values at
// src_v (0: their positions, argsort), into dst_k (not of an argsort) and
// dst_v, as the caller's keys.  whole: the source is the caller's (transformed
// on load).
template <bool K64, bool VALS, int BLOCK, int ITEMS>
DEV void block_range_sort(const FsArgs& a, uint64_t src_k, uint64_t src_v, bool whole, uint32_t len, uint64_t dst_k,
                          uint64_t dst_v, BlockSortLds<K64, VALS, BLOCK, ITEMS>& L) {
    typedef typename KeyT<K64>::type K;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    const bool put_keys = a.op != FSK_OP_ARGSORT;
    K xa, xb;
    xf_inv_masks<K64>(a.xform, xa, xb);
    GLOBAL K* dk = gptr<K>(dst_k);
    GLOBAL uint32_t* dv = gptr<uint32_t>(dst_v);
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
        if (tid == 0) bucket_pass_info<K64>(a, (uint64_t)(on & off), 0u);
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
        if (src_v == dst_v) __syncthreads();            // (uniform) in place: every value read before any is written
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            const uint32_t x = (uint32_t)i * BLOCK + tid;
            if (x < len) dv[x] = v[i];
        }
    }
    if (put_keys) {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            const uint32_t x = (uint32_t)i * BLOCK + tid;
            if (x < len) dk[x] = xf_inv_apply<K64>((K)(L.keys[x] + base), xa, xb);
        }
    }
}

// A sort of which some region overflowed, its keys incomplete in S1: every
// bucket's block gathers its keys from the caller's into S2, at their place in
// the output, and sorts them there; the block that ends last copies S2 back
// (the others may still read the caller's keys before).  start, len: the
// block's bucket by the partition's counts, which are whole.
template <bool K64, bool VALS, int BLOCK, int ITEMS>
DEV void sort_overflowed(const FsArgs& a, uint32_t start, uint32_t len, BlockSortLds<K64, VALS, BLOCK, ITEMS>& L) {
    typedef typename KeyT<K64>::type K;
    __shared__ uint32_t s_last;
    const uint32_t tid = threadIdx.x, nb = 1u << a.bk_lnb, j = blockIdx.x, n = (uint32_t)a.n;
    const bool put_keys = a.op != FSK_OP_ARGSORT, last = j + 1u == nb;
    GLOBAL uint32_t* tab = gptr<uint32_t>(a.bk_tab);
    const GLOBAL K* lbs = reinterpret_cast<const GLOBAL K*>(tab + FS_BK_LB);
    const K lo = lbs[j], hi = last ? (K)0 : lbs[j + 1u];
    const uint64_t k1 = a.s1k + (uint64_t)start * sizeof(K), v1 = a.s1v + (uint64_t)start * 4u;
    const uint64_t k2 = a.s2k + (uint64_t)start * sizeof(K), v2 = a.s2v + (uint64_t)start * 4u;
    K xa, xb;
    xf_inv_masks<K64>(a.xform, xa, xb);
    if (len) {                                           // (uniform, as every branch here)
        gather_bucket<K64, BLOCK>(a, a.keys, a.op == FSK_OP_PAIRS ? a.vals : 0u, true, n, lo, hi, last, k2, VALS ? v2 : 0u,
                                  len, reinterpret_cast<uint32_t*>(&L.red[0][0]));
        if (last ? lo == ~(K)0 : hi - lo == (K)1) {      // one value: in order as it is
            const K v = xf_inv_apply<K64>(lo, xa, xb);
            for (uint32_t p = tid; p < len; p += BLOCK) gptr<K>(k2)[p] = v;
        } else {
            // (also a bucket that LDS holds: the block sort, twice in the
            // kernel, took registers from every other sort: u64 argsort 100,003
            // keys 64.4 -> 65.9 us; here it saved 110 us of 1,530)
            slow_sort<K64, VALS, BLOCK, ITEMS>(a, k2, v2, false, k1, v1, k2, v2, k2, v2, len, L);
        }
    }
    __threadfence();                                     // the bucket in S2, before it is counted as done
    __syncthreads();
    if (tid == 0)
        s_last = __hip_atomic_fetch_add(&tab[FS_BK_DONE], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == nb - 1u;
    __syncthreads();
    if (!s_last) return;                                 // (uniform)
    __threadfence();
    if (put_keys)
        for (uint32_t p = tid; p < n; p += BLOCK) gptr<K>(a.keys)[p] = gptr<const K>(a.s2k)[p];
    if (VALS)
        for (uint32_t p = tid; p < n; p += BLOCK) gptr<uint32_t>(a.vals)[p] = gptr<const uint32_t>(a.s2v)[p];
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
    const uint32_t tid = threadIdx.x;
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
            if (c > cap) atomicAdd(&s_over, 1u);
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
            bucket_pass_info<K64>(a, ((uint64_t)(b[1] & b[3]) << 32) | (b[0] & b[2]), s_over);
        }
        if (s_over) {                                   // (uniform) a region overflowed
            __syncthreads();
            sort_overflowed<K64, VALS, BLOCK, ITEMS>(a, start, len, L);
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

    block_range_sort<K64, VALS, BLOCK, ITEMS>(a, src_k, src_v, whole, len, a.keys + (uint64_t)start * sizeof(K),
                                              a.vals + (uint64_t)start * 4u, L);
}

// ---------------------------------------------------------------------------
// fs_child_*, fs_rest_*: two levels of buckets
// ---------------------------------------------------------------------------

// Work for fs_rest_*: the two words of an entry.
DEV void push_rest(const FsArgs& a, uint32_t id, uint32_t what) {
    GLOBAL uint32_t* tab2 = gptr<uint32_t>(a.bk2_tab);
    const uint32_t at = __hip_atomic_fetch_add(&tab2[FS_BK2_RESTS], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (at < a.rest_cap) {
        GLOBAL uint32_t* e = gptr<uint32_t>(a.rest) + 2u * (uint64_t)at;
        e[0] = id;
        e[1] = what;
    } else {
        report(a, FS_DEVERR_BAD_PLAN);                   // (the host sized the list for every entry there can be)
    }
}

// The place of child `id`: its region in S2 and its keys' place in the output.
// false when there is nothing to do.  over: some child of its bucket outgrew
// its region (the bucket is then sorted from S1 instead).
struct ChildPlace {
    uint32_t start, len, base;
    bool over, one;
};
template <bool K64, int BLOCK>
DEV bool child_place(const FsArgs& a, uint32_t id, uint32_t* wsum, uint32_t* s_seg, ChildPlace& c) {
    typedef typename KeyT<K64>::type K;
    static_assert(BLOCK >= FS_BK2_NB, "a child per thread");
    const uint32_t tid = threadIdx.x, nb = 1u << a.bk2_lnb;
    const uint32_t par = id >> a.bk2_lnb, j = id & (nb - 1u);
    const CONSTANT uint32_t* tab2 = (const CONSTANT uint32_t*)(uintptr_t)a.bk2_tab;
    const CONSTANT uint32_t* info = tab2 + FS_BK2_INFO + par * FS_BK2_INFO_WORDS;
    if (info[0] == 0u || info[4]) return false;          // (uniform)
    const GLOBAL uint32_t* t = gptr<const uint32_t>(a.bk2_tab);
    const uint32_t n = tid < nb ? t[FS_BK2_CNT + par * FS_BK2_NB + tid] : 0u;
    const uint32_t cap = tid < nb ? t[FS_BK2_CAPS + par * FS_BK2_NB + tid] : 0u;
    if (tid == 0) s_seg[2] = 0u;
    const uint32_t ex = block_exclusive_scan<BLOCK>(n, wsum);
    if (n > cap) s_seg[2] = 1u;
    if (tid == j) {
        s_seg[0] = ex;
        s_seg[1] = n;
    }
    __syncthreads();
    const GLOBAL K* lb = reinterpret_cast<const GLOBAL K*>(t + FS_BK2_LB) + par * FS_BK2_NB;
    c.start = info[2] + s_seg[0];
    c.len = s_seg[1];
    c.base = tab2[FS_BK2_BASE + par * FS_BK2_NB + j];
    c.over = s_seg[2] != 0u;
    c.one = j + 1u < nb ? lb[j + 1u] - lb[j] == (K)1 && j != 0u : lb[j] == ~(K)0;
    return true;
}

// First launch: a small block per child (many to a CU) sorts it where the
// groups spread it; copies of one value are copied; the others (larger than
// the block, crowded) go to the rest list.
template <bool K64, bool VALS, int BLOCK, int ITEMS, int GB>
DEV void child_body(const FsArgs& a) {
    typedef typename KeyT<K64>::type K;
    constexpr uint32_t CAP = BLOCK * ITEMS;
    __shared__ BlockSortLds<K64, VALS, BLOCK, ITEMS, GB> L;
    __shared__ uint32_t s_seg[3];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    const uint32_t id = tile_of_block(blockIdx.x, gridDim.x);
    if (gridDim.x != 1u << (a.bk_lnb + a.bk2_lnb)) {
        if (tid == 0) report(a, FS_DEVERR_BAD_PLAN);
        return;
    }
    // The keys' region and their number are known at once; their loads are in
    // flight while the scan finds their place in the output.
    const CONSTANT uint32_t* ctab = (const CONSTANT uint32_t*)(uintptr_t)a.bk2_tab;
    const uint32_t child = (id >> a.bk2_lnb) * FS_BK2_NB + (id & ((1u << a.bk2_lnb) - 1u));
    const CONSTANT uint32_t* cinfo = ctab + FS_BK2_INFO + (id >> a.bk2_lnb) * FS_BK2_INFO_WORDS;
    if (ctab[FS_BK2_MODE] || cinfo[0] == 0u || cinfo[4]) return;   // (uniform)
    const uint32_t len0 = ctab[FS_BK2_CNT + child] <= CAP ? ctab[FS_BK2_CNT + child] : 0u;
    const uint32_t per = (len0 + BLOCK - 1u) / BLOCK, row0 = w * per * 64u + lane;
    const GLOBAL K* src = gptr<const K>(a.s2k) + ctab[FS_BK2_BASE + child];
    K k[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const uint32_t x = row0 + (uint32_t)i * 64u;
        k[i] = (uint32_t)i < per && x < len0 ? src[x] : ~(K)0;
    }
    ChildPlace c;
    if (!child_place<K64, BLOCK>(a, id, L.wsum, s_seg, c)) return;
    if (c.over) {                                        // (uniform)
        if (tid == 0 && (id & ((1u << a.bk2_lnb) - 1u)) == 0u) {
            __hip_atomic_fetch_add(gptr<uint32_t>(a.bk2_tab) + FS_BK2_OVERS, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            push_rest(a, id, FS_REST_BUCKET);
        }
        return;
    }
    if (c.len == 0u) return;
    if (c.len > CAP) {
        // copies of one value a few thousand at a time, anything else whole
        const uint32_t parts = c.one ? (c.len + FS_REST_KEYS - 1u) / FS_REST_KEYS : 1u;
        for (uint32_t i = tid; i < parts; i += BLOCK) push_rest(a, id, c.one ? i : FS_REST_SORT);
        return;
    }
    K least = 0, most = 0;
    block_fold<K64, VALS, BLOCK, ITEMS, false, GB>(k, c.len, per, L, least, most);
    const uint32_t bits = bit_length<K>(most - least);
    if (bits == 0u) {                                    // (uniform) one value: in order as it is
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            const uint32_t x = row0 + (uint32_t)i * 64u;
            if ((uint32_t)i >= per || x >= c.len) continue;
            L.keys[x] = 0;
            if constexpr (VALS) L.pos[x] = (uint16_t)x;
        }
        __syncthreads();
    } else {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i)
            if ((uint32_t)i < per && row0 + (uint32_t)i * 64u < c.len) k[i] -= least;
        if (!group_sort<K64, VALS, BLOCK, ITEMS, GB>(k, c.len, group_map<K64, GB>(least, most, false), per, L)) {
            if (tid == 0) push_rest(a, id, FS_REST_SORT);
            return;
        }
    }
    const GLOBAL uint32_t* sv = gptr<const uint32_t>(a.s2v) + c.base;
    K xa, xb;
    xf_inv_masks<K64>(a.xform, xa, xb);
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const uint32_t x = (uint32_t)i * BLOCK + tid;
        if (x >= c.len) continue;
        if constexpr (VALS) gptr<uint32_t>(a.vals)[c.start + x] = sv[L.pos[x]];
        if (!VALS || a.op != FSK_OP_ARGSORT) gptr<K>(a.keys)[c.start + x] = xf_inv_apply<K64>((K)(L.keys[x] + least), xa, xb);
    }
}

// Second launch: a small grid takes the rest list in turn: children on the
// one-level path's block sort (or through device memory when that is too
// small), pieces of a child of one value, whole buckets whose children
// outgrew their regions.
template <bool K64, bool VALS, int BLOCK, int ITEMS>
DEV void rest_body(const FsArgs& a) {
    typedef typename KeyT<K64>::type K;
    __shared__ BlockSortLds<K64, VALS, BLOCK, ITEMS> L;
    __shared__ uint32_t s_seg[3];
    const uint32_t tid = threadIdx.x;
    const CONSTANT uint32_t* tab1 = (const CONSTANT uint32_t*)(uintptr_t)a.bk_tab;
    const CONSTANT uint32_t* tab2 = (const CONSTANT uint32_t*)(uintptr_t)a.bk2_tab;
    if (tab2[FS_BK2_MODE]) return;                       // (uniform)
    if (blockIdx.x == 0 && tid == 0) {
        uint32_t b[4] = {0u, 0u, 0u, 0u};
#pragma unroll
        for (uint32_t i = 0; i < 4u * FS_BK_BIT_SLOTS; ++i) b[i % 4u] |= tab1[FS_BK_BITS + i];
        bucket_pass_info<K64>(a, ((uint64_t)(b[1] & b[3]) << 32) | (b[0] & b[2]), tab2[FS_BK2_OVER] + tab2[FS_BK2_OVERS]);
    }
    const uint32_t count = min(tab2[FS_BK2_RESTS], a.rest_cap);
    for (uint32_t e = blockIdx.x; e < count; e += gridDim.x) {
        const CONSTANT uint32_t* ent = (const CONSTANT uint32_t*)(uintptr_t)a.rest + 2u * (uint64_t)e;
        const uint32_t id = ent[0], what = ent[1];
        const uint32_t par = id >> a.bk2_lnb, nb = 1u << a.bk2_lnb;
        if (par >= 1u << a.bk_lnb) return;
        const CONSTANT uint32_t* info = tab2 + FS_BK2_INFO + par * FS_BK2_INFO_WORDS;
        ChildPlace c{0u, 0u, 0u, false, false};
        const bool bucket = what == FS_REST_BUCKET;      // (uniform, as every branch here)
        if (bucket || child_place<K64, BLOCK>(a, id, L.wsum, s_seg, c)) {
            __syncthreads();                             // (s_seg read by every thread)
            // a bucket from its region in S1 through its children's in S2; a
            // child the other way round (its bucket's keys in S1 are dead)
            const uint64_t in2 = bucket ? ((((uint64_t)info[2] * a.bk2_room) >> 8) + par * (32u * nb + 64u) + 15u) & ~15ull
                                        : (uint64_t)c.base;
            const uint64_t in1 = bucket ? (uint64_t)info[1] : (uint64_t)info[1] + (c.start - info[2]);
            const uint32_t start = bucket ? info[2] : c.start, len = bucket ? info[0] : c.len;
            const uint64_t k1 = a.s1k + in1 * sizeof(K), v1 = a.s1v + in1 * 4u;
            const uint64_t k2 = a.s2k + in2 * sizeof(K), v2 = a.s2v + in2 * 4u;
            const uint64_t sk = bucket ? k1 : k2, sv = bucket ? v1 : v2;
            if (bucket || what == FS_REST_SORT) {
                if (!bucket && len <= (uint32_t)(BLOCK * ITEMS))
                    block_range_sort<K64, VALS, BLOCK, ITEMS>(a, sk, VALS ? sv : 0u, false, len, a.keys + (uint64_t)start * sizeof(K),
                                                              a.vals + (uint64_t)start * 4u, L);
                else
                    slow_sort<K64, VALS, BLOCK, ITEMS>(a, sk, sv, false, bucket ? k2 : k1, bucket ? v2 : v1, sk, sv,
                                                       a.keys + (uint64_t)start * sizeof(K),
                                                       a.vals + (uint64_t)start * 4u, len, L);
            } else {
                const uint32_t p0 = what * FS_REST_KEYS, p1 = min(p0 + FS_REST_KEYS, c.len);
                K xa, xb;
                xf_inv_masks<K64>(a.xform, xa, xb);
                const K v = xf_inv_apply<K64>(gptr<const K>(sk)[0], xa, xb);
                for (uint32_t p = p0 + tid; p < p1; p += BLOCK) {
                    if (a.op != FSK_OP_ARGSORT) gptr<K>(a.keys)[c.start + p] = v;
                    if (VALS) gptr<uint32_t>(a.vals)[c.start + p] = gptr<const uint32_t>(sv)[p];
                }
            }
        }
        __syncthreads();                                // the entry's LDS is the next one's
    }
}

// Blocks per CU by LDS: the bucket kernels' registers leave room for them.
#define FS_BK_KERNELS(sfx, K64, VALS, PITEMS, BITEMS, WAVES)                                                      \
    extern "C" __global__ void __launch_bounds__(FS_BP_BLOCK) fs_part_##sfx(FsArgs a) {                           \
        part_body<K64, VALS, FS_BP_BLOCK, PITEMS, 0>(a);                                                          \
    }                                                                                                             \
    extern "C" __global__ void __launch_bounds__(FS_BK_BLOCK) FS_OCC(WAVES) fs_bucket_##sfx(FsArgs a) {           \
        bucket_body<K64, VALS, FS_BK_BLOCK, BITEMS>(a);                                                           \
    }
FS_BK_KERNELS(k32, false, false, FS_BP32_ITEMS, FS_BK32_ITEMS, FS_BK32_WAVES)
FS_BK_KERNELS(k32_v, false, true, FS_BP32_ITEMS, FS_BK32V_ITEMS, FS_BK32V_WAVES)
FS_BK_KERNELS(k64, true, false, FS_BP64_ITEMS, FS_BK64_ITEMS, FS_BK64_WAVES)
FS_BK_KERNELS(k64_v, true, true, FS_BP64_ITEMS, FS_BK64V_ITEMS, FS_BK64V_WAVES)

// Two levels.  The partition of the first has at most 256 buckets and larger
// tiles than one level's, so that a tile's runs of a bucket are long (f64
// 128M keys: 885 -> 659 us against 512 buckets of 5,120-key tiles).
#define FS_BK2_KERNELS(sfx, VALS, PITEMS, BITEMS, CITEMS, CWAVES, CGBITS)                                         \
    extern "C" __global__ void __launch_bounds__(FS_BP_BLOCK) fs_part1_##sfx(FsArgs a) {                          \
        part_body<true, VALS, FS_BP_BLOCK, PITEMS, 1>(a);                                                         \
    }                                                                                                             \
    extern "C" __global__ void __launch_bounds__(FS_BP_BLOCK) fs_part2_##sfx(FsArgs a) {                          \
        part_body<true, VALS, FS_BP_BLOCK, PITEMS, 2>(a);                                                         \
    }                                                                                                             \
    extern "C" __global__ void __launch_bounds__(FS_BC_BLOCK) FS_OCC(CWAVES) fs_child_##sfx(FsArgs a) {           \
        child_body<true, VALS, FS_BC_BLOCK, CITEMS, CGBITS>(a);                                                   \
    }                                                                                                             \
    extern "C" __global__ void __launch_bounds__(FS_BK_BLOCK) FS_OCC(2) fs_rest_##sfx(FsArgs a) {                 \
        rest_body<true, VALS, FS_BK_BLOCK, BITEMS>(a);                                                            \
    }
FS_BK2_KERNELS(k64, false, FS_BP2_64_ITEMS, FS_BK64_ITEMS, FS_BC64_ITEMS, FS_BC64_WAVES, FS_BC_GBITS)
FS_BK2_KERNELS(k64_v, true, FS_BP2_64V_ITEMS, FS_BK64V_ITEMS, FS_BC64V_ITEMS, FS_BC64V_WAVES, FS_BCV_GBITS)

extern "C" __global__ void __launch_bounds__(FS_BS_BLOCK) fs_split_k32(FsArgs a) {
    split_body<false, FS_BS_BLOCK, FS_BS_ITEMS, false>(a);
}
extern "C" __global__ void __launch_bounds__(FS_BS_BLOCK) fs_split_k64(FsArgs a) {
    split_body<true, FS_BS_BLOCK, FS_BS_ITEMS, false>(a);
}
extern "C" __global__ void __launch_bounds__(FS_BS_BLOCK) fs_split2_k64(FsArgs a) {
    split_body<true, FS_BS_BLOCK, FS_BS2_ITEMS, true>(a);
}
