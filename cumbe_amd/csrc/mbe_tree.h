// The pruned search of the default tree (included by mbe_kernel.hip).
//
// A level LEVEL(L, P, X, Q) holds the candidates to branch on (P), those that
// only take part in expansion (X, handed to another worker) and those already
// handled (Q). A candidate v of P whose row within L lies inside a Q row, or
// inside the row of a vertex already processed at this level, can never give
// a maximal biclique, neither at this level nor below a later sibling (every
// L' that holds v in R lies inside v's row, which the other vertex covers).
// Such a v leaves P and X and does not enter Q. The twins that iMBEA removes
// (Zhang et al., BMC Bioinformatics 2014) are the case of equal rows. What is
// left of the tree has one node per maximal biclique.
//
// With these rules a level is small: the problems of the benchmark workload
// average 4 candidates in P and 7 in Q. So the search runs on two tiers:
//
//  * wide: any size, one bit mask per set over the problem's candidates, rows
//    in LDS or the arena by word (rows[w][k]: 64 candidates are one coalesced
//    access). It descends until the child fits the tile.
//  * tile: at most 64 candidates in P and X, one per lane; at most 128 in Q,
//    two per lane; L of at most 8 words. All rows are in VGPRs, all sets are
//    64-bit scalars, and a node reads no memory: x is a scalar bit scan, L' a
//    lane read, and the check, absorption, P' and pruning are lane-parallel
//    compares whose ballots are the new sets. Frames are pushed on a descent
//    only, into registers too: frame f is lane f of the stack's registers.

constexpr uint32_t kTileP = 64;       // P and X candidates of a tile (lanes)
constexpr uint32_t kTileQ = 128;      // Q candidates of a tile (two per lane)
constexpr uint32_t kTileW = 8;        // words of L in a tile
constexpr uint32_t kTreeList = 0;     // LDS header: u32[192] gathered candidates
constexpr uint32_t kTreeHdr = 96;     // LDS words of the header
static_assert(kTreeHdr <= kLdsSec, "the section counters lie behind the header");

// Narrowing: below a vertex whose L' has at most 64 bits, a tile of more
// words goes on as a tile of one word over the bits of L', when P' holds at
// least kNarrowP candidates (gathering the bits takes about two microseconds).
// The narrow problem's memory: hash terms of the 64 bits and of the lanes,
// the lanes' rows and the Q rows, its own list.
constexpr uint32_t kNarrowP = 4;
constexpr uint32_t kNarrowWords = 64 + 64 + kTileP + kTileQ + (kTileP + kTileQ) / 2;

// frame words of a tile of W words: L, P, X, D, R hash sum, |R| and x. Frame
// f of a suspended tile is word f of each of these blocks of 64. Every descent
// takes at least x from the at most 64 candidates of P and X together, and a
// level is pushed only while it or its child has some in P, so 64 frames are
// enough.
__device__ __forceinline__ constexpr uint32_t tile_fw(uint32_t W) { return W + 5; }
__device__ __forceinline__ constexpr uint32_t save_words(uint32_t W) { return 64 * tile_fw(W); }
static_assert(save_words(1) + save_words(kTileW) + kNarrowWords == 1632 && kTileQ == 2 * 64,
              "see tree_wide_words");
// the tile classes: 1, 2, 4 or 8 words
__device__ __forceinline__ uint32_t tile_class(uint32_t W) {
    return W <= 1 ? 1 : W <= 2 ? 2 : W <= 4 ? 4 : 8;
}

// This wave's lane numbers, as a function's own: `const Here lane;` hides
// lane() in it. The compiler takes them as new at that point, so it computes
// addresses and masks from them there and not before the kernel's loop, where
// they would fill the registers of every tile search (384 VGPRs with them, 252
// without, and so one wave per SIMD instead of two).
struct Here {
    uint32_t v = lane();
    __device__ __forceinline__ Here() {
#ifdef __HIP_DEVICE_COMPILE__
        asm volatile("" : "+v"(v));
#endif
    }
    __device__ __forceinline__ uint32_t operator()() const { return v; }
};

__device__ __forceinline__ uint32_t wrlane32(uint32_t old, uint32_t v, uint32_t l) {
    return lane() == l ? v : old;
}
__device__ __forceinline__ u64 wrlane64(u64 old, u64 v, uint32_t l) { return lane() == l ? v : old; }
__device__ __forceinline__ uint32_t uni32(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ bool uni1(bool v) { return uni32(v) != 0; }
__device__ __forceinline__ u64 low_bits(uint32_t n) { return n >= 64 ? ~0ull : (1ull << n) - 1; }

// Relaxed device-scope accesses: words of another worker's slot and of the
// control block. They bypass the caches, so waiting for them orders them and
// no cache is ever written back or invalidated.
__device__ __forceinline__ void wait_mem() {
    wsync();
    __builtin_amdgcn_s_waitcnt(0);
    wsync();
}
// After a wave's own atomics on its own memory: they are complete and its
// later loads see them (same compute unit, so a workgroup-scope order; a
// device-scope acquire would invalidate the caches under every other worker).
__device__ __forceinline__ void sync_own() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    __builtin_amdgcn_s_waitcnt(0);
    wsync();
}
__device__ __forceinline__ void own_or(u64* p, u64 v) {
    __hip_atomic_fetch_or(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ uint32_t own_add(uint32_t* p, uint32_t v) {
    return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// What one worker carries through its tasks.
struct Walk {
    u64 cnt;         // bicliques of the task
    u64 hs;          // their hash: a sum per lane, reduced at the task's end
    u64 nodes, donated, words;
    u64 steps;       // vertices taken (the watchdog's and the donation's clock)
    u64 next_event;  // steps at which donation and the watchdog are looked at
    u64 charged;     // nodes charged against the node budget; without one, the
                     // steps at the last look at the abort flag
    u64 idle;        // lane i: idle workers of the i-th map word looked at
    uint32_t look;   // the first map word looked at
    uint32_t g, give;  // give: levels to give away at this event
    bool r_is_u, stop;
};

constexpr uint32_t kWatchSteps = 1024;  // some 100 us
__device__ __forceinline__ uint32_t give_interval(const KParams& kp) {
    return kp.donate_interval ? kp.donate_interval : 64;
}
// Steps between two events: the donation interval, but under a watchdog no
// more than kWatchSteps, and less under a node budget so that a small budget
// is seen in time.
__device__ __forceinline__ uint32_t event_interval(const KParams& kp) {
    return min(give_interval(kp), kp.node_budget ? 16u : kp.abort ? kWatchSteps : ~0u);
}

// Watchdog: charge the nodes since the last look (as mbe_result.nodes counts
// them; steps are no measure, a wide step counts for many), look at the abort
// flag. Every worker looks at the same line, so without a node budget it does
// every kWatchSteps and not at every event: with 2,048 workers that took a
// batch of 64 graphs under a time limit from 16 ms to 23.
__device__ __forceinline__ void watch(const KParams& kp, Walk& k) {
    if (!kp.abort) return;
    const u64 now = kp.node_budget ? k.nodes : k.steps;
    if (!kp.node_budget && now - k.charged < kWatchSteps) return;
    if (charge_nodes(kp, now - k.charged)) k.stop = true;
    k.charged = now;
}

// ------------------------------------------------------------ hand-over
// A donated level goes straight to an idle worker: it sets its bit in the
// idle map and watches its own flag word; a donor clears the bit (the one
// whose clear finds it set has the worker), writes the worker's slot and
// raises the flag. Nothing shared is polled: the flag has a line of its own,
// and a busy worker looks at a few words of the map once per event, each on a
// line of its own. (A shared ring that idle workers probe cost its users
// microseconds per access: the planted background took 15 ms with it and 4 ms
// with donation off. One count of idle workers that all read was the next
// limit: with 2,048 workers a batch of 64 graphs took 8.3 ms, and 4.5 with this
// map.)
// Control block (u64 words, 16 to a 128-byte line): [0] active workers,
// [16 (1 + i)] idle map word i, then one flag line per worker: 0
// none, 1 a level lies in the slot, 2 leave. A worker counts from its start
// on: the launch may hold more workers than are resident at once, and those
// that start late find the roots claimed and leave. It waits for its count to
// be performed before it claims a root: then whoever finds the roots claimed
// and the count at zero knows that nobody works, and that no level will be
// handed to the workers it sends away.
// Slot: [0] graph | r_is_u << 32, [1] W | np << 32, [2] nx | nq << 32, [3] R hash sum,
// [4] |R|, then hl[64 W], hc[np + nx], the rows of P, X and Q by word
// (W x (np + nx + nq)). It holds all that the level needs: a serving kernel's
// descriptors are written while it runs, and only the worker that claims a
// root has an acquire behind it.
__device__ __forceinline__ unsigned long long* idle_word(const KParams& kp, uint32_t i) {
    return kp.tctl + 16 * (1 + i);
}
__device__ __forceinline__ unsigned long long* flag_of(const KParams& kp, uint32_t w) {
    return kp.tctl + 16 * (1 + (kp.tworkers + 63) / 64 + w);
}
__device__ __forceinline__ u64* slot_of(const KParams& kp, uint32_t w) {
    return (u64*)kp.tslots + (size_t)w * kp.tslot_words;
}
// Look for idle workers at an event, in kLook words of the map from one that
// changes from event to event, and say how many levels may go to them: with
// few idle among many busy, most workers stay out of the race for them (about
// one donor per idle worker and interval: a claim that fails is an atomic
// lost); with many idle, more than one.
constexpr uint32_t kLook = 4, kMaxGive = 2;
__device__ __forceinline__ uint32_t map_words(const KParams& kp) { return (kp.tworkers + 63) / 64; }
__device__ __forceinline__ uint32_t may_give(const KParams& kp, Walk& k) {
    const Here lane;
    const uint32_t nw = map_words(kp), n = min(nw, kLook);
    const uint32_t h = (blockIdx.x * 0x9E3779B1u + (uint32_t)k.steps * 0x85EBCA6Bu) >> 8;
    k.look = h % nw;
    k.idle = lane() < n ? ld_rlx(idle_word(kp, (k.look + lane()) % nw)) : 0;
    if (!__ballot(k.idle != 0)) return 0;
    const uint32_t found = red_add32(__popcll(k.idle));
    return (h >> 6) % (64 * n) < found ? min(found, kMaxGive) : 0;
}
// Claim one of the idle workers seen, for a level of graph g; its number, or
// ~0. Whoever clears the worker's bit has it; this donor is active meanwhile,
// so counting the worker as active can follow.
__device__ __forceinline__ uint32_t claim_idle(const KParams& kp, Walk& k) {
    const Here lane;
    const uint32_t nw = map_words(kp), rot = (blockIdx.x * 0x9E3779B1u) >> 26;
    for (uint32_t tries = 0; tries < 4; tries++) {
        const u64 m = __ballot(k.idle != 0);
        if (!m) break;
        const uint32_t l = __builtin_ctzll(m);
        const uint32_t wi = (k.look + l) % nw;
        const u64 v = rdlane64(k.idle, l), up = v >> rot << rot;
        const uint32_t bit = __builtin_ctzll(up ? up : v);
        u64 old = 0;
        if (lane() == 0) old = atomicAnd(idle_word(kp, wi), ~(1ull << bit));
        old = uni64(old);
        // the word as it is now, without the worker tried
        k.idle = wrlane64(k.idle, old & ~(1ull << bit), l);
        if ((old >> bit) & 1) {
            if (lane() == 0) {
                atomicAdd(kp.tctl, 1ull);
                if (kp.remaining) atomicAdd(kp.remaining + 2 * (size_t)k.g, 1ull);
            }
            return wi * 64 + bit;
        }
    }
    return 0xFFFFFFFFu;
}
__device__ __forceinline__ void hand_over(const KParams& kp, uint32_t w) {
    wait_mem();  // the slot's words have reached the device's memory
    if (lane() == 0) st_rlx(flag_of(kp, w), 1ull);
}

// ------------------------------------------------------------------ wide
// A problem on the wide tier. rows[w * ncs + k] is word w of candidate k's
// row (ncs = nc rounded up to 64, the padding rows are never selected by a
// mask). Frame k: x, R hash sum, |R|, unused, then L (W words), P, X and Q
// (Wc words each).
struct Wide {
    uint32_t W, nc, Wc, ncs, fs, nlds, maxdepth;
    u64 *hl, *hc, *rows, *fbase, *hstack;
    u64* kcols;      // reduction scratch: 64 W columns of kWideKw words
    uint32_t* clist; // nc candidates
    size_t end;      // arena words in use
    __device__ __forceinline__ u64* frame(uint32_t k) const {
        const uint32_t i = k - 1;
        return i < nlds ? fbase + (size_t)i * fs : hstack + (size_t)(i - nlds) * fs;
    }
};
constexpr uint32_t kWideKw = kTileQ / 64;

// The LDS words problems may use: after the header (which the section
// counters follow when they are on), up to `end`.
struct LdsSpan {
    u64 *begin, *end;
};
__device__ __forceinline__ LdsSpan lds_span(const KParams& kp, u64* lds) {
    return {lds + (kp.sections ? kLdsHdr : kTreeHdr), lds + kp.lds_words};
}

// What a tile needs besides its source: where its frames go while it is
// suspended and, above one word, the narrow problem and that one's frames.
struct TileMem {
    u64 *save, *nar, *nsave;
};
// n words of LDS, when it has them and `spare` more, else of the arena
__device__ __forceinline__ u64* place(u64*& lp, const u64* lend, u64*& ap, size_t n, size_t spare) {
    u64*& at = n + spare <= (size_t)(lend - lp) ? lp : ap;
    u64* r = at;
    at += n;
    return r;
}

// Place a wide problem (W words, nc candidates of which np in P or X) from
// arena word off: the tile's memory, then the data and the reduction scratch,
// each in LDS when it fits, then as many frames as LDS holds.
__device__ __forceinline__ bool layout_wide(const KParams& kp, Wide& S, u64* arena, LdsSpan sp,
                                            size_t off, uint32_t W, uint32_t nc, uint32_t np,
                                            TileMem& M) {
    S.W = W;
    S.nc = nc;
    S.Wc = (nc + 63) >> 6;
    S.ncs = S.Wc * 64;
    S.fs = kFrameHdr + W + 3 * S.Wc;
    S.maxdepth = np + 2;
    u64* lp = sp.begin;
    u64* ap = arena + off;
    const uint32_t C = tile_class(W);
    M.nar = M.nsave = nullptr;
    if (C > 1) M.nar = place(lp, sp.end, ap, kNarrowWords, 0);
    S.hl = place(lp, sp.end, ap, (size_t)64 * W + nc + (size_t)S.ncs * W, 2 * S.fs);
    S.hc = S.hl + (size_t)64 * W;
    S.rows = S.hc + nc;
    S.kcols = place(lp, sp.end, ap, (size_t)64 * W * kWideKw + (nc + 1) / 2, 2 * S.fs);
    S.clist = (uint32_t*)(S.kcols + (size_t)64 * W * kWideKw);
    M.save = place(lp, sp.end, ap, save_words(C), 4 * S.fs);
    if (C > 1) M.nsave = place(lp, sp.end, ap, save_words(1), 4 * S.fs);
    S.nlds = (uint32_t)min((size_t)S.maxdepth, (size_t)(sp.end - lp) / S.fs);
    S.fbase = lp;
    S.hstack = ap;
    ap += (size_t)(S.maxdepth - S.nlds) * S.fs;
    S.end = (size_t)(ap - arena);
    return S.end <= kp.arena_words;
}

// Sum of the hash terms of the set bits of L (W words over hl).
__device__ __forceinline__ u64 sum_bits(const u64* hl, const u64* L, uint32_t W, uint32_t& nl) {
    const Here lane;
    u64 s = 0;
    uint32_t n = 0;
    for (uint32_t w = 0; w < W; w++) {
        const u64 word = uni64(L[w]);
        n += __popcll(word);
        if ((word >> lane()) & 1) s += hl[w * 64 + lane()];
    }
    nl = n;
    return red_add64(s);
}

// Materialisation of one biclique (see emit_biclique): room for the record
// and its head. Returns where the L' terms go, or null past the capacity.
__device__ __forceinline__ uint64_t* emit_head(const KParams& kp, uint32_t nl, u64 nr, u64 sr) {
    const Here lane;
    u64 at = 0;
    if (lane() == 0) {
        at = atomicAdd(&kp.emit_pos[0], (u64)nl + 2);
        atomicAdd(&kp.emit_pos[1], (u64)nl + nr + 2);
    }
    at = uni64(at);
    if (at + nl + 2 > kp.emit_cap) return nullptr;
    uint64_t* o = kp.emit + at;
    if (lane() == 0) {
        o[0] = (u64)nl | (nr << 32);
        o[1] = sr;
    }
    return o + 2;
}
// The terms of one word of L' (terms hl, one per bit), from position n on.
__device__ __forceinline__ void emit_word(uint64_t* o, uint32_t& n, u64 word, const u64* hl) {
    if ((word >> lane()) & 1) o[n + __popcll(word & lanemask_lt())] = hl[lane()];
    n += __popcll(word);
}

// ------------------------------------------------------------ Q reduction
// Keep the candidates of a list whose rows no other row of the list contains
// (see reduce_q for why the others decide nothing), in place; returns how
// many. Rows are taken in list order, 64 at a time: each is tested against
// the kept rows through their columns (kcols[j * kw + t]: the kept rows that
// hold bit j, 64 kw of them; later ones are kept without being indexed), then
// against the batch's other survivors. row(k, w): word w of candidate k's
// row. nk: how many kept rows are indexed. Rows are best given largest first:
// what is taken before a row that contains it stays.
template <class Row>
__device__ __forceinline__ bool inside_cols(const Row& row, uint32_t k, uint32_t W,
                                            const u64* kcols, uint32_t kw, uint32_t nk) {
    for (uint32_t t = 0; t * 64 < nk; t++) {
        u64 a = low_bits(nk - t * 64);
        for (uint32_t w = 0; w < W && a; w++) {
            u64 bits = row(k, w);
            while (bits && a) {
                a &= kcols[(size_t)(w * 64 + __builtin_ctzll(bits)) * kw + t];
                bits &= bits - 1;
            }
        }
        if (a) return true;
    }
    return false;
}
template <class Row>
__device__ __forceinline__ uint32_t reduce_rows(const Row& row, uint32_t W, uint32_t* list,
                                                uint32_t n, u64* kcols, uint32_t kw, uint32_t& nk) {
    const Here lane;
    for (uint32_t i = lane(); i < 64 * W * kw; i += 64) kcols[i] = 0;
    sync_own();
    uint32_t kept = 0, idx = 0;
    for (uint32_t b = 0; b < n; b += 64) {
        const bool valid = b + lane() < n;
        const uint32_t k = valid ? list[b + lane()] : 0;
        u64 m = __ballot(valid && !inside_cols(row, k, W, kcols, kw, idx));
        for (u64 todo = m; todo; todo &= todo - 1) {
            const uint32_t i = __builtin_ctzll(todo);
            const uint32_t ki = rdlane32(k, i);
            u64 out = 0;
            for (uint32_t w = 0; w < W; w++) out |= row(k, w) & ~row(ki, w);
            const u64 in = __ballot(out == 0) & ~(1ull << i) & m;
            m &= ~in;
            todo &= ~in;
        }
        const uint32_t cnt = __popcll(m);
        const bool mine = (m >> lane()) & 1;
        const uint32_t r = __popcll(m & lanemask_lt());
        if (mine) list[kept + r] = k;
        if (idx + cnt <= 64 * kw) {
            if (mine) {
                const uint32_t t = idx + r;
                for (uint32_t w = 0; w < W; w++)
                    for (u64 bits = row(k, w); bits; bits &= bits - 1)
                        own_or(&kcols[(size_t)(w * 64 + __builtin_ctzll(bits)) * kw + (t >> 6)],
                               1ull << (t & 63));
            }
            idx += cnt;
        }
        kept += cnt;
        sync_own();
    }
    nk = idx;
    return kept;
}
// Drop from a list of P candidates those inside an indexed row, in place.
template <class Row>
__device__ __forceinline__ uint32_t prune_rows(const Row& row, uint32_t W, uint32_t* list,
                                               uint32_t n, const u64* kcols, uint32_t kw,
                                               uint32_t nk) {
    const Here lane;
    uint32_t left = 0;
    for (uint32_t b = 0; b < n; b += 64) {
        const bool valid = b + lane() < n;
        const uint32_t k = valid ? list[b + lane()] : 0;
        const u64 m = __ballot(valid && !inside_cols(row, k, W, kcols, kw, nk));
        if ((m >> lane()) & 1) list[left + __popcll(m & lanemask_lt())] = k;
        left += __popcll(m);
        wsync();
    }
    return left;
}

// ------------------------------------------------------------------ tile
// The problem a tile is loaded from: rows[k * ks + w * ws], masked by L when
// it is given. Lane i's P, X or D candidate is k = list[i] (LDS header), Q
// candidates (nq of them) are list[kTileP ..]. P, X and D are the sets to
// start with; D holds handled vertices, which act as Q. Tile word i is source
// word (wmap >> 8 i) & 255. hc[cand[k]] (hc[k] without cand) is candidate k's
// hash term.
struct TileSrc {
    const u64 *rows, *hc, *L, *hl;
    const uint32_t* cand;
    size_t ks, ws;
    u64 wmap, P, X, D, sr;
    uint32_t W, nq, nr;
    __device__ __forceinline__ uint32_t word(uint32_t i) const { return (wmap >> (8 * i)) & 255; }
    __device__ __forceinline__ u64 row(uint32_t k, uint32_t i) const {
        return rows[k * ks + word(i) * ws];
    }
};

// How a search returns to run_tree.
enum Ret : int { kDone = 0, kToTile = 1, kEvent = 2, kToNarrow = 3 };
constexpr uint32_t kNoX = 64;  // x of a frame without one in progress

// An event: the watchdog, and how many levels this worker may give away.
// Returns whether the search has to stop for it.
__device__ __forceinline__ bool event(const KParams& kp, Walk& k) {
    k.next_event = k.steps + event_interval(kp);
    watch(kp, k);
    // the watchdog's events may be closer than the donation interval: then
    // donation takes one in so many, at random
    const uint32_t every = kp.abort ? give_interval(kp) / event_interval(kp) : 1;
    const uint32_t h = (blockIdx.x * 0x85EBCA6Bu + (uint32_t)k.steps * 0x9E3779B1u) >> 4;
    const uint32_t turn = every > 1 ? h % every : 0;
    k.give = kp.variant != kNoWS && !turn ? uni32(may_give(kp, k)) : 0;
    return k.stop || k.give;
}

// Search of a tile problem, from its start or (resume) from the frames that
// it left in save, dep of them, for an event or a narrow tile. Rows: rp (P, X
// and D, lane by lane), n0 and n1 (the complements of the Q rows; all ones
// where a lane holds none). Frame f is lane f of fr. A frame is pushed only
// when its level has candidates left, so a chain of last children returns in
// one step. The vertex test is a loop of its own: it carries P and X alone.
// nar: the narrow problem's memory (kNarrowWords), or null when this is one.
template <int W, bool SEC, bool EMIT>
__device__ __forceinline__ int tile_search(const KParams& kp, Walk& k, const TileSrc& src,
                                           const uint32_t* list, u64* save, uint32_t& dep,
                                           bool resume, u64* nar, TileSrc& nsrc, Sec& sec) {
    constexpr uint32_t FW = tile_fw(W);
    // uniform by construction, which the compiler cannot see through generic
    // loads and the task's loops: without this the sets are lane values
    uint32_t depth = resume ? uni32(dep) : 0;
    u64 rp[W], n0[W], n1[W], hcv;
    {
        const Here lane;
        const bool in = ((src.P | src.X | src.D) >> lane()) & 1;
        const uint32_t pk = in ? list[lane()] : 0;
        const uint32_t k0 = lane() < src.nq ? list[kTileP + lane()] : 0;
        const uint32_t k1 = lane() + 64 < src.nq ? list[2 * kTileP + lane()] : 0;
        hcv = in ? src.hc[src.cand ? src.cand[pk] : pk] : 0;
#pragma unroll
        for (int i = 0; i < W; i++) {
            const bool have = (uint32_t)i < src.W;
            const u64 m = have ? (src.L ? src.L[src.word(i)] : ~0ull) : 0;
            rp[i] = have && in ? src.row(pk, i) & m : 0;
            n0[i] = have && lane() < src.nq ? ~src.row(k0, i) : ~0ull;
            n1[i] = have && lane() + 64 < src.nq ? ~src.row(k1, i) : ~0ull;
        }
    }
    u64 P = uni64(src.P), X = uni64(src.X), D = uni64(src.D);
    u64 L[W];
#pragma unroll
    for (int i = 0; i < W; i++) L[i] = ~0ull;
    u64 sr = uni64(src.sr);
    uint32_t nr = uni32(src.nr), nrec = 0, steps = 0;
    uint32_t limit = uni32(k.next_event > k.steps ? (uint32_t)(k.next_event - k.steps) : 0);
    uint32_t all = 0;  // steps before the last event
    u64 fr[FW];
#pragma unroll
    for (uint32_t i = 0; i < FW; i++) fr[i] = 0;
    if (resume) {
        const Here lane;
#pragma unroll
        for (uint32_t i = 0; i < FW; i++) fr[i] = save[i * 64 + lane()];
    }
    int ret = kDone;
    if (resume) P = 0;  // the newest frame is taken first
    u64 recl[W], recs = 0;  // reports not hashed yet: lane i holds report i
    uint32_t recn = 0;
#pragma unroll
    for (int i = 0; i < W; i++) recl[i] = 0;

    // hash the reports: every lane sums the terms of its own L'
    auto flush = [&]() {
        const Here lane;
        u64 sl = 0;
        uint32_t nl = 0;
#pragma unroll
        for (int i = 0; i < W; i++) {
            u64 b = lane() < nrec ? recl[i] : 0;
            nl += __popcll(b);
            const u64* h = src.hl + src.word(i) * 64;
            while (b) {
                sl += h[__builtin_ctzll(b)];
                b &= b - 1;
            }
        }
        if (lane() < nrec)
            k.hs += k.r_is_u ? biclique_hash(recs, sl, recn, nl) : biclique_hash(sl, recs, nl, recn);
        k.cnt += nrec;
        k.nodes += nrec;
        nrec = 0;
    };
    auto push = [&](uint32_t x) {
#pragma unroll
        for (int i = 0; i < W; i++) fr[i] = wrlane64(fr[i], L[i], depth);
        fr[W] = wrlane64(fr[W], P, depth);
        fr[W + 1] = wrlane64(fr[W + 1], X, depth);
        fr[W + 2] = wrlane64(fr[W + 2], D, depth);
        fr[W + 3] = wrlane64(fr[W + 3], sr, depth);
        fr[W + 4] = wrlane64(fr[W + 4], (u64)nr | ((u64)x << 32), depth);
        depth++;
    };
    // whether an event is due that the search has to stop for
    auto due = [&]() {
        if (steps < limit) return false;
        k.steps += steps;
        all += steps;
        steps = 0;
        limit = event_interval(kp);
        return uni1(event(kp, k));
    };

    for (;;) {
        // the next vertex that gives a maximal biclique; what it or a Q row
        // or a handled vertex covers leaves P and X
        u64 Lp[W], C = 0, T = 0;
        uint32_t x = kNoX;
        u64 P0 = P, X0 = X;
        while (P) {
            const uint32_t v = __builtin_ctzll(P);
            u64 z0 = 0, z1 = 0, zc = 0, zt = 0, zd = 0;
#pragma unroll
            for (int i = 0; i < W; i++) {
                Lp[i] = rdlane64(rp[i], v) & L[i];
                z0 |= Lp[i] & n0[i];
                z1 |= Lp[i] & n1[i];
                const u64 t = rp[i] & Lp[i];
                zt |= t;
                zc |= t ^ Lp[i];
                zd |= rp[i] & (L[i] & ~Lp[i]);
            }
            C = __ballot(zc == 0);
            const u64 dead = __ballot(zd == 0);
            P0 = P;
            X0 = X;
            P &= ~dead;
            X &= ~dead;
            steps++;
            if (!(__ballot(z0 == 0) | __ballot(z1 == 0) | (C & D))) {
                T = __ballot(zt != 0);
                x = v;
                break;
            }
        }
        if (SEC) sec.mark(kSecSelect);
        if (x == kNoX) {
            if (depth == 0) break;
            depth--;  // ascend: the x in progress joins D
#pragma unroll
            for (int i = 0; i < W; i++) L[i] = rdlane64(fr[i], depth);
            P = rdlane64(fr[W], depth);
            X = rdlane64(fr[W + 1], depth);
            D = rdlane64(fr[W + 2], depth);
            sr = rdlane64(fr[W + 3], depth);
            const u64 nx = rdlane64(fr[W + 4], depth);
            nr = (uint32_t)nx;
            const uint32_t px = (uint32_t)(nx >> 32);
            if (px != kNoX) D |= 1ull << px;
            if (SEC) sec.mark(kSecLPrime);
            if (P && due()) {  // suspend: the level becomes a frame again
                push(kNoX);
                ret = kEvent;
                break;
            }
            continue;
        }
        const u64 live = P0 | X0, ab = live & C;  // x among them
        const u64 Pn = live & T & ~C;
        u64 sr2 = sr + rdlane64(hcv, x);
        for (u64 m = ab & ~(1ull << x); m; m &= m - 1) sr2 += rdlane64(hcv, __builtin_ctzll(m));
        const uint32_t nr2 = nr + __popcll(ab);
        if (SEC) sec.mark(kSecCheck);
#pragma unroll
        for (int i = 0; i < W; i++) recl[i] = wrlane64(recl[i], Lp[i], nrec);
        recs = wrlane64(recs, sr2, nrec);
        recn = wrlane32(recn, nr2, nrec);
        nrec++;
        if (EMIT && kp.emit_pos) {
            uint32_t nl = 0, n = 0;
#pragma unroll
            for (int i = 0; i < W; i++) nl += __popcll(Lp[i]);
            uint64_t* o = emit_head(kp, nl, nr2, sr2);
#pragma unroll
            for (int i = 0; i < W; i++)
                if (o) emit_word(o, n, Lp[i], src.hl + src.word(i) * 64);
        }
        if (nrec == 64) flush();
        if (SEC) sec.mark(kSecReport);
        if (!Pn) {
            D |= 1ull << x;
            continue;
        }
        bool narrow = false;
        if (W > 1 && (uint32_t)__popcll(Pn) >= kNarrowP) {
            uint32_t nl = 0;
#pragma unroll
            for (int i = 0; i < W; i++) nl += __popcll(Lp[i]);
            narrow = nl <= 64;
        }
        if (P || narrow) push(x);
        if (narrow) {
            // the bits of L' become bits 0, 1, ... of one word
            u64 a = 0, b0 = 0, b1 = 0;
            uint32_t t = 0;
            u64* hl = nar;
            const Here lane;
#pragma unroll
            for (int i = 0; i < W; i++) {
                const u64 m = Lp[i];
                if ((m >> lane()) & 1)
                    hl[t + __popcll(m & lanemask_lt())] = src.hl[src.word(i) * 64 + lane()];
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const uint32_t r = (uint32_t)(rp[i] >> (32 * h));
                    const uint32_t q0 = (uint32_t)(n0[i] >> (32 * h));
                    const uint32_t q1 = (uint32_t)(n1[i] >> (32 * h));
                    for (uint32_t mm = (uint32_t)(m >> (32 * h)); mm; mm &= mm - 1, t++) {
                        const uint32_t b = __builtin_ctz(mm);
                        a |= (u64)((r >> b) & 1) << t;
                        b0 |= (u64)((q0 >> b) & 1) << t;
                        b1 |= (u64)((q1 >> b) & 1) << t;
                    }
                }
            }
            const u64 all = low_bits(t);
            u64* hc = nar + 64;
            u64* rows = hc + 64;
            uint32_t* nl = (uint32_t*)(rows + kTileP + kTileQ);
            hc[lane()] = hcv;
            rows[lane()] = a;
            rows[kTileP + lane()] = ~b0 & all;
            rows[2 * kTileP + lane()] = ~b1 & all;
            for (uint32_t q = lane(); q < kTileP + kTileQ; q += 64) nl[q] = q;
            wsync();
            nsrc.rows = rows;
            nsrc.hc = hc;
            nsrc.L = nullptr;
            nsrc.hl = hl;
            nsrc.cand = nullptr;
            nsrc.ks = nsrc.ws = 1;
            nsrc.wmap = 0;
            nsrc.P = Pn;
            nsrc.X = 0;
            nsrc.D = D;
            nsrc.sr = sr2;
            nsrc.W = 1;
            nsrc.nq = src.nq;
            nsrc.nr = nr2;
            ret = kToNarrow;
            if (SEC) sec.mark(kSecCompact);
            break;
        }
#pragma unroll
        for (int i = 0; i < W; i++) L[i] = Lp[i];
        P = Pn;
        X = 0;
        sr = sr2;
        nr = nr2;
        if (SEC) sec.mark(kSecExpand);
        if (due()) {
            push(kNoX);
            ret = kEvent;
            break;
        }
    }
    if (nrec) flush();
    dep = depth;
    if (ret != kDone) {
        const Here lane;
#pragma unroll
        for (uint32_t i = 0; i < FW; i++) save[i * 64 + lane()] = fr[i];
    }
    k.steps += steps;
    k.words += (u64)(all + steps) * W * (src.nq + __popcll(src.P | src.X | src.D));
    wsync();
    return ret;
}

// --------------------------------------------------------------- wide walk
// Candidates of a bit mask (Wc words), ascending, into list; returns how many.
__device__ __forceinline__ uint32_t gather_bits(const u64* M, uint32_t Wc, uint32_t* list) {
    const Here lane;
    uint32_t n = 0;
    for (uint32_t b = 0; b < Wc; b++) {
        const u64 m = uni64(M[b]);
        if ((m >> lane()) & 1) list[n + __popcll(m & lanemask_lt())] = b * 64 + lane();
        n += __popcll(m);
    }
    return n;
}
// Lane i's word of L: word w0 + i.
__device__ __forceinline__ u64 word_of(const u64* L, uint32_t W, uint32_t w0) {
    const Here lane;
    return w0 + lane() < W ? L[w0 + lane()] : 0;
}
// Words of L (W of them) that are not zero, packed as a tile word map;
// returns how many, or kTileW + 1 when a tile cannot hold them.
__device__ __forceinline__ uint32_t word_map(const u64* L, uint32_t W, u64& wmap) {
    uint32_t n = 0;
    wmap = 0;
    if (W > 256) return kTileW + 1;
    for (uint32_t w = 0; w < W; w++)
        if (uni64(L[w])) {
            if (n < kTileW) wmap |= (u64)w << (8 * n);
            n++;
        }
    return min(n, kTileW + 1);
}

// A new level in frame F (P, X, Q): a tile (kToTile, src set), a level for
// the wide tier (kDone), or nothing left of P (kEvent). A level that does not
// fit the tile as it is loses the Q candidates that other Q candidates
// contain and the P candidates that Q candidates contain.
__device__ __forceinline__ int place_level(const Wide& S, u64* F, uint32_t pn, uint32_t xn,
                                           uint32_t qn, uint32_t* list, TileSrc& src) {
    const Here lane;
    const uint32_t W = uni32(S.W), Wc = uni32(S.Wc);
    const u64* L = F + kFrameHdr;
    u64* P = F + kFrameHdr + W;
    u64* Q = P + 2 * Wc;
    src.W = word_map(L, W, src.wmap);
    const bool fits = pn + xn <= kTileP && qn <= kTileQ && src.W <= kTileW;
    if (fits) {
        gather_bits(P, Wc, list);
        if (xn) gather_bits(P + Wc, Wc, list + pn);
        gather_bits(Q, Wc, list + kTileP);
        wsync();
    } else {
        if (qn == 0) return kDone;
        gather_bits(P, Wc, S.clist);
        gather_bits(Q, Wc, S.clist + pn);
        wsync();
        const auto row = [&](uint32_t k, uint32_t w) { return S.rows[(size_t)w * S.ncs + k] & L[w]; };
        uint32_t nk;
        const uint32_t p0 = pn;
        qn = reduce_rows(row, W, S.clist + p0, qn, S.kcols, kWideKw, nk);
        pn = prune_rows(row, W, S.clist, pn, S.kcols, kWideKw, nk);
        if (pn == 0) return kEvent;
        if (pn + xn <= kTileP && qn <= kTileQ && src.W <= kTileW) {
            for (uint32_t i = lane(); i < pn; i += 64) list[i] = S.clist[i];
            for (uint32_t i = lane(); i < qn; i += 64) list[kTileP + i] = S.clist[p0 + i];
            if (xn) gather_bits(P + Wc, Wc, list + pn);
            wsync();
        } else {
            for (uint32_t b = lane(); b < Wc; b += 64) P[b] = Q[b] = 0;
            sync_own();
            for (uint32_t i = lane(); i < pn; i += 64) own_or(&P[S.clist[i] >> 6], 1ull << (S.clist[i] & 63));
            for (uint32_t i = lane(); i < qn; i += 64)
                own_or(&Q[S.clist[p0 + i] >> 6], 1ull << (S.clist[p0 + i] & 63));
            sync_own();
            return kDone;
        }
    }
    src.rows = S.rows;
    src.ks = 1;
    src.ws = S.ncs;
    src.hc = S.hc;
    src.cand = nullptr;
    src.hl = S.hl;
    src.L = L;
    src.P = low_bits(pn);
    src.X = low_bits(pn + xn) & ~src.P;
    src.D = 0;
    src.nq = qn;
    src.sr = uni64(F[1]);
    src.nr = (uint32_t)uni64(F[2]);
    return kToTile;
}

// fn(i, row word) for the words w0 + i, i in m, of candidate block b, a
// candidate per lane; four loads in flight. m holds the words that L has bits
// in: below a hub root L' is a few bits, each in a word of its own, of a
// universe of many words. Five roots of 4,000 L bits against 900 candidates
// (63 words, a level's L' some 80 bits): 502 ms of kernel with every word read,
// 346 so; universes of a few words the same.
template <class F>
__device__ __forceinline__ void each_row(const Wide& S, uint32_t w0, uint32_t b, u64 m, F&& fn) {
    const Here lane;
    const u64* rows = S.rows + (size_t)w0 * S.ncs + b * 64 + lane();
    while (__popcll(m) >= 4) {
        uint32_t i[4];
        u64 r[4];
#pragma unroll
        for (int t = 0; t < 4; t++) {
            i[t] = __builtin_ctzll(m);
            m &= m - 1;
            r[t] = rows[(size_t)i[t] * S.ncs];
        }
#pragma unroll
        for (int t = 0; t < 4; t++) fn(i[t], r[t]);
    }
    for (; m; m &= m - 1) {
        const uint32_t i = __builtin_ctzll(m);
        fn(i, rows[(size_t)i * S.ncs]);
    }
}

// Walk the wide levels from level k until a child fits the tile (kToTile,
// src set; its level is k + 1), an event is due (kEvent) or the problem is
// finished (kDone). resume: level k's x in progress has just been handled.
template <bool SEC, bool EMIT>
__device__ __forceinline__ int wide_walk(const KParams& kp, Walk& wk, const Wide& S, uint32_t& k,
                                          bool resume, uint32_t* list, TileSrc& src, Sec& sec) {
    const Here lane;
    const uint32_t W = uni32(S.W), Wc = uni32(S.Wc);
    for (;;) {
        k = uni32(k);
        u64* F = S.frame(k);
        u64* L = F + kFrameHdr;
        u64* P = L + W;
        u64* X = P + Wc;
        u64* Q = X + Wc;
        if (resume) {  // the x in progress is handled: it joins Q
            if (lane() == 0) {
                const uint32_t x = (uint32_t)F[0];
                Q[x >> 6] |= 1ull << (x & 63);
            }
            wsync();
            resume = false;
        }
        if (wk.steps >= wk.next_event && uni1(event(kp, wk))) return kEvent;
        // the next x: the lowest candidate left in P
        uint32_t x = 0xFFFFFFFFu;
        for (uint32_t b0 = 0; b0 < Wc && x == 0xFFFFFFFFu; b0 += 64) {
            const u64 pw = b0 + lane() < Wc ? P[b0 + lane()] : 0;
            const u64 nz = __ballot(pw != 0);
            if (nz) {
                const uint32_t i = __builtin_ctzll(nz);
                x = (b0 + i) * 64 + __builtin_ctzll(rdlane64(pw, i));
            }
        }
        if (SEC) sec.mark(kSecSelect);
        if (x == 0xFFFFFFFFu) {
            if (--k == 0) return kDone;
            resume = true;
            continue;
        }
        // L'. A wide step counts for one tile step and for half a one per word of
        // candidates; it takes longer than as many, so events are further apart
        // in time here
        wk.steps += 1 + Wc / 2;
        u64* Fc = S.frame(k + 1);
        u64* Lc = Fc + kFrameHdr;
        u64* Pc = Lc + W;
        u64* Xc = Pc + Wc;
        u64* Qc = Xc + Wc;
        for (uint32_t w = lane(); w < W; w += 64) Lc[w] = S.rows[(size_t)w * S.ncs + x] & L[w];
        wsync();
        const u64 p0 = word_of(L, W, 0), c0 = word_of(Lc, W, 0);
        if (SEC) sec.mark(kSecLPrime);
        wk.words += (u64)W * S.nc;
        bool nonmax = false;
        uint32_t qn = 0;
        for (uint32_t b = 0; b < Wc; b++) {
            const u64 qw = uni64(Q[b]);
            u64 tm = 0;
            if (qw) {
                u64 miss = 0, touch = 0;
                for (uint32_t w0 = 0; w0 < W; w0 += 64) {
                    const u64 c = w0 ? word_of(Lc, W, w0) : c0;
                    each_row(S, w0, b, __ballot(c != 0), [&](uint32_t i, u64 r) {
                        const u64 l = rdlane64(c, i);
                        miss |= l & ~r;
                        touch |= r & l;
                    });
                }
                if (__ballot(miss == 0) & qw) {
                    nonmax = true;
                    break;
                }
                tm = __ballot(touch != 0) & qw;
                qn += __popcll(tm);
            }
            if (lane() == 0) Qc[b] = tm;
        }
        if (SEC) sec.mark(kSecCheck);
        uint32_t pn = 0, ab = 0;
        u64 abh = 0;
        for (uint32_t b = 0; b < Wc; b++) {
            const u64 pw = uni64(P[b]), xw = uni64(X[b]), live = pw | xw;
            u64 pm = 0;
            if (live) {
                u64 out = 0, miss = 0, touch = 0;
                for (uint32_t w0 = 0; w0 < W; w0 += 64) {
                    const u64 p = w0 ? word_of(L, W, w0) : p0, c = w0 ? word_of(Lc, W, w0) : c0;
                    each_row(S, w0, b, __ballot(p != 0), [&](uint32_t i, u64 r) {
                        const u64 l = rdlane64(c, i);
                        out |= r & rdlane64(p, i) & ~l;
                        miss |= l & ~r;
                        touch |= r & l;
                    });
                }
                const u64 dead = __ballot(out == 0);
                if (!nonmax) {
                    const u64 C = __ballot(miss == 0);
                    const u64 am = live & C;
                    pm = live & __ballot(touch != 0) & ~C;
                    ab += __popcll(am);
                    if ((am >> lane()) & 1) abh += S.hc[b * 64 + lane()];
                }
                if ((live & dead) && lane() == 0) {
                    P[b] = pw & ~dead;
                    X[b] = xw & ~dead;
                }
            }
            if (!nonmax) {
                if (lane() == 0) {
                    Pc[b] = pm;
                    Xc[b] = 0;
                }
                pn += __popcll(pm);
            }
        }
        wsync();
        if (nonmax) continue;
        wk.nodes++;
        uint32_t nl;
        const u64 sl = sum_bits(S.hl, Lc, W, nl);
        const u64 sr = uni64(F[1]) + red_add64(abh);
        const uint32_t nr = (uint32_t)uni64(F[2]) + ab;
        const u64 h = wk.r_is_u ? biclique_hash(sr, sl, nr, nl) : biclique_hash(sl, sr, nl, nr);
        wk.cnt++;
        if (lane() == 0) wk.hs += h;
        if (EMIT && kp.emit_pos) {
            uint32_t n = 0;
            uint64_t* o = emit_head(kp, nl, nr, sr);
            for (uint32_t w = 0; w < W && o; w++) emit_word(o, n, uni64(Lc[w]), S.hl + w * 64);
        }
        if (SEC) sec.mark(kSecExpand);
        if (lane() == 0) {
            F[0] = x;
            Fc[1] = sr;
            Fc[2] = nr;
        }
        wsync();
        if (pn == 0) {
            resume = true;  // a leaf: x joins Q
            continue;
        }
        const int r = place_level(S, Fc, pn, 0, qn, list, src);
        if (SEC) sec.mark(kSecCompact);
        if (r == kToTile) return r;
        if (r == kEvent)
            resume = true;  // nothing left of P': a leaf
        else
            k++;
    }
}

// -------------------------------------------------------------- donation
// What a level keeps of P when it gives: the first half, of which a level
// without an x in progress always has one; nothing when it gives the rest.
__device__ __forceinline__ uint32_t keep_of(uint32_t n, bool rest, bool running) {
    return running ? (rest ? 0 : n / 2) : max(1u, n / 2);
}
__device__ __forceinline__ u64 first_bits(u64 P, uint32_t n) {
    u64 r = P;
    for (uint32_t i = 0; i < n; i++) r &= r - 1;
    return P & ~r;
}
__device__ __forceinline__ size_t slot_need(uint32_t W, uint32_t npx, uint32_t nq) {
    return (size_t)kSlotHeaderWords + (size_t)64 * W + npx + (size_t)W * (npx + nq);
}
// Whether a donated level of this size fits a slot and any worker's arena.
__device__ __forceinline__ bool slot_fits(const KParams& kp, uint32_t W, uint32_t npx, uint32_t nq) {
    return slot_need(W, npx, nq) <= kp.tslot_words && tree_wide_words(W, npx + nq, npx) <= kp.arena_words;
}
__device__ __forceinline__ void slot_head(u64* slot, const Walk& wk, uint32_t W, uint32_t np,
                                          uint32_t nx, uint32_t nq, u64 sr, u64 nr) {
    if (lane() == 0) {
        st_rlx(slot, (u64)wk.g | ((u64)wk.r_is_u << 32));
        st_rlx(slot + 1, (u64)W | ((u64)np << 32));
        st_rlx(slot + 2, (u64)nx | ((u64)nq << 32));
        st_rlx(slot + 3, sr);
        st_rlx(slot + 4, nr);
    }
}

// Give away part of the shallowest wide level with unselected work: the donor
// keeps the first candidates A of P (keep_of) and moves the rest B to X; the
// thief gets P = B, X and Q u A u x. The order "x, A, B, X" is a valid order
// of the level, so both sides report exactly the bicliques of the sequential
// walk. Levels 1..cur have their x in progress; cur has none when idle_cur is
// set.
__device__ __forceinline__ bool donate_wide(const KParams& kp, const Wide& S, uint32_t cur,
                                            bool idle_cur, bool rest, Walk& wk) {
    const Here lane;
    const uint32_t W = S.W, Wc = S.Wc;
    const uint32_t top = kp.donate_depth ? min(cur, kp.donate_depth) : cur;
    for (uint32_t k = 1; k <= top; k++) {
        u64* F = S.frame(k);
        const u64* L = F + kFrameHdr;
        u64* P = F + kFrameHdr + W;
        u64* X = P + Wc;
        const u64* Q = X + Wc;
        uint32_t pc = 0;
        for (uint32_t b = lane(); b < Wc; b += 64) pc += __popcll(P[b]);
        pc = red_add32(pc);
        const bool running = k < cur || !idle_cur;
        if (pc == 0 || (!running && pc < 2)) continue;
        const uint32_t x = running ? uni32((uint32_t)F[0]) : 0xFFFFFFFFu;
        const uint32_t keep = keep_of(pc, rest, running), np = pc - keep;
        // sizes, and t = the first candidate of B
        uint32_t seen = 0, t = keep ? Wc * 64 : 0, nx = 0, nq = keep + (running ? 1 : 0);
        for (uint32_t b = 0; b < Wc; b++) {
            const u64 pw = uni64(P[b]);
            const uint32_t c = __popcll(pw);
            if (seen < keep && seen + c >= keep) {
                const u64 up = pw & ~first_bits(pw, keep - seen);
                t = b * 64 + (up ? __builtin_ctzll(up) : 64);
            }
            seen += c;
            nx += __popcll(uni64(X[b]));
            nq += __popcll(uni64(Q[b]));
        }
        const uint32_t npx = np + nx, n = npx + nq;
        if (!slot_fits(kp, W, npx, nq)) continue;
        const uint32_t to = uni32(claim_idle(kp, wk));
        if (to == 0xFFFFFFFFu) return false;
        u64* slot = slot_of(kp, to);
        u64* hl = slot + kSlotHeaderWords;
        u64* hc = hl + (size_t)64 * W;
        u64* rows = hc + npx;
        for (uint32_t i = lane(); i < 64 * W; i += 64) st_rlx(hl + i, S.hl[i]);
        uint32_t ip = 0, ix = np, iq = npx;
        for (uint32_t b = 0; b < Wc; b++) {
            const u64 pw = uni64(P[b]);
            const u64 aw = b * 64 >= t ? 0 : pw & low_bits(t - b * 64);
            const u64 bw = pw & ~aw, xw = uni64(X[b]);
            u64 qw = uni64(Q[b]) | aw;
            if (running && b == (x >> 6)) qw |= 1ull << (x & 63);
            const u64 all = bw | xw | qw;
            const uint32_t kk = b * 64 + lane();
            if ((all >> lane()) & 1) {
                const u64 lt = lanemask_lt();
                const uint32_t at = ((bw >> lane()) & 1)   ? ip + __popcll(bw & lt)
                                    : ((xw >> lane()) & 1) ? ix + __popcll(xw & lt)
                                                           : iq + __popcll(qw & lt);
                if (at < npx) st_rlx(hc + at, S.hc[kk]);
                for (uint32_t w = 0; w < W; w++)
                    st_rlx(rows + (size_t)w * n + at, S.rows[(size_t)w * S.ncs + kk] & L[w]);
            }
            ip += __popcll(bw);
            ix += __popcll(xw);
            iq += __popcll(qw);
        }
        slot_head(slot, wk, W, np, nx, nq, F[1], F[2]);
        hand_over(kp, to);
        for (uint32_t b = lane(); b < Wc; b += 64) {
            const u64 pw = P[b];
            const u64 aw = b * 64 >= t ? 0 : pw & low_bits(t - b * 64);
            X[b] |= pw & ~aw;
            P[b] = aw;
        }
        wsync();
        return true;
    }
    return false;
}

// The same from the frames of a suspended tile (depth of them; the newest may
// have no x in progress). Rows come from the tile's source; level: how many
// levels lie above.
__device__ __forceinline__ bool donate_tile(const KParams& kp, const TileSrc& src,
                                            const uint32_t* list, u64* save, uint32_t depth,
                                            uint32_t level, bool rest, Walk& wk) {
    const Here lane;
    const uint32_t W = src.W, C = tile_class(W);
    for (uint32_t f = 0; f < depth; f++) {
        if (kp.donate_depth && level + f + 1 > kp.donate_depth) return false;
        u64* F = save + f;
        const u64 P = uni64(F[64 * C]);
        const uint32_t x = uni32((uint32_t)(F[64 * (C + 4)] >> 32)), pc = __popcll(P);
        if (P == 0 || (x == kNoX && pc < 2)) continue;
        const u64 D = uni64(F[64 * (C + 2)]);
        const u64 A = first_bits(P, keep_of(pc, rest, x != kNoX)), B = P & ~A;
        const u64 X = uni64(F[64 * (C + 1)]);
        const u64 qp = (x == kNoX ? D : D | (1ull << x)) | A;  // lanes that become Q
        const uint32_t np = __popcll(B), nx = __popcll(X), npx = np + nx;
        const uint32_t nq = __popcll(qp) + src.nq, n = npx + nq;
        if (!slot_fits(kp, W, npx, nq)) continue;
        const uint32_t to = uni32(claim_idle(kp, wk));
        if (to == 0xFFFFFFFFu) return false;
        u64* slot = slot_of(kp, to);
        u64* hl = slot + kSlotHeaderWords;
        u64* hc = hl + (size_t)64 * W;
        u64* rows = hc + npx;
        const u64 lt = lanemask_lt(), me = 1ull << lane();
        const uint32_t at = (B & me)   ? __popcll(B & lt)
                            : (X & me) ? np + __popcll(X & lt)
                                       : npx + __popcll(qp & lt);
        const bool have = ((B | X | qp) & me) != 0;
        const uint32_t pk = have ? list[lane()] : 0;
        const uint32_t q0 = npx + __popcll(qp);
        if (have && at < npx) st_rlx(hc + at, src.hc[src.cand ? src.cand[pk] : pk]);
        for (uint32_t i = 0; i < W; i++) {
            const u64 L = F[64 * i] & (src.L ? src.L[src.word(i)] : ~0ull);
            u64* r = rows + (size_t)i * n;
            st_rlx(hl + i * 64 + lane(), src.hl[src.word(i) * 64 + lane()]);
            if (have) st_rlx(r + at, src.row(pk, i) & L);
            for (uint32_t q = lane(); q < src.nq; q += 64)
                st_rlx(r + q0 + q, src.row(list[kTileP + q], i) & L);
        }
        slot_head(slot, wk, W, np, nx, nq, uni64(F[64 * (C + 3)]), (uint32_t)uni64(F[64 * (C + 4)]));
        hand_over(kp, to);
        if (lane() == 0) {
            F[64 * C] = A;
            F[64 * (C + 1)] = X | B;
        }
        wsync();
        return true;
    }
    return false;
}

// ----------------------------------------------------------------- tasks
// The descriptors, which every lane holds alike, as the scalars they are: the
// compiler loses track of that where a root and a handed-over level merge, and
// lane values would cost a vector register each.
template <class T>
__device__ __forceinline__ void uni_one(T& v) {
#ifdef __HIP_DEVICE_COMPILE__
    if constexpr (sizeof(T) == 8)
        v = (T)uni64((u64)v);
    else
        v = (T)uni32((uint32_t)v);
#endif
}
template <class... T>
__device__ __forceinline__ void uni_all(T&... v) {
    (uni_one(v), ...);
}
__device__ __forceinline__ void make_uniform(Wide& S) {
    uni_all(S.W, S.nc, S.Wc, S.ncs, S.fs, S.nlds, S.maxdepth, S.hl, S.hc, S.rows, S.fbase, S.hstack,
            S.kcols, S.clist);
}
__device__ __forceinline__ void make_uniform(TileSrc& s) {
    uni_all(s.rows, s.hc, s.L, s.hl, s.cand, s.wmap, s.P, s.X, s.D, s.sr, s.ks, s.ws, s.W, s.nq, s.nr);
}
__device__ __forceinline__ void make_uniform(Walk& k) {
    uni_all(k.cnt, k.nodes, k.donated, k.words, k.steps, k.next_event, k.charged, k.look, k.g, k.give,
            k.r_is_u, k.stop);
}
__device__ __forceinline__ void make_uniform(TileMem& M) { uni_all(M.save, M.nar, M.nsave); }

// What a task starts with after localisation or a slot load.
enum TreeStart : int { kTreeOverflow = -1, kTreeDone = 0, kTreeTile = 1, kTreeWide = 2 };

// Place the memory and the 64 W hash terms of a task that starts as a tile,
// from arena word off; returns the arena words in use.
__device__ __forceinline__ size_t layout_tile(u64* arena, LdsSpan sp, size_t off, uint32_t W,
                                              TileMem& M, u64*& hl) {
    u64* lp = sp.begin;
    u64* ap = arena + off;
    const uint32_t C = tile_class(W);
    M.nar = M.nsave = nullptr;
    if (C > 1) M.nar = place(lp, sp.end, ap, kNarrowWords, 0);
    hl = place(lp, sp.end, ap, 64 * W, 0);
    M.save = place(lp, sp.end, ap, save_words(C), 0);
    if (C > 1) M.nsave = place(lp, sp.end, ap, save_words(1), 0);
    return (size_t)(ap - arena);
}

// Visit the entries (j, v) of N(u_j), u_j in N(x): 64 lists at a time, their
// bounds in LDS (lb: 128 words of u32), a group of g lanes per list with g
// near the lists' mean length, four lists per group in flight. fn(j, v) runs
// with lanes masked. Returns the number of entries.
template <class F>
__device__ __forceinline__ uint32_t for_entries(const DevGraph& G, const uint32_t* Nx, uint32_t d,
                                                uint32_t* lb, F&& fn) {
    const Here lane;
    uint32_t total = 0;
    for (uint32_t j0 = 0; j0 < d; j0 += 64) {
        const uint32_t n = min(64u, d - j0);
        uint32_t s = 0, l = 0;
        if (lane() < n) {
            const uint32_t u = Nx[j0 + lane()];
            s = G.offL[u];
            l = G.offL[u + 1] - s;
        }
        lb[lane()] = s;
        lb[64 + lane()] = l;
        const uint32_t sum = red_add32(l);
        total += sum;
        const uint32_t lg = sum > 32 * n ? 6 : sum > 16 * n ? 5 : sum > 8 * n ? 4 : 3;
        const uint32_t g = 1u << lg, ng = 64u >> lg, gi = lane() >> lg, li = lane() & (g - 1);
        wsync();
        for (uint32_t q0 = 0; q0 < n; q0 += 4 * ng) {
            uint32_t st[4], ln[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t q = q0 + i * ng + gi;
                st[i] = q < n ? lb[q] : 0;
                ln[i] = q < n ? lb[64 + q] : 0;
            }
            const uint32_t most = max(max(ln[0], ln[1]), max(ln[2], ln[3]));
            for (uint32_t t = li; __ballot(t - li < most); t += g) {
                uint32_t v[4];
#pragma unroll
                for (int i = 0; i < 4; i++) v[i] = t < ln[i] ? G.adjL[st[i] + t] : 0xFFFFFFFFu;
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (t < ln[i]) fn(j0 + q0 + i * ng + gi, v[i]);
            }
        }
        wsync();
    }
    return total;
}

// Local index of rank v among the marked ranks: the block's prefix (four
// words to a block) and the marks below v in the block.
__device__ __forceinline__ uint32_t marked_below(const u64* mark, const uint32_t* pre, uint32_t v) {
    const uint32_t b = v >> 8, wi = (v >> 6) & 3;
    const u64* m = mark + (size_t)b * 4;
    uint32_t c = pre[b];
#pragma unroll
    for (uint32_t i = 0; i < 4; i++)
        c += __popcll(m[i] & (i < wi ? ~0ull : i == wi ? (1ull << (v & 63)) - 1 : 0ull));
    return c;
}

// How a task whose first level lies in wide frame F starts.
__device__ __forceinline__ int place_start(const Wide& S, u64* F, uint32_t np, uint32_t nx,
                                           uint32_t nq, uint32_t* list, TileSrc& src) {
    const int r = place_level(S, F, np, nx, nq, list, src);
    return r == kToTile ? kTreeTile : r == kEvent ? kTreeDone : kTreeWide;
}

// Localise root x and process the root node. The distance-two candidates are
// marked in a bitmap over the ranks, which numbers them in rank order (P is
// the first kx of them); their rows over N(x) are built by word-wide ORs; the
// root node is decided on the rows; Q is reduced, and P loses what the kept Q
// rows contain. The bitmap, its prefix and the rows lie in LDS when they fit
// (the rows at its end, where the tile's stack does not reach), else in the
// worker's mark and rank tables and at the arena's tail. A problem that fits
// the tile is gathered from these rows as they are; any other is laid out by
// word for the wide tier.
template <bool EMIT>
__device__ __forceinline__ int build_tree_root(const KParams& kp, const DevGraph& G, uint32_t x,
                                               u64* arena, u64* lds, u64* gmark, uint32_t* cpos,
                                               Walk& wk, Wide& S, TileSrc& src, TileMem& M,
                                               uint32_t* list, u64& build) {
    const Here lane;
    const uint32_t s0 = uni32(G.offR[x]);
    const uint32_t d = uni32(G.offR[x + 1] - s0);
    const uint32_t* Nx = G.adjR + s0;
    if (d == 0) return kTreeDone;
    const uint32_t W = (d + 63) >> 6;
    LdsSpan sp = lds_span(kp, lds);
    const uint32_t nblk = (uni32(G.nR) + 255) >> 8, nwords = nblk * 4;
    u64* mark = gmark;
    uint32_t* pre = cpos;
    const bool lds_mark = sp.begin + nwords + (nblk + 1) / 2 <= sp.end;
    if (lds_mark) {
        mark = sp.begin;
        pre = (uint32_t*)(sp.begin + nwords);
    }
    for (uint32_t w = lane(); w < nwords; w += 64) mark[w] = 0;
    sync_own();
    const uint32_t T = for_entries(G, Nx, d, list, [&](uint32_t, uint32_t v) {
        if (v != x) own_or(&mark[v >> 6], 1ull << (v & 63));
    });
    build += T;
    sync_own();
    uint32_t nc = 0;
    for (uint32_t b0 = 0; b0 < nblk; b0 += 64) {
        const uint32_t b = b0 + lane();
        uint32_t c = 0;
        if (b < nblk)
            for (uint32_t i = 0; i < 4; i++) c += __popcll(mark[4 * b + i]);
        const uint32_t inc = scan_add32(c);
        if (b < nblk) pre[b] = nc + inc - c;
        nc += rdlane32(inc, 63);
    }
    sync_own();
    const uint32_t kx = uni32(marked_below(mark, pre, x));

    // arena: P's ranks, P and Q positions, then the problem; rows at the tail
    size_t off = kArenaHdr;
    uint32_t* cand = (uint32_t*)(arena + off);
    off += (kx + 1) / 2;
    uint32_t* kidx = (uint32_t*)(arena + off);
    off += nc + 1;  // P and Q positions, and the sorted Q
    const size_t row_words = (size_t)nc * W;
    const uint32_t lds_low = max(lds_mark ? nwords + (nblk + 1) / 2 : 0u,
                                 (W > 1 ? kNarrowWords : 0) + 64 * W);
    const bool lds_rows = row_words + lds_low <= (size_t)(sp.end - sp.begin);
    const size_t tail_words = lds_rows ? 0 : row_words;
    // roots that list mode suits (see build_root) and those whose rows do
    // not fit the arena are left to a later pass
    if (off + max(tail_words, (size_t)64 * W) > kp.arena_words ||
        (!kp.serve && kp.sparse_ratio && kx <= kSparseMaxP &&
         row_words + (size_t)d * ((nc + 63) >> 6) > (size_t)kp.sparse_ratio * T))
        return kTreeOverflow;
    u64* trow = lds_rows ? sp.end - row_words : arena + (kp.arena_words - row_words);
    if (lds_rows) sp.end = trow;
    for (size_t i = lane(); i < row_words; i += 64) trow[i] = 0;
    sync_own();
    for_entries(G, Nx, d, list, [&](uint32_t j, uint32_t v) {
        if (v != x)
            own_or(&trow[(size_t)marked_below(mark, pre, v) * W + (j >> 6)], 1ull << (j & 63));
    });
    for (uint32_t w = lane(); w <= (x >> 6); w += 64) {
        u64 m = mark[w];
        if (w == (x >> 6)) m &= (1ull << (x & 63)) - 1;
        uint32_t k = m ? marked_below(mark, pre, w * 64) : 0;
        while (m) {
            cand[k++] = w * 64 + __builtin_ctzll(m);
            m &= m - 1;
        }
    }
    sync_own();

    // root node: L' = N(x); a full Q row makes it non-maximal, full P rows
    // are absorbed, the other P candidates go to the head of kidx
    bool nonmax = false;
    uint32_t ab = 0, np = 0;
    u64 abh = 0;
    const uint32_t kq = kx & ~63u;  // Q first: most roots that fail, fail there
    for (uint32_t pass = 0; pass < 2 && !nonmax; pass++)
        for (uint32_t c0 = pass ? 0 : kq; c0 < (pass ? kx : nc) && !nonmax; c0 += 64) {
            const uint32_t k = c0 + lane();
            bool full = false;
            if (pass ? k < kx : k < nc && k >= kx) {
                uint32_t c = 0;
                for (uint32_t w = 0; w < W; w++) c += __popcll(trow[(size_t)k * W + w]);
                full = c == d;
            }
            if (!pass) {
                nonmax = __ballot(full) != 0;
                continue;
            }
            if (full) {
                ab++;
                abh += G.hR[cand[k]];
            }
            const u64 m = __ballot(k < kx && !full);
            if ((m >> lane()) & 1) kidx[np + __popcll(m & lanemask_lt())] = k;
            np += __popcll(m);
        }
    if (nonmax) {
        wk.nodes++;
        return kTreeDone;
    }
    ab = red_add32(ab);
    abh = red_add64(abh);
    const u64 sr = uni64(G.hR[x]) + abh;
    const uint32_t nr = 1 + ab;
    uint32_t nq = np ? nc - kx : 0;
    sync_own();
    for (uint32_t i = lane(); i < nq; i += 64) kidx[np + i] = kx + i;
    sync_own();
    if (np && nq && (np > kTileP || nq > kTileQ || W > kTileW)) {
        // reduce Q, largest rows first (a counting sort by size), then prune
        // P. The scratch goes to the LDS that the bitmap held, or to the
        // arena where the problem will be laid out.
        const auto row = [&](uint32_t k, uint32_t w) { return trow[(size_t)k * W + w]; };
        const size_t cols = (size_t)64 * W, histw = cols / 2 + 1, room = sp.end - sp.begin;
        u64* scr = sp.begin;
        uint32_t kw = room > histw ? (uint32_t)min((room - histw) / cols, (size_t)16) : 0;
        if (kw < kWideKw && off + histw + 16 * cols + tail_words <= kp.arena_words) {
            scr = arena + off;
            kw = 16;
        }
        uint32_t* ord = kidx + np + nq;  // room: see lists
        if (kw) {
            uint32_t* hist = (uint32_t*)scr;
            for (uint32_t i = lane(); i < 2 * histw; i += 64) hist[i] = 0;
            sync_own();
            auto size_of = [&](uint32_t k) {
                uint32_t c = 0;
                for (uint32_t w = 0; w < W; w++) c += __popcll(row(k, w));
                return c;
            };
            for (uint32_t i = lane(); i < nq; i += 64) own_add(&hist[cols - size_of(kx + i)], 1u);
            sync_own();
            uint32_t carry = 0;
            for (uint32_t b = 0; b < cols; b += 64) {
                const uint32_t c = hist[b + lane()];
                const uint32_t inc = scan_add32(c);
                hist[b + lane()] = carry + inc - c;
                carry += rdlane32(inc, 63);
            }
            sync_own();
            for (uint32_t i = lane(); i < nq; i += 64)
                ord[own_add(&hist[cols - size_of(kx + i)], 1u)] = kx + i;
            sync_own();
            uint32_t nk;
            nq = reduce_rows(row, W, ord, nq, scr + histw, kw, nk);
            np = prune_rows(row, W, kidx, np, scr + histw, kw, nk);
            for (uint32_t i0 = 0; i0 < nq; i0 += 64) {
                const uint32_t q = i0 + lane() < nq ? ord[i0 + lane()] : 0;
                wsync();
                if (i0 + lane() < nq) kidx[np + i0 + lane()] = q;
            }
            sync_own();
        }
    }
    const bool direct = np && np <= kTileP && nq <= kTileQ && W <= kTileW;
    u64* hl = arena + off;  // a leaf root's terms, for materialisation
    size_t end = off + (size_t)64 * W;
    if (direct) {
        end = layout_tile(arena, sp, off, W, M, hl);
    } else if (np) {
        if (!layout_wide(kp, S, arena, sp, off, W, np + nq, min(np, d), M)) return kTreeOverflow;
        hl = S.hl;
        end = S.end;
    }
    if (end + tail_words > kp.arena_words) return kTreeOverflow;
    // the root biclique (N(x), {x} u absorbed)
    wk.nodes++;
    wk.steps++;
    u64 sl = 0;
    for (uint32_t j = lane(); j < 64 * W; j += 64) {
        const u64 t = j < d ? G.hL[Nx[j]] : 0;
        hl[j] = t;
        sl += t;
    }
    sl = red_add64(sl);
    wk.cnt++;
    const u64 h = wk.r_is_u ? biclique_hash(sr, sl, nr, d) : biclique_hash(sl, sr, d, nr);
    if (lane() == 0) wk.hs += h;
    sync_own();
    if (EMIT && kp.emit_pos) {
        uint64_t* o = emit_head(kp, d, nr, sr);
        if (o)
            for (uint32_t j = lane(); j < d; j += 64) o[j] = hl[j];
    }
    if (!np) return kTreeDone;

    if (direct) {
        for (uint32_t i = lane(); i < np; i += 64) list[i] = kidx[i];
        for (uint32_t i = lane(); i < nq; i += 64) list[kTileP + i] = kidx[np + i];
        wsync();
        src.rows = trow;
        src.ks = W;
        src.ws = 1;
        src.hc = (const u64*)G.hR;
        src.hl = hl;
        src.L = nullptr;
        src.wmap = 0x0706050403020100ull;
        src.W = W;
        src.P = low_bits(np);
        src.X = src.D = 0;
        src.nq = nq;
        src.sr = sr;
        src.nr = nr;
        src.cand = cand;
        return kTreeTile;
    }
    // by word, P then Q; then level 1
    for (uint32_t k = lane(); k < S.ncs; k += 64) {
        const uint32_t o = k < S.nc ? kidx[k] : 0;
        if (k < np) S.hc[k] = G.hR[cand[o]];
        for (uint32_t w = 0; w < W; w++)
            S.rows[(size_t)w * S.ncs + k] = k < S.nc ? trow[(size_t)o * W + w] : 0;
    }
    u64* F1 = S.frame(1);
    u64* L1 = F1 + kFrameHdr;
    u64* P1 = L1 + W;
    for (uint32_t w = lane(); w < W; w += 64)
        L1[w] = (w == W - 1 && (d & 63)) ? low_bits(d & 63) : ~0ull;
    for (uint32_t b = lane(); b < S.Wc; b += 64) {
        const u64 pm = b * 64 >= np ? 0 : low_bits(np - b * 64);
        const u64 all = low_bits(S.nc - b * 64);
        P1[b] = pm;
        P1[S.Wc + b] = 0;
        P1[2 * S.Wc + b] = all & ~pm;
    }
    if (lane() == 0) {
        F1[1] = sr;
        F1[2] = nr;
    }
    sync_own();
    return place_start(S, F1, np, 0, nq, list, src);
}

// Copy a donated level out of the worker's slot: a tile as it is, or a wide
// problem, which is tried as a tile once more.
__device__ __forceinline__ int load_tree_slot(const KParams& kp, u64* slot, u64* arena,
                                              u64* lds, Wide& S, TileSrc& src, TileMem& M,
                                              uint32_t* list) {
    const Here lane;
    const u64 s1 = uni64(ld_rlx(slot + 1)), s2 = uni64(ld_rlx(slot + 2));
    const uint32_t W = (uint32_t)s1, np = (uint32_t)(s1 >> 32);
    const uint32_t nx = (uint32_t)s2, nq = (uint32_t)(s2 >> 32);
    const uint32_t npx = np + nx, n = npx + nq;
    u64* hl0 = slot + kSlotHeaderWords;
    u64* hc0 = hl0 + (size_t)64 * W;
    u64* rows0 = hc0 + npx;
    if (npx <= kTileP && nq <= kTileQ && W <= kTileW) {
        u64* hl;
        const size_t off = layout_tile(arena, lds_span(kp, lds), kArenaHdr, W, M, hl);
        u64* rows = arena + off;
        u64* hc = rows + (size_t)W * n;
        if (off + (size_t)W * n + npx > kp.arena_words) return kTreeOverflow;
        for (uint32_t i = lane(); i < 64 * W; i += 64) hl[i] = ld_rlx(hl0 + i);
        for (uint32_t i = lane(); i < W * n; i += 64) rows[i] = ld_rlx(rows0 + i);
        if (lane() < npx) hc[lane()] = ld_rlx(hc0 + lane());
        if (lane() < npx) list[lane()] = lane();
        for (uint32_t i = lane(); i < nq; i += 64) list[kTileP + i] = npx + i;
        wsync();
        src.rows = rows;
        src.ks = 1;
        src.ws = n;
        src.hc = hc;
        src.cand = nullptr;
        src.hl = hl;
        src.L = nullptr;
        src.wmap = 0x0706050403020100ull;
        src.W = W;
        src.P = low_bits(np);
        src.X = low_bits(npx) & ~src.P;
        src.D = 0;
        src.nq = nq;
        src.sr = uni64(ld_rlx(slot + 3));
        src.nr = (uint32_t)uni64(ld_rlx(slot + 4));
        return kTreeTile;
    }
    if (!layout_wide(kp, S, arena, lds_span(kp, lds), kArenaHdr, W, n, min(npx, 64 * W), M)) return kTreeOverflow;
    for (uint32_t i = lane(); i < 64 * W; i += 64) S.hl[i] = ld_rlx(hl0 + i);
    for (uint32_t k = lane(); k < S.ncs; k += 64) {
        if (k < n) S.hc[k] = k < npx ? ld_rlx(hc0 + k) : 0;
        for (uint32_t w = 0; w < W; w++)
            S.rows[(size_t)w * S.ncs + k] = k < n ? ld_rlx(rows0 + (size_t)w * n + k) : 0;
    }
    u64* F1 = S.frame(1);
    u64* L1 = F1 + kFrameHdr;
    u64* P1 = L1 + W;
    for (uint32_t w = lane(); w < W; w += 64) L1[w] = ~0ull;
    for (uint32_t b = lane(); b < S.Wc; b += 64) {
        const uint32_t o = b * 64;
        const u64 pm = o >= np ? 0 : low_bits(np - o), px = o >= npx ? 0 : low_bits(npx - o);
        P1[b] = pm;
        P1[S.Wc + b] = px & ~pm;
        P1[2 * S.Wc + b] = low_bits(n - o) & ~px;
    }
    if (lane() == 0) {
        F1[1] = ld_rlx(slot + 3);
        F1[2] = ld_rlx(slot + 4);
    }
    sync_own();
    return place_start(S, F1, np, nx, nq, list, src);
}

// Run a task from its start to its end: the wide walk, the tile it leads to,
// and the narrow tile that one leads to, whichever is current.
template <bool SEC, bool EMIT>
__device__ __forceinline__ void run_tree(const KParams& kp, Walk& wk, int start, const Wide& S,
                                         TileSrc& src, const TileMem& M, uint32_t* list,
                                         Sec& sec) {
    enum { kWideWalk, kTile, kNarrow };
    const bool wide = uni1(start == kTreeWide);
    uint32_t k = wide ? 1 : 0, depth = 0, ndepth = 0;
    int at = wide ? kWideWalk : kTile;
    bool resume = false;  // of a tile, or of level k after its x
    TileSrc nsrc{};
    for (;;) {
        int r;
        at = (int)uni32(at);
        k = uni32(k);
        depth = uni32(depth);
        ndepth = uni32(ndepth);
        resume = uni1(resume);
        make_uniform(wk);
        make_uniform(src);
        make_uniform(nsrc);
        const uint32_t cls = at == kTile ? tile_class(uni32(src.W)) : at == kNarrow ? 1 : 0;
        if (cls == 0) {
            r = wide_walk<SEC, EMIT>(kp, wk, S, k, resume, list, src, sec);
        } else if (cls == 1) {
            const bool n = at == kNarrow;
            TileSrc none;
            r = tile_search<1, SEC, EMIT>(
                kp, wk, n ? nsrc : src, n ? (uint32_t*)(nsrc.rows + kTileP + kTileQ) : list,
                n ? M.nsave : M.save, n ? ndepth : depth, resume, nullptr, none, sec);
        } else if (cls == 2) {
            r = tile_search<2, SEC, EMIT>(kp, wk, src, list, M.save, depth, resume, M.nar, nsrc, sec);
        } else if (cls == 4) {
            r = tile_search<4, SEC, EMIT>(kp, wk, src, list, M.save, depth, resume, M.nar, nsrc, sec);
        } else {
            r = tile_search<8, SEC, EMIT>(kp, wk, src, list, M.save, depth, resume, M.nar, nsrc, sec);
        }
        r = (int)uni32(r);
        make_uniform(wk);
        if (r == kEvent) {
            if (wk.stop) return;
            if (SEC) sec.mark(kSecOther);
            // half of the shallowest level with work left, then the rest of it
            bool rest = false;
            for (bool gave = true; wk.give && gave; wk.give--, rest = !rest) {
                // the levels above the current tier have their x in progress
                gave = wide && uni1(donate_wide(kp, S, k, at == kWideWalk, rest, wk));
                if (!gave && at != kWideWalk)
                    gave = uni1(donate_tile(kp, src, list, M.save, depth, k, rest, wk));
                if (!gave && at == kNarrow)
                    gave = uni1(donate_tile(kp, nsrc, (uint32_t*)(nsrc.rows + kTileP + kTileQ),
                                            M.nsave, ndepth, k + depth, rest, wk));
                wk.donated += gave;
                if (SEC) sec.mark(kSecDonate);
            }
            resume = at != kWideWalk;
        } else if (r == kToTile) {
            at = kTile;
            resume = false;
        } else if (r == kToNarrow) {
            at = kNarrow;
            resume = false;
        } else if (at == kNarrow) {
            at = kTile;
            resume = true;
        } else if (at == kTile && wide) {
            at = kWideWalk;
            resume = true;
        } else {
            return;
        }
    }
}

// ---------------------------------------------------------------- workers
// Claim a root of a served request (see serve_claim): an idle worker counts
// as active before it takes a root, so that no other worker leaves meanwhile.
__device__ __forceinline__ bool claim_served(const KParams& kp, uint32_t wid, bool idle, uint32_t& g,
                                             uint32_t& x) {
    const Here lane;
    u64 got = 0, gg = 0, xx = 0;
    if (lane() == 0) {
        ServeCtl* sc = kp.serve;
        const uint32_t pref = wid % kLargeShare == 0 ? 1 : 0;
        for (uint32_t i = 0; i < 2 && !got; i++) {
            const uint32_t ln = pref ^ i;
            for (;;) {
                const u64 la = __hip_atomic_load(&sc->lane_avail[ln], __ATOMIC_ACQUIRE,
                                                 __HIP_MEMORY_SCOPE_AGENT);
                const u64 f = ld_rlx(&sc->lane_first[ln]);
                if (f >= la) break;
                const uint32_t gl = kp.lane_list[(size_t)ln * kp.mail_cap + f];
                const u64 n = kp.graphs[gl].n_roots;
                if (idle) {
                    atomicAdd(kp.tctl, 1ull);
                    __builtin_amdgcn_s_waitcnt(0);
                }
                const u64 c = atomicAdd(&kp.root_cursor[gl], 1ull);
                if (c < n) {
                    got = 1;
                    gg = gl;
                    xx = c;
                    break;
                }
                if (idle) atomicAdd(kp.tctl, ~0ull);
                atomicMax(&sc->lane_first[ln], f + 1);
            }
        }
    }
    g = (uint32_t)uni64(gg);
    x = (uint32_t)uni64(xx);
    got = uni64(got);
    if (got) fence_acq();  // the loader published the graph's arrays with a release
    return got != 0;
}

// What bounds the kernel is one wave's chain of dependent vertex tests, so the
// registers are kept to what two waves per SIMD allow (256). A batch of 256
// graphs: 33.7 ms with 377 registers and one wave, 17.4 with two; bounds of
// three or four waves spill and were slower.
// One worker of the tree engine: roots first, then levels handed over by
// other workers; it leaves when every worker is idle (served kernels: once
// the host has closed the mailbox, too).
template <bool SEC, bool EMIT>
__global__ __launch_bounds__(64, 2) void mbe_tree(KParams kp) {
    extern __shared__ u64 lds_mem[];
    const uint32_t wid = blockIdx.x;
    u64* arena = (u64*)kp.arena + (size_t)wid * kp.arena_words;
    u64* mark = (u64*)kp.mark + (size_t)wid * kp.mark_words;
    uint32_t* cpos = kp.cpos + (size_t)wid * kp.cpos_len;
    uint32_t* list = (uint32_t*)(lds_mem + kTreeList);
    Sec sec;
    sec.init(SEC && kp.sections, lds_mem);
    Walk wk{};
    u64 roots = 0, ovf = 0, stolen = 0, dropped = 0, build = 0;
    bool roots_left = true, idle = false;
    uint32_t backoff = 1;
    const u64 my_bit = 1ull << (wid & 63);
    if (lane() == 0) atomicAdd(kp.tctl, 1ull);
    wait_mem();
    for (;;) {
        wsync();
        const bool stop = uni1(aborted(kp));
        if (stop) roots_left = false;
        Wide S{};
        TileSrc src{};
        TileMem M{};
        int start = kTreeDone;
        uint32_t x = 0;
        bool got = false, failed = false;
        u64 task = 0;
        wk.cnt = wk.hs = 0;
        wk.stop = false;
        // a task of less than an interval is not worth splitting
        wk.next_event = wk.steps + event_interval(kp);
        if (roots_left) {
            u64 t = 0;
            if (kp.serve) {
                got = claim_served(kp, wid, idle, wk.g, x);
            } else {
                t = uni64(lane() == 0 ? (u64)atomicAdd(kp.cursor, 1ull) : 0);
                got = t < kp.n_tasks;
                roots_left = got;
            }
            if (got && !kp.serve) {
                task = uni64(kp.task_list ? kp.task_list[t]
                                          : kp.task_first + t * (kp.task_step ? kp.task_step : 1));
                wk.g = uni32(find_graph(kp, kp.n_graphs, task));
            }
        }
        bool handed = false;
        if (idle) {
            // a served root was found, or a level may have been handed over;
            // a donor that has cleared the bit owns this worker
            u64 flag = 0;
            if (got) {
                u64 old = 0;
                if (lane() == 0) old = atomicAnd(idle_word(kp, wid >> 6), ~my_bit);
                idle = false;
                if (!(uni64(old) & my_bit)) {
                    // its level comes after this root; the donor counted this
                    // worker as active a second time
                    if (lane() == 0) atomicAdd(kp.tctl, ~0ull);
                    handed = true;
                }
            } else {
                flag = uni64(lane() == 0 ? ld_rlx(flag_of(kp, wid)) : 0);
                if (flag == 2) break;
            }
            if (flag == 1) {
                if (lane() == 0) st_rlx(flag_of(kp, wid), 0ull);
                idle = false;
                if (SEC) sec.mark(kSecWait);
                u64* slot = slot_of(kp, wid);
                const u64 s0 = uni64(ld_rlx(slot));
                wk.g = (uint32_t)s0;
                wk.r_is_u = uni1((s0 >> 32) != 0);
                start = stop ? kTreeOverflow : load_tree_slot(kp, slot, arena, lds_mem, S, src, M, list);
                failed = start < 0;
                dropped += failed && !stop;
                stolen++;
                got = true;
                x = 0xFFFFFFFFu;
                if (SEC) sec.mark(kSecFetch);
            }
        }
        if (got) {
            backoff = 1;
            if (x != 0xFFFFFFFFu) {
                const DevGraph G = kp.graphs[wk.g];
                wk.r_is_u = uni1(G.r_is_u);
                if (kp.serve) task = uni64(G.task_base) + x;
                else x = (uint32_t)(task - uni64(G.task_base));
                if (SEC) sec.mark(kSecOther);
                start = build_tree_root<EMIT>(kp, G, x, arena, lds_mem, mark, cpos, wk, S, src,
                                              M, list, build);
                if (SEC) sec.mark(kSecBuild);
                if (start < 0) {
                    ovf++;
                    if (lane() == 0) {
                        u64 idx = atomicAdd(kp.overflow_count, 1ull);
                        if (idx < kp.overflow_cap) kp.overflow_list[idx] = task;
                    }
                    failed = kp.serve != nullptr;  // served requests have no later pass
                } else {
                    roots++;
                }
            }
            start = (int)uni32(start);
            make_uniform(S);
            make_uniform(M);
            if (start > 0) run_tree<SEC, EMIT>(kp, wk, start, S, src, M, list, sec);
            if (kp.node_budget) watch(kp, wk);
            const u64 hs = red_add64(wk.hs);
            if (lane() == 0 && wk.cnt) {
                atomicAdd(&kp.results[2 * wk.g], wk.cnt);
                atomicAdd(&kp.results[2 * wk.g + 1], hs);
            }
            if (kp.remaining) finish_task(kp, wk.g, failed || aborted(kp));
            if (lane() == 0 && kp.progress) {
                __hip_atomic_store(&kp.progress[2 * wid], roots + ovf, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_SYSTEM);
                __hip_atomic_store(&kp.progress[2 * wid + 1], wk.nodes, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_SYSTEM);
            }
            if (handed) {  // wait for the level that a donor is writing
                while (uni64(lane() == 0 ? ld_rlx(flag_of(kp, wid)) : 0) != 1) __builtin_amdgcn_s_sleep(8);
                idle = true;  // taken on the next turn, as when idle
            }
            continue;
        }
        if (kp.serve && !stop && uni1(serve_load(kp))) {
            backoff = 1;
            continue;
        }
        if (!kp.serve && kp.variant == kNoWS) break;  // nothing is handed over
        if (!idle) {
            wait_mem();  // the slot's words have been read
            idle = true;
            u64 left = 0;
            if (lane() == 0) {
                atomicOr(idle_word(kp, wid >> 6), my_bit);
                left = atomicAdd(kp.tctl, ~0ull) - 1;
            }
            if (!kp.serve && uni64(left) == 0) {  // every worker is idle: all leave
                for (uint32_t w = lane(); w < kp.tworkers; w += 64) st_rlx(flag_of(kp, w), 2ull);
                break;
            }
        } else if (kp.serve) {
            if (uni1(serve_exit(kp, uni64(lane() == 0 ? ld_rlx(kp.tctl) : 0), stop))) break;
        }
        // served workers look at the mailbox ever less often, all of them at
        // the same lines; each watches its own flag all the while, or every
        // level handed over would first lie there for some 50 us
        for (uint32_t i = 0; i < backoff; i++) {
            __builtin_amdgcn_s_sleep(8);
            if (kp.serve && (i & 3) == 3 && uni64(lane() == 0 ? ld_rlx(flag_of(kp, wid)) : 0)) break;
        }
        backoff = min(backoff * 2, kp.serve ? 256u : 4u);
        if (SEC) sec.mark(kSecWait);
    }
    if (SEC) sec.mark(kSecWait);
    // nothing is handed to a worker that has left (under a watchdog others may
    // still be at work)
    if (idle && lane() == 0) atomicAnd(idle_word(kp, wid >> 6), ~my_bit);
    if (lane() == 0) {
        // a worker that found no task has nothing to add
        const u64 st[][2] = {{kStatNodes, wk.nodes},       {kStatRoots, roots},
                             {kStatDonated, wk.donated},   {kStatStolen, stolen},
                             {kStatOverflow, ovf},         {kStatBuildWords, build},
                             {kStatDropped, dropped},      {kStatWords, wk.words}};
#pragma unroll
        for (int i = 0; i < 8; i++)
            if (st[i][1]) atomicAdd(&kp.stats[st[i][0]], st[i][1]);
        if (SEC && kp.sections)
            for (int i = 0; i < kSecCount; i++) atomicAdd(&kp.sections[i], sec.t[i]);
        if (SEC && kp.worker_busy) {
            u64 busy = 0;
            for (int i = 0; i < kSecCount; i++)
                if (i != kSecWait) busy += sec.t[i];
            kp.worker_busy[wid] = busy;
        }
    }
}

