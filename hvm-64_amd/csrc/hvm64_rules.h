// Lane-level reduction rules of the engine (see hvm64_kernels.hip for the
// memory model and the linking protocol).  Compiled for gfx950 by the
// kernels; the memory primitives are the macros below.
#pragma once
#include "hvm64_engine.h"

#if defined(__HIPCC__) || defined(__HIP__)
#define DEV __device__ __forceinline__
#define NOINL __device__ __noinline__
#define HVM_LD(p) __hip_atomic_load((p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
#define HVM_ST(p, v) __hip_atomic_store((p), (v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
#define HVM_XCHG(p, v) __hip_atomic_exchange((p), (v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
#define HVM_FAA(p, v) __hip_atomic_fetch_add((p), (v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
#define HVM_CAS(p, e, v) \
  __hip_atomic_compare_exchange_strong((p), (e), (v), __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
#define HVM_LDS_FAA(p, v) atomicAdd((p), (v))
// True on any lane of the wave that is running.
#define HVM_ANY(c) (__ballot(c) != 0)
#define HVM_BALLOT(c) __ballot(c)
// Bits of a ballot below this lane.
#define HVM_BELOW(m) __builtin_amdgcn_mbcnt_hi((u32)((m) >> 32), __builtin_amdgcn_mbcnt_lo((u32)(m), 0u))
// Pinned host memory (serving rings): system-scope accesses.
#define HVM_LD_SYS(p) __hip_atomic_load((p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM)
#define HVM_ST_SYS(p, v) __hip_atomic_store((p), (v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM)
#define HVM_FENCE_SYS() __builtin_amdgcn_fence(__ATOMIC_RELEASE, "")
// A pointer known to address LDS (ds_* instructions, never flat ones).
typedef __attribute__((address_space(3))) unsigned long long lds_u64;
#define HVM_TO_LDS(p) ((lds_u64 *)(p))
// Retire every outstanding vector memory operation of this wave (vmcnt(0));
// no memory access moves across it.
#define HVM_PUBLISH() asm volatile("s_waitcnt vmcnt(0)" ::: "memory")
// The same wait, placed where nothing is outstanding but loads whose results
// are dead on some paths: it clears the compiler's record of them, which
// would otherwise put a vmcnt wait (that also waits for the stores issued
// since) at the top of every interpreter step.
#define HVM_SETTLE_LOADS() __builtin_amdgcn_s_waitcnt(0x0F70)
#else
#define DEV static inline
#define NOINL static
#define HVM_LD(p) __atomic_load_n((p), __ATOMIC_RELAXED)
#define HVM_ST(p, v) __atomic_store_n((p), (v), __ATOMIC_RELAXED)
#define HVM_XCHG(p, v) __atomic_exchange_n((p), (v), __ATOMIC_RELAXED)
#define HVM_FAA(p, v) __atomic_fetch_add((p), (v), __ATOMIC_RELAXED)
#define HVM_CAS(p, e, v) __atomic_compare_exchange_n((p), (e), (v), false, __ATOMIC_RELAXED, __ATOMIC_RELAXED)
#define HVM_LDS_FAA(p, v) __atomic_fetch_add((p), (v), __ATOMIC_RELAXED)
#define HVM_ANY(c) (c)
#define HVM_BALLOT(c) ((c) ? 1ull : 0ull)
#define HVM_BELOW(m) ((void)(m), 0u)
#define HVM_LD_SYS(p) __atomic_load_n((p), __ATOMIC_RELAXED)
#define HVM_ST_SYS(p, v) __atomic_store_n((p), (v), __ATOMIC_RELAXED)
#define HVM_FENCE_SYS() __atomic_thread_fence(__ATOMIC_RELEASE)
typedef unsigned long long lds_u64;
#define HVM_TO_LDS(p) ((lds_u64 *)(p))
#define HVM_PUBLISH() ((void)0)
#define HVM_SETTLE_LOADS() ((void)0)
#endif

namespace hvm {

// Wave-wide values.  Lane 0's value (of the lanes running) and a lane at a
// wave-uniform index.
#if defined(__HIPCC__) || defined(__HIP__)
DEV u32 uniform(u32 v) { return __builtin_amdgcn_readfirstlane(v); }
DEV u32 lane_at(u32 v, u32 i) { return __builtin_amdgcn_readlane(v, i); }
DEV u32 lane_from(u32 v, u32 i) { return (u32)__builtin_amdgcn_ds_bpermute((int)(i * 4), (int)v); }  // each lane its own i
#else
DEV u32 uniform(u32 v) { return v; }
DEV u32 lane_at(u32 v, u32) { return v; }
DEV u32 lane_from(u32 v, u32) { return v; }
#endif
DEV u64 uniform(u64 v) { return (u64)uniform((u32)v) | (u64)uniform((u32)(v >> 32)) << 32; }
DEV u64 lane_from(u64 v, u32 i) { return (u64)lane_from((u32)v, i) | (u64)lane_from((u32)(v >> 32), i) << 32; }
DEV u64 lane_at(u64 v, u32 i) { return (u64)lane_at((u32)v, i) | (u64)lane_at((u32)(v >> 32), i) << 32; }

static const u32 WAVES_PER_BLOCK = 4;
// Every wave keeps its pending redexes in LDS, in one ring per rule class, so
// that an iteration can run one rule on all 64 lanes.
// Definition calls go to NCALL rings by definition, so that the lanes of a
// call iteration mostly run the same definition in lockstep.
enum RedexClass : u32 { CLS_ANNI = 0, CLS_COMM = 1, CLS_OTHER = 2, CLS_CALL = 3, NCALL = 4, NCLS = CLS_CALL + NCALL };
static const u32 CLS_CAP = 128;    // redexes per anni / comm / other ring (power of two)
static const u32 CALL_CAP = 128;   // redexes per definition-call ring (power of two)
static const u32 RING_PAIRS = CLS_CALL * CLS_CAP + NCALL * CALL_CAP;  // per wave
DEV u32 ring_cap(u32 c) { return c < CLS_CALL ? CLS_CAP : CALL_CAP; }
DEV u32 ring_base(u32 c) { return c < CLS_CALL ? c * CLS_CAP : CLS_CALL * CLS_CAP + (c - CLS_CALL) * CALL_CAP; }
// Slot of a ring in the per-class statistics: anni, comm, call, other.
DEV u32 ring_stat(u32 c) { return c == CLS_OTHER ? 3u : c >= CLS_CALL ? 2u : c; }
static const u32 LDS_SLOTS = 10;   // trg registers per lane kept in LDS
static const u32 LINK_CAP = 6;     // deferred links per lane (LDS)
// A book of at most BOOK_LDS_WORDS words (definition records, instructions,
// label bits, compiled-definition records, templates) is copied into every
// block's LDS by the reduce kernel; of a larger one all but the instructions,
// when that fits.
static const u32 BOOK_LDS_WORDS = 6144;

// ---------------------------------------------------------------------------
// heap access
// ---------------------------------------------------------------------------
// Every heap address is checked: a bad port (an engine bug) is redirected to
// the sink words and recorded, so it can never touch memory outside the heap.
// Records the first error of a launch; `site` says which check found it.
NOINL void report_error(Globals *g, u32 code, u32 site = 0, u64 what = 0) {
  u32 zero = 0;
  if (HVM_CAS(&g->err, &zero, code)) {
    HVM_ST(&g->err_info, site);
    HVM_ST(&g->result, what);  // the offending address or port, for the message
  }
}

DEV u64 *hw(const Params &P, u64 addr) {
  u64 off = addr - HVM_HEAP_OFF;
  if (off >= P.heap_words * 8) {
    report_error(P.g, ERR_BADPTR, BAD_HEAP_ADDR, addr);
    off = DUMP_WORD * 8;
  }
  return P.heap + (off >> 3);
}
DEV u64 ld(const Params &P, u64 addr) { return HVM_LD(hw(P, addr)); }
struct Lane;
// The same check for a lane's accesses (below).
DEV u64 *hw(Lane &L, u64 addr);
// Both words of a node (16-byte aligned) in one agent-scope store.  A store
// ahead of a load delays that load until the store is acknowledged (the
// vector memory counter retires in order), so a node costs one store, not
// two.  The compiler does not count this store in its waits; since the
// counter retires in order, an uncounted store only makes later waits
// longer, never shorter, and a full wait (publish) covers it.
// gfx940 and later need two wait states before a VALU instruction may
// overwrite the data registers of a store wider than 64 bits; the compiler
// does not insert them after inline asm, so the asm ends with `s_nop 1`.
// The memory clobber, here and in the loads below, keeps them in order with
// the relaxed atomics on the same words (a fresh var cell's store and a later
// look at the cell); without it their order would rest on what the compiler
// happens to do.
DEV void st16(u64 *p, u64 w0, u64 w1) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef u64 u64x2 __attribute__((ext_vector_type(2)));
  const u64x2 d = {w0, w1};
  asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" ::"v"(p), "v"(d) : "memory");
#else
  HVM_ST(p, w0);
  HVM_ST(p + 1, w1);
#endif
}
DEV u64 gld(u64 *p) { return HVM_LD(p); }
DEV void gst(u64 *p, u64 v) { HVM_ST(p, v); }
DEV u32 gld32(u32 *p) { return HVM_LD(p); }
DEV void publish() { HVM_PUBLISH(); }

DEV u64 var_port(u64 cell) { return mkport(T_VAR, 0, cell); }
DEV u64 wire_port(u64 cell) { return mkport(T_RED, 0, cell); }
// Endpoints are stored as Var ports; the Red tag only marks trg registers
// that the interpreter may resolve (the reference's Trg::wire, linker.rs:233-281).
// (An endpoint's label is 0: only the tag changes.)
DEV u64 norm_endpoint(u64 p) { return is_endpoint(p) ? (p | T_VAR) : p; }

// ---------------------------------------------------------------------------
// per-lane state
// ---------------------------------------------------------------------------
// Two words side by side in LDS, moved by one 16-byte access.
struct alignas(16) pair {
  u64 a, b;
};

struct Lane {
  const Params *P;
  // allocator: this lane's slice of its wave's ring: the nodes at
  // slice + SLICE_STRIDE*i for i in [0, slice_n)
  u64 slice;
  u32 slice_n;
  u32 apos;            // allocations from the slice since the heap was reset
  u64 *apos_home;      // where apos is kept between launches
  u32 slice_rest;      // allocations left to take from the overflow ring
  u32 ov_left;         // nodes left in the current overflow run
  u32 ov_cur;          // next overflow-ring position of that run
  // (in_lds: the lane has redex rings and a free cache in LDS; a constant in
  // every kernel)
  bool in_lds;
  // free cache: nodes this lane consumed, oldest first: FC[i * 64] for
  // i < fcn
  u64 *FC;
  u32 fcn;
  // arenas: the net of the running task, and the lane's chunk of an arena
  // (nodes [a_pos, a_end) of net a_net; a_net = NO_NET: none)
  // (arenas: allocation from per-net arenas; a kernel that knows its mode
  // sets it to a constant after lane_init, and the compiler drops the other
  // mode's code from the inlined rules)
  bool arenas;
  // (serve: a serving launch, the arenas being request slots; also a
  // compile-time constant in the kernel that serves)
  bool serve;
  // the book and every definition's trg registers are in LDS: a constant in
  // the kernel instantiation for such books, which then carries no global
  // fallback reads nor the per-access branches that choose between the two
  bool lds_all;
  u32 lane_id;         // the lane's index in its wave
  u32 pushed;          // serving: redexes this task put in the wave's rings
  u32 inl_n;           // serving: redexes without a heap port waiting to run in this task
  u64 *inl;            // serving: their storage, SERVE_INL pairs
  u32 cur_net, a_net;
  u32 a_take;          // nodes of the lane's last take from a_net's arena
  // serving: the last task's change to its net's count, whose old value is
  // looked at only at the next loop pass (acct_delta 0: none)
  u32 acct_old, acct_delta, acct_net;
  u64 a_pos, a_end;
  // links deferred by the running task: pair i at PL[i * 64] (LDS)
  pair *PL;
  // trg registers: T[s * 64] (LDS for small definitions, else global)
  u64 *T_lds;
  u64 *T_glb;
  // LDS redex rings, RING_PAIRS pairs (without them redexes go straight to
  // the global ring); per-ring push counters and oldest entries
  pair *bag;
  u32 *bag_top;
  const u32 *bag_bot;
  // the book in LDS (nullptr: read it from global memory): definition
  // records at 0 (4 words each), instructions at book_ins (NO_INS: they are
  // read from global memory), label bits at book_lab, compiled-definition
  // records at book_cdef, templates at book_tmpl
  lds_u64 *book;
  u32 book_ins, book_lab, book_cdef, book_tmpl;
  // counters
  u32 rw[RW_SLOTS];
  // errors of this lane not yet reported (lane_report): the last address
  // outside the heap, bit 0 set (0: none; address 0, which a freed word holds,
  // counts), and the first other error's code and site
  u64 bad;
  u32 err;
};

// A lane records its errors in registers and goes on; the kernel reports
// them when the wave's tasks have ended (lane_report).  Reporting on the
// spot put a function call, and the register moves that a call's convention
// asks for, behind every heap access.
// (Bit 31: an address outside the heap was recorded before it.)
static const u32 ERR_AFTER_BAD = 1u << 31;
DEV void fail(Lane &L, u32 code, u32 site = 0) {
  if (L.err == 0) L.err = code | site << 16 | (L.bad ? ERR_AFTER_BAD : 0);
}

// Out of nodes.  Reported on the spot: the dump cell stands in for the missing
// node, and what this lane and, once it has linked, others find there would
// else be reported first, as an engine bug.  No call: the swap and the stores
// stand at the ends of the allocation paths.
DEV void out_of_nodes(Lane &L, u32 site = 0) {
  u32 zero = 0;
  if (HVM_CAS(&L.P->g->err, &zero, (u32)ERR_OOM)) {
    HVM_ST(&L.P->g->err_info, site);
    HVM_ST(&L.P->g->result, 0ull);
  }
  fail(L, ERR_OOM, site);
}

// The word at engine address `addr`; an address outside the heap is
// recorded and redirected to the dump words.  Selects, no branch: a branch
// that is never taken still costs its exec-mask bookkeeping on every access.
DEV u64 *hw(Lane &L, u64 addr) {
  const Params &P = *L.P;
  const u64 off = addr - HVM_HEAP_OFF;
  const bool out = off >= P.heap_words * 8;
  L.bad = out ? addr | 1 : L.bad;
  return (u64 *)((char *)P.heap + (out ? DUMP_WORD * 8 : off & ~7ull));
}
DEV u64 ld(Lane &L, u64 addr) { return HVM_LD(hw(L, addr)); }
DEV void st(Lane &L, u64 addr, u64 v) { HVM_ST(hw(L, addr), v); }
DEV u64 xchg(Lane &L, u64 addr, u64 v) { return HVM_XCHG(hw(L, addr), v); }

// Reports what the lane recorded (the first report of a launch is kept).
DEV void lane_report(Lane &L) {
  if (L.bad && (L.err == 0 || (L.err & ERR_AFTER_BAD)))
    report_error(L.P->g, ERR_BADPTR, BAD_HEAP_ADDR, L.bad & ~1ull);
  else if (L.err) report_error(L.P->g, L.err & 0xFFFF, L.err >> 16);
  L.bad = 0;
  L.err = 0;
}

// The book is read from LDS (L.book) rather than from global memory.
DEV bool has_book(const Lane &L) { return L.lds_all || L.book != nullptr; }
static const u32 NO_INS = 0xFFFFFFFFu;
// Its instructions too.
DEV bool has_ins(const Lane &L) { return L.lds_all || (L.book != nullptr && L.book_ins != NO_INS); }

DEV u64 dump_addr() { return HVM_HEAP_OFF + DUMP_WORD * 8; }

// Counters of rare events (interpreter shortcuts, allocation misses) go to
// the global counters at once: a per-lane register each would be kept for
// the whole launch.
DEV void count_rare(Lane &L, u32 k, u32 n) {
  if (n) HVM_FAA(&L.P->g->rw[k], (u64)n);
}

// Ring allocation.  Every wave owns a ring (a multiple of 64 nodes) and
// every lane a 1/64 slice of it (every 64th node, so lanes allocating
// together write adjacent nodes).  A slice's position counts its allocations since the heap
// was reset, so on the first lap every slot is known to be free and is taken
// without reading it.  Later laps take the next slot whose two words are
// FREE (frees write FREE in place, from any wave).  When SCAN_MISSES slots in
// a row are taken, the slice is treated as full for the next SLICE_REST
// allocations, which come from the shared overflow ring in runs of OV_RUN
// nodes (one atomic per run; a run in the overflow ring's first lap is free
// without reads, later laps check every slot).
static const u32 SCAN_MISSES = 8;
static const u32 FREE_CACHE = 4;  // nodes a lane keeps for reuse (LDS)
static const u32 SLICE_REST = 256;
static const u32 OV_RUN = 64;
static const u64 SLICE_STRIDE = 64 * 16;  // bytes between a slice's nodes
static_assert(TSLOT_STRIDE == SLICE_STRIDE, "a template's slots are consecutive nodes of a slice");

// One node past the slice's first lap (the free cache is empty).  Ring slots
// are in the heap by construction of the layout (no bounds check).
DEV u64 alloc_lapped(Lane &L) {
  const Params &P = *L.P;
  u64 *const heap = P.heap;
  if (L.slice_rest == 0) {
    for (u32 miss = 0; miss < SCAN_MISSES; miss++) {
      const u64 addr = L.slice + (u64)(L.apos % L.slice_n) * SLICE_STRIDE;
      if (++L.apos >= 1u << 31) {  // keep the position within 32 bits (the allocation count stays exact)
        const u32 whole = L.apos / L.slice_n * L.slice_n - L.slice_n;
        L.apos -= whole;
        count_rare(L, RW_REUSE, whole);
      }
      u64 *w = heap + ((addr - HVM_HEAP_OFF) >> 3);
      const u64 w0 = HVM_LD(w), w1 = HVM_LD(w + 1);
      if (w0 == P_FREE && w1 == P_FREE) return addr;
      count_rare(L, RW_ALLOC_MISS, 1);
    }
    L.slice_rest = SLICE_REST;
  } else {
    L.slice_rest--;
  }
  count_rare(L, RW_OV_ALLOC, 1);
  // Overflow slots are shared: a slot is taken by swapping its first word
  // from FREE (so two lanes whose runs alias the same slot a lap apart can
  // never both take it), and kept only if its second word is FREE too.
  for (u64 miss = 0; miss <= P.ov_nodes; miss++) {
    if (L.ov_left == 0) {
      L.ov_cur = (u32)HVM_FAA(&P.g->ov_pos, (u64)OV_RUN);
      L.ov_left = OV_RUN;
    }
    const u64 node = P.ov_node0 + (L.ov_cur++ & (P.ov_nodes - 1));
    L.ov_left--;
    u64 expect = P_FREE;
    if (HVM_CAS(heap + 2 * node, &expect, P_NONE)) {
      if (HVM_LD(heap + 2 * node + 1) == P_FREE) return HVM_HEAP_OFF + node * 16;
      HVM_ST(heap + 2 * node, P_FREE);  // second word in use: not a free node
    }
  }
  out_of_nodes(L);
  return dump_addr();
}

// Per-net arenas.  Net i's arena is a list of extents: its initial extent
// (arena_len[i] granules from granule arena_base0[i]) and refill extents of
// refill_of(i) granules taken from the shared pool.  One word per net,
// arena_word[i] = base granule of the current extent << 32 | nodes handed
// out of it, serves a lane's request with one atomic add.  The one lane
// whose add crosses the extent's end takes the next extent from the pool,
// names the net in the granule map for its granules and installs it; the
// lanes whose adds land past the end before it is installed take their
// nodes from the overflow region (node-granular, owned by no net).  No lane
// waits for another.  Requests never exceed one granule (the host bounds the
// chunk), so a fresh extent always holds the request that installed it.
static const u32 NO_NET = 0xFFFFFFFFu;
static const u32 ARENA_FIRST = 2;     // nodes taken right after the lane's net changed
static const u32 ARENA_MIN_REFILL = 16;  // granules of the smallest refill extent

struct ArenaChunk {
  u64 pos, end;
  u32 err, site;  // site: OOM_POOL or OOM_OVERFLOW
};

// Granules of a net's refill extents: half its initial extent (len
// granules), within [ARENA_MIN_REFILL, max_refill] (an extent must outlast
// the window in which it is replaced, or most requests would go to the
// overflow region).
DEV u64 refill_of(u64 len, u64 max_refill) {
  const u64 h = len >> 1;
  return h < ARENA_MIN_REFILL ? ARENA_MIN_REFILL : h > max_refill ? max_refill : h;
}

DEV ArenaChunk arena_take(u64 *word, u64 base0, u64 len0, u64 max_refill, u32 gs, u64 *pool_next, u64 pool_end,
                            u32 *gmap, u32 net, u64 *ov_next, u64 ov_end, u32 n) {
  ArenaChunk c;
  c.err = 0;
  c.site = 0;
  const u64 refill = refill_of(len0, max_refill);
  const u64 w = HVM_FAA(word, (u64)n);
  const u64 base = w >> 32, off = w & 0xFFFFFFFFull;
  const u64 len = (base == base0 ? len0 : refill) << gs;
  if (off + n <= len) {
    c.pos = (base << gs) + off;
    c.end = c.pos + n;
    return c;
  }
  if (off <= len) {  // this add crossed the end: the next extent is this lane's to install
    const u64 g = HVM_FAA(pool_next, refill);
    if (g + refill > pool_end) {
      c.err = ERR_OOM;
      c.site = OOM_POOL;
      c.pos = c.end = 0;
      return c;
    }
    for (u64 k = 0; k < refill; k++) HVM_ST(&gmap[g + k], net);
    HVM_ST(word, (g << 32) | n);
    c.pos = g << gs;
    c.end = c.pos + n;
    return c;
  }
  const u64 x = HVM_FAA(ov_next, (u64)n);
  if (x + n > ov_end) {
    c.err = ERR_OOM;
    c.site = OOM_OVERFLOW;
    c.pos = c.end = 0;
    return c;
  }
  c.pos = x;
  c.end = x + n;
  return c;
}

// A port that reaches a heap node or cell (and so names its net).
DEV bool reaches_heap(u64 p) { return ptag(p) >= T_OP || (ptag(p) == T_REF && addr_in_heap(paddr(p))); }

// The net a redex belongs to: the arena of the node (or ExpandDef cell) it
// reaches.  Two nilary ports allocate nothing, and a granule of the pool
// whose owner this lane does not see yet names no net: the lane keeps its
// net.
DEV u32 net_of_port(const Params &P, u64 p, u32 dflt) {
  if (!reaches_heap(p)) return dflt;
  const u64 g = ((paddr(p) - HVM_HEAP_OFF) >> 4) >> P.gran_shift;
  if (g >= P.gmap_len) {
    report_error(P.g, ERR_BADPTR, BAD_NET, p);
    return dflt;
  }
  // (serving: the map never changes, so its words may come from the caches)
  const u32 net = P.serve ? P.gmap[g] : HVM_LD(&P.gmap[g]);
  return net < P.n_nets ? net : dflt;
}

// Serving: a slot's arena is SERVE_SUB sub-arenas of `len` nodes, side by
// side.  Sub-arena k has two words: words[2k] counts the nodes asked of it,
// and never goes back while the slot's net runs; the one request that crosses
// the end leaves what was left behind (first node << 32 | end) in words[2k+1],
// where later requests that fit take from its front.  A request that does not
// fit therefore changes nothing that another request counts on.  (Adding, and
// giving back what did not fit, handed nodes out twice: with two such
// requests under way, one's return brings the count back below the end while
// it still holds the other's, and that one's return then takes away a third
// request's nodes.)
//
// `n` consecutive nodes of a slot, from sub-arena k0 on; the first node's
// place in the slot's arena, or NO_NODES.  One add where there is room; only
// once sub-arena k0 is short are the others looked at, and nothing is refused
// while a sub-arena changes hands.  No wave waits for another beyond the
// store that leaves the rest.
static const u64 NO_NODES = ~0ull;
static const u32 SERVE_ROUNDS = 1u << 16;

DEV u64 serve_add(u64 *words, u64 len, u32 k, u32 n) {
  const u64 used = HVM_FAA(&words[2 * k], (u64)n);
  if (used + n <= len) return k * len + used;
  if (used <= len) HVM_ST(&words[2 * k + 1], used << 32 | len);
  return NO_NODES;
}

DEV u64 serve_take(u64 *words, u64 len, u32 k0, u32 n) {
  u64 at = NO_NODES;
  if (n <= len) at = serve_add(words, len, k0 & (SERVE_SUB - 1), n);
  bool moved = n <= len;
  for (u32 round = 0; at == NO_NODES && moved && round < SERVE_ROUNDS; round++) {
    moved = false;
    for (u32 j = 0; j < SERVE_SUB && at == NO_NODES; j++) {
      const u32 k = (k0 + j) & (SERVE_SUB - 1);
      const u64 used = HVM_LD(&words[2 * k]);
      if (used <= len) {
        if (used + n <= len) {
          at = serve_add(words, len, k, n);
          moved = true;
        }
        continue;
      }
      u64 rest = HVM_LD(&words[2 * k + 1]);
      const u64 pos = rest >> 32, end = rest & 0xFFFFFFFFull;
      if (rest == 0) moved = true;  // on its way
      else if (pos + n <= end) {
        if (HVM_CAS(&words[2 * k + 1], &rest, rest + ((u64)n << 32))) at = k * len + pos;
        moved = true;
      }
    }
  }
  return at;
}

// A slot's sub-arenas as they are before its net: nothing asked of any.
DEV void serve_clear(u64 *words) {
  for (u32 k = 0; k < 2 * SERVE_SUB; k++) HVM_ST(&words[k], 0ull);
}

// Serving: the lanes of a wave that take nodes together and are on the same
// slot take them with one atomic add: exactly `need` nodes each, side by
// side.  (Every serving lane takes at nearly every task, since its slot may
// restart in between; with an atomic per lane the words of a few dozen slots
// were the hottest lines of the launch.)
// The lanes first find their slot's sum and their place in it, without a
// memory access; then the first lane of every slot adds, all of them at once,
// and the others take the result from it.  (Each slot's add waited for before
// the next slot's turn: 128 requests on 32 slots 137 ms; this way 131 ms.)
// Where no sub-arena holds a slot's sum, its lanes take what they need one by
// one: 64 lanes may ask for more than a whole sub-arena (1,024 nodes in the
// smallest slot) together, and what is left of a nearly full slot lies in
// pieces.
DEV void arena_room_serve(Lane &L, u32 need) {
  const Params &P = *L.P;
  u32 lead = 0, before = 0, sum = 0;
  for (u64 todo = HVM_BALLOT(true); todo;) {
    const u32 first = (u32)__builtin_ctzll(todo);
    const bool mine = L.cur_net == lane_at(L.cur_net, first);
    u32 all = 0, below = 0;
    for (u32 b = 0; HVM_ANY(need >> b != 0); b++) {
      const u64 m = HVM_BALLOT(mine && ((need >> b) & 1));
      all += (u32)__builtin_popcountll(m) << b;
      below += HVM_BELOW(m) << b;
    }
    lead = mine ? first : lead;
    sum = mine ? all : sum;
    before = mine ? below : before;
    todo &= ~HVM_BALLOT(mine);
  }
  const u64 len = (u64)P.sub_granules << P.gran_shift;
  u64 w = NO_NODES;
  u64 *const words = &P.arena_word[(u64)L.cur_net * SERVE_WORDS];
#pragma unroll 1
  for (u32 alone = 0; alone < 2 && HVM_ANY(w == NO_NODES); alone++) {
    if (w == NO_NODES && (alone || L.lane_id == lead))
      w = serve_take(words, len, L.rw[RW_POPS] + L.lane_id, alone ? need : sum);
    if (!alone) {
      w = lane_from(w, lead);
      w = w == NO_NODES ? w : w + before;
    }
  }
  const bool fits = w != NO_NODES;
  const u64 slot0 = ((u64)P.serve_first << P.gran_shift) + (u64)L.cur_net * SERVE_SUB * len;
  L.a_pos = fits ? slot0 + w : 0;
  L.a_end = fits ? L.a_pos + need : 0;
  if (!fits) out_of_nodes(L, OOM_POOL);
}

// Makes room for `need` consecutive nodes of the running task's net.  Right
// after the lane's net changed it takes little (a lane's next task is often
// another net's, and the rest of a chunk would stay unused); while it stays
// on one net each take doubles, up to the chunk.
DEV void arena_room(Lane &L, u32 need) {
  if (L.serve) {
    arena_room_serve(L, need);
    return;
  }
  const bool same = L.a_net == L.cur_net;
  if (same && L.a_pos + need <= L.a_end) return;
  const Params &P = *L.P;
  u32 t = same ? L.a_take * 2 : ARENA_FIRST;
  t = t > P.arena_chunk ? P.arena_chunk : t;
  L.a_take = t;
  const u32 net = L.cur_net;
  const ArenaChunk c = arena_take(&P.arena_word[net], P.arena_base0[net], P.arena_len[net], P.refill_granules,
                                  P.gran_shift, P.pool_next, P.pool_end, P.gmap, net, P.ov_next, P.ov_end,
                                  need > t ? need : t);
  L.a_net = L.cur_net;
  L.a_pos = c.pos;
  L.a_end = c.end;
  if (c.err) {
    out_of_nodes(L, c.site);
    L.a_end = L.a_pos;  // every later allocation reports again
  }
}

// `need` (at most N) nodes, each on its own: out[0 .. need).  From the free
// cache, newest first, then from the slice's first lap; both are address
// arithmetic without a branch.  Past the first lap one by one, in a loop, so
// that the scan is in the code once per call site.
template <u32 N>
DEV void alloc_nodes(Lane &L, u32 need, u64 (&out)[N]) {
  if (L.arenas) {
    // the last nodes of a chunk that holds fewer than `need`, then the next
    // chunk's (a serving lane has no chunk: it takes what it needs)
    u32 rest = 0;
    const u64 last = L.a_pos;
    if (!L.serve) {
      const u64 left = L.a_net == L.cur_net ? L.a_end - L.a_pos : 0;
      rest = left < need ? (u32)left : 0;
      L.a_pos += rest;
    }
    const u32 more = need - rest;
    if (more) arena_room(L, more);
    const bool ok = L.a_pos + more <= L.a_end;
#pragma unroll
    for (u32 j = 0; j < N; j++)
      out[j] = j < rest || ok ? HVM_HEAP_OFF + ((j < rest ? last : L.a_pos - rest) + j) * 16 : dump_addr();
    L.a_pos += ok ? more : 0;
    return;
  }
  const u32 used = L.in_lds ? (L.fcn < need ? L.fcn : need) : 0;
  const u32 apos = L.apos + need - used;
  if (need > used && apos > L.slice_n) {
    for (u32 j = 0; j < need; j++) {
      u64 v;
      if (L.in_lds && L.fcn) {
        v = L.FC[--L.fcn * 64];
        L.rw[RW_REUSE]++;
      } else if (L.apos < L.slice_n) {
        v = L.slice + (u64)L.apos++ * SLICE_STRIDE;
      } else {
        v = alloc_lapped(L);
      }
#pragma unroll
      for (u32 k = 0; k < N; k++) out[k] = k == j ? v : out[k];
    }
    return;
  }
#pragma unroll
  for (u32 j = 0; j < N; j++) {
    const u64 fresh = L.slice + (u64)(L.apos + j - used) * SLICE_STRIDE;
    if (L.in_lds && j < FREE_CACHE) {
      const u64 cached = L.FC[(j < used ? L.fcn - 1 - j : 0) * 64];
      out[j] = j < used ? cached : fresh;
    } else {
      out[j] = fresh;
    }
  }
  L.apos = apos;
  if (L.in_lds) L.fcn -= used;
  L.rw[RW_REUSE] += used;
}

DEV u64 alloc_node(Lane &L) {
  u64 n[1];
  alloc_nodes(L, 1, n);
  return n[0];
}

// Two node words.  Agent-scope stores: a plain store may stay in the
// writing XCD's L2, where lanes on the other XCDs would not see it.
DEV void st2(Lane &L, u64 addr, u64 w0, u64 w1) { st16(hw(L, addr), w0, w1); }

// Both words of a published node (immutable until taken) in one 16-byte
// agent-scope load; two nodes: two loads and one wait.  The compiler does not
// track these loads, so the asm waits for them itself.
DEV void ld16x2(const u64 *p, const u64 *q, u64 &p0, u64 &p1, u64 &q0, u64 &q1) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef u64 u64x2 __attribute__((ext_vector_type(2)));
  u64x2 dp, dq;
  asm volatile("global_load_dwordx4 %0, %2, off sc1\n\tglobal_load_dwordx4 %1, %3, off sc1\n\ts_waitcnt vmcnt(0)"
               : "=&v"(dp), "=&v"(dq)
               : "v"(p), "v"(q)
               : "memory");
  p0 = dp.x;
  p1 = dp.y;
  q0 = dq.x;
  q1 = dq.y;
#else
  p0 = HVM_LD(p);
  p1 = HVM_LD(p + 1);
  q0 = HVM_LD(q);
  q1 = HVM_LD(q + 1);
#endif
}
DEV void ld16(const u64 *p, u64 &p0, u64 &p1) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef u64 u64x2 __attribute__((ext_vector_type(2)));
  u64x2 dp;
  asm volatile("global_load_dwordx4 %0, %1, off sc1\n\ts_waitcnt vmcnt(0)" : "=v"(dp) : "v"(p) : "memory");
  p0 = dp.x;
  p1 = dp.y;
#else
  p0 = HVM_LD(p);
  p1 = HVM_LD(p + 1);
#endif
}

// One fresh var cell; the node's other word stays FREE.
DEV u64 alloc_var1(Lane &L) {
  u64 n = alloc_node(L);
  st2(L, n, P_NONE, P_FREE);
  return n;
}

// Two words of a node this lane has just allocated (always in the heap).
DEV void st2_new(const Params &P, u64 addr, u64 w0, u64 w1) {
  st16(P.heap + ((addr - HVM_HEAP_OFF) >> 3), w0, w1);
}
// The same for a node's aux ports.
DEV void node_new(const Params &P, u64 addr, u64 p1, u64 p2) {
  st2_new(P, addr, norm_endpoint(p1), norm_endpoint(p2));
}

// A node this lane has consumed (its words already read).  Per-net arenas
// never reuse a node, so it is simply dropped; with the allocation rings it
// goes to the lane's free cache, from which the lane's next allocations are
// taken, or, when the cache is full, it is marked FREE for the ring scan.  A
// cached node is never marked: the scan skips it as live until it is reused.
DEV void drop_node(Lane &L, u64 *w) {
  if (L.arenas) return;
  const u64 off = (u64)(w - L.P->heap);
  if (L.in_lds && L.fcn < FREE_CACHE && off >= RESERVED_WORDS) {
    L.FC[L.fcn++ * 64] = HVM_HEAP_OFF + off * 8;
    return;
  }
  st16(w, P_FREE, P_FREE);
}

// Consume a binary node: read both aux words, then drop the node.
DEV void take(Lane &L, u64 p, u64 &x, u64 &y) {
  u64 a = paddr(p);
  u64 *w = hw(L, a & ~15ull);
  ld16(w, x, y);
  drop_node(L, w);
}

// take() of two nodes, their loads in flight together.
DEV void take2(Lane &L, u64 p, u64 q, u64 &p1, u64 &p2, u64 &q1, u64 &q2) {
  u64 *wp = hw(L, paddr(p) & ~15ull), *wq = hw(L, paddr(q) & ~15ull);
  ld16x2(wp, wq, p1, p2, q1, q2);
  drop_node(L, wp);
  drop_node(L, wq);
}

// A var cell both of whose sides have arrived: marked FREE for the ring scan
// (arenas never reuse it).
DEV void free_cell(Lane &L, u64 c) {
  if (!L.arenas) st(L, c, P_FREE);
}

// ---------------------------------------------------------------------------
// redexes
// ---------------------------------------------------------------------------
// Push one redex to the global ring (retires the lane's stores first).
DEV void push_global(u64 *queue, u64 qmask, Globals *g, u64 a, u64 b) {
  publish();
  u64 pos = HVM_FAA(&g->q_tail, 1ull);
  u64 *s = queue + (pos & qmask) * 2;
  gst(s, a);
  gst(s + 1, b);
  publish();
  u64 old = HVM_FAA(&g->S, 1ull << 32);
  if ((old >> 32) + 1 > (qmask + 1) / 2) report_error(g, ERR_QUEUE);
}

DEV void global_push1(Lane &L, u64 a, u64 b) {
  // serving: a redex in the global ring can be taken and finished by another
  // wave before this task ends, so it is counted for its net at once
  if (L.serve) HVM_FAA(&L.P->pending[(u64)L.cur_net * PENDING_STRIDE], 1u);
  push_global(L.P->queue, L.P->qmask, L.P->g, a, b);
}

// The rule a redex will take, grouped: the arms of interact.rs:6-44 that run
// anni2, comm22, a definition call (a non-ERA Ref), and everything else.
// Calls go to the ring of the definition's group (DefRec::group, by
// instruction count), read from the book in LDS; a wave runs one call ring
// per iteration and waits for its longest definition, so definitions of
// similar length share a ring.  Without the LDS book: definition modulo NCALL.
// An ExpandDef (a Ref to a heap cell) goes to the first.
// No branches: the redexes of a wave's lanes are of all kinds.
DEV u32 redex_class(u64 a, u64 b, const lds_u64 *book, bool lds, u32 ndefs) {
  const u32 at = ptag(a), bt = ptag(b), la = plab(a), lb = plab(b);
  const bool aref = (at == T_REF) & (a != P_ERA), bref = (bt == T_REF) & (b != P_ERA);
  const u64 r = aref ? a : b;
  const bool call = aref | bref, heap = addr_in_heap(paddr(r));
  const u32 di = def_index((u64)(u32)paddr(r));
  u32 g;
  if (lds) g = (u32)book[4 * ((call & !heap & (di < ndefs)) ? di : 0u) + 3];
  else g = di;
  g = heap ? 0u : g % NCALL;
  const bool same = (at == bt) & (at >= T_OP), ctrs = same & (at == T_CTR);
  const bool anni = same & (!ctrs | (la == lb));
  const bool op_ctr = (at ^ bt) == (T_CTR ^ T_OP) && (at == T_CTR || bt == T_CTR);
  const bool swi_ctr = (at ^ bt) == (T_CTR ^ T_SWI) && (at == T_CTR || bt == T_CTR);
  const bool comm = (ctrs & (la != lb)) | op_ctr | (swi_ctr & ((at == T_CTR ? la : lb) != 0));
  return call ? CLS_CALL + g : anni ? CLS_ANNI : comm ? CLS_COMM : CLS_OTHER;
}

// linker.rs:70-85: skippable pairs count as an erasure and are dropped.
DEV void redux(Lane &L, u64 a, u64 b) {
  const bool skip = is_skippable(a) & is_skippable(b);
  L.rw[RW_ERAS] += skip;
  if (skip) return;
  if (L.serve) {
    if (!reaches_heap(a) && !reaches_heap(b)) {  // no net to count it for: run it in this task
      if (L.inl_n >= SERVE_INL) {
        fail(L, ERR_QUEUE);
        return;
      }
      L.inl[2 * L.inl_n] = a;
      L.inl[2 * L.inl_n + 1] = b;
      L.inl_n++;
      return;
    }
  }
  if (L.in_lds) {
    const u32 c = redex_class(a, b, L.book, has_book(L), L.P->ndefs);
    const u32 idx = HVM_LDS_FAA(&L.bag_top[c], 1u);
    if (idx - L.bag_bot[c] < ring_cap(c)) {
      L.bag[ring_base(c) + (idx & (ring_cap(c) - 1))] = pair{a, b};
      if (L.serve) L.pushed++;  // counted when the task ends (a full ring's redex is counted at once, below)
      return;
    }
  }
  global_push1(L, a, b);
}

// Linking.  A link step either meets two principal ports (a redex) or swaps a
// port into the var cell of an endpoint: the first endpoint to arrive leaves
// its port there; the second finds it, frees the cell and links on.
//
// Rules never link directly: they append (a, b) pairs to the lane's link
// list (LDS, LINK_CAP pairs), and its task loop (run_tasks, run_def) links the
// whole list at one place in the code, four swaps in flight at a time.  A
// swap that finds the other endpoint's port frees the cell and appends the
// continuation link to the list.  Every continuation consumes a var cell, so
// a longer run than MAX_CHAIN rounds means a corrupted net.
static const u32 MAX_CHAIN = 1u << 24;

// A lane on a long chain, every CHAIN_LOOK rounds: has the launch failed?
// After an allocation failed the dump cell stands in for the missing node,
// and lanes that meet there hand each other's ports round for as long as
// MAX_CHAIN lets them (a planned batch that ran out of nodes took 30 to 90 s
// to report it; it takes as long as the launch up to there).  What the lane
// recorded itself counts: it is reported when its task ends.  (Reporting it
// here put a function call into every link loop: tree-sum 18 5.49 ms, this
// way 4.67.)
static const u32 CHAIN_LOOK = 256;
DEV bool launch_failed(const Lane &L) { return L.bad != 0 || L.err != 0 || HVM_LD(&L.P->g->err) != 0; }

// Every producer checks the room it needs (interp_run: one link per
// instruction; a rule: at most four, into an empty list).
DEV void push_link(Lane &L, u32 &np, u64 a, u64 b) {
  L.PL[np * 64] = pair{a, b};
  np++;
}

// Links every pair of the list (the list is empty afterwards), four at a
// time: a pair of principal ports is a redex; the others swap their value
// into the endpoint's cell, the (up to) four swaps in flight together.
// The redexes go to the rings while the stores of new nodes retire, in as
// many passes as the lane with the most of them has.
DEV void flush_links(Lane &L, u32 &np) {
  for (u32 round = 0; np > 0; round++) {
    if (round % CHAIN_LOOK == CHAIN_LOOK - 1) {
      if (round > MAX_CHAIN) fail(L, ERR_BADPTR, BAD_CHAIN);
      if (launch_failed(L)) {
        np = 0;
        return;
      }
    }
    const u32 cnt = np < 4 ? np : 4;
    np -= cnt;
    pair p[4];
    u32 red = 0, cell = 0;  // bit j: pair j is a redex / swaps
#pragma unroll
    for (u32 j = 0; j < 4; j++) p[j] = L.PL[(np + j) * 64];  // np + j < LINK_CAP: np > 0 only when cnt == 4
#pragma unroll
    for (u32 j = 0; j < 4; j++) {
      // the endpoint (if there is one) to `a`
      const bool ea = is_endpoint(p[j].a), eb = is_endpoint(p[j].b), in = j < cnt;
      const u64 a = ea ? p[j].a : p[j].b, b = ea ? p[j].b : p[j].a;
      red |= (in & !ea & !eb) ? 1u << j : 0u;
      cell |= (in & (ea | eb)) ? 1u << j : 0u;
      p[j].a = a;
      p[j].b = b;
    }
    while (red) {
      // (a redex's two sides were exchanged above: exchange them back)
      u64 a = p[3].b, b = p[3].a;
#pragma unroll
      for (u32 j = 3; j-- > 0;) {
        const bool here = (red >> j) & 1;
        a = here ? p[j].b : a;
        b = here ? p[j].a : b;
      }
      red &= red - 1;
      redux(L, a, b);
    }
    // (the nodes these ports lead to; the later rounds' are the other side's)
    if (round == 0) publish();
    u64 o[4];
#pragma unroll
    for (u32 j = 0; j < 4; j++) {
      u64 *const w = hw(L, (cell >> j) & 1 ? paddr(p[j].a) : dump_addr());
      o[j] = P_NONE;
      if ((cell >> j) & 1) o[j] = HVM_XCHG(w, norm_endpoint(p[j].b));
      p[j].a = paddr(p[j].a);
    }
#pragma unroll
    for (u32 j = 0; j < 4; j++) {
      if (o[j] != P_NONE) {  // second arrival: free the cell, link on
        free_cell(L, p[j].a);
        push_link(L, np, o[j], p[j].b);
      }
    }
  }
}

// Follow a wire endpoint whose other side has already linked (the
// reference's Trg::target on a wire, linker.rs:278-280), when `go`.  The
// caller owns the endpoint, so once a cell holds a port the cell is ours to
// free.
DEV u64 follow(Lane &L, u64 p, bool go) {
  for (u32 hop = 0; HVM_ANY(go); hop++) {
    if (go) {
      u64 *const w = hw(L, paddr(p));
      const u64 v = HVM_LD(w);
      go = v != P_NONE;
      if (go) {
        if (!L.arenas) HVM_ST(w, P_FREE);
        p = v;
        go = is_endpoint(v);
      }
    }
    if (hop % CHAIN_LOOK == CHAIN_LOOK - 1 && go) {
      if (hop >= MAX_CHAIN) fail(L, ERR_BADPTR, BAD_RESOLVE);
      if (launch_failed(L)) {
        p = P_ERA;
        go = false;
      }
    }
  }
  return p;
}

DEV u64 as_wire(u64 p) { return is_endpoint(p) ? p & ~(u64)T_VAR : p; }

// operate_binary, whose unsigned operations that neither divide nor shift
// are computed here: they are nearly all of a program's, and the general
// function is a call (and a second one inside), with its result by memory.
DEV u32 num_binary(Lane &L, u32 a, u32 op, u32 b) {
  const u32 p = num_u24(a), q = num_u24(b);
  u32 r = op == N_ADD ? p + q : op == N_SUB ? p - q : op == N_SUBS ? q - p : op == N_MUL ? p * q
          : op == N_EQ ? (u32)(p == q) : op == N_NE ? (u32)(p != q) : op == N_LT ? (u32)(p < q)
          : op == N_GT ? (u32)(p > q) : op == N_AND ? (p & q) : op == N_OR ? (p | q) : (p ^ q);
  const u32 fast = 1u << N_ADD | 1u << N_SUB | 1u << N_SUBS | 1u << N_MUL | 1u << N_EQ | 1u << N_NE | 1u << N_LT |
                   1u << N_GT | 1u << N_AND | 1u << N_OR | 1u << N_XOR;
  u32 out = num_new_u24(r);
  if (num_tag(a) != N_U24 || num_tag(b) != N_U24 || op >= N_TAGS || !((fast >> op) & 1)) {
    bool div0 = false;
    out = operate_binary(a, op, b, &div0);
    if (div0) fail(L, ERR_DIV0);
  }
  return out;
}

// ---------------------------------------------------------------------------
// interaction rules (interact.rs); each appends at most 4 links
// ---------------------------------------------------------------------------
DEV void anni2(Lane &L, u32 &np, u64 a, u64 b) {
  L.rw[RW_ANNI]++;
  u64 a1, a2, b1, b2;
  take2(L, a, b, a1, a2, b1, b2);
  push_link(L, np, a1, b1);
  push_link(L, np, a2, b2);
}

DEV void comm22(Lane &L, u32 &np, u64 a, u64 b) {
  const Params &P = *L.P;
  L.rw[RW_COMM]++;
  u64 a1, a2, b1, b2;
  take2(L, a, b, a1, a2, b1, b2);
  u64 n[6];
  alloc_nodes(L, 6, n);
  const u64 v1 = var_port(n[0]), v2 = var_port(n[0] + 8), v3 = var_port(n[1]), v4 = var_port(n[1] + 8);
  st2_new(P, n[0], P_NONE, P_NONE);
  st2_new(P, n[1], P_NONE, P_NONE);
  st2_new(P, n[2], v1, v2);
  st2_new(P, n[3], v3, v4);
  st2_new(P, n[4], v1, v3);
  st2_new(P, n[5], v2, v4);
  push_link(L, np, a1, mkport(ptag(b), plab(b), n[4]));
  push_link(L, np, a2, mkport(ptag(b), plab(b), n[5]));
  push_link(L, np, b1, mkport(ptag(a), plab(a), n[2]));
  push_link(L, np, b2, mkport(ptag(a), plab(a), n[3]));
}

DEV void comm02(Lane &L, u32 &np, u64 a, u64 b) {
  L.rw[RW_COMM]++;
  u64 b1, b2;
  take(L, b, b1, b2);
  push_link(L, np, b1, a);
  push_link(L, np, b2, a);
}

// The redexes of CLS_OTHER (the arms of interact.rs:6-44 that are neither
// an annihilation, a comm22 nor a call): an eraser or a number meeting a
// node.  One node is read, whichever the rule; a number meeting a Ctr, and
// an eraser, are copied onto both aux ports (comm02, interact.rs:162-168).
DEV void rule_other(Lane &L, u32 &np, u64 a, u64 b) {
  const Params &P = *L.P;
  const bool bin_a = is_binary(a);
  const u64 y = bin_a ? a : b, n = bin_a ? b : a;  // the node, the nilary port
  const u32 yt = ptag(y), nt = ptag(n);
  if (!is_binary(y) || is_endpoint(y)) {
    if (is_principal(a) && is_principal(b)) L.rw[RW_ERAS]++;
    else fail(L, ERR_UNIMPL);
    return;
  }
  const bool copy = n == P_ERA || (nt == T_NUM && yt == T_CTR);
  const bool oper = nt == T_NUM && yt == T_OP, swi = nt == T_NUM && yt == T_SWI;
  if (!(copy || oper || swi)) {  // Switch-Ctr(0), Op-Switch: unimplemented!() in the reference
    fail(L, ERR_UNIMPL);
    return;
  }
  u64 y1, y2;
  take(L, y, y1, y2);
  L.rw[RW_COMM] += copy;
  const u32 num = pnum(n);
  // op_num (interact.rs:251-270): the node's operand, when it has arrived
  y1 = follow(L, y1, oper && is_endpoint(y1));
  const bool done = oper && ptag(y1) == T_NUM;  // both operands: the result
  // switch_num (interact.rs:201-223)
  const u32 v = num_tag(num) == N_U24 ? num_u24(num) : 0;
  L.rw[RW_OPER] += done || swi;
  u64 m[2];
  const u32 need = swi ? (v ? 2u : 1u) : oper && !done ? 1u : 0u;
  if (need) alloc_nodes(L, need, m);
  if (copy) {
    push_link(L, np, y1, n);
    push_link(L, np, y2, n);
  } else if (swi) {
    if (v == 0) node_new(P, m[0], y2, P_ERA);
    else {
      node_new(P, m[1], numport(num_new_u24(v - 1)), y2);
      node_new(P, m[0], P_ERA, mkport(T_CTR, 0, m[1]));
    }
    push_link(L, np, y1, mkport(T_CTR, 0, m[0]));
  } else if (done) {
    push_link(L, np, y2, numport(num_binary(L, num, plab(y), pnum(y1))));
  } else {
    node_new(P, m[0], numport(operate_unary(plab(y), num)), y2);
    push_link(L, np, y1, mkport(T_OP, N_SYM, m[0]));
  }
}

// ---------------------------------------------------------------------------
// definitions: call, instruction interpreter, ExpandDef
// ---------------------------------------------------------------------------
// A definition record, from the LDS copy of the book when there is one.
DEV DefRec load_def(const Lane &L, u32 di) {
  if (has_book(L)) {
    DefRec d;
    u64 w0 = L.book[4 * di], w1 = L.book[4 * di + 1], w2 = L.book[4 * di + 2];
    d.ioff = (u32)w0;
    d.ilen = (u32)(w0 >> 32);
    d.nslots = (u32)w1;
    d.labs_off = (u32)(w1 >> 32);
    d.labs_words = (u32)w2;
    d.min_safe = (u32)(w2 >> 32);
    d.group = (u32)L.book[4 * di + 3];
    d.flags = (u32)(L.book[4 * di + 3] >> 32);
    return d;
  }
  return L.P->defs[di];
}

DEV bool labs_has(const Lane &L, const DefRec &d, u32 lab) {  // def.rs:30-37
  if (lab >= d.min_safe) return false;
  u32 idx = lab >> 6;
  if (idx >= d.labs_words) return false;
  u64 w = has_book(L) ? L.book[L.book_lab + d.labs_off + idx] : L.P->labbits[d.labs_off + idx];
  return (w >> (lab & 63)) & 1;
}

// Definition instructions (def.rs:217-289, instruction.rs:110-210).
//
// A definition runs as a sequence of steps with the same shape for every
// instruction kind, so that lanes running different definitions stay
// converged on the memory operations: (1) the trg operand is read and, if it
// is a wire, followed (Trg::target); (2) a CTR meeting a CTR of its own label
// takes that node (the annihilation fast path of do_ctr); (3) the kind's own
// work, which only allocates and stores; (4) the link it asks for, if any,
// is appended to the lane's link list.  The list is linked when it is full
// and when the definition ends.  Deferring a link inside a definition changes
// nothing a later instruction relies on: a trg read in (1) sees either the
// port the link would have parked or the unresolved wire, and both lead to
// the same net with the same rewrite counts (each fast path counts what the
// interaction it replaces counts).
struct Interp {
  u32 ipw;        // next instruction's first word in the instruction array
                  // (of the LDS copy of the book, from L.book_ins)
  lds_u64 *Tl;    // trg registers 0 .. LDS_SLOTS-1 (LDS, stride 64)
  u64 *Tg;        // trg registers LDS_SLOTS .. (global, stride 64)
  u32 left;       // instructions left; 0: no definition running
  bool t_lds;     // every trg register is in LDS (else all in global memory)
  u64 tbase;      // compiled definition: address of its first template slot
  u64 tstride;    // bytes between its slots
};

// Trg register s of this lane: in LDS when every definition of the book
// fits there (a kernel-wide choice, so the branch is uniform), else in the
// lane's global trg area.
DEV u64 t_get(const Interp &I, u32 s) { return I.t_lds ? I.Tl[s * 64] : I.Tg[(u64)s * 64]; }
DEV void t_set(Interp &I, u32 s, u64 v) {
  if (I.t_lds) I.Tl[s * 64] = v;
  else I.Tg[(u64)s * 64] = v;
}

// The instruction kinds other than Ctr that read a trg or make registers
// (instruction.rs:134-203), and the nodes each takes with its operand `p`.
DEV u32 other_need(u32 kind, u64 p) {
  if (kind == I_WIRES) return 1;
  if (kind == I_CONST || p == P_ERA) return 0;
  if (ptag(p) != T_NUM) return 2;
  if (kind == I_OPNUM) return 0;
  if (kind == I_OP) return 2;
  return num_tag(pnum(p)) == N_U24 && num_u24(pnum(p)) != 0 ? 3 : 2;  // I_SWITCH
}

// `m`: the nodes other_need asked for.
DEV void exec_other(Lane &L, Interp &I, u64 w0, u64 w1, u64 p, const u64 (&m)[3], u32 &np) {
  const Params &P = *L.P;
  const u32 kind = (u32)(w0 & 0xFF), lab = (u32)(w1 & 0xFFFF);
  const u32 a = (u32)(w0 >> 16) & 0xFFFF, b = (u32)(w0 >> 32) & 0xFFFF, c = (u32)(w0 >> 48);
  if (kind == I_CONST) {
    t_set(I, a, w1);
    return;
  }
  if (kind == I_WIRES) {
    st2_new(P, m[0], P_NONE, P_NONE);
    t_set(I, a, var_port(m[0]));
    t_set(I, b, wire_port(m[0]));
    t_set(I, c, var_port(m[0] + 8));
    t_set(I, lab, wire_port(m[0] + 8));
    return;
  }
  const bool num = ptag(p) == T_NUM, one = kind == I_OPNUM;  // one: a single result, in c
  const u32 n = pnum(p);
  u64 rb, rc;
  if (p == P_ERA) {
    count_rare(L, kind == I_OP ? SC_OP_ERA : one ? SC_OPNUM_ERA : SC_SWITCH_ERA, 1);
    L.rw[RW_ERAS] += kind == I_SWITCH;
    rb = rc = P_ERA;
  } else if (!num) {  // a node of the instruction's kind, linked to the operand
    const u32 rhs = (u32)(w1 >> 32);
    st2_new(P, m[0], P_NONE, one ? P_FREE : P_NONE);
    st2_new(P, m[1], one ? numport(rhs) : var_port(m[0]), one ? var_port(m[0]) : var_port(m[0] + 8));
    push_link(L, np, p, kind == I_SWITCH ? mkport(T_SWI, 0, m[1]) : mkport(T_OP, lab, m[1]));
    rb = var_port(m[0]);
    rc = one ? var_port(m[0]) : var_port(m[0] + 8);
  } else if (one) {
    L.rw[RW_OPER]++;
    rb = rc = numport(num_binary(L, n, lab, (u32)(w1 >> 32)));
  } else if (kind == I_OP) {
    st2_new(P, m[0], P_NONE, P_FREE);
    st2_new(P, m[1], numport(operate_unary(lab, n)), var_port(m[0]));
    rb = mkport(T_OP, N_SYM, m[1]);
    rc = var_port(m[0]);
  } else {  // I_SWITCH
    L.rw[RW_OPER]++;
    const u32 v = num_tag(n) == N_U24 ? num_u24(n) : 0;
    st2_new(P, m[0], P_NONE, P_FREE);
    if (v == 0) {
      st2_new(P, m[1], var_port(m[0]), P_ERA);
      rb = mkport(T_CTR, 0, m[1]);
    } else {
      st2_new(P, m[1], numport(num_new_u24(v - 1)), var_port(m[0]));
      st2_new(P, m[2], P_ERA, mkport(T_CTR, 0, m[1]));
      rb = mkport(T_CTR, 0, m[2]);
    }
    rc = wire_port(m[0]);
  }
  if (!one) t_set(I, b, rb);
  t_set(I, c, rc);
}

// A template word spec (hvm64_engine.h) as the word it stands for.  Every
// candidate is computed and one is selected, with no branch: the lanes of a
// wave write different templates, and a branch per tag costs each word the
// exec-mask bookkeeping of every arm.  The register read uses register 0
// for words that name none (every definition has it: t0).
DEV u64 tspec(const Interp &I, u64 s) {
  // slot, half and register numbers are small: their arithmetic is 32-bit
  const u32 lo = (u32)s, hi = (u32)(s >> 32), t = lo & 7, k = lo >> 3, var = t == T_VAR;
  const u64 addr = I.tbase + ((k >> var) * (u32)I.tstride + (k & var) * 8);
  // a slot's port; a Var spec's label is 0, so var_port(addr)
  const u64 rel = addr | t | (u64)(hi & 0xFFFF0000u) << 32;
  const bool reg = (t == T_RED) & (hi == 0);  // P_NONE and P_FREE have high words
  const u64 rv = norm_endpoint(t_get(I, reg ? k : 0u));
  const bool lit = ((t == T_REF) | (t == T_NUM) | (t == T_RED)) & !reg;
  return lit ? s : reg ? rv : rel;
}

// I_TEMPLATE: writes every slot of the running definition's template (one
// 16-byte store each), pushes its redexes and adds the counts of the
// instructions the compiler evaluated.  The slots were reserved when the
// call began (interp_begin).
DEV void run_template(Lane &L, Interp &I, u32 off) {
  const Params &P = *L.P;
  const bool lds = has_book(L);
  const u32 base = lds ? L.book_tmpl + off : off;
#define HVM_TW(i) (lds ? (u64)L.book[base + (i)] : P.tmpl[base + (i)])
  const u64 h0 = HVM_TW(0), h1 = HVM_TW(1);
  const u32 S = (u32)(h0 & 0xFF), R = (u32)((h0 >> 16) & 0xFF);
  for (u32 j = 0; j < S; j++)
    st2_new(P, I.tbase + j * I.tstride, tspec(I, HVM_TW(2 + 2 * j)), tspec(I, HVM_TW(3 + 2 * j)));
  for (u32 r = 0; r < R; r++) redux(L, tspec(I, HVM_TW(2 + 2 * S + 2 * r)), tspec(I, HVM_TW(3 + 2 * S + 2 * r)));
#undef HVM_TW
  if (h1) {
#pragma unroll
    for (u32 k = 0; k < 5; k++) L.rw[k] += (u32)((h1 >> (8 * k)) & 0xFF);
    if (h1 >> 40) {  // the interpreter shortcuts the compiler took (rare)
#pragma unroll
      for (u32 k = 5; k < 8; k++) count_rare(L, k, (u32)((h1 >> (8 * k)) & 0xFF));
    }
  }
}

// One Ctr / Op / OpNum / Switch / Const / Wires instruction
// (instruction.rs:110-210).  Every lane goes through the same sequence (read
// the trg, follow it, take the node, take fresh nodes, write two registers),
// with a branch only around what touches memory: a wave executes the union
// of its lanes' paths.
DEV void exec_step(Lane &L, Interp &I, u64 w0, u64 w1, u32 &np) {
  const Params &P = *L.P;
  const u32 kind = (u32)(w0 & 0xFF);
  const u32 a = (u32)(w0 >> 16) & 0xFFFF, b = (u32)(w0 >> 32) & 0xFFFF, c = (u32)(w0 >> 48);
  const bool ctr = kind == I_CTR;
  u64 p = t_get(I, a);  // every kind's `a` is a register of the definition (checked at book load)
  // the trg, followed if it is a wire
  const u32 pt = ptag(p);
  p = follow(L, p, (kind - I_CTR <= I_SWITCH - I_CTR) & ((pt == T_RED) | ((pt == T_VAR) & ((w0 & I_ASWIRE) != 0))));
  const u32 lab = (u32)(w1 & 0xFFFF);
  const bool match = ctr & (ptag(p) == T_CTR) & (plab(p) == lab);  // do_ctr's fast path (instruction.rs:116-121)
  u64 x = 0, y = 0;
  if (match) take(L, p, x, y);
  L.rw[RW_ANNI] += match;
  if (ctr) {
    if (!match) {  // instruction.rs:126-131
      u64 m[2];
      alloc_nodes(L, 2, m);
      st2_new(P, m[0], P_NONE, P_NONE);
      x = var_port(m[0]);
      y = var_port(m[0] + 8);
      st2_new(P, m[1], x, y);
      push_link(L, np, p, mkport(T_CTR, lab, m[1]));
    }
    t_set(I, b, match ? as_wire(x) : x);
    t_set(I, c, match ? as_wire(y) : y);
  }
  if (HVM_ANY(!ctr)) {
    if (!ctr) {
      u64 m[3] = {0, 0, 0};
      const u32 need = other_need(kind, p);
      if (need) alloc_nodes(L, need, m);
      exec_other(L, I, w0, w1, p, m, np);
    }
  }
}

// def.rs:217-289: start the definition whose record is `d`, with t0 = `t0`.
// The compiled-definition record of definition di (0: none, or compiled
// definitions are off).
DEV u64 load_cdef(const Lane &L, u32 di) {
  if (!L.P->compiled) return 0;
  return has_book(L) ? (u64)L.book[L.book_cdef + di] : L.P->cdefs[di];
}

// A compiled definition runs when its template's slots fit, as one block, in
// what is left of the first lap of the lane's allocation slice (consecutive
// slice positions are TSLOT_STRIDE bytes apart), or in the lane's chunk of
// the net's arena (consecutive nodes); otherwise the definition's
// own instructions run.
DEV void interp_begin(Lane &L, Interp &I, const DefRec &d, u64 t0, u64 cdef) {
  const Params &P = *L.P;
  I.Tl = HVM_TO_LDS(L.T_lds);
  I.Tg = L.T_glb;
  I.t_lds = L.lds_all || (P.t_lds && L.T_lds);
  I.tstride = L.arenas ? 16 : TSLOT_STRIDE;
  u32 ioff = d.ioff, ilen = d.ilen, nslots = d.nslots;
  I.tbase = 0;
  if (cdef) {
    const u32 ts = cdef_tslots(cdef);
    bool fits = false;
    if (L.arenas) {  // arenas: consecutive nodes of the lane's chunk
      if (ts) arena_room(L, ts);
      fits = L.a_pos + ts <= L.a_end;
      if (fits) {
        I.tbase = HVM_HEAP_OFF + L.a_pos * 16;
        L.a_pos += ts;
      }
    } else if (L.apos + ts <= L.slice_n) {
      I.tbase = L.slice + (u64)L.apos * SLICE_STRIDE;
      L.apos += ts;
      fits = true;
    }
    if (fits) {
      ioff = cdef_ioff(cdef);
      ilen = cdef_ilen(cdef);
      nslots = cdef_nslots(cdef);
    }
  }
  I.ipw = ioff * 2;
  I.left = ilen;
  // the trg area is sized for the book, and is in LDS only for books that fit
  if (nslots > (I.t_lds ? LDS_SLOTS : P.trg_slots)) {
    fail(L, ERR_BADPTR, BAD_SLOTS);
    I.left = 0;
    return;
  }
  t_set(I, 0, t0);
}

// The next instruction's two words.
DEV void fetch(const Lane &L, const Interp &I, u64 &w0, u64 &w1) {
  if (has_ins(L)) {
    w0 = L.book[L.book_ins + I.ipw];
    w1 = L.book[L.book_ins + I.ipw + 1];
  } else {
    w0 = L.P->instrs[I.ipw];
    w1 = L.P->instrs[I.ipw + 1];
    HVM_SETTLE_LOADS();
  }
}

// Runs instructions until the definition ends or the link list is full.
// A wave executes the union of what its lanes do at one step, so the kinds
// run in three loops, each reconverging before the next: every lane's
// pattern steps; then the templates of all the lanes that reached theirs, at
// once; then the links.  A compiled program has exactly that order, so its
// lanes go through once; an interpreted program, whose links stand among its
// patterns, goes round again.
DEV void interp_run(Lane &L, Interp &I, u32 &np) {
  const u32 LINKS = 1u << I_LINK | 1u << I_LINKCONST | 1u << I_LINKT;
  HVM_SETTLE_LOADS();
  u64 w0 = 0, w1 = 0;
  u32 kb = 0;  // bit of the instruction that ended the loop
  while ((I.left > 0) & (np < LINK_CAP)) {
    fetch(L, I, w0, w1);
    kb = 1u << (w0 & 0x1F);
    if (kb & (LINKS | 1u << I_TEMPLATE)) break;
    exec_step(L, I, w0, w1, np);
    I.ipw += 2;
    I.left -= 1;
  }
  if ((I.left > 0) & (np < LINK_CAP) & ((kb >> I_TEMPLATE) & 1)) {
    run_template(L, I, (u32)w1);
    I.ipw += 2;
    I.left -= 1;
  }
  while ((I.left > 0) & (np < LINK_CAP)) {
    fetch(L, I, w0, w1);
    kb = 1u << (w0 & 0x1F);
    if (!(kb & LINKS)) break;
    const u64 t_a = t_get(I, (u32)(w0 >> 16) & 0xFFFF), t_b = t_get(I, (u32)(w0 >> 32) & 0xFFFF);
    u64 v = (kb >> I_LINK) & 1 ? t_b : w1;
    if (HVM_ANY((kb >> I_LINKT) & 1)) v = (kb >> I_LINKT) & 1 ? tspec(I, w1) : v;
    push_link(L, np, t_a, v);
    I.ipw += 2;
    I.left -= 1;
  }
}

// The running definition (if any) to its end, and every link the task asks
// for.
DEV void run_program(Lane &L, Interp &I, u32 &np) {
  for (;;) {
    if (I.left > 0) interp_run(L, I, np);
    if (np == LINK_CAP || I.left == 0) flush_links(L, np);
    if (I.left == 0) break;
  }
}

DEV u64 expand_ref(u64 cell) { return mkport(T_REF, 0xFFFF, cell); }

// net.rs:82-109.  `cell` holds the ExpandDef's `out` endpoint.
DEV void expand_call(Lane &L, Interp &I, u32 &np, u64 cell, u64 port) {
  const Params &P = *L.P;
  if (ptag(port) == T_REF && port != P_ERA) {
    u64 oaddr = paddr(port);
    if (addr_in_heap(oaddr)) {
      u64 x = ld(L, cell), y = ld(L, oaddr);
      st(L, cell, P_FREE);
      st(L, oaddr, P_FREE);
      push_link(L, np, x, y);
      return;
    }
    // net.call(port, Ref(self)): the book def meets this ExpandDef, which is
    // never a Ctr, so the call always dereferences (def.rs:182-188).
    if (oaddr == 0 || def_index(oaddr) >= P.ndefs) {
      fail(L, ERR_BADPTR, BAD_DEF_EXPAND);
      return;
    }
    L.rw[RW_DREF]++;
    interp_begin(L, I, load_def(L, def_index(oaddr)), expand_ref(cell), load_cdef(L, def_index(oaddr)));
    return;
  }
  u64 out = ld(L, cell);
  st(L, cell, P_FREE);
  u32 t = ptag(port);
  if (t == T_REF || t == T_NUM || t == T_VAR || t == T_RED) {
    push_link(L, np, out, port);
    return;
  }
  u64 p1, p2, m[3];
  take(L, port, p1, p2);
  alloc_nodes(L, 3, m);  // the node's var cells, the two ExpandDefs' cells, the node
  st2_new(P, m[0], P_NONE, P_NONE);
  st2_new(P, m[1], var_port(m[0]), var_port(m[0] + 8));
  st2_new(P, m[2], var_port(m[0]), var_port(m[0] + 8));
  push_link(L, np, out, mkport(t, plab(port), m[2]));
  push_link(L, np, p1, expand_ref(m[1]));
  push_link(L, np, p2, expand_ref(m[1] + 8));
}

// def.rs:177-189
// Records (port, trg) in the captured list; the host puts the list back
// among the net's pending redexes after the launch.
DEV void capture_redex(Lane &L, u64 port, u64 trg) {
  const Params &P = *L.P;
  const u64 i = HVM_FAA(&P.g->captured_n, 1ull);
  if (i >= P.captured_cap) {
    fail(L, ERR_OOM);
    return;
  }
  HVM_ST(&P.captured[2 * i], port);
  HVM_ST(&P.captured[2 * i + 1], trg);
}

// The redexes of the call rings: a Ref that is not the eraser on at least
// one side.  The arms of interact.rs:6-44 that apply, in their order: of two
// nilary ports the first one that is not skippable is called (neither: an
// erasure); of a nilary port and a node, the Ref is called, unless the node
// is a Ctr whose label is not below the Ref's (comm02).  Then Net::call
// (def.rs:177-189): a Ctr whose label the definition's set does not hold is
// copied too; anything else starts the definition.
DEV void call_redex(Lane &L, Interp &I, u32 &np, u64 a, u64 b) {
  const Params &P = *L.P;
  const u32 at = ptag(a), bt = ptag(b);
  const bool aref = (at == T_REF) & (a != P_ERA);
  const bool nil = !is_binary(a) & !is_binary(b);
  const bool call_a = nil ? aref & !is_skippable(a) : aref;
  const u64 port = call_a ? a : b, trg = call_a ? b : a;
  if (nil & is_skippable(port)) {
    L.rw[RW_ERAS]++;
    return;
  }
  const u64 addr = paddr(port);
  const bool ctr = ptag(trg) == T_CTR;
  const u32 lab = plab(trg);
  const u32 di = def_index((u64)(u32)addr);
  const bool heap = addr_in_heap(addr), def = !heap & (addr != 0) & (di < P.ndefs);
  const DefRec d = load_def(L, def ? di : 0);
  const u64 cdef = load_cdef(L, def ? di : 0);
  const bool copy = ctr & ((lab >= plab(port)) | (def && !labs_has(L, d, lab)));
  if (copy) {
    comm02(L, np, port, trg);
    return;
  }
  if (!def && !heap) {
    fail(L, ERR_BADPTR, BAD_DEF_CALL);
    return;
  }
  L.rw[RW_DREF]++;
  if (heap) {  // ExpandDef: LabSet::ALL
    expand_call(L, I, np, addr, trg);
    return;
  }
  if (d.flags & DEF_INERT) {  // InertDef::call (pre_reduce.rs:108-115)
    capture_redex(L, port, trg);
    return;
  }
  interp_begin(L, I, d, trg, cdef);
}

// Serving: slot `s`'s net is normal.  Its root port (following parked
// ports) and tag go to the completion ring in host memory (the entry's
// sequence word last), then the slot is reset and handed back for admission.
DEV void serve_complete(Lane &L, u32 s) {
  const Params &P = *L.P;
  u64 p = var_port(HVM_LD(&P.slot_root[s]));
  for (u32 hop = 0; hop < MAX_CHAIN && is_endpoint(p); hop++) {
    const u64 v = ld(L, paddr(p));
    if (v == P_NONE) break;
    p = v;
  }
  u64 *const sv = P.serve_ctl;
  const u64 idx = HVM_FAA(&sv[SV_DONE_TAIL], 1ull);
  if (idx - HVM_LD_SYS(&P.host_ctl[SH_DONE_READ]) > P.done_mask) {  // the host fell behind by a whole ring
    fail(L, ERR_QUEUE);
    return;
  }
  u64 *e = P.done + (idx & P.done_mask) * 4;
  HVM_ST_SYS(e + 1, HVM_LD(&P.slot_tag[s]));
  HVM_ST_SYS(e + 2, p);
  HVM_FENCE_SYS();
  HVM_ST_SYS(e, idx + 1);
  // the slot again: its arena restarts (lanes drop their chunks at every
  // task, so no chunk of the old net is used again), then it is freed
  serve_clear(&P.arena_word[(u64)s * SERVE_WORDS]);
  publish();
  const u64 pos = HVM_FAA(&sv[SV_FREE_TAIL], 1ull);
  HVM_ST(&P.free_ring[pos % P.serve_slots], (u64)s + 1);
  publish();
  HVM_FAA(&sv[SV_FREE_COUNT], 1ull);
}

// Serving: the running task changed its net's count of redexes by `delta`
// (the redexes it put in rings, less the one it consumed); the task that
// brings the count to 0 completes the net.
// Serving, at the end of a task: the change is sent now, its old value
// looked at in serve_settle at the wave's next loop pass, so the lane does not
// wait for the atomic here.  Every path that shows this task's redexes to
// another wave first retires the wave's memory operations (this one too),
// and the wave pops its own rings only after serve_settle, so no consumer's
// decrement can overtake it.
// One atomic per slot and wave: the changes of the lanes on a slot are summed,
// and the first of those lanes sends the sum and looks at it later (an atomic
// per lane, all slots' words on a few lines, held every iteration up: 128
// requests on 32 slots, 350 ms; with this and arena_room_serve 131 ms).  All
// lanes call it; `ran`: the lane ran a task or a boot.
DEV void serve_account_deferred(Lane &L, bool ran) {
  L.acct_delta = 0;
  const u32 delta = L.pushed;  // of the redexes put in rings; one was consumed by each lane
  for (u64 todo = HVM_BALLOT(ran); todo;) {
    const u32 lead = (u32)__builtin_ctzll(todo);
    const u32 net = lane_at(L.cur_net, lead);
    const u64 same = HVM_BALLOT(ran && L.cur_net == net);
    u32 sum = 0u - (u32)__builtin_popcountll(same);
    for (u32 b = 0; HVM_ANY(delta >> b != 0); b++)
      sum += (u32)__builtin_popcountll(HVM_BALLOT(ran && L.cur_net == net && ((delta >> b) & 1))) << b;
    if (L.lane_id == lead && sum != 0) {
      L.acct_delta = sum;
      L.acct_net = net;
      L.acct_old = HVM_FAA(&L.P->pending[(u64)net * PENDING_STRIDE], sum);
    }
    todo &= ~same;
  }
}

DEV void serve_settle(Lane &L) {
  if (L.acct_delta != 0 && L.acct_old + L.acct_delta == 0) serve_complete(L, L.acct_net);
  L.acct_delta = 0;
}

DEV Interp interp_none(const Lane &L) {
  Interp I;
  I.left = 0;
  I.ipw = 0;
  I.Tl = nullptr;
  I.Tg = nullptr;
  I.t_lds = L.lds_all;  // a constant where the kernel knows it
  I.tbase = 0;
  I.tstride = L.arenas ? 16 : TSLOT_STRIDE;
  return I;
}

// Runs definition `di` with t0 (Net::boot, Host::encode_net), outside the
// reduction kernel.
DEV void run_def(Lane &L, u32 di, u64 t0) {
  Interp I = interp_none(L);
  u32 np = 0;
  interp_begin(L, I, load_def(L, di), t0, load_cdef(L, di));
  run_program(L, I, np);
  // nodes a template wrote may be reached only through the redexes it
  // pushed: retire their stores before any lane reads them
  publish();
}

// What an iteration takes is the instructions one wave issues (a few
// thousand, four cycles each) plus its dependent round trips to memory
// (about 1,000 cycles each): in a bitonic sort of 2^16 keys 38% and 55% of a
// busy wave's cycles, by the counters.  The lane's state is therefore small, its rare
// parts are in LDS, and nothing on the way is a function call: every call
// and every divergent merge costs moves of whatever lives across it.  With
// the state in registers, calls in the access path and one interaction
// switch for all classes, an iteration of rules that read one node took
// 9,240 cycles and a call iteration 27,800; this way 7,000 and 26,200
// (bitonic 2^6: 8.32 -> 7.08 ms, 2^16: 118 -> 109 ms, tree-sum 18: 5.46 ->
// 4.70 ms).
//
// One iteration of a wave: every lane with `has` runs the redex (a, b) of
// ring class `cls` (wave-uniform: each class has its code, entered by a
// scalar branch), then links everything it asks for.  Serving: then the
// redexes without a heap port that made, each in turn (they are calls: a
// pair of which neither side can be called was dropped).  `booting`
// (serving): the lane starts definition `di` with `t0` instead, its net's
// root link already in the list.
DEV void run_tasks(Lane &L, u32 cls, bool has, u64 a, u64 b, bool booting, u32 di, u64 t0, u32 np) {
  Interp I = interp_none(L);
  if (L.arenas && has) L.cur_net = net_of_port(*L.P, a, net_of_port(*L.P, b, L.cur_net));
  if (L.serve) {
    L.pushed = 0;
    if (!booting) L.a_net = NO_NET;  // a slot's arena restarts when its net completes
  }
  for (;;) {
    if (cls == CLS_ANNI) {
      if (has) anni2(L, np, a, b);
      flush_links(L, np);
    } else if (cls == CLS_COMM) {
      if (has) comm22(L, np, a, b);
      flush_links(L, np);
    } else if (cls == CLS_OTHER) {
      if (has) rule_other(L, np, a, b);
      flush_links(L, np);
    } else {
      if (has) call_redex(L, I, np, a, b);
      if (L.serve && booting) interp_begin(L, I, load_def(L, di), t0, load_cdef(L, di));
      run_program(L, I, np);
    }
    if (!L.serve) break;
    has = L.inl_n > 0;
    if (!HVM_ANY(has)) break;
    if (has) {
      L.inl_n--;
      a = L.inl[2 * L.inl_n];
      b = L.inl[2 * L.inl_n + 1];
    }
    cls = CLS_CALL;
    booting = false;
  }
}

// Serving: sets a lane up to boot a request into free slot s as Net::boot +
// the expansion of Net::normal (net.rs:30-32, 55-69) would; run_tasks then
// runs its definition with the port returned as t0, the link of the new root
// already in the list.  The slot's count is held at 1 while the boot runs,
// so that a redex the boot sends to the global ring cannot complete the net
// early.
DEV u64 serve_boot(Lane &L, u32 s, u64 tag, u32 &np) {
  const Params &P = *L.P;
  L.cur_net = s;
  L.a_net = NO_NET;
  HVM_FAA(&P.pending[(u64)s * PENDING_STRIDE], 1u);
  HVM_ST(&P.slot_tag[s], tag);
  u64 m[2];
  alloc_nodes(L, 2, m);
  st2_new(P, m[0], P_NONE, var_port(m[0]));
  st2_new(P, m[1], P_NONE, P_FREE);
  HVM_ST(&P.slot_root[s], m[0]);
  L.rw[RW_DREF]++;
  push_link(L, np, var_port(m[1]), expand_ref(m[0] + 8));
  return var_port(m[1]);
}

// ---------------------------------------------------------------------------
// lane setup / teardown
// ---------------------------------------------------------------------------
DEV void lane_init(Lane &L, const Params &P, u32 gwave, u32 lane) {
  L.P = &P;
  L.slice = HVM_HEAP_OFF + (P.ring_node0 + (u64)gwave * P.wave_nodes + lane) * 16;
  L.slice_n = (u32)(P.wave_nodes / 64);
  L.apos_home = &P.alloc_pos[(u64)gwave * 64 + lane];
  L.apos = (u32)*L.apos_home;
  L.slice_rest = 0;
  L.ov_left = 0;
  L.ov_cur = 0;
  L.fcn = 0;
  L.FC = nullptr;
  L.in_lds = false;
  L.arenas = P.gmap != nullptr;
  L.cur_net = 0;
  L.serve = false;  // set by the serving kernel
  L.lane_id = lane;
  L.pushed = 0;
  L.inl_n = 0;
  L.inl = P.inl ? P.inl + ((u64)gwave * 64 + lane) * SERVE_INL * 2 : nullptr;
  L.a_net = NO_NET;
  L.a_take = 0;
  L.acct_old = L.acct_delta = L.acct_net = 0;
  L.a_pos = 0;
  L.a_end = 0;
  L.T_lds = nullptr;
  L.PL = nullptr;
  L.T_glb = P.trg_buf + (u64)gwave * P.trg_slots * 64 + lane;
  L.bag = nullptr;
  L.bag_top = nullptr;
  L.bag_bot = nullptr;
  L.book = nullptr;
  L.lds_all = false;
  L.book_ins = 0;
  L.book_lab = 0;
  L.book_cdef = 0;
  L.book_tmpl = 0;
#pragma unroll
  for (u32 k = 0; k < RW_SLOTS; k++) L.rw[k] = 0;
  L.bad = 0;
  L.err = 0;
}

DEV void lane_finish(Lane &L) {
  *L.apos_home = L.apos;
  lane_report(L);
}

}  // namespace hvm
