// Host build of single rules of the device (hvm64_rules.h), one case a run
// (argv[1]).  Prints "ok" or what differs; exits 1 if something does.
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "hvm64_rules.h"

using namespace hvm;

// One lane with a small heap.
struct Bench {
  std::vector<u64> heap = std::vector<u64>(1 << 12, P_FREE);
  std::vector<u64> queue = std::vector<u64>(2 << 8, 0);
  std::vector<u64> alloc_pos = std::vector<u64>(64, 0);
  std::vector<u64> trg = std::vector<u64>(64 * 64, 0);
  std::vector<u64> on_chip = std::vector<u64>(64 * 64, 0);
  std::vector<pair> links = std::vector<pair>(64 * 64);
  Globals g{};
  Params P{};
  Lane L;
  Bench() {
    P.heap = heap.data();
    P.heap_words = heap.size();
    P.ring_node0 = RESERVED_WORDS / 2;
    P.wave_nodes = (heap.size() - RESERVED_WORDS) / 2 / 64 * 64;
    P.queue = queue.data();
    P.qmask = (1 << 8) - 1;
    P.alloc_pos = alloc_pos.data();
    P.trg_buf = trg.data();
    P.trg_slots = 16;
    P.g = &g;
    P.limit = ~0ull;
    lane();
  }
  void lane() {
    lane_init(L, P, 0, 0);
    L.PL = links.data();
    L.T_lds = on_chip.data();
  }
};

static bool same(const char *what, u64 got, u64 want) {
  if (got == want) return true;
  std::printf("%s: got %llx, want %llx\n", what, (unsigned long long)got, (unsigned long long)want);
  return false;
}

// A definition of more registers than are kept on chip is refused where the
// launch keeps them there, and nothing is written behind them.
static bool wide_definition() {
  bool ok = true;
  for (u32 nslots : {LDS_SLOTS, LDS_SLOTS + 1, 16u}) {
    for (u32 t_lds : {0u, 1u}) {
      Bench b;
      std::vector<u64> instrs;
      for (u32 s = 1; s < nslots; s++) {
        instrs.push_back(instr_w0(I_CONST, s, 0, 0));
        instrs.push_back(numport(num_new_u24(s)));
      }
      instrs.push_back(instr_w0(I_LINKCONST, 0, 0, 0));
      instrs.push_back(P_ERA);
      DefRec d{};
      d.ilen = (u32)instrs.size() / 2;
      d.nslots = nslots;
      b.P.defs = &d;
      b.P.instrs = instrs.data();
      b.P.ndefs = 1;
      b.P.t_lds = t_lds;
      run_def(b.L, 0, numport(num_new_u24(0)));
      lane_finish(b.L);
      const bool refused = t_lds && nslots > LDS_SLOTS;
      ok &= same("error", b.g.err, refused ? ERR_BADPTR : 0);
      ok &= same("site", b.g.err_info, refused ? BAD_SLOTS : 0);
      ok &= same("erasures", b.L.rw[RW_ERAS], refused ? 0 : 1);
      for (u32 s = LDS_SLOTS; s < 64; s++) ok &= same("word behind the registers", b.on_chip[s * 64], 0);
    }
  }
  return ok;
}

// The error reported is the one that came first.
static bool first_error() {
  bool ok = true;
  for (u32 order = 0; order < 4; order++) {  // bit 0: a bad address first; bit 1: both kinds
    Bench b;
    const u64 bad = 0x20;
    if (order & 1) hw(b.L, bad);
    if (order != 1) fail(b.L, ERR_UNIMPL);
    if (order == 2) hw(b.L, bad);
    lane_report(b.L);
    ok &= same("error", b.g.err, order & 1 ? ERR_BADPTR : ERR_UNIMPL);
    ok &= same("address", b.g.result, order & 1 ? bad : 0);
  }
  return ok;
}

// A lane without a node reports it before anything can be found in the dump
// cell: at once, in each way that nodes are allocated.
static bool out_of_nodes_first() {
  bool ok = true;
  for (u32 way = 0; way < 3; way++) {
    Bench b;
    b.P.ov_nodes = 64;
    b.P.ov_node0 = b.P.ring_node0 + b.P.wave_nodes - 64;
    b.P.wave_nodes = 64;
    u64 word = 1ull << 32, base0 = 1, pool_next = 2, ov_next = 256;
    std::vector<u32> gmap(1 << 8, 0);
    u32 len = 1;
    u64 slot[SERVE_WORDS] = {};
    if (way) {
      b.P.gmap = gmap.data();
      b.P.gmap_len = gmap.size();
      b.P.gran_shift = 4;
      b.P.n_nets = 1;
      b.P.arena_word = way == 1 ? &word : slot;
      b.P.arena_base0 = &base0;
      b.P.arena_len = &len;
      b.P.pool_next = &pool_next;
      b.P.pool_end = 2;
      b.P.ov_next = &ov_next;
      b.P.ov_end = 256;
      b.P.refill_granules = 1;
      b.P.arena_chunk = 8;
      b.P.sub_granules = 1;
      b.P.serve_first = 1;
    }
    b.lane();
    b.L.serve = way == 2;
    u32 n = 0;
    for (; n < 1000 && b.g.err == 0; n++) {
      const u64 a = alloc_node(b.L);
      if (a != dump_addr()) st2(b.L, a, P_NONE, P_NONE);
    }
    ok &= same("allocations until none is left", n < 1000, 1);
    ok &= same("error", b.g.err, ERR_OOM);
    ok &= same("site", b.g.err_info, way ? OOM_POOL : 0);
    hw(b.L, 0x20);
    lane_report(b.L);
    ok &= same("error after a bad address", b.g.err, ERR_OOM);
  }
  return ok;
}

// An access outside the heap is reported, whichever address it has: 0 too,
// which the word of a freed cell holds.
static bool outside_the_heap() {
  bool ok = true;
  Bench top;
  const u64 end = HVM_HEAP_OFF + top.P.heap_words * 8;
  for (u64 addr : {(u64)0, (u64)8, (u64)0x20, HVM_HEAP_OFF - 8, HVM_HEAP_OFF, end - 8, end, ADDR_MASK}) {
    Bench b;
    const bool out = addr < HVM_HEAP_OFF || addr >= end;
    ok &= same("word", (u64)(hw(b.L, addr) - b.P.heap), out ? DUMP_WORD : (addr - HVM_HEAP_OFF) / 8);
    lane_report(b.L);
    ok &= same("error", b.g.err, out ? ERR_BADPTR : 0);
    ok &= same("site", b.g.err_info, out ? BAD_HEAP_ADDR : 0);
    ok &= same("address", b.g.result, out ? addr : 0);
  }
  Bench b;  // a wire whose cell was freed
  const u64 cell = HVM_HEAP_OFF + RESERVED_WORDS * 8;
  st(b.L, cell, P_FREE);
  follow(b.L, wire_port(cell), true);
  lane_report(b.L);
  ok &= same("freed cell", b.g.err, ERR_BADPTR);
  return ok;
}

// A lane of a planned batch hands out every node of its chunks, in order,
// whatever the sizes of its requests: the chunks (8 nodes after the first few)
// end within requests of 1 to 6 nodes.
static bool arena_remainders() {
  bool ok = true;
  for (u32 first = 1; first <= 6; first++) {
    Bench b;
    const u64 nodes = 214;
    u64 word = 1ull << 32, base0 = 1, pool_next = 1 + nodes / 2, ov_next = 1000;
    std::vector<u32> gmap(1 << 10, 0);
    u32 len = nodes / 2;
    b.P.gmap = gmap.data();
    b.P.gmap_len = gmap.size();
    b.P.gran_shift = 1;
    b.P.n_nets = 1;
    b.P.arena_word = &word;
    b.P.arena_base0 = &base0;
    b.P.arena_len = &len;
    b.P.pool_next = &pool_next;
    b.P.pool_end = pool_next;
    b.P.ov_next = &ov_next;
    b.P.ov_end = 1000;
    b.P.refill_granules = 4;
    b.P.arena_chunk = 8;
    b.lane();
    for (u64 at = 0, need = first; at + need + 8 <= nodes; at += need, need = need % 6 + 1) {
      u64 out[6];
      alloc_nodes(b.L, (u32)need, out);
      for (u64 j = 0; j < need; j++) ok &= same("node", out[j], HVM_HEAP_OFF + (2 + at + j) * 16);
    }
    ok &= same("error", b.g.err, 0);
  }
  return ok;
}

int main(int, char **argv) {
  const std::string c = argv[1];
  bool ok = false;
  if (c == "wide definition") ok = wide_definition();
  if (c == "first error") ok = first_error();
  if (c == "out of nodes first") ok = out_of_nodes_first();
  if (c == "outside the heap") ok = outside_the_heap();
  if (c == "arena remainders") ok = arena_remainders();
  if (ok) std::printf("ok\n");
  return ok ? 0 : 1;
}
