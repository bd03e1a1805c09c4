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

int main(int, char **argv) {
  const std::string c = argv[1];
  bool ok = false;
  if (c == "wide definition") ok = wide_definition();
  if (ok) std::printf("ok\n");
  return ok ? 0 : 1;
}
