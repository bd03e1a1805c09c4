// Host::encode_net on the one-lane device of fake_device.cpp, through the C
// interface: argv[1] a book, argv[2] a net, argv[3] 1 with and 0 without
// compiled definitions.  The net is encoded and reduced, then the book's
// `main` is booted on the same handle and reduced.  Prints the rewrite counts
// of both; exits 1 if a register was written outside its area, 2 on an error.
#include <cstdint>
#include <cstdio>
#include <cstdlib>

#include "fake_device.h"
#include "hvm64_amd.h"

static hvm_gpu *h;

static void ok(int rc, const char *what) {
  if (rc == 0 && fake_guard_intact()) return;
  std::printf("%s: %s (guard words %s)\n", what, rc ? hvm_gpu_last_error(h) : "ok",
              fake_guard_intact() ? "intact" : "overwritten");
  std::exit(rc ? 2 : 1);
}

static void counts() {
  uint64_t rw[5];
  ok(hvm_gpu_rewrites(h, rw), "rewrites");
  for (uint64_t c : rw) std::printf("%llu ", (unsigned long long)c);
  std::printf("\n");
}

int main(int, char **argv) {
  uint32_t main_id = 0;
  ok(hvm_gpu_open_grid(0, 64 << 20, 1, &h), "open");
  ok(hvm_gpu_set_compiled(h, std::atoi(argv[3]), nullptr), "set_compiled");
  ok(hvm_gpu_load_book_text(h, argv[1]), "book");
  ok(hvm_gpu_reset(h), "reset");
  ok(hvm_gpu_encode_net_text(h, argv[2]), "encode");
  ok(hvm_gpu_normal(h), "normal");
  counts();
  ok(hvm_gpu_def_id(h, "main", &main_id), "main");
  ok(hvm_gpu_reset(h), "reset");
  ok(hvm_gpu_boot(h, main_id), "boot");
  ok(hvm_gpu_normal(h), "normal");
  counts();
  hvm_gpu_close(h);
  return 0;
}
