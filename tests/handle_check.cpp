// Launches that the host loses (the wait for the stream fails) on the one-lane
// device of fake_device.cpp.  After a Net::normal the handle's root cell stays
// one of the heap's, the net's own or its expansion's, whatever was reduced
// before; after a Net::reduce a reset clears every redex that it left.
// Prints "ok" or what differs; exits 1 if something does.
#include <cstdint>
#include <cstdio>
#include <cstdlib>

#include "fake_device.h"
#include "hvm64_amd.h"

static hvm_gpu *h;

static void ok(bool good, const char *what) {
  if (good) return;
  std::printf("%s: %s\n", what, hvm_gpu_last_error(h));
  std::exit(1);
}

static uint64_t root() {
  hvm_net_image img;
  ok(hvm_gpu_snapshot(h, &img, 0, 0, nullptr) == 0, "snapshot");
  return img.root_cell;
}

int main() {
  uint32_t main_id = 0;
  ok(hvm_gpu_open_grid(0, 64 << 20, 1, &h) == 0, "open");
  ok(hvm_gpu_load_book_text(h, "@main = a & @f ~ (1 b) & @f ~ (b a)\n@f = (x y) & @g ~ (x y)\n@g = (x x)") == 0, "book");
  ok(hvm_gpu_def_id(h, "main", &main_id) == 0, "main");
  for (int reduced_before = 0; reduced_before < 2; reduced_before++) {
    ok(hvm_gpu_reset(h) == 0, "reset");
    ok(hvm_gpu_boot(h, main_id) == 0, "boot");
    if (reduced_before) ok(hvm_gpu_normal(h) == 0, "normal");
    const uint64_t before = root();
    fake_fail_next_sync();
    ok(hvm_gpu_normal(h) != 0, "a failed wait is an error");
    ok(root() == before, "the root cell after a failed wait");
    ok(hvm_gpu_reset(h) == 0, "reset");
    ok(hvm_gpu_boot(h, main_id) == 0, "boot");
    const uint64_t booted = root();
    ok(hvm_gpu_normal(h) == 0, "normal");
    ok(root() != 0 && root() != booted, "the root cell after normal");
  }
  ok(hvm_gpu_reset(h) == 0, "reset");
  ok(hvm_gpu_boot(h, main_id) == 0, "boot");
  fake_fail_next_sync();
  ok(hvm_gpu_reduce(h, 1, nullptr, nullptr) != 0, "a failed wait is an error");
  ok(!fake_ring_clear(), "the reduction left redexes");
  ok(hvm_gpu_reset(h) == 0, "reset");
  ok(fake_ring_clear(), "the redex ring after a reset");
  hvm_gpu_close(h);
  std::printf("ok\n");
  return 0;
}
