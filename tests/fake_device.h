// Test hooks of the host-memory device (fake_device.cpp).
#pragma once

// False: the last launch wrote behind the registers it has on chip.
bool fake_guard_intact();
// The next wait for the stream fails.
void fake_fail_next_sync();
// The global redex ring holds no redex.
bool fake_ring_clear();
