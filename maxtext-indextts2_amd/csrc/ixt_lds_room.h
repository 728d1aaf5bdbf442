// ixt_lds_room.h -- which devices know how much LDS a kernel's launches ask for.
//
// More than 64 KiB of dynamic LDS has to be asked for ahead of a launch, and what is granted holds for the current device alone: a process that drives several asks once on each.
// Host code of its own: no GPU header.
#pragma once
#include <stddef.h>

#include <atomic>

class IxtLdsRoom {
 public:
  // give() asks the runtime for `bytes` on `device` and returns 0 when it has them; not called where as much was given before.  From several threads: asked once too often at most
  template <typename Give>
  int ask(int device, size_t bytes, Give give) {
    std::atomic<size_t>* given = device >= 0 && device < MOST ? &given_[device] : nullptr;
    if (given != nullptr && given->load(std::memory_order_acquire) >= bytes) return 0;
    const int rc = give();
    if (rc != 0 || given == nullptr) return rc;
    size_t had = given->load(std::memory_order_relaxed);
    while (had < bytes && !given->compare_exchange_weak(had, bytes, std::memory_order_release)) {}
    return 0;
  }

 private:
  static constexpr int MOST = 64;                        // (devices beyond ask every time)
  std::atomic<size_t> given_[MOST] = {};
};
