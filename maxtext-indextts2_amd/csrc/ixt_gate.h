// ixt_gate.h -- which pass may take the launches whose blocks wait for each other (k_step, k_mid, k_attn_split).
//
// One such grid ends beside anything that ends by itself (ixt_step.h, ixt_small.h).  Two of them need not: each could hold the compute units that a block of the other has to start on.  So a pass takes these
// forms only while no other context has a pass on the GPU, and otherwise the forms without waits, which give the same bits.  Nobody stands still for the answer.  (A turn that
// kernels wait for needs a launch behind them to give it on, which a hardware queue shared with another stream may hold back, or which an error on the way may never send.)
//
// That the other's pass counts whatever its form is a matter of speed: a grid of k_step beside launches of another pass slows both.  Two engines of the 1B model on two streams, ms for
// a step of both, 1 + 1 / 8 + 8 / 48 + 48 / 1 + 48 slots: a turn for the waiting forms 1.24 / 1.55 / 2.79 / 2.05, one pass with them and the other without 1.44 / 1.78 / 2.64 / 2.13, both without 1.32 / 1.60 / 2.42 / 2.04.
//
// Between processes a record lock on a file per GPU does the same, for as long as a process has contexts whose passes asked for these forms; the others' passes take the forms without waits.
// Processes that do not see each other's /tmp are not told apart: there the waits' bounds end them, and the caller gets an error.
//
// Host code of its own: no GPU header.
#pragma once
#include <errno.h>
#include <fcntl.h>
#include <sys/stat.h>
#include <unistd.h>

#include <map>
#include <mutex>
#include <string>
#include <utility>

class IxtGate {
 public:
  explicit IxtGate(std::string lock_file = "") : file_(std::move(lock_file)) {}
  // Context `who` comes, with an event of its own (any pointer).  `settle` waits for the GPU: passes of a context that was alone have no event behind them.
  template <typename Settle>
  void join(const void* who, void* event, Settle settle) {
    std::map<const void*, long> open;
    {
      std::lock_guard<std::mutex> lk(mu_);
      users_[who].event = event;
      for (auto& u : users_)
        if (u.second.state == OPEN) open[u.first] = u.second.passes;
    }
    if (open.empty() || !settle()) return;
    std::lock_guard<std::mutex> lk(mu_);
    for (auto& o : open) {
      auto u = users_.find(o.first);
      if (u != users_.end() && u->second.state == OPEN && u->second.passes == o.second) u->second.state = NONE;
    }
  }
  // `who` is about to go, with nothing of it left on the GPU
  void forget(const void* who) {
    std::lock_guard<std::mutex> lk(mu_);
    users_.erase(who);
    for (auto& u : users_)
      if (u.second.passes > 0) return;
    if (fd_ >= 0) (void)close(fd_);              // (and with it the lock)
    fd_ = -1;
  }
  // A pass of `who` (the caller orders those of one context) is about to be enqueued: may it take the forms that wait?  leave() follows in either case.
  // `ended`: has everything in front of the last record of this event ended?
  template <typename Ended>
  bool enter(const void* who, Ended ended) {
    std::lock_guard<std::mutex> lk(mu_);
    bool alone = true;
    for (auto& u : users_) {
      if (u.first == who) continue;
      if (u.second.state == MARKED && ended(u.second.event)) u.second.state = NONE;
      alone = alone && u.second.state == NONE;
    }
    User& me = users_[who];
    me.state = OPEN;
    ++me.passes;
    return alone && claim();
  }
  // It is enqueued; `mark` records the event behind it, which the only context of a GPU is spared (3 us of a pass).
  template <typename Mark>
  void leave(const void* who, Mark mark) {
    std::lock_guard<std::mutex> lk(mu_);
    User& me = users_[who];
    if (users_.size() < 2) return;
    if (mark(me.event)) me.state = MARKED;
    else ++me.passes;                            // (a join that is waiting for the GPU may have begun before this pass)
  }

 private:
  enum State { NONE, OPEN, MARKED };             // of a context's last pass: ended; enqueued or being enqueued; with the event behind it
  struct User {
    void* event = nullptr;
    State state = NONE;
    long passes = 0;
  };
  // the file's lock.  A record lock: a child of fork() has no part in it, and cannot keep it.
  bool claim() {
    if (fd_ >= 0) return true;
    int fd = open(file_.c_str(), O_RDWR | O_CLOEXEC | O_NOFOLLOW);
    if (fd < 0 && errno == ENOENT) {
      fd = open(file_.c_str(), O_RDWR | O_CLOEXEC | O_NOFOLLOW | O_CREAT, 0666);
      if (fd >= 0) (void)fchmod(fd, 0666);       // for the processes of other users
    }
    struct flock whole = {};
    whole.l_type = F_WRLCK;
    whole.l_whence = SEEK_SET;
    if (fd >= 0 && fcntl(fd, F_SETLK, &whole) != 0) {
      (void)close(fd);
      fd = -1;
    }
    fd_ = fd;
    return fd_ >= 0;
  }

  std::mutex mu_;
  std::map<const void*, User> users_;
  const std::string file_;
  int fd_ = -1;
};
