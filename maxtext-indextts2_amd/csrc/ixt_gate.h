// ixt_gate.h -- which pass may take the launches whose blocks wait for each other (k_step, k_mid, k_attn_split).
//
// One such grid ends beside anything that ends by itself (ixt_step.h, ixt_small.h).  Two of them need not: each could hold the compute units that a block of the other has to start on.  So a pass takes these
// forms only while no other context has a pass on another stream of the GPU, and otherwise the forms without waits, which give the same bits.  Nobody stands still for the answer.  (A turn that
// kernels wait for needs a launch behind them to give it on, which a hardware queue shared with another stream may hold back, or which an error on the way may never send.)
//
// That the other's pass counts whatever its form is a matter of speed: a grid of k_step beside launches of another pass slows both.  Two engines of the 1B model on two streams, ms for
// a step of both, 1 + 1 / 8 + 8 / 48 + 48 / 1 + 48 slots: a turn for the waiting forms 1.24 / 1.55 / 2.79 / 2.05, one pass with them and the other without 1.44 / 1.78 / 2.64 / 2.13, both without 1.32 / 1.60 / 2.42 / 2.04.
//
// Between processes a record lock on a file per GPU does the same, for as long as a process has contexts whose passes asked for these forms; the others' passes take the forms without waits.
// Processes that do not see each other's file are not told apart: there the waits' bounds end them, and the caller gets an error.
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
#include <thread>
#include <utility>
#include <vector>

class IxtGate {
 public:
  using Lane = std::pair<const void*, std::thread::id>;      // a stream; the thread where the handle means another stream in each
  // the first of the files that can be opened counts; none: no pass takes the forms that wait
  explicit IxtGate(std::vector<std::string> lock_files) : files_(std::move(lock_files)) {}
  // A pass of `who` (the caller orders those of one context) is about to be enqueued on stream `lane`: may it take the forms that wait?  leave() follows in either case.
  // event: the context's own, for leave() to record; ended: has all in front of its last record ended?  settle: waits for the GPU; for passes without an event behind them.
  template <typename Ended, typename Settle>
  bool enter(const void* who, Lane lane, void* event, Ended ended, Settle settle) {
    std::lock_guard<std::mutex> lk(mu_);
    bool alone = true, settled = false;
    for (auto& u : users_) {
      User& other = u.second;
      if (u.first == who || other.state == NONE || other.lane == lane) continue;       // (passes of one stream run one after the other)
      lanes_ = true;
      if (other.state == OPEN && !settled) settled = settle();
      if ((other.state == OPEN && settled) || (other.state == MARKED && ended(other.event))) other.state = NONE;
      else alone = false;
    }
    users_[who] = User{BEGUN, lane, event};
    return alone && claim();
  }
  // It is enqueued; `mark` records the event behind it, which passes are spared (3 us of the host) until a second stream is seen.
  template <typename Mark>
  void leave(const void* who, Mark mark) {
    std::lock_guard<std::mutex> lk(mu_);
    User& me = users_[who];
    me.state = lanes_ && mark(me.event) ? MARKED : OPEN;
  }
  // `who` is about to go, with nothing of it left on the GPU
  void forget(const void* who) {
    std::lock_guard<std::mutex> lk(mu_);
    users_.erase(who);
    if (users_.size() < 2) lanes_ = false;
    if (!users_.empty() || fd_ < 0) return;
    (void)close(fd_);                            // (and with it the lock)
    fd_ = -1;
  }

 private:
  enum State { NONE, BEGUN, OPEN, MARKED };      // of a context's last pass: it has ended; is being enqueued; is enqueued; with the event behind it
  struct User {
    State state = NONE;
    Lane lane{};
    void* event = nullptr;
  };
  // the file's lock.  A record lock: a child of fork() has no part in it, and cannot keep it.
  bool claim() {
    for (size_t i = 0; i < files_.size() && fd_ < 0; ++i) {
      int fd = open(files_[i].c_str(), O_RDWR | O_CLOEXEC | O_NOFOLLOW);
      if (fd < 0 && errno == ENOENT) {
        fd = open(files_[i].c_str(), O_RDWR | O_CLOEXEC | O_NOFOLLOW | O_CREAT, 0666);
        if (fd >= 0) (void)fchmod(fd, 0666);     // for the processes of other users
      }
      if (fd < 0) continue;
      struct flock whole = {};
      whole.l_type = F_WRLCK;
      whole.l_whence = SEEK_SET;
      if (fcntl(fd, F_SETLK, &whole) != 0) {
        (void)close(fd);
        return false;
      }
      fd_ = fd;
    }
    return fd_ >= 0;
  }

  std::mutex mu_;
  std::map<const void*, User> users_;            // contexts whose passes asked
  bool lanes_ = false;           // on different streams
  const std::vector<std::string> files_;
  int fd_ = -1;
};
