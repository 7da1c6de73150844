// Host side of the resident solves (persist.h): room on a device, and when a
// result stands.  Plain C++ and POSIX, so it can be compiled and tested
// without a GPU.
#pragma once

#include <fcntl.h>
#include <sys/stat.h>
#include <unistd.h>

#include <algorithm>
#include <cerrno>
#include <cstdint>
#include <mutex>
#include <string>

namespace xcal {

// Whether a case's resident solve is complete, from its state after the
// launch: `stop` says that the case's first workgroup finished, `gave_up` that
// some workgroup of it left early, without its rows of the solution.  Both can
// be set, when the one that left had published its last sums: the solve is
// then incomplete whatever `stop` says.  Launch chains never set `gave_up`.
inline bool resident_done(int stop, int gave_up) { return stop != 0 && gave_up == 0; }

// The workgroups a device holds at once, one per compute unit, shared by every
// stream, thread and process that starts resident solves on it: two solves
// that each got part of the device would wait for each other.  A device's
// compute units are up to 64 chunks; a solve takes whole chunks.  Between
// processes a chunk is a byte of a file in shared memory, locked by its
// holder, so that the kernel gives it back when a process dies.  Without the
// file (or where processes see different ones) only this process is counted,
// and a wait between processes ends at its bound.
class ResidentRoom {
 public:
  // Takes room for nwg of cap workgroups; 0: there is none.
  uint64_t acquire(int nwg, int cap) {
    if (nwg <= 0 || nwg > cap) return 0;
    std::lock_guard<std::mutex> lk(mu);
    (void)file();
    const int chunk = (cap + 63) / 64, total = cap / chunk, need = (nwg + chunk - 1) / chunk;
    if (need > total) return 0;  // cap is not a multiple of a chunk
    uint64_t got = 0;
    int have = 0;
    // the first free run that is long enough, or else single chunks
    for (int c = 0, run = 0; c < total && have < need; ++c) {
      run = mine >> c & 1 ? 0 : run + 1;
      if (run < need) continue;
      if (!lock(c + 1 - need, need, F_WRLCK)) break;
      got = mask(c + 1 - need, need);
      have = need;
    }
    for (int c = 0; c < total && have < need; ++c)
      if (!(mine >> c & 1) && lock(c, 1, F_WRLCK)) {
        got |= 1ull << c;
        ++have;
      }
    if (have < need) {
      unlock(got);
      return 0;
    }
    mine |= got;
    return got;
  }
  void release(uint64_t chunks) {
    std::lock_guard<std::mutex> lk(mu);
    unlock(chunks);
    mine &= ~chunks;
  }
  // The file that stands for the device, before the first acquire().
  void share(const std::string& file) {
    std::lock_guard<std::mutex> lk(mu);
    if (path.empty()) path = file;
  }

 private:
  static uint64_t mask(int first, int count) {
    return (count == 64 ? ~0ull : (1ull << count) - 1) << first;
  }
  // Locks belong to the open file, not to the process, so a fork would share
  // them: a child opens the file anew.
  int file() {
    if (fd >= 0 && pid != getpid()) {
      close(fd);  // the parent's locks stay: it holds the open file too
      fd = -1;
      tried = false;
      mine = 0;
    }
    if (!tried && !path.empty()) {
      tried = true;
      pid = getpid();
      const int flags = O_RDWR | O_CLOEXEC | O_NOFOLLOW;
      fd = open(path.c_str(), flags);
      if (fd < 0) {
        fd = open(path.c_str(), flags | O_CREAT | O_EXCL, 0666);
        if (fd >= 0) (void)!fchmod(fd, 0666);  // other users' processes too
        else fd = open(path.c_str(), flags);   // another process was first
      }
    }
    return fd;
  }
  // False only where another process holds one of the chunks.
  bool lock(int first, int count, short type) {
    const int f = file();
    if (f < 0) return true;
    struct flock l {};
    l.l_type = type;
    l.l_whence = SEEK_SET;
    l.l_start = first;
    l.l_len = count;
    return fcntl(f, F_OFD_SETLK, &l) == 0 || (errno != EAGAIN && errno != EACCES);
  }
  void unlock(uint64_t chunks) {
    for (int c = 0; c < 64;) {
      int n = 0;
      while (c + n < 64 && chunks >> (c + n) & 1) ++n;
      if (n > 0) (void)lock(c, n, F_UNLCK);
      c += std::max(n, 1);
    }
  }
  std::mutex mu;
  std::string path;
  uint64_t mine = 0;  // chunks this process holds
  int fd = -1;
  pid_t pid = 0;
  bool tried = false;
};

// Room held from a launch until its stream has been waited for.
class ResidentLease {
 public:
  ResidentLease() = default;
  ResidentLease(const ResidentLease&) = delete;
  ResidentLease& operator=(const ResidentLease&) = delete;
  ~ResidentLease() { release(); }
  bool acquire(ResidentRoom& r, int nwg, int cap) {
    release();
    chunks = r.acquire(nwg, cap);
    room = chunks ? &r : nullptr;
    return chunks != 0;
  }
  void release() {
    if (room) room->release(chunks);
    room = nullptr;
  }

 private:
  ResidentRoom* room = nullptr;
  uint64_t chunks = 0;
};

}  // namespace xcal
