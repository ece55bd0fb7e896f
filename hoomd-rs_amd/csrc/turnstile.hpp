// A lock between the processes of a machine that serves them in turn.
//
// Two record locks of one file per key: a process that wants the lock first takes
// the second record, the place at the head of the queue, waits there for the first,
// and gives the head up once it has it.  A process that gives the lock up and wants it
// again at once so comes behind one that waited.  The records belong to the open file
// (not to the thread), and the system gives them up when the process ends.
#pragma once
#include <cerrno>
#include <cstdint>
#include <fcntl.h>
#include <unistd.h>

namespace hmc {

class Turnstile {
 public:
  // The lock `key` of the file at `path`, which must be there and writable.
  bool open(const char* path, uint64_t key) {
    fd_ = ::open(path, O_RDWR | O_CLOEXEC);
    at_ = (off_t)(2 * key);
    return fd_ >= 0;
  }
  // Waits for the lock.
  bool enter() const {
    if (!record(at_ + 1, F_WRLCK)) return false;
    const bool got = record(at_, F_WRLCK);
    (void)record(at_ + 1, F_UNLCK);
    return got;
  }
  void leave() const { (void)record(at_, F_UNLCK); }
  // Whether another process waits for it.
  bool wanted() const {
    struct flock r = range(at_ + 1, F_WRLCK);
    return fcntl(fd_, F_OFD_GETLK, &r) == 0 && r.l_type != F_UNLCK;
  }

 private:
  static struct flock range(off_t byte, short type) {
    struct flock r {};
    r.l_type = type;
    r.l_whence = SEEK_SET;
    r.l_start = byte;
    r.l_len = 1;
    return r;
  }
  bool record(off_t byte, short type) const {
    struct flock r = range(byte, type);
    int rc;
    while ((rc = fcntl(fd_, F_OFD_SETLKW, &r)) != 0 && errno == EINTR) {
    }
    return rc == 0;
  }
  int fd_ = -1;
  off_t at_ = 0;
};

}  // namespace hmc
