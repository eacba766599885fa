// claims.hpp -- which process's waiting kernels a device may hold.
//
// The entries of turns.hpp cover the solvers of one process.  Workgroups of
// kernels from several processes share the device unseen: two tile kernels fit
// beside each other, but three, or one beside a grid-wide sweep, may each be
// partly resident and wait for workgroups that cannot start.  So a process holds
// a lock on a file of the device: alone while it has solvers with tiles, shared
// while it has solvers of grid-wide kernels (a cooperative launch, as always,
// leaves other processes' to the driver).  A solver that does not get its lock
// keeps to kernels that end by themselves.  The locks go with the process,
// however it ends; the file stays.  Processes that do not share /dev/shm (other
// containers) do not see each other.
//
// No HIP calls: the caller names the device.
#pragma once
#include <errno.h>
#include <fcntl.h>
#include <sys/stat.h>
#include <unistd.h>

#include <cstdint>
#include <map>
#include <mutex>
#include <string>

namespace avbd {

enum class Claim : unsigned char { None, Shared, Alone };

class Claims {
 public:
  explicit Claims(std::string dir = "/dev/shm") : dir_(std::move(dir)) {}
  // One more holder of `what` in this process; false where another process's lock forbids it.
  bool take(const std::string& device, Claim what) {
    std::lock_guard<std::mutex> g(m_);
    Held& h = held_[device];
    const bool first = h.alone + h.shared == 0;
    if (first) h.fd = open_file(device);
    const bool raise = what == Claim::Alone ? h.alone == 0 : first;
    if (h.fd < 0 || (raise && !lock(h.fd, what == Claim::Alone ? F_WRLCK : F_RDLCK))) {
      if (first) drop(h);
      return false;
    }
    (what == Claim::Alone ? h.alone : h.shared)++;
    return true;
  }
  void give(const std::string& device, Claim what) {
    std::lock_guard<std::mutex> g(m_);
    Held& h = held_[device];
    uint32_t& n = what == Claim::Alone ? h.alone : h.shared;
    if (n == 0) return;
    n--;
    if (h.alone + h.shared == 0) drop(h);
    else if (h.alone == 0) lock(h.fd, F_RDLCK);  // atomic: no other process gets in between
  }

 private:
  struct Held {
    int fd = -1;
    uint32_t alone = 0, shared = 0;
  };
  static void drop(Held& h) {
    if (h.fd >= 0) close(h.fd);
    h.fd = -1;
  }
  // Locks of the open file, not of the process: another part of the program
  // that opens and closes the file does not end them.
  static bool lock(int fd, short type) {
    struct flock f = {};
    f.l_type = type;
    f.l_whence = SEEK_SET;
    return fcntl(fd, F_OFD_SETLK, &f) == 0;
  }
  // Made for every user, and opened without creating it where it is there: a
  // sticky folder refuses to open another user's file for creation.
  int open_file(const std::string& device) const {
    std::string path = dir_ + "/avbd_device_";
    for (char c : device) path += (c >= '0' && c <= '9') || (c >= 'a' && c <= 'z') || (c >= 'A' && c <= 'Z') ? c : '_';
    const int flags = O_RDWR | O_CLOEXEC | O_NOFOLLOW;
    int fd = -1;
    for (int i = 0; i < 3 && fd < 0; i++) {
      fd = open(path.c_str(), flags);
      if (fd >= 0 || errno != ENOENT) break;
      fd = open(path.c_str(), flags | O_CREAT | O_EXCL, 0666);
      if (fd >= 0) fchmod(fd, 0666);
      else if (errno != EEXIST) break;
    }
    struct stat st;
    if (fd >= 0 && (fstat(fd, &st) != 0 || !S_ISREG(st.st_mode))) {
      close(fd);
      fd = -1;
    }
    return fd;
  }

  std::string dir_;
  std::mutex m_;
  std::map<std::string, Held> held_;
};

}  // namespace avbd
