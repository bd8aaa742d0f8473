#include "resident.h"

#include <fcntl.h>
#include <sys/file.h>

#include <cctype>
#include <cerrno>
#include <mutex>
#include <string>

#include "device.h"

namespace cavs {

namespace {
constexpr int kDevices = 64;
struct Gpu {
  std::mutex m;
  bool tried = false;
  int fd = -1;  // -1 behind tried: no such file here, every claim is granted
  int users = 0;
};
Gpu &gpu(int device) {
  static Gpu *all = new Gpu[kDevices];  // (outlives every static destructor)
  return all[device];
}
}  // namespace

bool ResidentClaim::take(int device) {
  if (device_ >= 0) return true;
  if (device < 0 || device >= kDevices) return false;
  Gpu &g = gpu(device);
  std::lock_guard<std::mutex> lock(g.m);
  if (g.users == 0) {
    if (!g.tried) {
      g.tried = true;
      char id[32] = "";
      if (cavs_device_bus_id(device, id, sizeof id) == CAVS_OK) {
        std::string path = "/sys/bus/pci/devices/";
        for (const char *c = id; *c; c++) path += (char)std::tolower(*c);
        g.fd = open((path + "/vendor").c_str(), O_RDONLY | O_CLOEXEC);
      }
    }
    if (g.fd >= 0 && flock(g.fd, LOCK_EX | LOCK_NB) != 0 && errno == EWOULDBLOCK) return false;
  }
  g.users++;
  device_ = device;
  return true;
}

void ResidentClaim::give() {
  if (device_ < 0) return;
  Gpu &g = gpu(device_);
  device_ = -1;
  std::lock_guard<std::mutex> lock(g.m);
  if (--g.users == 0 && g.fd >= 0) (void)flock(g.fd, LOCK_UN);
}

}  // namespace cavs
