// A kernel's dynamic LDS limit is a setting of the device that is current, which need not be the context's: this program stands in
// for the two runtime calls and counts what reaches each device.  Exits with 0 when every device has been set, once for each larger
// size.
#include <cstdio>
#include <map>

namespace tpuhip {
bool raise_lds_limit(int device, const void *kernel, unsigned bytes);
}

namespace {
int current = 0, calls[2] = {0, 0};
std::map<const void *, int> limit[2];
bool refuse = false;
}  // namespace

extern "C" int hipSetDevice(int d) {
  current = d;
  return 0;
}
extern "C" int hipFuncSetAttribute(const void *kernel, int, int bytes) {
  ++calls[current];
  if (refuse) return 1;
  limit[current][kernel] = bytes;
  return 0;
}

int main() {
  int device;
  static const int a = 0, b = 0;
  bool ok = true;
  auto expect = [&](bool held, const char *what) {
    if (!held) fprintf(stderr, "%s\n", what), ok = false;
  };
  for (int turn = 0; turn < 2; ++turn)
    for (device = 0; device < 2; ++device) {
      expect(tpuhip::raise_lds_limit(device, &a, 100 << 10) && tpuhip::raise_lds_limit(device, &b, 120 << 10), "refused");
      expect(limit[device][&a] >= 100 << 10 && limit[device][&b] >= 120 << 10, "a device's limit was not raised");
    }
  expect(calls[0] == 2 && calls[1] == 2, "not once per device and kernel");
  device = 1;
  expect(tpuhip::raise_lds_limit(device, &a, 160 << 10) && limit[1][&a] == 160 << 10, "a larger size was not set");
  expect(tpuhip::raise_lds_limit(device, &a, 80 << 10) && limit[1][&a] == 160 << 10, "a smaller size took the larger one back");
  device = 0;
  refuse = true;
  expect(!tpuhip::raise_lds_limit(device, &a, 160 << 10), "another device's size stands for this one");
  refuse = false;
  expect(tpuhip::raise_lds_limit(device, &a, 160 << 10) && limit[0][&a] == 160 << 10, "a refusal was remembered");
  return ok ? 0 : 1;
}
