// How many CPUs this process may keep busy: those of its affinity mask, or of its control groups' quota where that is less
// (a container that may use 2 of 128 CPUs has all of them in the mask).
#pragma once

#include <sched.h>

#include <algorithm>
#include <cstdlib>
#include <fstream>
#include <string>

namespace tpuhip {

// whole CPUs of a quota in files of `folder`, at least 1; 0: there is none
inline int cpus_of_quota(const std::string &folder) {
  auto read = [&](const char *file, std::string *first, std::string *second) {
    std::ifstream in(folder + "/" + file);
    in >> *first;
    if (second) in >> *second;
  };
  std::string quota, period;
  read("cpu.max", &quota, &period);                            // "max 100000", "150000 100000"
  if (quota.empty()) {
    read("cpu.cfs_quota_us", &quota, nullptr);                 // -1: none
    read("cpu.cfs_period_us", &period, nullptr);
  }
  const long q = atol(quota.c_str()), p = atol(period.c_str());
  return q > 0 && p > 0 ? (int)std::max(1l, q / p) : 0;
}

// the tightest quota of the groups that the lines of `groups` ("0::/a/b", "4:cpu,cpuacct:/a/b") name, and of those they lie in
inline int cpus_of_groups(const std::string &groups, const std::string &mount) {
  int least = 0;
  std::ifstream in(groups);
  for (std::string line; std::getline(in, line);) {
    const size_t a = line.find(':'), b = a == std::string::npos ? a : line.find(':', a + 1);
    if (b == std::string::npos) continue;
    const std::string controllers = "," + line.substr(a + 1, b - a - 1) + ",";
    const bool unified = controllers == ",,";
    if (!unified && controllers.find(",cpu,") == std::string::npos) continue;
    const std::string root = unified ? mount : mount + "/cpu";
    for (std::string path = line.substr(b + 1);;) {
      if (const int n = cpus_of_quota(root + path)) least = least ? std::min(least, n) : n;
      const size_t up = path.rfind('/');
      if (up == std::string::npos || path.empty()) break;
      path.resize(up);
    }
  }
  return least;
}

inline int usable_cpus() {
  cpu_set_t set;
  int cpus = 1;
  if (sched_getaffinity(0, sizeof(set), &set) == 0) cpus = CPU_COUNT(&set);
  const int quota = cpus_of_groups("/proc/self/cgroup", "/sys/fs/cgroup");
  return quota ? std::min(cpus, quota) : cpus;
}

}  // namespace tpuhip
