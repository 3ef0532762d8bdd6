// Calls that would rather have more memory, or threads, do without them: this program defines the functions that the library
// gets them by, refuses what the running case says (memory with the runtime's own error), and checks the results.
// `doing_without_example <case> [model.mlir]` exits with 0 when they are right.
#include <dlfcn.h>
#include <pthread.h>

#include <cerrno>

#include <cmath>
#include <cstdio>
#include <cstring>
#include <functional>
#include <vector>

#include "tpuhip/interpreter.hpp"

using namespace tpuhip;

namespace {
std::function<bool(size_t)> refuse;   // whether an allocation of that many bytes fails
bool no_threads = false;
int refused = 0;
constexpr size_t kNever = (size_t)1 << 60;

template <class F>
F next(const char *name) {
  return reinterpret_cast<F>(dlsym(RTLD_NEXT, name));
}
}  // namespace

extern "C" int hipMalloc(void **p, size_t bytes) {
  static const auto real = next<int (*)(void **, size_t)>("hipMalloc");
  if (refuse && refuse(bytes)) ++refused, bytes = kNever;
  return real(p, bytes);
}
extern "C" int hipHostMalloc(void **p, size_t bytes, unsigned flags) {
  static const auto real = next<int (*)(void **, size_t, unsigned)>("hipHostMalloc");
  if (refuse && refuse(bytes)) ++refused, bytes = kNever;
  return real(p, bytes, flags);
}

extern "C" int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *arg) {
  static const auto real = next<int (*)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *)>("pthread_create");
  if (no_threads) {
    ++refused;
    return EAGAIN;
  }
  return real(t, a, f, arg);
}

namespace {

void check(int status) {
  if (status != TPUHIP_OK) throw std::runtime_error(tpuhip_last_error());
}
void expect(bool ok, const char *what) {
  if (!ok) throw std::runtime_error(what);
}

OpDesc op(const char *type, const std::string &name, SyncedDataShape shape, std::vector<std::string> operands) {
  OpDesc d;
  d.type = type;
  d.name = name;
  d.shape = std::move(shape);
  d.operands = std::move(operands);
  return d;
}

std::vector<int8_t> values(size_t n, unsigned seed) {
  std::vector<int8_t> v(n);
  for (auto &x : v) x = (int8_t)((seed = seed * 1664525u + 1013904223u) >> 24);
  return v;
}

// an output that is complete before the last kernel, read after every invoke
void early_output() {
  const SyncedDataShape shape = {1, 70, 50, 41};
  const size_t n = 70 * 50 * 41;
  ModuleDesc m;
  m.ops = {op("tpu.input", "x", shape, {}), op("tpu.relu", "first", shape, {"x"}), op("tpu.relu", "second", shape, {"x"})};
  m.returns = {"first", "second"};
  ModuleInterpreter interp;
  interp.loadModule(m);
  for (unsigned k = 0; k < 5; ++k) {
    const auto x = values(n, k);
    interp.setTensorI8("x", x.data(), n, 0);
    refuse = [](size_t bytes) { return bytes > (128 << 10); };   // only what is laid out early is as large by now
    if (k == 0) refuse = nullptr;
    interp.invoke(0);
    for (const char *name : {"first", "second"}) {
      std::vector<int8_t> y(n);
      interp.getTensorI8(name, y.data(), n, 0);
      for (size_t i = 0; i < n; ++i) expect(y[i] == (x[i] < 0 ? 0 : x[i]), name);
    }
  }
  refuse = nullptr;
  expect(refused > 0, "nothing was refused");
}

// a global average over a large map, whose partial sums would go to a workspace
void pool_workspace() {
  tpuhip_ctx *ctx = nullptr;
  check(tpuhip_ctx_create(0, &ctx));
  const int n = 2, c = 120, h = 60, w = 50, cs = 128;
  const auto x = values((size_t)n * c * h * w, 3);
  void *dense = nullptr, *in = nullptr, *out = nullptr;
  check(tpuhip_malloc(ctx, x.size(), &dense));
  check(tpuhip_malloc(ctx, (size_t)n * h * w * cs, &in));
  check(tpuhip_malloc(ctx, (size_t)n * cs, &out));
  check(tpuhip_upload(ctx, dense, x.data(), x.size()));
  check(tpuhip_nchw_to_nhwc_i8(ctx, dense, in, n, c, h, w, cs));
  const tpuhip_pool_desc d = {n, c, h, w, 1, 1, h, w, 1, 1, 0, 0, 0, 0, cs, cs};
  std::vector<int8_t> got[2];
  for (int with = 0; with < 2; ++with) {
    refuse = [with](size_t) { return with == 0; };
    check(tpuhip_memset(ctx, out, 0x55, (size_t)n * cs));
    check(tpuhip_pool_avg_i8(ctx, &d, in, out, 81, 13));
    got[with].resize((size_t)n * cs);
    check(tpuhip_download(ctx, got[with].data(), out, got[with].size()));
  }
  refuse = nullptr;
  for (void *p : {dense, in, out}) check(tpuhip_free(ctx, p));
  check(tpuhip_ctx_destroy(ctx));
  expect(refused > 0, "nothing was refused");
  expect(got[0] == got[1], "the averages differ");
  for (int k = 0; k < c; ++k) {
    int32_t s = 0;
    for (int i = 0; i < h * w; ++i) s += x[(size_t)k * h * w + i];
    const float q = std::fmin(std::fmax((float)s * 81.0f / 8192.0f, -128.0f), 127.0f);   // sat8
    expect(std::fabs((float)got[0][k] - q) <= 0.5f, "an average is wrong");
  }
}

// a module loads where there is no room for the slabs that its tensors and weights would share
void slab() {
  const SyncedDataShape shape = {1, 16, 20, 20};
  const size_t n = 16 * 20 * 20;
  ModuleDesc m;
  m.ops = {op("tpu.input", "x", shape, {}), op("tpu.relu", "y", shape, {"x"}), op("tpu.relu", "z", shape, {"y"})};
  m.returns = {"z"};
  refuse = [](size_t bytes) { return bytes >= ((size_t)16 << 20); };
  for (int again = 0; again < 2; ++again) {   // and gives its memory back
    ModuleInterpreter interp;
    interp.loadModule(m);
    const auto x = values(n, 5);
    interp.setTensorI8("x", x.data(), n, 0);
    interp.invoke(0);
    std::vector<int8_t> y(n);
    interp.getTensorI8("z", y.data(), n, 0);
    for (size_t i = 0; i < n; ++i) expect(y[i] == (x[i] < 0 ? 0 : x[i]), "z");
  }
  refuse = nullptr;
  expect(refused > 0, "nothing was refused");
}

// several tensors to the host at once, whose dense forms would lie on the device together
void many_results() {
  const SyncedDataShape shape = {1, 70, 61, 67};
  const size_t n = 70 * 61 * 67;
  ModuleDesc m;
  m.ops = {op("tpu.input", "x", shape, {}), op("tpu.relu", "y", shape, {"x"}), op("tpu.relu", "z", shape, {"y"})};
  m.returns = {"z"};
  ModuleInterpreter interp;
  interp.loadModule(m);
  const auto x = values(n, 11);
  interp.setTensorI8("x", x.data(), n, 0);
  interp.invoke(0);
  const std::vector<std::string> names = {"x", "y", "z"};
  for (int with = 0; with < 2; ++with) {
    std::vector<std::vector<float>> got(3, std::vector<float>(n));
    std::vector<float *> to = {got[0].data(), got[1].data(), got[2].data()};
    // one alone has room, and the pinned buffer, a power of two
    refuse = [with, n](size_t bytes) { return with == 0 && bytes > 2 * n && (bytes & (bytes - 1)); };
    interp.getTensors(names, to, {n, n, n}, 0);
    for (size_t i = 0; i < n; ++i)
      expect(got[0][i] == x[i] && got[1][i] == (x[i] < 0 ? 0 : x[i]) && got[2][i] == got[1][i], "a result is wrong");
  }
  refuse = nullptr;
  expect(refused > 0, "nothing was refused");
}

// the host passes of large tensors and the reading of weights beside the text
void threads(const char *model) {
  const SyncedDataShape shape = {4, 64, 128, 128};
  const size_t n = (size_t)4 * 64 * 128 * 128;
  ModuleDesc m;
  m.ops = {op("tpu.input", "x", shape, {}), op("tpu.relu", "y", shape, {"x"})};
  m.returns = {"y"};
  ModuleInterpreter interp;
  interp.loadModule(m);
  std::string in = "x";
  const auto x = values(n, 7);
  interp.setTensorI8(in, x.data(), n, 0);   // on one thread: what the runtime starts for transfers, it has started then
  interp.invoke(0);
  interp.sync();
  for (bool without : {true, false}) {
    no_threads = without;
    std::vector<float> f(n), got(n);
    for (size_t i = 0; i < n; ++i) f[i] = (float)(without ? x[i] : x[n - 1 - i]);
    interp.setTensor(in, f, 0);
    interp.invoke(0);
    interp.getTensor("y", got.data(), n, 0);
    for (size_t i = 0; i < n; ++i) expect(got[i] == (f[i] < 0 ? 0 : f[i]), "y");
  }
  ModuleInterpreter first, second;
  std::vector<float> results[2];
  for (int k = 0; k < 2; ++k) {
    ModuleInterpreter &file = k ? second : first;
    no_threads = k == 0;
    file.loadModuleFile(model);
    const size_t count = file.input_details[0].second;
    const auto v = values(count, 9);
    file.setTensorI8(file.input_details[0].first, v.data(), count, 0);
    file.invoke(0);
    no_threads = false;
    std::string out = file.output_details[0];
    results[k] = *file.getTensor(out, 0);
  }
  expect(results[0] == results[1], "the results differ");
  expect(refused > 1, "nothing was refused");
}

}  // namespace

int main(int argc, char **argv) {
  if (argc < 2) return 2;
  try {
    const std::string which = argv[1];
    if (which == "early_output") early_output();
    else if (which == "pool_workspace") pool_workspace();
    else if (which == "slab") slab();
    else if (which == "many_results") many_results();
    else if (which == "threads" && argc == 3) threads(argv[2]);
    else return 2;
  } catch (const std::exception &e) {
    refuse = nullptr;
    no_threads = false;
    fprintf(stderr, "%s\n", e.what());
    return 1;
  }
  return 0;
}
