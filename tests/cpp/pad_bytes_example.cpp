// Loads a module into device memory that other tensors of the same context had filled, runs it and counts, per tensor, the
// bytes between its channels and its channel stride that are not zero: `pad_bytes_example model.mlir input.npz all.npz`
// prints "<tensor> <nonzero pad bytes> <pad bytes>" per line and writes every tensor to the last file.
#include <cstdio>
#include <fstream>
#include <iterator>
#include <vector>

#include "tpuhip/interpreter.hpp"
#include "tpuhip/mlir_text.hpp"
#include "tpuhip/tensor_file.hpp"

using namespace tpuhip;

int main(int argc, char **argv) {
  if (argc != 4) return 2;
  try {
    ModuleInterpreter interp;
    auto check = [](int status) {
      if (status != TPUHIP_OK) throw std::runtime_error(tpuhip_last_error());
    };
    // tensors by the names of the model's ops: each is freed when the model's own takes its place
    ModuleDesc before;
    const SyncedDataShape shape = {1, 64, 128, 128};
    OpDesc op;
    op.shape = shape;
    op.type = "tpu.input";
    op.name = "filled_input";
    before.ops.push_back(op);
    op.type = "tpu.relu";
    op.operands = {"filled_input"};
    std::ifstream file(argv[1]);
    const std::string text((std::istreambuf_iterator<char>(file)), std::istreambuf_iterator<char>());
    const MlirModule model = moduleFromMlir(parseMlirText(text));
    for (auto &o : model.module.ops) {
      if (o.type == "tpu.input") continue;
      op.name = o.name;
      before.ops.push_back(op);
    }
    before.returns = {before.ops.back().name};
    interp.loadModule(before);
    for (auto &kv : interp.activationMapping)
      check(tpuhip_memset(interp.context(), kv.second->data(), 0x55, kv.second->slot_bytes()));
    interp.loadModuleFile(argv[1]);
    auto inputs = openInputTensorFile(argv[2]);
    std::vector<std::string> names;
    std::vector<std::vector<float>> values;
    std::vector<std::vector<int64_t>> shapes;
    inputs->readAllTensors(names, values, shapes);
    for (size_t i = 0; i < names.size(); ++i) interp.setTensor(names[i], values[i], 0);
    interp.invoke(0);
    interp.sync();
    auto out = openOutputTensorFile(argv[3]);
    for (auto &kv : interp.valueMapping) {
      std::string name = kv.first;
      out->addTensor(name, interp.getTensor(name, 0)->data(), interp.getTensorShape(name));
      const TensorData &t = *kv.second;
      if (t.f32 || !t.materialized) continue;
      std::vector<int8_t> bytes(t.slot_bytes());
      check(tpuhip_download(interp.context(), bytes.data(), t.data(), bytes.size()));
      size_t nonzero = 0, pads = 0;
      for (size_t p = 0; p < bytes.size(); p += (size_t)t.cs)
        for (int c = t.c; c < t.cs; ++c, ++pads) nonzero += bytes[p + (size_t)c] != 0;
      printf("%s %zu %zu\n", kv.first.c_str(), nonzero, pads);
    }
    out->keep();
  } catch (const std::exception &e) {
    fprintf(stderr, "%s\n", e.what());
    return 1;
  }
  return 0;
}
