// launch_recorder.cpp -- a stand-in for the HIP runtime calls that libtcrv_hip.so makes, which
// records every kernel launch (name, grid, block) instead of running it.  Loaded before the
// library with RTLD_GLOBAL, it shows on a machine without a GPU which kernels an entry
// launches for given arguments (tests/launches.py).  Device pointers are never followed.
#include <cxxabi.h>

#include <cstdint>
#include <cstdlib>
#include <map>
#include <string>

namespace {

struct Dim3 {
  uint32_t x, y, z;
};

struct Config {
  Dim3 grid, block;
  size_t shared;
  void *stream;
};

std::map<const void *, std::string> &names() {
  static std::map<const void *, std::string> m;
  return m;
}
Config pushed;
std::string launches;
unsigned char scratch[16];

// "void tcrv::gemm_batch<true, 8, false>(unsigned char const*, ...)" -> "gemm_batch<true, 8, false>"
std::string short_name(const char *mangled) {
  int status = 0;
  char *text = abi::__cxa_demangle(mangled, nullptr, nullptr, &status);
  std::string s = text ? text : mangled;
  std::free(text);
  for (const char *cut : {"void ", "(anonymous namespace)::", "tcrv::"})
    for (size_t at; (at = s.find(cut)) != std::string::npos;)
      s.erase(at, std::string(cut).size());
  int depth = 0;
  for (size_t i = 0; i < s.size(); ++i) {  // up to the parameter list
    depth += s[i] == '<' ? 1 : s[i] == '>' ? -1 : 0;
    if (s[i] == '(' && depth == 0)
      return s.substr(0, i);
  }
  return s;
}

}  // namespace

extern "C" {

void **__hipRegisterFatBinary(const void *) {
  static void *handle;
  return &handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *device, unsigned, void *,
                           void *, void *, void *, int *) {
  names()[host] = short_name(device);
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t shared, void *stream) {
  pushed = {grid, block, shared, stream};
  return 0;
}
int __hipPopCallConfiguration(Dim3 *grid, Dim3 *block, size_t *shared, void **stream) {
  *grid = pushed.grid;
  *block = pushed.block;
  *shared = pushed.shared;
  *stream = pushed.stream;
  return 0;
}
int hipLaunchKernel(const void *f, Dim3 g, Dim3 b, void **, size_t, void *) {
  const auto it = names().find(f);
  launches += it == names().end() ? "?" : it->second;
  for (uint32_t v : {g.x, g.y, g.z, b.x, b.y, b.z})
    launches += "|" + std::to_string(v);
  launches += "\n";
  return 0;
}
int hipGetLastError() { return 0; }
const char *hipGetErrorString(int) { return "recorded"; }
int hipGetDevice(int *d) {
  *d = 0;
  return 0;
}
int hipSetDevice(int) { return 0; }
int hipStreamGetDevice(void *, int *d) {
  *d = 0;
  return 0;
}
int hipStreamSynchronize(void *) { return 0; }
int hipGetSymbolAddress(void **p, const void *) {
  *p = scratch;
  return 0;
}

// The launches since the last call, a line each: name|grid x|y|z|block x|y|z.
const char *recorder_take() {
  static std::string out;
  out.swap(launches);
  launches.clear();
  return out.c_str();
}

}  // extern "C"
