// TEST INFRASTRUCTURE ONLY: which kernels a call of the built kernel library (libugache_hip.so) launches, in which order and
// with which arguments, without a GPU.  This executable defines the runtime's launch calls itself, in front of those of
// libamdhip64, and notes every launch instead of performing it; device pointers are made up and never followed.
//
// usage: launch_order <libugache_hip.so> <call> <number>; prints a line per launch: the kernel and its arguments
#include <cxxabi.h>
#include <dlfcn.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {
struct Dim3 {
  uint32_t x, y, z;
};
struct Config {
  Dim3 grid, block;
  size_t shared;
  void *stream;
} g_config;
std::map<const void *, std::string> &kernels() {  // registered while the library is loaded
  static std::map<const void *, std::string> k;
  return k;
}

// the types between the outer parentheses of a demangled kernel
std::vector<std::string> parameters(const std::string &name) {
  std::vector<std::string> out;
  int angle = 0, depth = 0;
  size_t begin = 0, open = name.size();
  for (size_t i = 0; i < name.size(); ++i) {  // (anonymous namespace) and template arguments come in front
    if (name[i] == '<') ++angle;
    if (name[i] == '>') --angle;
    if (name[i] == '(' && angle == 0 && name.compare(i, 21, "(anonymous namespace)") != 0) {
      open = i;
      break;
    }
  }
  begin = open + 1;
  for (size_t i = begin; i < name.size(); ++i) {
    const char c = name[i];
    if (c == '(' || c == '<') ++depth;
    if (depth == 0 && (c == ',' || c == ')')) {
      if (i > begin) out.push_back(name.substr(begin, i - begin));
      begin = i + 2;
      if (c == ')') break;
    }
    if ((c == ')' || c == '>') && depth > 0) --depth;
  }
  return out;
}
}  // namespace

extern "C" {
void **__hipRegisterFatBinary(const void *) {
  static void *handle;
  return &handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *, int *) {
  int rc = 0;
  char *text = abi::__cxa_demangle(name, nullptr, nullptr, &rc);
  kernels()[host] = text ? text : name;
  free(text);
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t shared, void *stream) {
  g_config = Config{grid, block, shared, stream};
  return 0;
}
int __hipPopCallConfiguration(Dim3 *grid, Dim3 *block, size_t *shared, void **stream) {
  *grid = g_config.grid, *block = g_config.block, *shared = g_config.shared, *stream = g_config.stream;
  return 0;
}
int hipGetDevice(int *dev) {
  *dev = 0;
  return 0;
}
int hipDeviceGetAttribute(int *value, int, int) {
  *value = 256;
  return 0;
}
int hipGetLastError() { return 0; }
int hipLaunchKernel(const void *f, Dim3, Dim3, void **args, size_t, void *stream) {
  const std::string &name = kernels()[f];
  std::string line = name.substr(0, name.find("_kernel") + 7);
  line = line.substr(line.rfind("::") == std::string::npos ? 0 : line.rfind("::") + 2);
  printf("%s stream=%llx", line.c_str(), (unsigned long long)(uintptr_t)stream);
  const std::vector<std::string> types = parameters(name);
  for (size_t i = 0; i < types.size(); ++i) {
    unsigned long long v = 0;
    const std::string &t = types[i];
    if (t.find('*') != std::string::npos || t == "unsigned long" || t == "long" || t == "unsigned long long" || t == "long long")
      memcpy(&v, args[i], 8);
    else if (t == "unsigned int" || t == "int")
      memcpy(&v, args[i], 4);
    else
      continue;  // structures by value
    printf(" %llx", v);
  }
  printf("\n");
  return 0;
}
}

int main(int argc, char **argv) {
  if (argc != 4) return 2;
  void *lib = dlopen(argv[1], RTLD_NOW);
  if (!lib) {
    fprintf(stderr, "%s\n", dlerror());
    return 1;
  }
  const uint64_t number = strtoull(argv[3], nullptr, 0);
  const auto dev = [](uint64_t k) { return reinterpret_cast<void *>(0x100000000000ull + (k << 32)); };
  if (strcmp(argv[2], "place_with_ticket") == 0) {
    typedef int (*fn_t)(void *, uint64_t, uint64_t, void *, void *, void *, int, void *, void *, void *, void *, void *, uint32_t,
                        void *);
    const fn_t fn = reinterpret_cast<fn_t>(dlsym(lib, "ugk_rank_place_observed_ticket"));
    // evict and insert workspaces at 7 and 8, the ticket is 0xabcd
    return !fn || fn(dev(1), number, number / 2, dev(2), dev(3), dev(4), 1, dev(6), dev(7), dev(8), dev(9), dev(10), 0xabcd, dev(11));
  }
  return 2;
}
