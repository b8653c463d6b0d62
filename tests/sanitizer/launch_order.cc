// TEST INFRASTRUCTURE ONLY: which kernels a call of the built kernel library (libugache_hip.so) launches, in which order and
// with which arguments, without a GPU.  This executable defines the runtime's launch calls itself, in front of those of
// libamdhip64, and notes every launch instead of performing it; device pointers are made up and never followed.
//
// usage: launch_order <libugache_hip.so> place <rows>                          a placement with a ticket
//                                       gather <row bytes> <rows> <words>
//                                       scatter <row bytes> <rows> <words>            and a direct gather behind it
//                                       mix <row bytes> <rows> <words>
//                                       pool <id bytes> <row bytes> <ids> <samples> <max norm> <words>
//                                       lists <bits>                                  one out of a bitmap, two out of two
// words: 0: nobody polls, 1: words are asked for (ugk_leave_done_words), 2: where they are faster, 3: and a key with them.
// Prints a line per launch, the kernel, its template arguments, the stream, workgroups x threads and the other arguments, and how
// many words the call says it leaves.
#include <cxxabi.h>
#include <dlfcn.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "ugache_hip.h"

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
std::vector<std::string> parameters(const std::string &name, size_t *open_at) {
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
  *open_at = open;
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
int hipLaunchKernel(const void *f, Dim3 grid, Dim3 block, void **args, size_t, void *stream) {
  const std::string &name = kernels()[f];
  const size_t end = name.find("_kernel") + 7, begin = name.rfind("::", end) == std::string::npos ? 0 : name.rfind("::", end) + 2;
  size_t open = 0;
  const std::vector<std::string> types = parameters(name, &open);
  std::string templ = name.substr(end, open - end);
  for (size_t i; (i = templ.find(' ')) != std::string::npos;) templ.erase(i, 1);
  printf("%s %s stream=%llx %ux%u", name.substr(begin, end - begin).c_str(), templ.empty() ? "<>" : templ.c_str(),
         (unsigned long long)(uintptr_t)stream, grid.x, block.x);
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
  if (argc < 4) return 2;
  void *lib = dlopen(argv[1], RTLD_NOW);
  if (!lib) {
    fprintf(stderr, "%s\n", dlerror());
    return 1;
  }
  const auto dev = [](uint64_t k) { return reinterpret_cast<void *>(0x100000000000ull + (k << 32)); };
  const auto number = [&](int i) { return i < argc ? strtoull(argv[i], nullptr, 0) : 0ull; };
  const std::string call = argv[2];
  ugk_done_t done{};
  done.words_host = static_cast<uint64_t *>(dev(20)), done.counters_dev = static_cast<uint64_t *>(dev(21)), done.tag = 1;
  const auto ask = [&](uint64_t words) {
    done.where_faster = words >= 2;
    if (words == 3) done.keys_host = dev(22), done.num_keys = 1;
    return words == 0 || reinterpret_cast<decltype(&ugk_leave_done_words)>(dlsym(lib, "ugk_leave_done_words"))(&done) == 0;
  };
  uint32_t *u32 = static_cast<uint32_t *>(dev(9));
  int rc = 2;
  if (call == "place") {  // evict and insert workspaces at 7 and 8, the ticket is 0xabcd
    const auto fn = reinterpret_cast<decltype(&ugk_rank_place_observed_ticket)>(dlsym(lib, "ugk_rank_place_observed_ticket"));
    rc = fn(static_cast<uint32_t *>(dev(1)), number(3), number(3) / 2, dev(2), static_cast<uint64_t *>(dev(3)),
            static_cast<uint64_t *>(dev(4)), 1, static_cast<uint64_t *>(dev(6)), dev(7), dev(8), u32, static_cast<uint32_t *>(dev(10)),
            0xabcd, dev(11));
  } else if (call == "lists") {
    const auto one = reinterpret_cast<decltype(&ugk_bitmap_emit)>(dlsym(lib, "ugk_bitmap_emit"));
    const auto two = reinterpret_cast<decltype(&ugk_bitmap_emit_diff)>(dlsym(lib, "ugk_bitmap_emit_diff"));
    uint64_t *a = static_cast<uint64_t *>(dev(1)), *b = static_cast<uint64_t *>(dev(2));
    rc = one(a, nullptr, 0, number(3), dev(7), u32, number(3), dev(11)) ||
         two(a, b, number(3), dev(7), dev(8), u32, number(3), static_cast<uint32_t *>(dev(10)), number(3), dev(11));
  } else if (call == "gather" && argc == 6 && ask(number(5))) {
    const auto fn = reinterpret_cast<decltype(&ugk_gather_direct_i64)>(dlsym(lib, "ugk_gather_direct_i64"));
    rc = fn(dev(1), 1000, static_cast<int64_t *>(dev(2)), number(4), dev(3), number(3), 0, u32, nullptr, dev(11));
  } else if (call == "scatter" && argc == 6 && ask(number(5))) {
    const auto fn = reinterpret_cast<decltype(&ugk_gather_scatter_i64)>(dlsym(lib, "ugk_gather_scatter_i64"));
    const auto next = reinterpret_cast<decltype(&ugk_gather_direct_i64)>(dlsym(lib, "ugk_gather_direct_i64"));
    rc = fn(dev(1), 1000, static_cast<int64_t *>(dev(2)), static_cast<uint32_t *>(dev(4)), number(4), dev(3), 1000, number(3), 0, u32,
            nullptr, dev(11)) ||
         next(dev(1), 1000, static_cast<int64_t *>(dev(2)), number(4), dev(3), number(3), 0, u32, nullptr, dev(11));
  } else if (call == "mix" && argc >= 6 && ask(number(5))) {
    ugk_table_t flat{};
    flat.kind = argc > 6 ? (int32_t)number(6) : 1, flat.table = dev(4), flat.size = flat.kind == 1 ? 1000 : 1024;
    const auto fn = reinterpret_cast<decltype(&ugk_extract_mix_i64)>(dlsym(lib, "ugk_extract_mix_i64"));
    rc = fn(flat, static_cast<int64_t *>(dev(2)), number(4), dev(1), 1000, dev(5), 1000, dev(3), number(3), u32, nullptr, nullptr,
            nullptr, UGK_HINT_UNKNOWN, dev(11));
  } else if (call == "pool" && argc == 9 && ask(number(8))) {
    ugk_table_t none{};
    const auto run = [&](auto fn, auto *ids) {
      return fn(none, ids, static_cast<int64_t *>(dev(2)), nullptr, number(6), number(5), 0, 4, (float)number(7), nullptr, 0, dev(3),
                1000, dev(4), number(4), u32, nullptr, nullptr, nullptr, dev(11));
    };
    rc = number(3) == 4 ? run(reinterpret_cast<decltype(&ugk_extract_pool_clip_u32)>(dlsym(lib, "ugk_extract_pool_clip_u32")),
                              static_cast<uint32_t *>(dev(1)))
                        : run(reinterpret_cast<decltype(&ugk_extract_pool_clip_i64)>(dlsym(lib, "ugk_extract_pool_clip_i64")),
                              static_cast<int64_t *>(dev(1)));
  }
  if (rc == 0) printf("words %u\n", done.num_words);
  return rc;
}
