// Stands in front of the HIP runtime (LD_PRELOAD) for tests of a kernel library's
// host code on a machine without a GPU: launches are noted, not run.
#include <stdint.h>
#include <string.h>

#include <map>
#include <string>
#include <vector>

namespace {
struct Dim3 {
  uint32_t x, y, z;
};
struct Launch {
  std::string name;
  Dim3 grid, block;
  std::vector<uint64_t> words;      // of the watched argument
};
struct Config {
  Dim3 grid, block;
  size_t shmem;
  void* stream;
};
std::map<const void*, std::string>& names() {
  static auto& n = *new std::map<const void*, std::string>;
  return n;
}
std::vector<Launch> launches;
Config pushed;
// the leading words of an argument of the kernels whose names contain a text
std::string watched;
int watched_argument = 0;
size_t watched_words = 0;
int compute_units = 256;      // of every stream; 0: the query fails
int queries = 0;
int last_error = 0;
}  // namespace

extern "C" {
int launch_log_size() { return (int)launches.size(); }
void launch_log_clear() { launches.clear(), queries = 0; }
const char* launch_log_name(int i) { return launches[i].name.c_str(); }
unsigned launch_log_grid(int i) { return launches[i].grid.x * launches[i].grid.y; }
unsigned launch_log_block(int i) { return launches[i].block.x; }
void launch_log_set_compute_units(int n) { compute_units = n; }
void launch_log_watch(const char* name, int argument, int words) {
  watched = name;
  watched_argument = argument;
  watched_words = words;
}
int launch_log_words(int i) { return (int)launches[i].words.size(); }
uint64_t launch_log_word(int i, int k) { return launches[i].words[k]; }
int launch_log_queries() { return queries; }
int launch_log_kernels() { return (int)names().size(); }
const char* launch_log_kernel(int i) {
  auto it = names().begin();
  while (i--) ++it;
  return it->second.c_str();
}

void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*,
                           void*, void*, void*, int*) {
  names()[host] = name;
}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t shmem, void* stream) {
  pushed = {grid, block, shmem, stream};
  return 0;
}
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* shmem, void** stream) {
  *grid = pushed.grid;
  *block = pushed.block;
  *shmem = pushed.shmem;
  *stream = pushed.stream;
  return 0;
}
int hipLaunchKernel(const void* f, Dim3 grid, Dim3 block, void** args, size_t, void*) {
  launches.push_back({names().count(f) ? names()[f] : "unknown", grid, block, {}});
  if (watched_words && launches.back().name.find(watched) != std::string::npos) {
    launches.back().words.resize(watched_words);
    memcpy(launches.back().words.data(), args[watched_argument], watched_words * 8);
  }
  return 0;
}
int hipExtStreamGetCUMask(void*, uint32_t words, uint32_t* mask) {
  ++queries;
  if (compute_units == 0) return last_error = 1;
  memset(mask, 0, words * sizeof(uint32_t));
  for (int b = 0; b < compute_units; ++b) mask[b / 32] |= 1u << (b % 32);
  return 0;
}
int hipGetLastError() {
  const int e = last_error;
  last_error = 0;
  return e;
}
}
