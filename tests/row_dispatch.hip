// row_dispatch.hip -- the launches that the row kernels' dispatch makes, without a GPU.
//
// Compiled for the host only and linked without the HIP runtime: enqueue() is
// replaced by a recorder, so every accepted shape of the three row entries and of
// the quantizer can be asked for its launches.  For each shape the recorded
// launches must together cover every row once, in order, each with fewer than 2^32
// threads and at most 160 KiB of LDS, by a kernel whose threads and chunks hold the
// row.  Prints one line per fault, then the names of all kernels chosen.
#include <dlfcn.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <set>
#include <string>
#include <vector>

#include "../v7multiplikator_amd/csrc/v7g_device.h"
#include "../v7multiplikator_amd/csrc/v7g_internal.h"

struct Launch {
  const void *kernel;
  dim3 grid, block;
  unsigned lds;
  uintptr_t out;  // the launch's first argument: o, or the codes
};
static std::vector<Launch> launches;

namespace v7g {
template <typename... K, typename First, typename... A>
static void record(void (*kernel)(K...), dim3 grid, dim3 block, unsigned lds, hipStream_t, First out, A...) {
  launches.push_back({reinterpret_cast<const void *>(kernel), grid, block, lds, reinterpret_cast<uintptr_t>(out)});
}
}  // namespace v7g

#define enqueue record
#include "../v7multiplikator_amd/csrc/k_add_rmsnorm.hip"
#include "../v7multiplikator_amd/csrc/k_swiglu_q8.hip"
#undef enqueue

// The registration hooks of the host object; nothing is registered or launched.
extern "C" {
void **__hipRegisterFatBinary(const void *) { return nullptr; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, void *, void *, int *) {}
}

static std::set<std::string> names;
static int faults = 0;
static void fault(const char *what, const char *op, long long rows, long long dim, int gs, const char *kernel) {
  if (++faults <= 40) std::printf("FAULT %s: %s [%lld, %lld] gs %d: %s\n", what, op, rows, dim, gs, kernel);
}

static std::string name_of(const void *kernel) {
  Dl_info d;
  if (!dladdr(kernel, &d) || !d.dli_sname) return "?";
  return d.dli_sname;
}

// Template arguments of a mangled kernel name: the integers of its ILi..ELi.. list.
static std::vector<long> ints_of(const std::string &s, size_t from) {
  std::vector<long> v;
  for (size_t i = from; i + 1 < s.size(); ++i)
    if (s[i] == 'L' && (s[i + 1] == 'i' || s[i + 1] == 'b')) v.push_back(std::strtol(s.c_str() + i + 2, nullptr, 10));
  return v;
}

static const uintptr_t kBase = (uintptr_t)1 << 40;  // never dereferenced

template <typename Call>
static void check(const char *op, int rows, int dim, int gs, unsigned elem, Call call) {
  launches.clear();
  call();
  if (launches.empty()) return fault("nothing launched", op, rows, dim, gs, "");
  long long done = 0;
  for (const Launch &l : launches) {
    const std::string n = name_of(l.kernel);
    names.insert(n);
    const unsigned long long threads = (unsigned long long)l.grid.x * l.block.x;
    if (threads >= 1ull << 32 || l.grid.y != 1 || l.grid.z != 1) fault("grid of 2^32 threads", op, rows, dim, gs, n.c_str());
    if (l.block.x == 0 || l.block.x > 1024 || l.lds > 160 * 1024) fault("block or LDS", op, rows, dim, gs, n.c_str());
    if (l.out != kBase + (unsigned long long)done * dim * elem) fault("rows out of order", op, rows, dim, gs, n.c_str());
    done += l.grid.x;
    const size_t chain = n.find("rmsnorm_row_kernelI"), q8 = n.find("rmsnorm_q8_row_kernelI"),
                 pad = n.find("padded_row_kernelI"), row16 = n.find("norm_q8_row16_kernelI");
    if (row16 != std::string::npos) {
      if (l.block.x * 16 != (unsigned)dim || l.lds < 5u * dim) fault("row16 shape", op, rows, dim, gs, n.c_str());
      continue;
    }
    const bool padded = pad != std::string::npos;
    const size_t at = padded ? pad : q8 != std::string::npos ? q8 : chain;
    if (at == std::string::npos) {
      fault("unknown kernel", op, rows, dim, gs, n.c_str());
      continue;
    }
    const std::vector<long> t = ints_of(n, at);  // TPR, KMAX, ...
    const long tpr = t[0], kmax = t[1];
    if (l.block.x != (unsigned)tpr || 4 * tpr * kmax < dim) fault("row does not fit", op, rows, dim, gs, n.c_str());
    if (padded) {
      const bool fix = t[3], left = t[4];
      const int m = dim / 4 - 1;
      if ((fix && dim != 4 * tpr * kmax) || left != (dim % 32 != 0) || l.lds < 4u * (4 * (m + (m >> 2)) + 4) ||
          l.lds < 80)
        fault("padded shape", op, rows, dim, gs, n.c_str());
    } else {
      const bool left = q8 == std::string::npos && t[3];
      if (left != (dim % 32 != 0)) fault("leftover blocks", op, rows, dim, gs, n.c_str());
      if (!left && 4 * tpr * (kmax - 1) > dim) fault("more than the last chunk past the row", op, rows, dim, gs, n.c_str());
    }
  }
  if (done != rows) fault("rows missing or twice", op, rows, dim, gs, "");
}

int main() {
  std::vector<int> rows;
  for (int r : {1, 2, 8, 200, 256, 257, 320, 384, 385, 400, 448, 449, 512, 513, 576, 577, 640, 700, 768, 769, 900, 1000,
                1024, 1025, 1100, 1152, 1153, 1280, 1281, 1400, 1536, 1537, 1700, 1792, 1793, 2048, 2049, 3000, 5000,
                5001, 6144, 6145, 7000, 8191, 8192, 20000, 1 << 20, (1 << 22) - 1, 1 << 22, 1 << 23, 1 << 24,
                (1 << 24) + 3, 1 << 25, 1 << 26, 2147483647})
    rows.push_back(r);
  float *o = reinterpret_cast<float *>(kBase), *x = reinterpret_cast<float *>(kBase * 2);
  const float *add = reinterpret_cast<const float *>(kBase * 3), *w = reinterpret_cast<const float *>(kBase * 4);
  float *qs = reinterpret_cast<float *>(kBase * 5);
  for (int dim = 8; dim <= 16384; dim += 8)
    for (int r : rows) {
      check("add+rmsnorm", r, dim, 0, 4, [&] { v7g::launch_fused_add_rmsnorm(o, x, add, w, r, dim, 1e-6f, nullptr); });
      if (dim % 32) continue;
      check("rmsnorm", r, dim, 0, 4, [&] { v7g::launch_rmsnorm(o, x, w, r, dim, 1e-6f, nullptr); });
      for (int gs : {32, 64}) {
        if (dim % gs) continue;
        for (int off : {0, 4}) {  // aligned codes, and codes 4 bytes off: the recorded address then ends in 4
          int8_t *q = reinterpret_cast<int8_t *>(kBase) + off;
          const long long bytes = (long long)r * dim;
          if (!off && r > 256 && dim >= 512 && dim <= 12288 && bytes >= 1ll << 36) continue;  // beyond any memory
          for (const float *a : {(const float *)nullptr, add})
            check(a ? "add+rmsnorm->q8" : "rmsnorm->q8", r, dim, gs, 1, [&] {
              v7g::launch_rmsnorm_quantize(q, qs, x, a, w, r, dim, gs, 1e-6f, nullptr);
              for (Launch &l : launches) l.out -= off;
            });
        }
      }
    }
  // The quantizer: fewer than 2^32 threads for every accepted size.
  const float *in = reinterpret_cast<const float *>(kBase);
  int8_t *q = reinterpret_cast<int8_t *>(kBase * 2);
  for (int gs : {1, 3, 16, 32, 64, 100, 128, 256, 512, 4096})
    for (long long len : {1ll, 64ll, 4096ll, 12288ll, 16385ll, 1ll << 20, 1ll << 30})
      for (long long n : {1ll << 20, (1ll << 34) - 4096, 1ll << 34, (1ll << 34) + (1ll << 20), 1ll << 36, (1ll << 40) - 1}) {
        const long long r = n / len;
        if (r < 1 || r > 2147483647 || r * ((len + gs - 1) / gs) >= 1ll << 38) continue;
        for (int off : {0, 1}) {
          launches.clear();
          v7g::launch_quantize_q8(q + off, qs, in, nullptr, nullptr, (int)r, (int)len, gs, nullptr);
          if (launches.size() != 1) fault("quantizer launches", "quantize", r, len, gs, "");
          for (const Launch &l : launches)
            if ((unsigned long long)l.grid.x * l.block.x >= 1ull << 32)
              fault("grid of 2^32 threads", "quantize", r, len, gs, name_of(l.kernel).c_str());
        }
      }
  for (const std::string &n : names) std::printf("KERNEL %s\n", n.c_str());
  std::printf("%d faults\n", faults);
  return faults != 0;
}
