#include <vector>

#include "registry.hpp"

namespace bosss {

static const std::vector<KernelSet>& all_sets() {
  static std::vector<KernelSet> sets = [] {
    std::vector<KernelSet> v;
    register_sip(v);
    register_advdiff(v);
    register_euler(v);
    return v;
  }();
  return sets;
}

const KernelSet* find_kernels(int kind, int D, int N, int K1, int precision) {
  for (const KernelSet& k : all_sets())
    if (k.kind == kind && k.D == D && k.N == N && k.K1 == K1) {
      if (precision == 1 && !k.k32[KernelSet::RES]) return nullptr;
      return &k;
    }
  return nullptr;
}

int KernelSet::prepare(bool fp32, bool tensor, const bool* split) const {
  for (int i = 0; i < NVARIANT; i++) {
    const void* k;
    size_t lds;
    if (!tensor) {
      k = fp32 ? (const void*)k32[i] : (const void*)k64[i];
      lds = fp32 ? lds32 : lds64;
    } else {
      k = fp32 ? (const void*)(split[i] ? kts32 : kt32)[i] : (const void*)(split[i] ? kts64 : kt64)[i];
      lds = fp32 ? ktlds32[i] : ktlds64[i];
    }
    if (k && hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) return 1 + i;
  }
  return 0;
}

}  // namespace bosss
