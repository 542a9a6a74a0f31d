// gfx950 kernels of the N-fold way (the body, shared with the run-time
// specialised kernels, is in clexmc_nfold.h).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "clexmc_nfold.h"

namespace clexmc {

size_t nfold_lds_bytes(int pad_sites, int n_sites, int nb_max, int nb_total, int n_sublat) {
  const int n_groups = (n_sites + 63) / 64;
  return nfold_align16((size_t)image_bytes(pad_sites, false)) + nfold_align16((size_t)n_groups * 64 * 4) +
         nfold_align16((size_t)n_groups * 8) + 2 * nfold_align16((size_t)nb_max * 4) + kNfoldSelBytes +
         kNfoldNbBeginBytes + nfold_align16((size_t)nb_total * 4) + (size_t)n_sublat * (1 + kMaxOcc) * 4;
}

template <bool BIN>
__global__ __launch_bounds__(kNfoldMaxThreads) void nfold_kernel(NfoldArgs na) {
  nfold_body<BIN, GenericField>(na);
}

template <bool BIN>
__global__ __launch_bounds__(128, kNfoldSingleWaves) void nfold_own_books_kernel(NfoldArgs na) {
  nfold_body<BIN, GenericField, true>(na);
}

hipError_t launch_nfold(const NfoldArgs &a, bool binary, int n_chains, int threads, bool own_books, size_t lds,
                        hipStream_t st) {
  void (*fn)(NfoldArgs) = own_books ? (binary ? nfold_own_books_kernel<true> : nfold_own_books_kernel<false>)
                                    : (binary ? nfold_kernel<true> : nfold_kernel<false>);
  hipError_t e = hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(fn, dim3(n_chains), dim3(threads), lds, st, a);
  return hipGetLastError();
}

}  // namespace clexmc
