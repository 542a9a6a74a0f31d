// gfx950 kernels of the N-fold way (the body, shared with the run-time
// specialised kernels, is in clexmc_nfold.h).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "clexmc_nfold.h"

namespace clexmc {

size_t nfold_lds_bytes(int pad_sites, int n_sites, int nb_max, int nb_total, int n_sublat) {
  return nfold_lds(pad_sites, n_sites, nb_max, nb_total, n_sublat).bytes;
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
