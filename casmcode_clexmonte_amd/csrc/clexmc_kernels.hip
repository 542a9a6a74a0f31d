// gfx950 kernels of the clexmc Metropolis hot path.
//
//  metropolis_kernel   one workgroup per chain; the chain's occupation lives
//                      in LDS as a halo-padded image (int8 per site, or 2 bits
//                      per site packed 16 to a 32-bit word when the int8 image
//                      does not fit: up to 4 occupants); sites are updated
//                      class by class (independent sets: no cluster contains
//                      two sites of one class), so all proposals of a class
//                      are evaluated and applied concurrently and exactly.
//                      Binary (+-1) expansions use integer cluster-product
//                      counts per orbit (K_a, exact), FP32 dE = dphi*sum w_a K_a
//                      and exact int64 correlation counts C_a per chain; other
//                      expansions use FP32 flower tables (staged in LDS) and
//                      an FP64 running energy.  Philox4x32-10 supplies the
//                      uniforms; lane accumulators are reduced per wavefront
//                      with cross-lane shuffles.
//  delta_batch_kernel  per-proposal dE (BaseMontePotential::occ_delta_per_supercell)
//  corr_count_kernel   decoration counts per orbit and
//  corr_finish_kernel  full per-supercell correlations in FP64 from them
//  philox_kernel       device Philox for known-answer checks
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <type_traits>

#include "clexmc_device.h"
#include "clexmc_kernels.h"
#include "clexmc_metropolis.h"

namespace clexmc {

// ---------------------------------------------------------------------------
// Persistent Metropolis kernel (generic site programs)
// ---------------------------------------------------------------------------
template <bool BIN, int KIND, bool PACK>
__global__ __launch_bounds__(512) void metropolis_kernel(RunArgs args) {
  metropolis_body<BIN, KIND, PACK, GenericField>(args, BlockRole{(int)blockIdx.x, args.chain_map, args.slabs});
}

// binary path, two lanes per site in the class sweeps (up to 1024 threads)
template <int KIND, bool PACK>
__global__ __launch_bounds__(1024) void metropolis_split_kernel(RunArgs args) {
  metropolis_body<true, KIND, PACK, GenericField, 2>(args, BlockRole{(int)blockIdx.x, args.chain_map, args.slabs});
}

// ---------------------------------------------------------------------------
// Per-proposal dE on the unpadded occupation (periodic wrap): one wavefront
// per proposal, one cluster of the site per lane and turn, the FP32 table
// values times the FP32 site-function differences summed in FP64.  A proposal
// is bound by three dependent loads (cluster, occupants, table), so clusters
// run side by side: one swap on FCC 12^3 took 187 us in one thread and takes
// 8.9 us, 65,536 swaps on BCC 32^3 797 us and 214 us.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void delta_batch_kernel(DeltaArgs a) {
  const int p = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
  const int lane = threadIdx.x & 63;
  if (p >= a.n_prop) return;
  cptr<DevSystem> sys = cst(a.sys);
  const int chain = __builtin_amdgcn_readfirstlane(a.chain[p]);
  cptr<ChainParams> cp = cst(a.params + chain);
  cptr<DevSupercell> sc = cst(a.scs + cp->sc);
  const int8_t *__restrict__ occ = a.occ + cp->occ_offset;
  const int L1 = sc->L1, L2 = sc->L2, L3 = sc->L3, n_cells = sc->n_cells;
  const bool near = sc->h <= L1 && sc->h <= L2 && sc->h <= L3;  // a coordinate wraps by one period at most
  const int m = a.sites_per_prop;
  int site[kMaxSitesPerProp], nocc[kMaxSitesPerProp];
#pragma unroll
  for (int i = 0; i < kMaxSitesPerProp; ++i) {
    site[i] = i < m ? __builtin_amdgcn_readfirstlane(a.sites[(long long)p * m + i]) : -1;
    nocc[i] = i < m ? __builtin_amdgcn_readfirstlane(a.new_occ[(long long)p * m + i]) : 0;
  }
  double dE = 0.0;  // this lane's share
#pragma unroll
  for (int i = 0; i < kMaxSitesPerProp; ++i) {
    if (i >= m) break;
    const int l = site[i];
    const int b = l / n_cells;
    const int c = l - b * n_cells;
    const int i0 = c % L1, j0 = (c / L1) % L2, k0 = c / (L1 * L2);
    // occupant of site x with the earlier changes of this proposal applied
    auto occ_of = [&](int x) -> int {
      int o = occ[x];
#pragma unroll
      for (int j = 0; j < i; ++j) o = site[j] == x ? nocc[j] : o;
      return o;
    };
    const int o = __builtin_amdgcn_readfirstlane(occ_of(l));
    const int nw = nocc[i];
    if (nw == o) continue;
    const int nf = sys->n_func[b];
    double ds[kMaxFunc];
#pragma unroll
    for (int f = 0; f < kMaxFunc; ++f) ds[f] = f < nf ? (double)(sys->site_func[b][f][nw] - sys->site_func[b][f][o]) : 0.0;
    const int e1 = sys->flower_begin[b + 1];
    for (int e = sys->flower_begin[b] + lane; e < e1; e += 64) {
      int idx = 0;
      for (int q = sys->entry_site_begin[e]; q < sys->entry_site_begin[e + 1]; ++q) {
        const int4 d = sys->entry_sites[q];
        int ii = i0 + d.y, jj = j0 + d.z, kk = k0 + d.w;
        if (!near) {
          ii %= L1;
          jj %= L2;
          kk %= L3;
        }
        ii += ii < 0 ? L1 : 0;
        jj += jj < 0 ? L2 : 0;
        kk += kk < 0 ? L3 : 0;
        ii -= ii >= L1 ? L1 : 0;
        jj -= jj >= L2 ? L2 : 0;
        kk -= kk >= L3 ? L3 : 0;
        idx += occ_of(d.x * n_cells + ii + L1 * (jj + L2 * kk)) * sys->entry_mul[q];
      }
      const float *V = sys->flower_tables + sys->entry_table[e] + idx * nf;
      dE += ds[0] * (double)V[0];
      if (nf > 1) dE += ds[1] * (double)V[1];
      if (nf > 2) dE += ds[2] * (double)V[2];
    }
    if (a.include_chem && lane == 0) dE -= (double)(cp->chem[b * kMaxOcc + nw] - cp->chem[b * kMaxOcc + o]);
  }
  dE = wave_sum(dE);
  if (lane == 0) a.dE[p] = (float)dE;
}

// ---------------------------------------------------------------------------
// Full correlations.  An orbit's functions depend on its clusters only through
// how often each decoration tau occurs: corr_f = sum_tau count[tau] T[tau][f]
// / mult.  So the lattice is walked once per orbit, not once per function,
// with exact integer counts, and the FP64 sum runs over decorations.
//
// corr_count_kernel: a block counts the decorations of one orbit over a range
// of cells of one chain (grid: cell ranges of one orbit after the other, chains) in LDS, with up
// to 16 copies of every counter (by lane) so that the few decorations of a
// pair do not serialise the lanes.  `direct` (a chain's cells in one block):
// it forms the correlations at once.  Else the counts go to a.hist and
// corr_finish_kernel forms them, by the same sum (corr_sum): a chain's
// correlations do not depend on the form, and so not on the chains beside it.  Orbits with more than kCorrLdsBins
// decorations count in global memory.  Bound by the address arithmetic of the
// cluster sites (about 10 VALU operations per site).
// BCC quaternary 32^3, 8 chains loaded and every correlation read one chain
// at a time: 1.29 ms (counting 23 us per chain); one FP64 walk of the lattice
// per function took 17.2 ms.
// ---------------------------------------------------------------------------
constexpr int kCorrThreads = 512;
constexpr int kCorrLdsBins = 8192;  // counters in LDS (32 KB)

// decoration counts of one orbit over the cells [c0, c1); K: sites per
// cluster (-1: any), NEAR: every site offset is at most one period.  SHARE
// (fewer cells than threads): groups of wavefronts share the orbit's elements;
// one cell's elements one after the other are a chain of load latencies (BCC
// 8^3, correlations of one chain: 54 us, 35 us so with the sums below)
template <int K, bool NEAR, bool SHARE, class ADD>
__device__ __forceinline__ void corr_count(cptr<DevSystem> sys, const DevSupercell &sc, const int8_t *__restrict__ occ,
                                           const int4 *elem_sites, int ne, int k_rt, int c0, int c1, ADD add) {
  const int k = K >= 0 ? K : k_rt;
  const int L1 = sc.L1, L2 = sc.L2, L3 = sc.L3, n_cells = sc.n_cells;
  cptr<int4> es = cst(elem_sites);
  const int w = SHARE ? (c1 - c0 + 63) & ~63 : kCorrThreads, groups = SHARE ? kCorrThreads / w : 1;
  const int group = SHARE ? __builtin_amdgcn_readfirstlane((int)threadIdx.x / w) : 0;
  if (group >= groups) return;
  for (int c = c0 + (int)threadIdx.x - group * w; c < c1; c += w) {
    const int i0 = c % L1, j0 = (c / L1) % L2, k0 = c / (L1 * L2);
#pragma unroll 2
    for (int e = group; e < ne; e += groups) {
      int tau = 0, mul = 1;
#pragma unroll
      for (int q = 0; q < k; ++q) {
        const int bq = es[e * k + q].x, dy = es[e * k + q].y, dz = es[e * k + q].z, dw = es[e * k + q].w;
        int ii = i0 + dy, jj = j0 + dz, kk = k0 + dw;
        if (NEAR) {
          ii += ii < 0 ? L1 : 0;
          jj += jj < 0 ? L2 : 0;
          kk += kk < 0 ? L3 : 0;
          ii -= ii >= L1 ? L1 : 0;
          jj -= jj >= L2 ? L2 : 0;
          kk -= kk >= L3 ? L3 : 0;
        } else {
          ii %= L1;
          jj %= L2;
          kk %= L3;
          ii += ii < 0 ? L1 : 0;
          jj += jj < 0 ? L2 : 0;
          kk += kk < 0 ? L3 : 0;
        }
        tau += occ[bq * n_cells + ii + L1 * (jj + L2 * kk)] * mul;
        mul *= sys->n_occ[bq];
      }
      add(tau);
    }
  }
}

// Correlation f of an orbit from its decoration counts (count(t) occurrences of
// decoration t), one wavefront: products and sums carry their rounding errors
// along (Dekker's two-product by fma, Knuth's two-sum), so that the sum is
// rounded once before the division by the multiplicity.
template <class COUNT>
__device__ __forceinline__ double corr_sum(int ntau, const double *T, int nf, int f, int mult, COUNT count) {
#pragma clang fp contract(off)
  double hi = 0.0, lo = 0.0;
  auto add = [&](double p, double err) {
#pragma clang fp contract(off)
    const double s = hi + p, q = s - hi;
    lo += ((hi - (s - q)) + (p - q)) + err;
    hi = s;
  };
#pragma unroll 4
  for (int t = threadIdx.x & 63; t < ntau; t += 64) {
    const double n = (double)count(t), v = T[t * nf + f], p = n * v;
    if (n > 0.0) add(p, __builtin_fma(n, v, -p));
  }
  for (int o = 32; o > 0; o >>= 1) {
    const double h2 = __shfl_xor(hi, o), l2 = __shfl_xor(lo, o);
    add(h2, l2);
  }
  return (hi + lo) / (double)mult;
}

__global__ __launch_bounds__(kCorrThreads) void corr_count_kernel(CorrArgs a) {
  __shared__ unsigned bins[kCorrLdsBins];
  const int tid = threadIdx.x;
  const int orb = (int)blockIdx.x / a.n_ranges;
  const int chain = a.chain0 + blockIdx.y;
  cptr<DevSystem> sys = cst(a.sys);
  const ChainParams &cp = a.params[chain];
  const DevSupercell &sc = a.scs[cp.sc];
  const int8_t *__restrict__ occ = a.occ + cp.occ_offset;
  const int nf = sys->orbit_nfunc[orb];
  const int c0 = ((int)blockIdx.x - orb * a.n_ranges) * a.cells_per_block;
  if (nf <= 0 || c0 >= sc.n_cells) return;
  const int c1 = min(c0 + a.cells_per_block, sc.n_cells);
  const int k = sys->orbit_k_all[orb];
  const int ne = sys->corr_orbit_begin[orb + 1] - sys->corr_orbit_begin[orb];
  const int4 *es = sys->corr_elem_sites + sys->corr_elem_begin[orb];
  const int ntau = sys->orbit_ntau[orb];
  const bool in_lds = ntau <= kCorrLdsBins;
  int copies = 1;
  while (in_lds && copies < 16 && ntau * copies * 2 <= kCorrLdsBins) copies *= 2;
  unsigned long long *hist = a.hist ? a.hist + (long long)blockIdx.y * a.n_bins + sys->orbit_bin0[orb] : nullptr;
  if (in_lds)
    for (int t = tid; t < ntau * copies; t += kCorrThreads) bins[t] = 0u;
  __syncthreads();
  const bool near = a.elem_reach <= sc.L1 && a.elem_reach <= sc.L2 && a.elem_reach <= sc.L3;
  if (in_lds) {
    unsigned *mine = bins + (tid & (copies - 1));
    auto add = [&](int tau) { atomicAdd(&mine[tau * copies], 1u); };
    auto count = [&](auto share) {
      constexpr bool S = decltype(share)::value;
      if (!near) corr_count<-1, false, S>(sys, sc, occ, es, ne, k, c0, c1, add);
      else if (k == 1) corr_count<1, true, S>(sys, sc, occ, es, ne, k, c0, c1, add);
      else if (k == 2) corr_count<2, true, S>(sys, sc, occ, es, ne, k, c0, c1, add);
      else if (k == 3) corr_count<3, true, S>(sys, sc, occ, es, ne, k, c0, c1, add);
      else if (k == 4) corr_count<4, true, S>(sys, sc, occ, es, ne, k, c0, c1, add);
      else corr_count<-1, true, S>(sys, sc, occ, es, ne, k, c0, c1, add);
    };
    if (c1 - c0 <= kCorrThreads / 2) count(std::true_type{});
    else count(std::false_type{});
  } else {
    auto add = [&](int tau) { atomicAdd(&hist[tau], 1ull); };
    corr_count<-1, false, false>(sys, sc, occ, es, ne, k, c0, c1, add);
  }
  __syncthreads();
  if (!in_lds) return;
  // the copies of a counter, added from another one on in every lane (lanes a
  // multiple of the copies apart would read one LDS bank)
  for (int t = tid; t < ntau; t += kCorrThreads) {
    unsigned v = 0u;
    for (int q = 0; q < copies; ++q) v += bins[t * copies + ((q + t) & (copies - 1))];
    if (a.direct) bins[t * copies] = v;
    else if (v) atomicAdd(&hist[t], (unsigned long long)v);
  }
  if (!a.direct) return;
  __syncthreads();
  const double *T = sys->orbit_tables + sys->orbit_table_offset[orb];
  const int f0 = sys->orbit_func_begin[orb];
  for (int f = tid >> 6; f < nf; f += kCorrThreads / 64) {
    const double v = corr_sum(ntau, T, nf, f, sys->orbit_mult[orb],
                              [&](int t) -> unsigned long long { return bins[t * copies]; });
    if ((tid & 63) == 0) a.out[(long long)blockIdx.y * a.n_corr + f0 + f] = v;
  }
}

// correlations from the decoration counts: one block per (orbit, chain), one
// wavefront per function
__global__ __launch_bounds__(1024) void corr_finish_kernel(CorrArgs a) {
  const int orb = blockIdx.x;
  cptr<DevSystem> sys = cst(a.sys);
  const int nf = sys->orbit_nfunc[orb], f0 = sys->orbit_func_begin[orb], ntau = sys->orbit_ntau[orb];
  const double *T = sys->orbit_tables + sys->orbit_table_offset[orb];
  const unsigned long long *hist = a.hist + (long long)blockIdx.y * a.n_bins + sys->orbit_bin0[orb];
  for (int f = threadIdx.x >> 6; f < nf; f += 16) {
    const double v = corr_sum(ntau, T, nf, f, sys->orbit_mult[orb], [&](int t) { return hist[t]; });
    if ((threadIdx.x & 63) == 0) a.out[(long long)blockIdx.y * a.n_corr + f0 + f] = v;
  }
}

// The first n samples of every chain's row of `cap` samples, rows put next to
// each other (E, and the occupant counts as one int4 per sample; one block row
// per chain), so that a read is one contiguous copy: the row-by-row copy it
// replaces took 3.3 ms for 256 chains of 20 samples.  Bound by its launch.
__global__ __launch_bounds__(256) void pack_samples_kernel(const double *E, const int4 *N, int cap, int n, double *outE,
                                                           int4 *outN) {
  const int s = blockIdx.x * 256 + threadIdx.x;
  if (s >= n) return;
  const long long src = (long long)blockIdx.y * cap + s, dst = (long long)blockIdx.y * n + s;
  outE[dst] = E[src];
  outN[dst] = N[src];
}

__global__ void philox_kernel(int n, const uint4 *ctr, const uint2 *key, uint4 *out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = philox4x32_10(ctr[i], key[i].x, key[i].y);
}

// ---------------------------------------------------------------------------
// launch wrappers
// ---------------------------------------------------------------------------
// launch == false: only set the kernel's dynamic LDS limit (not a stream
// operation, so it stays outside graph capture)
template <bool BIN, int KIND, bool PACK>
static hipError_t launch_metro(const RunArgs &args, int n_chains, int threads, size_t lds, hipStream_t st,
                               bool launch) {
  auto kern = metropolis_kernel<BIN, KIND, PACK>;
  if (!launch) return hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  hipLaunchKernelGGL(kern, dim3(n_chains), dim3(threads), lds, st, args);
  return hipGetLastError();
}

template <int KIND, bool PACK>
static hipError_t launch_split(const RunArgs &args, int n_chains, int threads, size_t lds, hipStream_t st,
                               bool launch) {
  auto kern = metropolis_split_kernel<KIND, PACK>;
  if (!launch) return hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  hipLaunchKernelGGL(kern, dim3(n_chains), dim3(threads), lds, st, args);
  return hipGetLastError();
}

hipError_t launch_metropolis_split(const RunArgs &args, int kind, bool packed, int n_chains, int threads, size_t lds,
                                   hipStream_t st, bool launch) {
  if (packed)
    return kind == 0 ? launch_split<0, true>(args, n_chains, threads, lds, st, launch)
                     : launch_split<1, true>(args, n_chains, threads, lds, st, launch);
  return kind == 0 ? launch_split<0, false>(args, n_chains, threads, lds, st, launch)
                   : launch_split<1, false>(args, n_chains, threads, lds, st, launch);
}

hipError_t launch_metropolis(const RunArgs &args, bool binary, int kind, bool packed, int n_chains, int threads,
                             size_t lds, hipStream_t st, bool launch) {
  // kind 0 canonical, 1 semi-grand canonical, 2 semi-grand canonical with multiswaps
  if (packed) {
    if (binary)
      return kind == 0   ? launch_metro<true, 0, true>(args, n_chains, threads, lds, st, launch)
             : kind == 1 ? launch_metro<true, 1, true>(args, n_chains, threads, lds, st, launch)
                         : launch_metro<true, 2, true>(args, n_chains, threads, lds, st, launch);
    return kind == 0   ? launch_metro<false, 0, true>(args, n_chains, threads, lds, st, launch)
           : kind == 1 ? launch_metro<false, 1, true>(args, n_chains, threads, lds, st, launch)
                       : launch_metro<false, 2, true>(args, n_chains, threads, lds, st, launch);
  }
  if (binary)
    return kind == 0   ? launch_metro<true, 0, false>(args, n_chains, threads, lds, st, launch)
           : kind == 1 ? launch_metro<true, 1, false>(args, n_chains, threads, lds, st, launch)
                       : launch_metro<true, 2, false>(args, n_chains, threads, lds, st, launch);
  return kind == 0   ? launch_metro<false, 0, false>(args, n_chains, threads, lds, st, launch)
         : kind == 1 ? launch_metro<false, 1, false>(args, n_chains, threads, lds, st, launch)
                     : launch_metro<false, 2, false>(args, n_chains, threads, lds, st, launch);
}

// ---------------------------------------------------------------------------
// After a slab launch (RunArgs::slabs > 1), one thread per chain: sums the
// slabs' records in pass order (what each slab had added since the launch
// started, at every sampled pass and at the last pass), writes the samples,
// then the chain's energy, counts and exact binary counts, and advances the
// pass and draw counters, which the slabs read but do not change.
// ---------------------------------------------------------------------------
__global__ void slab_post_kernel(RunArgs a, int n_chains) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n_chains) return;
  const int chain = a.chain_map ? a.chain_map[i] : i;
  const DevSystem *sys = a.sys;
  ChainState *cs = a.state + chain;
  const bool bin = sys->binary != 0;
  long long *C = a.binC + (long long)chain * a.n_orbits;
  const double E0 = cs->E;
  const unsigned long long pass0 = cs->pass_base;
  constexpr int nI = kMaxSlots + kMaxOcc + 2;
  long long tot[nI];
  double totE = 0.0;
  int j = 0;
  for (int p = 0; p < a.n_passes; ++p) {
    const bool due = ((pass0 + (unsigned long long)p + 1ull) % (unsigned long long)a.sample_period) == 0ull;
    if (!due && p != a.n_passes - 1) continue;
    for (int q = 0; q < nI; ++q) tot[q] = 0;
    totE = 0.0;
    for (int s = 0; s < a.slabs; ++s) {
      const SlabRecord &r = a.slab_rec[((long long)chain * kSlabMax + s) * kSlabRecords + j];
      totE += r.dE;
      for (int q = 0; q < nI; ++q) tot[q] += r.dI[q];
    }
    ++j;
    if (!due) continue;
    double E;
    if (bin) {
      E = 0.0;
      for (int o = 0; o < a.n_orbits; ++o) {
        long long c = C[o];
        for (int q = 0; q < sys->n_slots; ++q)
          if (sys->slot_orbit[q] == o) c += tot[q];
        E += sys->bin_w64[o] * (double)c;
      }
    } else {
      E = E0 + totE;
    }
    long long cnt[kMaxOcc];
    for (int q = 0; q < kMaxOcc; ++q) cnt[q] = cs->counts[q] + tot[kMaxSlots + q];
    const int idx = a.sample_count[chain];
    if (idx < a.sample_cap) {
      const long long o = (long long)chain * a.sample_cap + idx;
      a.sampE[o] = E;
      for (int q = 0; q < kMaxOcc; ++q) a.sampN[o * kMaxOcc + q] = (int)cnt[q];
      a.sample_count[chain] = idx + 1;
    }
    const double n1 = (double)cnt[1];
    cs->sumE += E;
    cs->sumE2 += E * E;
    cs->sumN1 += n1;
    cs->sumN12 += n1 * n1;
    cs->sumEN1 += E * n1;
    cs->n_samples_acc += 1;
  }
  // the last record holds the launch's totals
  if (bin) {
    for (int q = 0; q < sys->n_slots; ++q) C[sys->slot_orbit[q]] += tot[q];
    double E = 0.0;
    for (int o = 0; o < a.n_orbits; ++o) E += sys->bin_w64[o] * (double)C[o];
    cs->E = E;
  } else {
    cs->E = E0 + totE;
  }
  for (int q = 0; q < kMaxOcc; ++q) cs->counts[q] += tot[kMaxSlots + q];
  cs->n_attempt += tot[kMaxSlots + kMaxOcc];
  cs->n_accept += tot[kMaxSlots + kMaxOcc + 1];
  cs->pass_base += (unsigned long long)a.n_passes;
  const unsigned long long next = cs->draw_hi + 1ull;
  if (next > cs->draw_base) cs->draw_base = next;
}

hipError_t launch_slab_post(const RunArgs &a, int n_chains, hipStream_t st) {
  if (n_chains <= 0) return hipSuccess;
  hipLaunchKernelGGL(slab_post_kernel, dim3((n_chains + 63) / 64), dim3(64), 0, st, a, n_chains);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// LDS read-throughput probe: every lane reads LDS in a loop and folds the
// values into a checksum (written out so that nothing is optimised away).
// mode 0: byte gathers, lanes of a wavefront 3 bytes apart (the stride of
// independent-set class sites along a row) at 8 offsets per iteration;
// mode 1: 16-byte reads, lanes 16 bytes apart (bank-conflict free).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(512) void lds_probe_kernel(int mode, int iters, unsigned *sink) {
  extern __shared__ __align__(16) unsigned char lds[];
  const int tid = threadIdx.x;
  const int bytes = 32768;
  for (int i = tid; i < bytes / 4; i += blockDim.x) ((unsigned *)lds)[i] = (unsigned)(i * 2654435761u);
  __syncthreads();
  unsigned acc = 0u;
  if (mode == 0) {
    const int base = (tid & 63) * 3 + (tid >> 6) * 211;
    for (int it = 0; it < iters; ++it) {
      const int o = (it * 97) & 4095;
#pragma unroll
      for (int k = 0; k < 8; ++k) acc += lds[(base + o + k * 401) & (bytes - 1)];
    }
  } else {
    const uint4 *v = (const uint4 *)lds;
    const int base = tid & 511;
    for (int it = 0; it < iters; ++it) {
      const int o = (it * 64) & 1023;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const uint4 x = v[(base + o + k * 256) & 2047];
        acc += x.x ^ x.y ^ x.z ^ x.w;
      }
    }
  }
  sink[blockIdx.x * blockDim.x + tid] = acc;
}

hipError_t launch_lds_probe(int mode, int iters, int blocks, unsigned *sink, hipStream_t st) {
  hipLaunchKernelGGL(lds_probe_kernel, dim3(blocks), dim3(512), 32768, st, mode, iters, sink);
  return hipGetLastError();
}

// Staging array of clexmc_delta_energy_batch_noalloc: each GPU holds its own
// copy at its own address until the process ends.  Host code never passes
// the name itself to a kernel (in host code it is a stand-in, not a device
// address); it uses the address hipGetSymbolAddress returns for the device.
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

hipError_t noalloc_scratch(int device, unsigned char **ptr) {
  static std::mutex mu;
  static std::map<int, unsigned char *> by_device;
  std::lock_guard<std::mutex> lock(mu);
  auto it = by_device.find(device);
  if (it != by_device.end()) {
    *ptr = it->second;
    return hipSuccess;
  }
  void *p = nullptr;
  const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess) return e;
  by_device[device] = (unsigned char *)p;
  *ptr = (unsigned char *)p;
  return hipSuccess;
}

hipError_t launch_delta_batch(const DeltaArgs &a, hipStream_t st) {
  hipLaunchKernelGGL(delta_batch_kernel, dim3((unsigned)(((long long)a.n_prop + 3) / 4)), dim3(256), 0, st, a);
  return hipGetLastError();
}

bool corr_direct(long long max_cells, int max_elem, int max_ntau) {
  // one block per (orbit, chain) up to 32,768 clusters: the two further
  // launches of the split form (about 10 us) cost more than the longer loop
  return max_cells * max_elem <= 32768 && max_ntau <= kCorrLdsBins;
}

// cells per block of the split form: about 64K clusters of the largest orbit,
// fewer while that leaves the device short of blocks, at least one per thread
int corr_cells_per_block(long long max_cells, int max_elem, int n_orbits, int n_chains, int n_cu) {
  long long cells = std::max(1, 65536 / std::max(1, max_elem));
  cells = std::max(cells, max_cells * n_orbits >> 30);  // (the grid is bounded)
  while (cells > kCorrThreads && (max_cells + cells - 1) / cells * n_orbits * n_chains < 4ll * n_cu) cells /= 2;
  return (int)((cells + kCorrThreads - 1) / kCorrThreads * kCorrThreads);
}

hipError_t launch_corr(const CorrArgs &a, long long max_cells, int n_orbits, int n_chains, hipStream_t st) {
  // the grid's y extent is bounded: chains in slices
  for (int z0 = 0; z0 < n_chains; z0 += 32768) {
    CorrArgs s = a;
    const int nz = std::min(32768, n_chains - z0);
    s.chain0 = a.chain0 + z0;
    s.out = a.out + (long long)z0 * a.n_corr;
    if (a.hist) s.hist = a.hist + (long long)z0 * a.n_bins;
    s.n_ranges = a.direct ? 1 : (int)((max_cells + a.cells_per_block - 1) / a.cells_per_block);
    hipLaunchKernelGGL(corr_count_kernel, dim3((unsigned)s.n_ranges * n_orbits, nz), dim3(kCorrThreads), 0, st, s);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess && !a.direct) {
      hipLaunchKernelGGL(corr_finish_kernel, dim3(n_orbits, nz), dim3(1024), 0, st, s);
      e = hipGetLastError();
    }
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_pack_samples(const double *E, const int *N, int cap, int n_samples, int n_chains, double *outE,
                               int *outN, hipStream_t st) {
  static_assert(kMaxOcc == 4, "occupant counts of a sample are one int4");
  for (int c0 = 0; c0 < n_chains; c0 += 32768) {
    const int nc = std::min(32768, n_chains - c0);
    hipLaunchKernelGGL(pack_samples_kernel, dim3((n_samples + 255) / 256, nc), dim3(256), 0, st, E + (size_t)c0 * cap,
                       (const int4 *)N + (size_t)c0 * cap, cap, n_samples, outE + (size_t)c0 * n_samples,
                       (int4 *)outN + (size_t)c0 * n_samples);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_philox(int n, const uint4 *ctr, const uint2 *key, uint4 *out, hipStream_t st) {
  hipLaunchKernelGGL(philox_kernel, dim3((n + 63) / 64), dim3(64), 0, st, n, ctr, key, out);
  return hipGetLastError();
}

size_t metropolis_lds_bytes(int pad_sites, int n_tab, bool binary, int n_func_max, int max_class, bool packed) {
  size_t img = (size_t)image_bytes(pad_sites, packed);
  size_t tab = binary ? 0 : (size_t)((n_tab * 4 + 15) & ~15);
  const int n_islot = (binary ? kMaxSlots : 0) + kMaxOcc + 2;
  size_t red = (size_t)n_islot * 16 * sizeof(int) + 16 * sizeof(double) + 16 + 128 + kMswapLdsBytes +
               kChainLdsBytes;
  const int nfs = binary ? 1 : n_func_max;
  size_t scratch = (size_t)nfs * max_class * sizeof(float) + (binary ? (size_t)kMaxSlots * max_class : 0);
  return img + tab + red + scratch + 64;
}

}  // namespace clexmc
