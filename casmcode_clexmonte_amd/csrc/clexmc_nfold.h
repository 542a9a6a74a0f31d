// Device code of the N-fold way (rejection-free, Bortz-Kalos-Lebowitz) semi-grand canonical
// sampling: the reference's nfold method
// (include/casm/clexmonte/nfold/nfold_impl.hh:18-98: events are the
// semi-grand canonical changes of single sites; rates
// src/casm/clexmonte/nfold/nfold_events.cc:28-62: 1 if dE <= 0, else
// exp(-beta dE), dE the semi-grand potential change).
//
// The events are those of the plain semi-grand canonical proposal (a site
// and a uniformly chosen other occupant): a site's rate is the mean
// Metropolis acceptance of its changes, (1/(n_occ-1)) sum_o' min(1,
// exp(-beta dOmega)); binary expansions have one change per site.
//
// One workgroup per chain.  LDS holds the padded int8 image, the FP32 rate
// of every site and FP64 sums of the rates over groups of 64 sites.  Per
// event:
//  * wavefront 0 forms the total rate R (FP64), draws a 53-bit uniform u,
//    finds the group by a scan over per-lane chunks of group sums, then the
//    site by a scan of the group's 64 rates (FP64 wavefront scans), so a rate
//    is drawn in proportion to its value however small it is next to R;
//  * wavefront 0 applies the change (the new occupant drawn in proportion to
//    its rate; every periodic copy of the site, one per lane), then the lanes
//    recompute the rates of the site and of its interaction neighbours (each
//    neighbour once), and the sum of every group holding one of them is
//    formed again from its 64 rates, four lanes per group;
//  * meanwhile one lane of the last wavefront (OWN_BOOKS: afterwards one lane
//    of the first) weights the state the event leaves by its expected residence time w = n_mutable / R in Metropolis
//    steps (the jump chain visits states in proportion to pi(x) R(x); weights
//    1/R recover pi) and keeps the counts (binary: exact integer cluster
//    counts, general: FP64 energy).
//    Group sums are never updated by differences, so they carry no
//    cancellation error when rates of very different size come and go;
//  * if R falls below 1e-30 (every rate of the chain within a few decades of
//    FP32 underflow, beta dE > ~69 for all changes) the chain stops and
//    records the condition in its state; the host reports it as an error.
//
// nfold_body<BIN, FIELD>: FIELD is GenericField (interpreted site programs,
// clexmc_nfold.hip) or the run-time specialised JitField (clexmc_jit.cpp);
// both sum the clusters in the same order, so the results are identical.
#pragma once
#include "clexmc_metropolis.h"

namespace clexmc {

// LDS of an N-fold workgroup: byte offsets behind the padded image
struct NfoldLds {
  size_t rate;   // [n_groups * 64] FP32 rates, zero past n_sites (rate_at)
  size_t G;      // [n_groups] FP64 group sums
  size_t aff;    // [nb_max] linear indices of the sites whose rates change
  size_t affp;   // [nb_max] their padded addresses
  size_t sel;    // the event's record (kNfoldSelBytes)
  size_t nb_begin;  // [n_sublat + 1] starts of the neighbour lists
  size_t nb;     // [nb_total] sublattice, di, dj, dk of a neighbour, a byte each
  size_t n_occ;  // [n_sublat]
  size_t chem;   // [n_sublat][kMaxOcc]
  size_t bytes;
};
__host__ __device__ inline NfoldLds nfold_lds(int pad_sites, int n_sites, int nb_max, int nb_total, int n_sublat) {
  auto up = [](size_t x) { return (x + 15) & ~(size_t)15; };
  const size_t n_groups = (size_t)((n_sites + 63) / 64);
  NfoldLds o;
  o.rate = (size_t)image_bytes(pad_sites, false);
  o.G = o.rate + n_groups * 64 * 4;
  o.aff = o.G + up(n_groups * 8);
  o.affp = o.aff + up((size_t)nb_max * 4);
  o.sel = o.affp + up((size_t)nb_max * 4);
  o.nb_begin = o.sel + kNfoldSelBytes;
  o.nb = o.nb_begin + kNfoldNbBeginBytes;
  o.n_occ = o.nb + up((size_t)nb_total * 4);
  o.chem = o.n_occ + (size_t)n_sublat * 4;
  o.bytes = o.chem + (size_t)n_sublat * kMaxOcc * 4;
  return o;
}
__host__ __device__ inline uint32_t nfold_pack_nb(int b, int di, int dj, int dk) {
  return (uint32_t)(b & 0xff) | (uint32_t)(di & 0xff) << 8 | (uint32_t)(dj & 0xff) << 16 | (uint32_t)(dk & 0xff) << 24;
}
__host__ __device__ inline int4 nfold_unpack_nb(uint32_t v) {
  return make_int4((int)(v & 0xff), (int)(int8_t)(v >> 8), (int)(int8_t)(v >> 16), (int)v >> 24);
}

// x of the lane that DPP control CTRL names (0 where it names none, and in
// the rows ROW_MASK leaves out), the two halves moved separately
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ double dpp_d(double x) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(x);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, ROW_MASK, 0xf, false);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, ROW_MASK, 0xf, false);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Inclusive prefix sum (FP64) over the 64 lanes of a full wave: shifted adds
// within rows of 16 lanes (DPP row_shr 1, 2, 4, 8), then row 0's total into
// row 1 and row 2's into row 3 (row_bcast 15), then rows 0-1's total into
// rows 2-3 (row_bcast 31).  VALU only: no LDS round trips.
__device__ __forceinline__ double wave_scan_incl_d(double v) {
  v += dpp_d<0x111, 0xf>(v);
  v += dpp_d<0x112, 0xf>(v);
  v += dpp_d<0x114, 0xf>(v);
  v += dpp_d<0x118, 0xf>(v);
  v += dpp_d<0x142, 0xa>(v);
  v += dpp_d<0x143, 0xc>(v);
  return v;
}

// x of lane l (l the same in every lane)
__device__ __forceinline__ double lane_d(double x, int l) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(x);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, l);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), l);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Orders the wavefront's LDS accesses: what any lane stored before, every lane
// reads after.  (No instruction: a wavefront's LDS operations are in order; the
// compiler must keep them so.)
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// first lane whose inclusive prefix exceeds t; if rounding leaves none, the
// last lane with a positive value (-1 if there is none)
__device__ __forceinline__ int pick_lane(double incl, double v, double t) {
  const unsigned long long m = __ballot(incl > t && v > 0.0);
  if (m) return __ffsll((long long)m) - 1;
  const unsigned long long m2 = __ballot(v > 0.0);
  return m2 ? 63 - __clzll((long long)m2) : -1;
}

// uniform double in [0, 1) from 53 random bits of two words
__device__ __forceinline__ double u01_53(uint32_t a, uint32_t b) {
  return ((double)(a >> 5) * 67108864.0 + (double)(b >> 6)) * (1.0 / 9007199254740992.0);
}

// Place of site l's rate: its group's 64 rates stay together, but the 16
// blocks of four are permuted by the group number, so that lanes that walk
// different groups in step read different LDS banks (with plain rows every
// group's block q lies in the same four banks: 860 conflict cycles per event)
__host__ __device__ __forceinline__ int rate_at(int l) {
  return (l & ~63) | ((((l >> 2) ^ (l >> 6)) & 15) << 2) | (l & 3);
}

// Sum of the 64 FP32 rates of group g in FP64: lane q of a quad adds the rates
// 4 p + q, p = 0..15, then (q0 + q1) + (q2 + q3) over the quad (DPP), so the
// order is fixed and every lane of the quad has the sum.  All four lanes must
// be active.
__device__ __forceinline__ double group_rate_sum(const float *rate, int g, int q) {
  const float *r = rate + g * 64 + q;
  double a = 0.0;
#pragma unroll
  for (int p = 0; p < 16; ++p) a += (double)r[(p ^ (g & 15)) << 2];
  a += dpp_d<0xB1, 0xf>(a);
  return a + dpp_d<0x4E, 0xf>(a);
}
// the same sum, bit for bit, in one lane (in one or two wavefronts four lanes
// per group would take four times the turns)
__device__ __forceinline__ double group_rate_sum_lane(const float *rate, int g) {
  const float4 *r = (const float4 *)(rate + g * 64);
  double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
#pragma unroll
  for (int p = 0; p < 16; ++p) {
    const float4 v = r[p ^ (g & 15)];
    a0 += (double)v.x;
    a1 += (double)v.y;
    a2 += (double)v.z;
    a3 += (double)v.w;
  }
  return (a0 + a1) + (a2 + a3);
}

// x / d for 0 <= x < 2^18 and 1 <= d < 2^14 or d > x, by one high product (on
// the scalar unit for a uniform x): m = floor(2^32 / d) + 1 exceeds 2^32 / d
// by at most 1, so x m / 2^32 exceeds x / d by less than 2^-14 < 1 / d (and
// by less than 2^-14 below 1 for d > x); d = 1 has m = 0.  Fewer than 2^15
// sites (kNfoldMaxLds) keep x and d there: a d of 2^14 or more is the cells of
// the one sublattice, or an axis longer than the site's index.
__host__ __device__ __forceinline__ uint32_t div_magic(int d) {
  return d > 1 ? (uint32_t)(4294967296ull / (uint32_t)d) + 1u : 0u;
}
__host__ __device__ __forceinline__ int div_small(int x, uint32_t m) {
  return m ? (int)(((unsigned long long)(uint32_t)x * m) >> 32) : x;
}

// The padded image of a supercell (cells of one sublattice after the other)
struct NfoldShape {
  int L1, L2, L3, h, P1, P12, S, n_cells;
  bool near;  // h <= L on every axis: a coordinate wraps by one period at most
};
// Neighbour o (nfold_unpack_nb; offsets within the halo) of the site in cell
// (i, j, k): its linear index and its address in the padded image.
__host__ __device__ __forceinline__ void nfold_place(const NfoldShape &g, const int4 &o, int i, int j, int k, int &lt,
                                                     int &pt) {
  int it = i + o.y, jt = j + o.z, kt = k + o.w;
  if (g.near) {
    it += it < 0 ? g.L1 : 0;
    jt += jt < 0 ? g.L2 : 0;
    kt += kt < 0 ? g.L3 : 0;
    it -= it >= g.L1 ? g.L1 : 0;
    jt -= jt >= g.L2 ? g.L2 : 0;
    kt -= kt >= g.L3 ? g.L3 : 0;
  } else {
    it = pad_wrap(it + g.h, g.h, g.L1);
    jt = pad_wrap(jt + g.h, g.h, g.L2);
    kt = pad_wrap(kt + g.h, g.h, g.L3);
  }
  lt = o.x * g.n_cells + it + g.L1 * (jt + g.L2 * kt);
  pt = o.x * g.S + (kt + g.h) * g.P12 + (jt + g.h) * g.P1 + (it + g.h);
}
// Address a of a copy of the site in cell (i, j, k) of sublattice b, per axis
// shifted by 0 (digit 0), +1 (1) or -1 (2) period, and whether the image has
// such a copy (near shapes only).
__host__ __device__ __forceinline__ bool nfold_copy(const NfoldShape &g, int cpi, int cpj, int cpk, int b, int i, int j,
                                                   int k, int &a) {
  const int qi = i + g.h + (cpi == 1 ? g.L1 : (cpi == 2 ? -g.L1 : 0)), qj = j + g.h + (cpj == 1 ? g.L2 : (cpj == 2 ? -g.L2 : 0)),
            qk = k + g.h + (cpk == 1 ? g.L3 : (cpk == 2 ? -g.L3 : 0));
  const bool vi = cpi == 0 || (cpi == 1 ? i < g.h : i >= g.L1 - g.h), vj = cpj == 0 || (cpj == 1 ? j < g.h : j >= g.L2 - g.h),
             vk = cpk == 0 || (cpk == 1 ? k < g.h : k >= g.L3 - g.h);
  a = b * g.S + qk * g.P12 + qj * g.P1 + qi;
  return vi && vj && vk;
}

// smallest total rate a chain may reach before it stops with an error
constexpr double kNfoldMinTotalRate = 1e-30;

// The books of a chain, kept by one lane: the energy and occupant counts of the
// state it is in, the moments of the current block and the time samples.
template <bool BIN>
struct NfoldBooks {
  long long C[kMaxSlots];        // binary: cluster-count changes per slot
  long long cnt[kMaxOcc], n_done;
  double E_run;                  // general: running energy
  double mom[kNfoldBlockSums];   // residence-weighted moments (kNfoldBlockSums layout)
  double n_mutable, T_now;
  // binary: the weight of each slot's orbit, read once (the energy of a state
  // is formed at every event), and the energy of the exact counts at launch
  double wslot[kMaxSlots], E0;
  int s_base, n_rec;

  __device__ __forceinline__ void open(const NfoldArgs &na, cptr<DevSystem> sys, const ChainState *cs, int chain,
                                       int n_cells) {
    const RunArgs &args = na.a;
#pragma unroll
    for (int q = 0; q < kMaxOcc; ++q) cnt[q] = cs->counts[q];
    E_run = cs->E;
#pragma unroll
    for (int q = 0; q < kNfoldBlockSums; ++q) mom[q] = 0.0;
    n_done = 0;
    n_mutable = 0.0;
    for (int b = 0; b < sys->n_sublat; ++b)
      if (sys->n_occ[b] >= 2) n_mutable += (double)n_cells;
#pragma unroll
    for (int j = 0; j < kMaxSlots; ++j) {
      C[j] = 0;
      wslot[j] = (BIN && j < sys->n_slots) ? sys->bin_w64[sys->slot_orbit[j]] : 0.0;
    }
    E0 = 0.0;
    if (BIN) {
      const long long *C0 = args.binC + (long long)chain * args.n_orbits;
      for (int a = 0; a < args.n_orbits; ++a) E0 += sys->bin_w64[a] * (double)C0[a];
    }
    // (the sample storage is only passed in for time sampling)
    s_base = na.n_time_samples > 0 ? args.sample_count[chain] : 0;
    T_now = 0.0;
    n_rec = 0;
  }

  // The state the event leaves, weighted by its expected Metropolis steps (R:
  // its total rate); true: time sampling has taken every sample.
  __device__ __forceinline__ bool leave(const NfoldArgs &na, int chain, int n_slots, double R) {
    const RunArgs &args = na.a;
    double E = E0;
    if (BIN) {
#pragma unroll
      for (int j = 0; j < kMaxSlots; ++j)
        if (j < n_slots) E += wslot[j] * (double)C[j];
    } else {
      E = E_run;
    }
    const double w = n_mutable / R;
    // every sample time in this state's residence interval
    // [T, T + w / n_mutable) (in passes) samples it
    if (na.n_time_samples > 0) {
      const double t1 = T_now + w / n_mutable;
      while (n_rec < na.n_time_samples && (double)n_rec * na.sample_dt < t1) {
        const long long so = (long long)chain * args.sample_cap + (s_base + n_rec);
        args.sampE[so] = E;
#pragma unroll
        for (int q = 0; q < kMaxOcc; ++q) args.sampN[so * kMaxOcc + q] = (int)cnt[q];
        ++n_rec;
      }
      T_now = t1;
    }
    mom[0] += w;
    mom[1] += w * E;
    mom[2] += w * E * E;
    int t = 0;
#pragma unroll
    for (int o = 0; o < kMaxOcc; ++o) {
      const double wn = w * (double)cnt[o];
      mom[3 + o] += wn;
      mom[17 + o] += wn * E;
#pragma unroll
      for (int q = o; q < kMaxOcc; ++q, ++t) mom[7 + t] += wn * (double)cnt[q];
    }
    return na.n_time_samples > 0 && n_rec >= na.n_time_samples;
  }

  // Event `ev` has been applied; sel: its record.
  __device__ __forceinline__ void applied(const NfoldArgs &na, int chain, int ev, const int *sel) {
    const int o = sel[4], nw = sel[5];
    if (BIN) {
      const int sk = o ? -2 : 2;
#pragma unroll
      for (int a = 0; a < kMaxSlots; ++a) C[a] += (long long)sk * sel[8 + a];
    } else {
      E_run += (double)__int_as_float(sel[6]);
    }
#pragma unroll
    for (int q = 0; q < kMaxOcc; ++q) cnt[q] += (q == nw ? 1 : 0) - (q == o ? 1 : 0);
    ++n_done;
    if ((ev + 1) % na.events_per_block == 0) {
      const int blk = (ev + 1) / na.events_per_block - 1;
      if (blk < na.n_blocks) {
        double *out = na.blocks + ((long long)chain * na.n_blocks + blk) * kNfoldBlockSums;
#pragma unroll
        for (int q = 0; q < kNfoldBlockSums; ++q) out[q] = mom[q];
      }
#pragma unroll
      for (int q = 0; q < kNfoldBlockSums; ++q) mom[q] = 0.0;
    }
  }

  __device__ __forceinline__ void close(const NfoldArgs &na, cptr<DevSystem> sys, ChainState *cs, int chain,
                                        int n_slots, unsigned long long ev0) const {
    const RunArgs &args = na.a;
    if (BIN) {
      long long *Cg = args.binC + (long long)chain * args.n_orbits;
#pragma unroll
      for (int j = 0; j < kMaxSlots; ++j)
        if (j < n_slots) Cg[sys->slot_orbit[j]] += C[j];
      double E = 0.0;
      for (int a = 0; a < args.n_orbits; ++a) E += sys->bin_w64[a] * (double)Cg[a];
      cs->E = E;
    } else {
      cs->E = E_run;
    }
#pragma unroll
    for (int q = 0; q < kMaxOcc; ++q) cs->counts[q] = cnt[q];
    if (na.n_time_samples > 0) args.sample_count[chain] = s_base + n_rec;
    cs->n_attempt += n_done;
    cs->n_accept += n_done;
    cs->pass_base = ev0 + (unsigned long long)na.n_events;
  }
};

// OWN_BOOKS: the first wavefront keeps the books as well, after each event,
// instead of a wavefront of their own (many chains per compute unit).
template <bool BIN, class FIELD, bool OWN_BOOKS = false>
__device__ __forceinline__ void nfold_body(const NfoldArgs &na) {
  extern __shared__ __align__(16) unsigned char smem[];
  const RunArgs &args = na.a;
  const int chain = blockIdx.x;
  const int tid = threadIdx.x;
  const int nthr = blockDim.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n_waves = nthr >> 6;
  cptr<DevSystem> sys = cst(args.sys);
  cptr<ChainParams> cp = cst(args.params + chain);
  ChainState *cs = args.state + chain;
  cptr<DevSupercell> sc = cst(args.scs + cp->sc);

  const int L1 = sc->L1, L2 = sc->L2, L3 = sc->L3, h = sc->h;
  const int P1 = sc->P1, P12 = sc->P1 * sc->P2, S = sc->S;
  const int n_cells = sc->n_cells, n_sites = sc->n_sites, pad_bytes = sc->pad_bytes;
  const int n_slots = sys->n_slots;
  const int n_groups = (n_sites + 63) / 64;

  ImgU8 img;
  img.p = (uint8_t *)smem;
  const NfoldLds lds = nfold_lds(pad_bytes, n_sites, sc->nb_max, sc->nb_begin[sys->n_sublat], sys->n_sublat);
  float *rate = (float *)(smem + lds.rate);
  double *G = (double *)(smem + lds.G);
  int *aff = (int *)(smem + lds.aff);
  int *affp = (int *)(smem + lds.affp);
  // the event: [0] site (-2: stopped), [1], [2] random words, [3] time
  // sampling complete, [4], [5] old and new occupant, [6] energy change (FP32,
  // general), [8..] cluster sums of the flipped site, and the total rate
  int *sel = (int *)(smem + lds.sel);
  double *selR = (double *)(sel + 16);
  // the interaction-neighbour offsets of every sublattice, staged once: an
  // event reads them right after its flip
  int *nbB = (int *)(smem + lds.nb_begin);
  uint32_t *nbL = (uint32_t *)(smem + lds.nb);
  // occupant counts and chemical potentials per sublattice: the rate of a
  // neighbour reads them for its sublattice (a per-lane index)
  int *noccL = (int *)(smem + lds.n_occ);
  float *chemL = (float *)(smem + lds.chem);

  // ---- padded image, neighbour lists
  const int8_t *__restrict__ occG = args.occ + cp->occ_offset;
  for (int p = tid; p < pad_bytes; p += nthr) {
    const int b = p / S;
    const int r = p - b * S;
    const int pk = r / P12, pj = (r - pk * P12) / P1, pi = r - pk * P12 - pj * P1;
    const int i = pad_wrap(pi, h, L1), j = pad_wrap(pj, h, L2), k = pad_wrap(pk, h, L3);
    img.p[p] = (uint8_t)occG[b * n_cells + i + L1 * (j + L2 * k)];
  }
  {
    const int n_sub = sys->n_sublat;
    const int nb_tot = sc->nb_begin[n_sub];
    for (int t = tid; t < nb_tot; t += nthr) {
      const int4 o = sc->nb_cell[t];
      nbL[t] = nfold_pack_nb(o.x, o.y, o.z, o.w);
    }
    if (tid <= n_sub) nbB[tid] = sc->nb_begin[tid];
    if (tid < n_sub) noccL[tid] = sys->n_occ[tid];
    if (tid < n_sub * kMaxOcc) chemL[tid] = cp->chem[tid];
  }
  __syncthreads();
  const int P3 = S / P12;
  const float beta = cp->beta;
  cptr<int> bin_off = cst(sc->bin_off);
  auto main_addr = [&](int l) {
    const int b = l / n_cells;
    const int c = l - b * n_cells;
    const int i = c % L1, j = (c / L1) % L2, k = c / (L1 * L2);
    return b * S + (k + h) * P12 + (j + h) * P1 + (i + h);
  };
  const float *tab = sys->flower_tables;
  cptr<int> gen_prog = cst(sc->gen_prog);
  const FieldCtx fctx{sc, bin_off, gen_prog, n_slots};
  // rate of one change o -> nw of a general site with cluster sums G
  auto change_rate = [&](int b, int o, int nw, const float (&G)[kMaxFunc]) -> float {
    const float dE = general_dE(sys, b, o, nw, G) - (chemL[b * kMaxOcc + nw] - chemL[b * kMaxOcc + o]);
    return dE <= 0.0f ? 1.0f : __expf(-beta * dE);
  };
  // rate of the site at padded address pa on sublattice b (0 for fixed
  // sites); binary: its cluster sums K (which do not depend on the site itself)
  auto site_rate_at = [&](int b, int pa, int (&K)[kMaxSlots]) -> float {
    const int no = noccL[b];
    if (no < 2) return 0.0f;
    const int o = img.get(pa);
    if (BIN) {
      const float F = FIELD::bin(fctx, img, b, pa, o, K);
      const float chem0 = chemL[b * kMaxOcc + 0], chem1 = chemL[b * kMaxOcc + 1];
      const float dE = (o ? -2.0f : 2.0f) * F - (o ? (chem0 - chem1) : (chem1 - chem0));
      return dE <= 0.0f ? 1.0f : __expf(-beta * dE);
    }
    float G[kMaxFunc];
    FIELD::gen(fctx, img, b, pa, tab, G);
    float r = 0.0f;
    for (int q = 0; q < no; ++q)
      if (q != o) r += change_rate(b, o, q, G);
    return r / (float)(no - 1);
  };
  auto site_rate = [&](int l) -> float {
    int K[kMaxSlots];
    return site_rate_at(l / n_cells, main_addr(l), K);
  };
  for (int l = tid; l < n_groups * 64; l += nthr) rate[rate_at(l)] = l < n_sites ? site_rate(l) : 0.0f;
  __syncthreads();
  for (int w = tid; w < 4 * n_groups; w += nthr) {
    const double s = group_rate_sum(rate, w >> 2, w & 3);
    if ((w & 3) == 0) G[w >> 2] = s;
  }
  __syncthreads();

  const uint32_t m1_ = div_magic(L1), m2_ = div_magic(L2), mc_ = div_magic(n_cells);
  const unsigned long long ev0 = cs->pass_base;
  // sampling by N-fold time (na.n_time_samples > 0): samples at times
  // 0, dt, 2 dt, ... (passes since the launch) of the state occupied then
  const int n_tsamp = na.n_time_samples;
  const bool distinct = sc->nb_distinct != 0;  // no duplicate sites: no list in LDS, no search
  if (tid == 0) sel[3] = 0;

  // The last wavefront keeps the books; the others make the events.  Both
  // loops pass the same barriers per event:
  //  A  the event is chosen (sel, selR)
  // [T  time sampling: the state's samples are taken; sel[3] ends the run]
  // [B  the flip and the neighbour list; not where the first wavefront, which
  //     makes the flip, takes all rates itself: at most 64 distinct sites]
  //  C  the rates
  //  D  the group sums
  // The event's record (sel[4..15]) stands until the next flip, after the next
  // A, so the books take it in while the next event is being chosen.
  auto list_in_first_wave = [&](int sb) { return distinct && nbB[sb + 1] - nbB[sb] <= 64; };
  if (!OWN_BOOKS && wave == n_waves - 1) {
    NfoldBooks<BIN> books;
    books.open(na, sys, cs, chain, n_cells);
    for (int ev = 0; ev < na.n_events; ++ev) {
      __syncthreads();  // A
      const int site = __builtin_amdgcn_readfirstlane(sel[0]);
      if (site < 0) break;
      // in time sampling the state is left before the event is applied
      for (int turn = 0; turn < 2; ++turn) {
        if (lane == 0 && turn == (n_tsamp > 0 ? 0 : 1))
          if (books.leave(na, chain, n_slots, *selR)) sel[3] = 1;  // stop before this event
        if (turn == 0) {
          if (n_tsamp > 0) __syncthreads();  // T
          if (n_tsamp > 0 && __builtin_amdgcn_readfirstlane(sel[3])) break;
          if (!list_in_first_wave(div_small(site, mc_))) __syncthreads();  // B
        }
      }
      if (n_tsamp > 0 && __builtin_amdgcn_readfirstlane(sel[3])) break;  // (uniform across the workgroup)
      __syncthreads();  // C
      __syncthreads();  // D
      if (lane == 0) books.applied(na, chain, ev, sel);
    }
    if (lane == 0) books.close(na, sys, cs, chain, n_slots, ev0);
  } else {
    const NfoldShape shape{L1, L2, L3, h, P1, P12, S, n_cells, h <= L1 && h <= L2 && h <= L3};
    const int n_work = OWN_BOOKS ? nthr : nthr - 64;  // threads that make the events
    NfoldBooks<BIN> books;
    if (OWN_BOOKS && wave == 0) books.open(na, sys, cs, chain, n_cells);
    // this lane's periodic copy in a flip
    const int cpk = lane / 9, cpj = (lane / 3) % 3, cpi = lane % 3;
    uint4 rv = make_uint4(0u, 0u, 0u, 0u);  // wavefront 0: the random words of events ev0 + 64 m + lane
    for (int ev = 0; ev < na.n_events; ++ev) {
      // ---- select an event (wavefront 0)
      int site = -1;
      if (wave == 0) {
        const int chunk = (n_groups + 63) / 64;
        const int g0 = min(lane * chunk, n_groups), g1 = min(g0 + chunk, n_groups);
        // (four group sums on their way at a time; adding 0 leaves a sum as it is)
        double ls = 0.0, v0 = 0.0, v1 = 0.0, v2 = 0.0, v3 = 0.0;
        for (int g = g0; g < g0 + chunk; g += 4) {
          v0 = g < g1 ? G[g] : 0.0;
          v1 = g + 1 < g1 ? G[g + 1] : 0.0;
          v2 = g + 2 < g1 ? G[g + 2] : 0.0;
          v3 = g + 3 < g1 ? G[g + 3] : 0.0;
          ls += v0;
          ls += v1;
          ls += v2;
          ls += v3;
        }
        const double incl = wave_scan_incl_d(ls);
        const double R = lane_d(incl, 63);
        if ((ev & 63) == 0) {
          const unsigned long long gev = ev0 + (unsigned long long)(ev + lane);
          rv = philox4x32_10(make_uint4(0x4E464C44u, (uint32_t)gev, (uint32_t)(gev >> 32), (uint32_t)chain), cp->key0,
                             cp->key1);
        }
        const uint32_t rx = (uint32_t)__builtin_amdgcn_readlane((int)rv.x, ev & 63),
                       ry = (uint32_t)__builtin_amdgcn_readlane((int)rv.y, ev & 63);
        const double t = u01_53(rx, ry) * R;
        const bool live = R >= kNfoldMinTotalRate;
        const int L = live ? pick_lane(incl, ls, t) : -1;
        if (L >= 0) {
          const double before = lane_d(incl, L) - lane_d(ls, L);
          const int gl0 = __builtin_amdgcn_readlane(g0, L), gl1 = __builtin_amdgcn_readlane(g1, L);
          // the chunk's groups: at most four come from the registers of lane L
          // and need the scan's first two steps only (the others add 0)
          double gv, gi;
          if (chunk <= 4) {
            const double c0 = lane_d(v0, L), c1 = lane_d(v1, L), c2 = lane_d(v2, L), c3 = lane_d(v3, L);
            gv = lane == 0 ? c0 : (lane == 1 ? c1 : (lane == 2 ? c2 : (lane == 3 ? c3 : 0.0)));
            gi = gv + dpp_d<0x111, 0xf>(gv);
            gi += dpp_d<0x112, 0xf>(gi);
          } else {
            gv = (gl0 + lane < gl1) ? G[gl0 + lane] : 0.0;
            gi = wave_scan_incl_d(gv);
          }
          const double t2 = t - before;
          const int lg = pick_lane(gi, gv, t2);
          if (lg >= 0) {
            const int g = gl0 + lg;
            const double before2 = lane_d(gi, lg) - lane_d(gv, lg);
            const double rg = (double)rate[rate_at(g * 64 + lane)];
            const double ri = wave_scan_incl_d(rg);
            const int ls2 = pick_lane(ri, rg, t2 - before2);
            if (ls2 >= 0) site = g * 64 + ls2;
          }
        }
        if (lane == 0) {
          // a chain whose total rate vanished (or a group sum without a
          // positive rate, which exact group sums rule out) stops: -2
          sel[0] = site >= 0 ? site : -2;
          *selR = R;
        }
        // the new occupant (general sites): 53-bit uniform
        const int rz = __builtin_amdgcn_readlane((int)rv.z, ev & 63), rw = __builtin_amdgcn_readlane((int)rv.w, ev & 63);
        if (lane == 1) sel[1] = rz;
        if (lane == 2) sel[2] = rw;
      }
      __syncthreads();  // A
      // the same in every lane (the first wavefront has it in a register)
      if (wave != 0) site = sel[0];
      site = __builtin_amdgcn_readfirstlane(site);
      if (site < 0) {
        // uniform across the workgroup: record the stall for the host
        if (tid == 0) cs->flags |= kChainFlagNfoldStalled;
        break;
      }
      if (n_tsamp > 0) {
        if (OWN_BOOKS && tid == 0)
          if (books.leave(na, chain, n_slots, *selR)) sel[3] = 1;
        __syncthreads();  // T
        if (__builtin_amdgcn_readfirstlane(sel[3])) break;  // time sampling complete (uniform across the workgroup)
      }
      // ---- apply the change (first wavefront); binary: its cluster sums K come
      // with its new rate below; general: the new occupant in proportion to its
      // rate
      const int sb = div_small(site, mc_), scell = site - sb * n_cells;
      const int srow = div_small(scell, m1_);
      const int ci = scell - srow * L1, ck = div_small(srow, m2_), cj = srow - ck * L2;
      if (wave == 0) {
        const int b = sb;
        const int pa = b * S + (ck + h) * P12 + (cj + h) * P1 + (ci + h);
        const int o = img.get(pa);
        int nw = 1 - o;
        if (!BIN) {
          const int no = noccL[b];
          float Gf[kMaxFunc];
          FIELD::gen(fctx, img, b, pa, tab, Gf);
          double rq[kMaxOcc] = {0.0, 0.0, 0.0, 0.0}, tot = 0.0;
          for (int q = 0; q < no; ++q)
            if (q != o) {
              rq[q] = (double)change_rate(b, o, q, Gf);
              tot += rq[q];
            }
          const double t = u01_53((uint32_t)sel[1], (uint32_t)sel[2]) * tot;
          double acc = 0.0;
          nw = -1;
          for (int q = 0; q < no; ++q) {
            if (q == o) continue;
            acc += rq[q];
            if (nw < 0 && t < acc) nw = q;
          }
          if (nw < 0) nw = (o + 1 < no) ? no - 1 : no - 2;  // rounding: the last other occupant
          if (lane == 0) sel[6] = __float_as_int(general_dE(sys, b, o, nw, Gf));
        }
        // every lane has read the site before a copy of it is written
        wave_sync();
        if (lane == 0) {
          sel[4] = o;
          sel[5] = nw;
        }
        // the site and every periodic copy of it in the padded image: padded
        // coordinate (i + h) + d L for every d that stays inside [0, L + 2h)
        if (shape.near) {
          // d in {0, +1 (i < h), -1 (i >= L - h)}: at most three per axis, one
          // combination per lane
          int copy;
          if (nfold_copy(shape, cpi, cpj, cpk, b, ci, cj, ck, copy) && lane < 27) img.p[copy] = (uint8_t)nw;
        } else if (lane == 0) {
          const int m1 = (h + L1 - 1) / L1, m2 = (h + L2 - 1) / L2, m3 = (h + L3 - 1) / L3;
          for (int dk = -m3; dk <= m3; ++dk) {
            const int qk = ck + h + dk * L3;
            if (qk < 0 || qk >= P3) continue;
            for (int dj = -m2; dj <= m2; ++dj) {
              const int qj = cj + h + dj * L2;
              if (qj < 0 || qj >= P12 / P1) continue;
              for (int di = -m1; di <= m1; ++di) {
                const int qi = ci + h + di * L1;
                if (qi < 0 || qi >= P1) continue;
                img.p[b * S + qk * P12 + qj * P1 + qi] = (uint8_t)nw;
              }
            }
          }
        }
        // the copies, written by many lanes, are there for every lane of this
        // wavefront (barrier B is for the others, and left out where only this
        // one reads them)
        wave_sync();
      }
      // ---- rates of the site and its interaction neighbours
      {
        const int nb0 = nbB[sb], nb1 = nbB[sb + 1];
        auto place = [&](int t, int &lt, int &pt) {
          nfold_place(shape, nfold_unpack_nb(nbL[nb0 + t]), ci, cj, ck, lt, pt);
        };
        if (!distinct)
          for (int t = tid; t < nb1 - nb0; t += n_work) {
            int lt, pt;
            place(t, lt, pt);
            aff[t] = lt;
            affp[t] = pt;
          }
        // the flip and the list before any rate is read (a list of at most 64
        // distinct sites stays in the first wavefront, which made the flip)
        if (!list_in_first_wave(sb)) __syncthreads();  // B
        for (int t = tid; t < nb1 - nb0; t += n_work) {
          int lt, pt;
          if (distinct) {
            place(t, lt, pt);
          } else {
            lt = aff[t];
            pt = affp[t];
          }
          bool dup = false;
          if (!distinct)
            for (int q = 0; q < t; ++q) dup = dup || (aff[q] == lt);
          if (distinct) aff[t] = lt;  // the groups to sum again below
          if (!dup) {
            int K[kMaxSlots];
            rate[rate_at(lt)] = site_rate_at((int)(nbL[nb0 + t] & 0xff), pt, K);
            if (BIN && t == 0) {
              // the flipped site itself (first in the list): its cluster sums
#pragma unroll
              for (int a = 0; a < kMaxSlots; ++a) sel[8 + a] = K[a];
            }
          }
        }
        __syncthreads();  // C
        // the groups of the changed rates, summed again from their 64 rates by
        // four lanes each (several quads may form one group's sum: they write
        // the same value)
        if constexpr (OWN_BOOKS) {
          for (int t = tid; t < nb1 - nb0; t += n_work) {
            const int g = aff[t] >> 6;
            G[g] = group_rate_sum_lane(rate, g);
          }
        } else
        for (int w = tid; w < 4 * (nb1 - nb0); w += n_work) {
          const int g = aff[w >> 2] >> 6;
          const double s = group_rate_sum(rate, g, w & 3);
          if ((w & 3) == 0) G[g] = s;
        }
        __syncthreads();  // D
      }
      if (OWN_BOOKS && tid == 0) {
        if (n_tsamp == 0) (void)books.leave(na, chain, n_slots, *selR);
        books.applied(na, chain, ev, sel);
      }
    }
    if (OWN_BOOKS && tid == 0) books.close(na, sys, cs, chain, n_slots, ev0);
  }

  // ---- write back: occupation, exact counts, energy, counters
  int8_t *occW = args.occ + cp->occ_offset;
  for (int l = tid; l < n_sites; l += nthr) occW[l] = (int8_t)img.get(main_addr(l));
}

}  // namespace clexmc
