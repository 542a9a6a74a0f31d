// Host check of the N-fold kernel's LDS layout and index arithmetic: the
// kernel's own functions over every site, neighbour, copy, group and lane of
// a shape.  Reads shapes from stdin, per shape: n_sublat L1 L2 L3 h row_pitch,
// then per sublattice the list's length and its neighbours (b di dj dk, the
// site itself first); prints "lds <bytes> errors <n>" per shape.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <vector>

#include "../../casmcode_clexmonte_amd/csrc/clexmc_nfold.h"

using namespace clexmc;

int main() {
  int n_sub, L1, L2, L3, h, pitch;
  while (std::scanf("%d %d %d %d %d %d", &n_sub, &L1, &L2, &L3, &h, &pitch) == 6) {
    long long bad = 0;
    auto check = [&](bool ok) { bad += ok ? 0 : 1; };
    std::vector<std::vector<int4>> nb(n_sub);
    int nb_max = 0, nb_total = 0;
    for (auto &list : nb) {
      int n = 0;
      if (std::scanf("%d", &n) != 1) return 2;
      list.resize(n);
      for (auto &o : list)
        if (std::scanf("%d %d %d %d", &o.x, &o.y, &o.z, &o.w) != 4) return 2;
      nb_max = n > nb_max ? n : nb_max;
      nb_total += n;
    }
    NfoldShape g;
    g.L1 = L1, g.L2 = L2, g.L3 = L3, g.h = h;
    g.P1 = L1 + 2 * h + pitch, g.P12 = g.P1 * (L2 + 2 * h), g.S = g.P12 * (L3 + 2 * h);
    g.n_cells = L1 * L2 * L3;
    g.near = h <= L1 && h <= L2 && h <= L3;
    const int pad = n_sub * g.S, n_sites = n_sub * g.n_cells, n_groups = (n_sites + 63) / 64;
    const NfoldLds o = nfold_lds(pad, n_sites, nb_max, nb_total, n_sub);
    // regions one after the other, each large and aligned enough
    const size_t groups = (size_t)n_groups;
    check(o.rate >= (size_t)pad && o.rate % 16 == 0);
    check(o.G >= o.rate + groups * 64 * 4 && o.G % 8 == 0);
    check(o.aff >= o.G + groups * 8 && o.affp >= o.aff + (size_t)nb_max * 4 && o.sel >= o.affp + (size_t)nb_max * 4);
    check(o.sel % 8 == 0 && o.nb_begin >= o.sel + 16 * 4 + 8);
    check(o.nb >= o.nb_begin + (n_sub + 1) * 4 && o.n_occ >= o.nb + (size_t)nb_total * 4);
    check(o.chem >= o.n_occ + n_sub * 4 && o.bytes >= o.chem + n_sub * kMaxOcc * 4 && o.nb % 4 == 0 && o.chem % 4 == 0);
    // rates: a permutation within every group, whose sum reads exactly its own
    std::vector<int> hit(n_groups * 64, 0);
    for (int l = 0; l < n_groups * 64; ++l) {
      const int a = rate_at(l);
      check(a >= 0 && a < n_groups * 64 && a / 64 == l / 64);
      if (a >= 0 && a < n_groups * 64) ++hit[a];
    }
    for (int v : hit) check(v == 1);
    for (int gr = 0; gr < n_groups; ++gr)
      for (int q = 0; q < 4; ++q)
        for (int p = 0; p < 16; ++p) {
          const int a = gr * 64 + q + ((p ^ (gr & 15)) << 2);  // group_rate_sum
          check(a == rate_at(gr * 64 + 4 * p + q));
        }
    // every site as the event's: its cell by the quick division, its copies,
    // its neighbours
    const uint32_t m1 = div_magic(L1), m2 = div_magic(L2), mc = div_magic(g.n_cells);
    std::vector<int> home(pad, -1);  // site of each padded address, by the copies
    for (int site = 0; site < n_sites; ++site) {
      const int b = div_small(site, mc), cell = site - b * g.n_cells, row = div_small(cell, m1);
      const int i = cell - row * L1, k = div_small(row, m2), j = row - k * L2;
      check(b == site / g.n_cells && i == cell % L1 && j == (cell / L1) % L2 && k == cell / (L1 * L2));
      const int pa = b * g.S + (k + h) * g.P12 + (j + h) * g.P1 + (i + h);
      check(pa >= 0 && pa < pad);
      if (g.near)
        for (int c = 0; c < 27; ++c) {
          int a = -1;
          if (!nfold_copy(g, c % 3, (c / 3) % 3, c / 9, b, i, j, k, a)) continue;
          check(a >= 0 && a < pad && (c > 0 || a == pa));
          if (a >= 0 && a < pad) {
            check(home[a] == -1);
            home[a] = site;
          }
        }
      for (auto const &n : nb[b]) {
        const int4 u = nfold_unpack_nb(nfold_pack_nb(n.x, n.y, n.z, n.w));
        check(u.x == n.x && u.y == n.y && u.z == n.z && u.w == n.w);
        int lt = -1, pt = -1;
        nfold_place(g, u, i, j, k, lt, pt);
        auto md = [](int x, int m) { return ((x % m) + m) % m; };
        const int ii = md(i + n.y, L1), jj = md(j + n.z, L2), kk = md(k + n.w, L3);
        check(lt == n.x * g.n_cells + ii + L1 * (jj + L2 * kk));
        check(pt == n.x * g.S + (kk + h) * g.P12 + (jj + h) * g.P1 + (ii + h) && pt >= 0 && pt < pad);
      }
    }
    // every cell of the image but the row pitch is a copy of one site
    if (g.near)
      for (int p = 0; p < pad; ++p) check((p % g.P1 < L1 + 2 * h) == (home[p] >= 0));
    std::printf("lds %zu errors %lld\n", o.bytes, bad);
  }
  return 0;
}
