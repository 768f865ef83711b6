// Pure integer logic shared by the device code, the host code and the CPU
// checks (this header needs no HIP: it also compiles with a plain C++
// compiler, which is how the CPU tests exercise it).
//
//  * the chunk geometry of the gen support gather (A_S x_S);
//  * the form a plan's solve runs in, and the teams a batch's does;
//  * the names of the ten algorithms, indexed by the Alg codes;
//  * the autotuner's cache key of a batch.
#pragma once
#include <algorithm>
#include <cmath>
#include <string>
#include <vector>
#if defined(__HIPCC__) || defined(__HIP__)
#define XCS_HD __host__ __device__
#else
#define XCS_HD
#endif

namespace xcs {

constexpr int MAXCH = 64;    // gen gather: column chunks (rows of the partials buffer)
constexpr int SLDS = 4096;   // gen gather: support entries staged in LDS per pass
constexpr int GATHER_BLOCK = MAXCH * SLDS;  // support entries per gather block

// Geometry of one gather block of `cnt` support entries (0 <= cnt <=
// GATHER_BLOCK): chunks of `cs` consecutive entries (at least 8), `nch` of
// them (nch <= MAXCH, one partials row each), staged `cpp` whole chunks per
// LDS pass (cpp >= 1 because cs <= SLDS).
struct GatherGeom {
  int cs, nch, cpp;
};
XCS_HD inline GatherGeom gather_geom(int cnt) {
  GatherGeom g;
  int cs = (cnt + MAXCH - 1) / MAXCH;
  if (cs < 8) cs = 8;
  g.cs = cs;
  g.nch = (cnt + cs - 1) / cs;
  g.cpp = SLDS / cs;
  return g;
}
// Number of gather blocks for a support of cnt entries (at least one, so an
// empty support still writes its zero output).
XCS_HD inline int gather_blocks(int cnt) {
  const int b = (cnt + GATHER_BLOCK - 1) / GATHER_BLOCK;
  return b < 1 ? 1 : b;
}

// The form of a single solve: the general one (solve_coop_kernel), or the ones with
// the vectors in LDS.  A plan is laid out for one of them; a solve from a warm start
// (a given support) runs in the general form, the only one that reads it, on the
// plan's team (at most one workgroup per CU, which the general form always fits).
enum SolveForm { FORM_GENERAL = 0, FORM_RESIDENT = 1, FORM_SPLIT = 2 };
inline int solve_form(int planned, bool warm) { return warm ? FORM_GENERAL : planned; }

// Teams of c workgroups for up to `want` instances, of `resident` workgroups in all:
// whole groups of eight (one per XCD), with a few spare teams where the chip has room
// for them rather than a few instances that wait.
inline int batch_teams(int resident, int want, int c) {
  const int most = resident / c;
  const int teams = std::min(want, most);
  if (c == 1 || teams < 8) return teams;
  return (teams + 7) / 8 * 8 <= most ? (teams + 7) / 8 * 8 : teams - teams % 8;
}

// The geometry of one batch solve without a tail schedule: teams of c for the `big`
// largest of `count` instances, single workgroups for the others.  With `grow`, in
// larger teams where the chip has room for them.  A workgroup streams about 100 GB/s,
// so a large instance on a few workgroups takes long after the others are done.
// Teams of twice the size are taken, again and again, while every large instance
// still has its team at once, a workgroup keeps GROW_BYTES a product (below that the
// team's barriers take the time) and the longest wait shrinks: the bytes a workgroup
// streams for the largest instance (`most`) and, where the other instances can't all
// run beside the teams, for the largest of those after it (`most1`).
// Measured on MI355X, ms per solve before and after: instances of both ensembles, n =
// 1024 to 8192, the largest quarter in teams of 4, CGIHT: 256 of them 21.0 -> 16.6, 128
// 14.7 -> 10.5, 64 9.4 -> 4.2, 16 5.6 -> 3.6; 20 of 2048 x 8192 in teams of 4 16.2 -> 7.4.
constexpr double GROW_BYTES = 2e6;
struct BatchPick {
  int c, teams;
};
inline BatchPick batch_pick(int count, int big, int c, int resident, int max_team, double most, double most1,
                            bool grow) {
  const int small = count - big;
  BatchPick best{c, 0};
  double wait = 0.0;
  for (int d = c; d == c || (grow && d <= std::min(resident, max_team) && most / d >= GROW_BYTES); d *= 2) {
    const int teams = batch_teams(resident, big + (small + d - 1) / d, d);
    const double w = most / d + ((long)teams * d >= (long)big * d + small ? 0.0 : most1);
    if (d > c && teams < big) break;
    if (d > c && w >= wait) continue;
    wait = w;
    best = BatchPick{d, teams};
  }
  return best;
}

constexpr int NUM_ALGS = 10;
// Algorithm names as the reference's option strings spell them
// (GAGA/gaga/gaga_gen.cu:65, 625-634); index = the Alg code.
inline const char *alg_name(int alg) {
  static const char *const names[NUM_ALGS] = {"NIHT", "HTP", "CSMPSP", "CGIHT", "IHT",
                                              "ThresholdSD", "ThresholdCG", "FIHT", "ALPS",
                                              "CGIHTprojected"};
  return (alg >= 0 && alg < NUM_ALGS) ? names[alg] : "unknown";
}

// Key of a batch in the autotuner's cache file: algorithm, instance count,
// then per ensemble the instance count, the n range and log2 of the matrix
// bytes, and the probe length.  One entry per instance: ensemble code (0 gen,
// 1 smv, 2 dct), n, the leading dimension lda (gen) and nz (smv).
struct SigInstance {
  int ens, n, lda, nz;
};
inline std::string batch_signature_text(int alg, const std::vector<SigInstance> &inst,
                                        int probe_iters) {
  static const char *const ens_names[3] = {"gen", "smv", "dct"};
  std::string s = std::string(alg_name(alg)) + ":count=" + std::to_string(inst.size());
  for (int e = 0; e < 3; e++) {
    int cnt = 0, nmin = 1 << 30, nmax = 0;
    double bytes = 0.0;
    for (const SigInstance &P : inst)
      if (P.ens == e) {
        cnt++;
        nmin = std::min(nmin, P.n);
        nmax = std::max(nmax, P.n);
        bytes += e == 0 ? 4.0 * P.lda * P.n : e == 1 ? 8.0 * P.nz : 24.0 * P.n;
      }
    if (cnt)
      s += std::string(":") + ens_names[e] + "=" + std::to_string(cnt) + "/" +
           std::to_string(nmin) + "-" + std::to_string(nmax) + "/2^" +
           std::to_string((int)std::lround(std::log2(std::max(bytes, 1.0))));
  }
  return s + ":probe=" + std::to_string(probe_iters);
}

}  // namespace xcs
