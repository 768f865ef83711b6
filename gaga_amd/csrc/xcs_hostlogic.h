// Pure integer logic shared by the device code, the host code and the CPU
// checks (this header needs no HIP: it also compiles with a plain C++
// compiler, which is how the CPU tests exercise it).
//
//  * the chunk geometry of the gen support gather (A_S x_S);
//  * the form a plan's solve runs in;
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
