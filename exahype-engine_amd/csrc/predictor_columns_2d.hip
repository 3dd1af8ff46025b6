// The column / line predictor for the compiled 2D shapes (predictor_columns.h).
#include "predictor_columns.h"

namespace exa {
namespace {

struct Entry {
  int B, V, NP;
  int (*run)(const KernelCfg&, hipStream_t, long, const double*, const double*, const double*, double*, double*,
             double*, int*, const LaunchOpts&);
};

#define EXA_COLUMNS(D, B, V, NP) Entry{B, V, NP, &columns::Launch<D, B, V, NP>::run}

const Entry kEntries[] = {
    EXA_COLUMNS(2, 2, 5, 0),
    EXA_COLUMNS(2, 3, 5, 0),
    EXA_COLUMNS(2, 4, 5, 0),
    EXA_COLUMNS(2, 5, 5, 0),
    EXA_COLUMNS(2, 6, 5, 0),
    EXA_COLUMNS(2, 7, 5, 0),
    EXA_COLUMNS(2, 4, 5, 1),
    EXA_COLUMNS(2, 4, 1, 0),
    EXA_COLUMNS(2, 4, kUserNVar, 0),
    EXA_COLUMNS(2, 5, kUserNVar, 0),
};

}  // namespace

int launch_predictor_columns_2d(const KernelCfg& k, hipStream_t s, long n, const double* luh, const double* h,
                                const double* dt, double* lduh, double* qb, double* fb, int* pic,
                                const LaunchOpts& o) {
  for (const Entry& e : kEntries)
    if (e.B == k.order + 1 && e.V == k.nvar && e.NP == k.npar)
      return e.run(k, s, n, luh, h, dt, lduh, qb, fb, pic, o);
  return -1;
}

}  // namespace exa
