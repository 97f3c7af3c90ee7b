// The default Euler predictors (aderdg_history.h), orders 1..8: FP64, FP32
// sweeps before the FP64 correction sweeps, and the latter's variant for
// meshes with many uniform cells (orders up to 7, the adaptive mesh's range).
#include "aderdg_history.h"
#include "predictor_tu.h"

namespace {
template <int N>
PredFn pick(bool mixed, int fp64_sweeps, bool uskip) {
  if (!mixed) return &exa::k_predictor_history<N, false, false, false>;
  if constexpr (N <= 7) {
    if (uskip)
      return fp64_sweeps == 1 ? &exa::k_predictor_history<N, true, true, true>
                              : &exa::k_predictor_history<N, true, false, true>;
  }
  return fp64_sweeps == 1 ? &exa::k_predictor_history<N, true, true, false>
                          : &exa::k_predictor_history<N, true, false, false>;
}
}  // namespace

PredFn exa_pred_history_kernel(int order, bool mixed, int fp64_sweeps, bool uskip) {
  switch (order) {
    case 1: return pick<1>(mixed, fp64_sweeps, uskip);
    case 2: return pick<2>(mixed, fp64_sweeps, uskip);
    case 3: return pick<3>(mixed, fp64_sweeps, uskip);
    case 4: return pick<4>(mixed, fp64_sweeps, uskip);
    case 5: return pick<5>(mixed, fp64_sweeps, uskip);
    case 6: return pick<6>(mixed, fp64_sweeps, uskip);
    case 7: return pick<7>(mixed, fp64_sweeps, uskip);
    case 8: return pick<8>(mixed, fp64_sweeps, uskip);
    default: return nullptr;
  }
}

namespace {
template <int N>
int lds_bytes(bool fp64_sweeps, bool one_sweep) {
  return exa::HistOrd<N>::lds_doubles(fp64_sweeps, one_sweep) * (int)sizeof(double);
}
}  // namespace

int exa_pred_history_lds_bytes(int order, bool mixed, int fp64_sweeps, bool uskip) {
  const bool one = mixed && fp64_sweeps == 1, f64 = !one || uskip;  // the sweeps that the kernel holds
  switch (order) {
    case 1: return lds_bytes<1>(f64, one);
    case 2: return lds_bytes<2>(f64, one);
    case 3: return lds_bytes<3>(f64, one);
    case 4: return lds_bytes<4>(f64, one);
    case 5: return lds_bytes<5>(f64, one);
    case 6: return lds_bytes<6>(f64, one);
    case 7: return lds_bytes<7>(f64, one);
    case 8: return lds_bytes<8>(f64, one);
    default: return 0;
  }
}

hipError_t exa_pred_history_init(const DGTables* tab, const DGTablesF* tabf) {
  hipError_t e = hipMemcpyToSymbol(HIP_SYMBOL(c_tab), tab, sizeof(DGTables) * (EXA_MAX_ORDER + 1));
  if (e != hipSuccess) return e;
  e = hipMemcpyToSymbol(HIP_SYMBOL(c_tabf), tabf, sizeof(DGTablesF) * (EXA_MAX_ORDER + 1));
  if (e != hipSuccess) return e;
  exa::HistTables<double> ht[EXA_MAX_ORDER + 1] = {};
  exa::fill_hist_tables(tab, ht);
  exa::HistTables<float> htf[EXA_MAX_ORDER + 1] = {};
  for (int n = 1; n <= EXA_MAX_ORDER; ++n)
    for (int i = 0; i < EXA_NB; ++i) {
      htf[n].a[i] = (float)ht[n].a[i];
      htf[n].b[i] = (float)ht[n].b[i];
      for (int j = 0; j < exa::EXA_NH && i < exa::EXA_NH; ++j) {
        htf[n].ev[i][j] = (float)ht[n].ev[i][j];
        htf[n].od[i][j] = (float)ht[n].od[i][j];
      }
    }
  e = hipMemcpyToSymbol(HIP_SYMBOL(exa::c_ht), ht, sizeof(ht));
  if (e != hipSuccess) return e;
  e = hipMemcpyToSymbol(HIP_SYMBOL(exa::c_htf), htf, sizeof(htf));
  if (e != hipSuccess) return e;
  for (int order = EXA_HISTORY_MIN_ORDER; order <= EXA_HISTORY_MAX_ORDER; ++order)
    for (int var = 0; var < 5; ++var) {  // FP64; mixed with one and with more FP64 sweeps, each with uskip
      const bool mixed = var > 0, uskip = var > 2;
      const int sweeps = 1 + (var & 1);
      e = hipFuncSetAttribute(reinterpret_cast<const void*>(exa_pred_history_kernel(order, mixed, sweeps, uskip)),
                              hipFuncAttributeMaxDynamicSharedMemorySize,
                              exa_pred_history_lds_bytes(order, mixed, sweeps, uskip));
      if (e != hipSuccess) return e;
    }
  return hipSuccess;
}
