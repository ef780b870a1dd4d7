// Compile-time-size FFT kernels (declarations).
#pragma once

#include "wh_fft.h"

namespace wh {

struct TplKernels {
  void (*zinv)(const StickPlanDev&, const FftItem*, int, const z64*, long, const z64*, long, void*, int, hipStream_t);
  void (*zfwd)(const StickPlanDev&, const FftItem*, int, const void*, const z64*, long, z64*, long, const ZfwdArgs&,
               hipStream_t);
  // occ: workgroups per CU the plane kernel's LDS is sized for (1..max_occ)
  void (*vloc)(const StickPlanDev&, const FftItem*, int, const void*, void*, const double*, long, double, int,
               hipStream_t);
  void (*to_real)(const StickPlanDev&, const FftItem*, int, const void*, double*, long, hipStream_t);
  // density(P, npert, nband, sticks in, occ, sticks out, scratch, stream): scratch holds
  // density_scratch n3 reals per perturbation (may be null when that is 0)
  void (*density)(const StickPlanDev&, int, int, const void*, const double*, void*, void*, hipStream_t);
  long density_scratch;   // per plane; 0: none needed; -1: this grid has no density kernel
  int max_occ;
};

// FP32 operator (sticks, vectors and potential in FP32)
struct TplKernels32 {
  void (*zinv)(const StickPlanDev&, const FftItem*, int, const z32*, long, const z32*, long, void*, int, hipStream_t);
  void (*zfwd)(const StickPlanDev&, const FftItem*, int, const void*, const z32*, long, z32*, long, const ZfwdArgs&,
               hipStream_t);
  void (*vloc)(const StickPlanDev&, const FftItem*, int, const void*, void*, const float*, long, double, int,
               hipStream_t);
  int max_occ;
};

// FP64: plane kernels specialised on N = nr1 = nr2 (any nr3) and z kernels on
// N = nr3, or null when that length is not one of the compiled sizes (the
// runtime-size kernels are used then); FP32: cubic grids only
const TplKernels* tpl_kernels_f64(const StickPlanDev& P);
const TplKernels* tpl_z_kernels_f64(const StickPlanDev& P);
const TplKernels32* tpl_kernels_f32(const StickPlanDev& P);

}  // namespace wh
