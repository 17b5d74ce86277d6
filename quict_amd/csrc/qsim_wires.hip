// Tile passes planned in wires: kernel instances and their launch.
//
// A translation unit of its own because it is compiled with
// -structurizecfg-skip-uniform-regions: the op switch is uniform, and without the
// flag the compiler rebuilds it as nested regions that carry the whole tile from
// one to the next (two register sets, up to 64 moves an op).
#include "qsim_wire_kernel.hpp"

namespace qs {

template <typename R, int RB, int TB>
void launch_wires(cx<R>* v, uint64_t tiles, const PassHdr& hd, const PassHdr* dh, const WireOp<R>* ops, const cx<R>* coef,
                  const uint32_t* aux, uint32_t nsmall, const PassStart& S, size_t lds, hipStream_t s) {
  if (hd.has_dk)
    hipLaunchKernelGGL((k_wires<R, RB, TB, true>), dim3((unsigned)tiles), dim3(1 << TB), lds, s, v, dh, ops, coef, aux,
                       nsmall, S);
  else
    hipLaunchKernelGGL((k_wires<R, RB, TB, false>), dim3((unsigned)tiles), dim3(1 << TB), lds, s, v, dh, ops, coef,
                       aux, nsmall, S);
}

template <typename R, int RB, int TB> void wires_lds_attr() {
  const int bytes = (int)((1u << (RB + TB - 1)) * sizeof(cx<R>) + FMAX_PASS_COEF * sizeof(cx<R>));
  (void)hipFuncSetAttribute((const void*)k_wires<R, RB, TB, true>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  (void)hipFuncSetAttribute((const void*)k_wires<R, RB, TB, false>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
}

template <typename R>
void launch_jobs(cx<R>* psi, cx<R>* lam, const char* image, const WireJobs& jobs, uint32_t blocks, bool heavy, double* partial,
                 size_t lds, int cus, hipStream_t s) {
  static bool attr = false;  // two images, tables and gradient rows can pass 64 KiB
  if (!attr) {
    const int bytes = 150 * 1024;
    (void)hipFuncSetAttribute((const void*)k_jobs<R, 1, 1, false>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    (void)hipFuncSetAttribute((const void*)k_jobs<R, 1, 1, true>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    (void)hipFuncSetAttribute((const void*)k_jobs<R, 2, 1, false>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    (void)hipFuncSetAttribute((const void*)k_jobs<R, 2, 2, false>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    (void)hipFuncSetAttribute((const void*)k_jobs<R, 2, 2, true>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    attr = true;
  }
  const dim3 g(blocks), t(256);
  // One image for both vectors where a CU gets more than the two workgroups that fit
  // with one each.  1024 variational circuits 6.5 -> 6.1 ms; with a workgroup a CU (20
  // qubits) two images cost nothing and save barriers.
  const bool shared = lam && !heavy && sizeof(R) == 8 && blocks > 2u * (uint32_t)cus && lds >= 2 * (sizeof(cx<R>) << 11);
  if (!lam && heavy) hipLaunchKernelGGL((k_jobs<R, 1, 1, true>), g, t, lds, s, psi, lam, image, jobs, partial);
  else if (!lam) hipLaunchKernelGGL((k_jobs<R, 1, 1, false>), g, t, lds, s, psi, lam, image, jobs, partial);
  else if (heavy) hipLaunchKernelGGL((k_jobs<R, 2, 2, true>), g, t, lds, s, psi, lam, image, jobs, partial);
  else if (shared)
    hipLaunchKernelGGL((k_jobs<R, 2, 1, false>), g, t, lds - (sizeof(cx<R>) << 11), s, psi, lam, image, jobs, partial);
  else hipLaunchKernelGGL((k_jobs<R, 2, 2, false>), g, t, lds, s, psi, lam, image, jobs, partial);
}

template void launch_jobs<double>(cx<double>*, cx<double>*, const char*, const WireJobs&, uint32_t, bool, double*,
                                  size_t, int, hipStream_t);
template void launch_jobs<float>(cx<float>*, cx<float>*, const char*, const WireJobs&, uint32_t, bool, double*, size_t, int,
                                 hipStream_t);

#define QS_WIRES(R, TB)                                                                                          \
  template void launch_wires<R, 4, TB>(cx<R>*, uint64_t, const PassHdr&, const PassHdr*, const WireOp<R>*,       \
                                       const cx<R>*, const uint32_t*, uint32_t, const PassStart&, size_t, hipStream_t); \
  template void wires_lds_attr<R, 4, TB>();
QS_WIRES(double, 7)
QS_WIRES(double, 8)
QS_WIRES(double, 9)
QS_WIRES(float, 8)
QS_WIRES(float, 9)

}  // namespace qs
