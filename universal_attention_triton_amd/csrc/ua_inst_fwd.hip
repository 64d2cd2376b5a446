// Instantiations and launchers of the forward kernels.
#include <algorithm>
#include <cstdint>
#include <cstdlib>
#include "ua_fused.hpp"
#include "ua_fwd.hpp"
#include "ua_internal.hpp"

namespace ua {

template <class K>
static void allow_lds(K kernel, size_t bytes) {
  (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

template <class T, int D>
static hipError_t carry_t(const void* Kp, const float* lsrc, const float* ldest, float* C, int Lp, int Zk, int tiled,
                          const float* knorm2, const float* qnorm2, int R, int* reach, hipStream_t s, void* Bt,
                          int variant) {
  constexpr int NST = 2;
  _Float16* none = nullptr;
  // bias tiles, variant 1: 4-wave workgroups (launches of under two 8-wave workgroups per CU are bound by the latency
  // of a workgroup's serial sweep and run faster as twice as many 4-wave workgroups)
  // variant 2: the same with two key groups per workgroup (see k_carry2)
  if (tiled && Bt && sizeof(T) == 2 && (variant == 1 || variant == 2))
    hipLaunchKernelGGL((k_carry2<T, D, NST, true, true, 4>), dim3(variant == 2 ? (Lp / 64 + 1) / 2 : Lp / 64, Zk), dim3(256), 0, s, (const T*)Kp, lsrc, ldest, C, Lp, knorm2, qnorm2, R, reach, (_Float16*)Bt);
  else if (tiled && Bt && sizeof(T) == 2) hipLaunchKernelGGL((k_carry2<T, D, NST, true, true>), dim3(Lp / 128, Zk), dim3(512), 0, s, (const T*)Kp, lsrc, ldest, C, Lp, knorm2, qnorm2, R, reach, (_Float16*)Bt);
  else if constexpr (D == 256) return hipErrorInvalidValue;
  else if (tiled) hipLaunchKernelGGL((k_carry2<T, D, NST, true, false, 4>), dim3(Lp / 64, Zk), dim3(256), 0, s, (const T*)Kp, lsrc, ldest, C, Lp, knorm2, qnorm2, R, reach, none);
  else hipLaunchKernelGGL((k_carry2<T, D, NST, false, false>), dim3(Lp / 128, Zk), dim3(512), 0, s, (const T*)Kp, lsrc, ldest, C, Lp, knorm2, qnorm2, R, reach, none);
  return hipGetLastError();
}
hipError_t launch_carry(int dtype, int D, const void* Kp, const float* lsrc, const float* ldest, float* C, int Lp, int Zk,
                        int tiled, const float* knorm2, const float* qnorm2, int R, int* reach, hipStream_t s,
                        void* Bt, int variant) {
#define UA_ARGS Kp, lsrc, ldest, C, Lp, Zk, tiled, knorm2, qnorm2, R, reach, s, Bt, variant
  if (D == 256) return (dtype == 1 && tiled && Bt) ? carry_t<bf16, 256>(UA_ARGS) : hipErrorInvalidValue;   // bias tiles only
  if (dtype == 1) return D == 64 ? carry_t<bf16, 64>(UA_ARGS) : carry_t<bf16, 128>(UA_ARGS);
  return D == 64 ? carry_t<float, 64>(UA_ARGS) : carry_t<float, 128>(UA_ARGS);
#undef UA_ARGS
}

// explicit instantiations (the implicit ones are not emitted on the host side for these kernels)
#define UA_INST3(T, D, NST, NW, CH, BI, RB)                                                                             \
  template __global__ void k_fwd_fused2<T, D, NST, NW, CH, BI, RB>(RowsOut, const T*, const T*, const T*, const float*, const float*, \
                                                               const float*, T*, float*, float*, const int*, \
                                                               int, int, int, int, ChunkOut<T>, const _Float16*);
#define UA_INST2(T, D, NST, NW, CH, BI) UA_INST3(T, D, NST, NW, CH, BI, 1)
#define UA_INST(T, D, NST, NW, CH) UA_INST2(T, D, NST, NW, CH, false)
UA_INST3(bf16, 256, 1, 8, false, true, 2) UA_INST3(bf16, 256, 1, 8, false, true, 4) UA_INST2(bf16, 256, 1, 8, false, true)
#define UA_INSTF_(D, RB, NW, KS, PR)                                                                                              \
  template __global__ void k_fwd_tiles<D, RB, NW, KS, PR>(RowsOut, const bf16*, const bf16*, const bf16*, bf16*, float*, float*, \
                                                          const int*, int, int, int, int, const _Float16*, int);
#define UA_INSTF(RB, NW, KS) UA_INSTF_(64, RB, NW, KS, false) UA_INSTF_(64, RB, NW, KS, true) UA_INSTF_(128, RB, NW, KS, false) UA_INSTF_(128, RB, NW, KS, true)
UA_INSTF(1, 4, 1) UA_INSTF(2, 4, 1) UA_INSTF(4, 4, 1) UA_INSTF(1, 8, 2) UA_INSTF(2, 8, 2) UA_INSTF(4, 8, 2) UA_INSTF(1, 8, 4)
#undef UA_INSTF
#undef UA_INSTF_
UA_INST(bf16, 64, 1, 8, false) UA_INST(bf16, 64, 2, 8, false) UA_INST(bf16, 64, 2, 12, false) UA_INST(bf16, 64, 2, 16, false)
UA_INST(bf16, 128, 2, 4, false) UA_INST(bf16, 64, 2, 4, false) UA_INST(bf16, 128, 1, 8, false) UA_INST(bf16, 128, 2, 8, false) UA_INST(bf16, 128, 2, 12, false) UA_INST(bf16, 128, 2, 16, false)
UA_INST(bf16, 64, 2, 8, true) UA_INST(bf16, 128, 2, 8, true) UA_INST(float, 64, 1, 8, true) UA_INST(float, 128, 1, 8, true)
#define UA_INSTS(D, NST, NW, KS)                                                                                                      \
  template __global__ void k_fwd_split<D, NST, NW, KS>(RowsOut, const float*, const float*, const float*, const float*, const float*, \
                                                       const float*, float*, float*, float*, const int*, int, int, int, int);
UA_INSTS(64, 1, 4, 2) UA_INSTS(128, 1, 4, 2) UA_INSTS(64, 2, 4, 4) UA_INSTS(128, 1, 4, 4)
#undef UA_INSTS
#undef UA_INST
#undef UA_INST2
#undef UA_INST3

template <class T, int D, int NST, int NW>
static hipError_t fused_t(const void* Qp, const void* Kp, const void* VT, const float* lsrc, const float* ldest,
                          const float* C, void* O, float* lse, float* lse2, const int* reach, int R, int L,
                          int Lp, int d, int Zq, const RowsOut& orow, hipStream_t s) {
  const _Float16* none = nullptr;
  hipLaunchKernelGGL((k_fwd_fused2<T, D, NST, NW, false>), dim3((Lp / 16 + NW - 1) / NW, Zq), dim3(64 * NW), 0, s, orow, (const T*)Qp,
                     (const T*)Kp, (const T*)VT, lsrc, ldest, C, (T*)O, lse, lse2, reach, R, L, Lp, d, ChunkOut<T>{}, none);
  return hipGetLastError();
}
// bf16 with bias tiles from launch_carry, head dims up to 128.  prune: the pre-pass left out tiles (UA_FLAG_PRUNE).
// variant (UA_TUNE_FWD_TILES): 0 = 4 waves, one key split; 1, 2 = 8 waves, two and four.
template <int D, int RB, int NW, int KS>
static hipError_t fwd_tiles_t(bool prune, const void* Qp, const void* Kp, const void* VT, void* O, float* lse, float* lse2,
                              const int* reach, int R, int L, int Lp, int d, int Zq, const RowsOut& orow, hipStream_t s, const void* Bt) {
  constexpr int nb = NW / KS / RB;
  const int n_blk = (Lp / 32 + nb - 1) / nb;
  // Two query blocks per workgroup where these make whole rounds of the CUs, or many: equal workgroups, half as many changes.
  const long pairs = (long)((n_blk + 1) / 2) * (Zq / RB);
  // (b = 2 h = 16 L = 2048 d = 64, two key splits: 512 blocks 62 us, 256 pairs 46; one and a half rounds of pairs cost more than
  // three of single blocks, heaviest first.)
  const bool pair = pairs >= 4L * device_cus() || (pairs >= device_cus() && pairs % device_cus() == 0);
  const int gx = pair ? (n_blk + 1) / 2 : n_blk;
#define UA_FT(PR_)                                                                                                               \
  hipLaunchKernelGGL((k_fwd_tiles<D, RB, NW, KS, PR_>), dim3(gx, Zq / RB), dim3(64 * NW), 0, s, orow, (const bf16*)Qp, (const bf16*)Kp, \
                     (const bf16*)VT, (bf16*)O, lse, lse2, reach, R, L, Lp, d, (const _Float16*)Bt, n_blk)
  if (prune) UA_FT(true); else UA_FT(false);
#undef UA_FT
  return hipGetLastError();
}
template <int D, int RB>
static hipError_t fwd_tiles_rb(int variant, bool prune, const void* Qp, const void* Kp, const void* VT, void* O, float* lse, float* lse2,
                               const int* reach, int R, int L, int Lp, int d, int Zq, const RowsOut& orow, hipStream_t s, const void* Bt) {
#define UA_ARGS prune, Qp, Kp, VT, O, lse, lse2, reach, R, L, Lp, d, Zq, orow, s, Bt
  if constexpr (RB == 1) { if (variant == 2) return fwd_tiles_t<D, RB, 8, 4>(UA_ARGS); }
  return variant == 1 ? fwd_tiles_t<D, RB, 8, 2>(UA_ARGS) : fwd_tiles_t<D, RB, 4, 1>(UA_ARGS);
#undef UA_ARGS
}
template <int D>
static hipError_t fwd_tiles(int variant, bool prune, const void* Qp, const void* Kp, const void* VT, void* O, float* lse, float* lse2,
                            const int* reach, int R, int L, int Lp, int d, int Zq, const RowsOut& orow, hipStream_t s, const void* Bt) {
#define UA_ARGS variant, prune, Qp, Kp, VT, O, lse, lse2, reach, R, L, Lp, d, Zq, orow, s, Bt
  return R % 4 == 0 ? fwd_tiles_rb<D, 4>(UA_ARGS) : R % 2 == 0 ? fwd_tiles_rb<D, 2>(UA_ARGS) : fwd_tiles_rb<D, 1>(UA_ARGS);
#undef UA_ARGS
}
// head dim above 128: 16 queries per wave (the accumulators of a 32-query block do not fit), 8-wave workgroups of 128 queries; the
// groups of a kv head share the tiles of a 32-query block (see RB)
static hipError_t fwd_tiles_256(const void* Qp, const void* Kp, const void* VT, const float* lsrc, const float* ldest, const float* C, void* O,
                                float* lse, float* lse2, const int* reach, int R, int L, int Lp, int d, int Zq, const RowsOut& orow,
                                hipStream_t s, const void* Bt) {
#define UA_SHARED(RB_)                                                                                                           \
  hipLaunchKernelGGL((k_fwd_fused2<bf16, 256, 1, 8, false, true, RB_>), dim3(Lp / (128 / RB_), Zq / RB_), dim3(512), 0, s, orow,  \
                     (const bf16*)Qp, (const bf16*)Kp, (const bf16*)VT, lsrc, ldest, C, (bf16*)O, lse, lse2, reach, R, L, Lp, d, \
                     ChunkOut<bf16>{}, (const _Float16*)Bt)
  if (R % 4 == 0) UA_SHARED(4);
  else if (R % 2 == 0) UA_SHARED(2);
  else UA_SHARED(1);
#undef UA_SHARED
  return hipGetLastError();
}
// float32: two key splits, or four where those workgroups (of 32 queries) would leave CUs without one
template <int D>
static hipError_t fwd_split(const void* Qp, const void* Kp, const void* VT, const float* lsrc, const float* ldest, const float* C, void* O,
                            float* lse, float* lse2, const int* reach, int R, int L, int Lp, int d, int Zq, const RowsOut& orow, hipStream_t s) {
#define UA_FS(NST_, KS_)                                                                                                       \
  hipLaunchKernelGGL((k_fwd_split<D, NST_, 4, KS_>), dim3(Lp / (64 / KS_), Zq), dim3(256), 0, s, orow, (const float*)Qp, (const float*)Kp, \
                     (const float*)VT, lsrc, ldest, C, (float*)O, lse, lse2, reach, R, L, Lp, d)
  if ((long)(Lp / 32) * Zq < device_cus()) UA_FS((D == 64 ? 2 : 1), 4);
  else UA_FS(1, 2);
#undef UA_FS
  return hipGetLastError();
}
// variants (bf16): 0 = 8 waves, double-buffered stages; 1 = 8 waves, single stage; 2 = 12 waves; 3 = 16 waves
// (both double-buffered).
int fwd_fused_variants(int dtype, int D) { (void)D; return dtype == 1 ? 5 : 1; }
template <class T, int D>
static hipError_t fused_v(int variant, const void* Qp, const void* Kp, const void* VT, const float* lsrc, const float* ldest,
                          const float* C, void* O, float* lse, float* lse2, const int* reach, int R, int L,
                          int Lp, int d, int Zq, const RowsOut& orow, hipStream_t s) {
#define UA_ARGS Qp, Kp, VT, lsrc, ldest, C, O, lse, lse2, reach, R, L, Lp, d, Zq, orow, s
  switch (variant) {
    case 1: return fused_t<T, D, 1, 8>(UA_ARGS);
    case 2: return fused_t<T, D, 2, 12>(UA_ARGS);
    case 3: return fused_t<T, D, 2, 16>(UA_ARGS);
    case 4: return fused_t<T, D, 2, 4>(UA_ARGS);
    default: return fused_t<T, D, 2, 8>(UA_ARGS);
  }
#undef UA_ARGS
}
hipError_t launch_fwd_fused(int dtype, int D, int variant, const void* Qp, const void* Kp, const void* VT,
                            const float* lsrc, const float* ldest, const float* C, void* O, float* lse, float* lse2,
                            const int* reach, int R, int L, int Lp, int d, int Zq, const RowsOut& orow, hipStream_t s,
                            const void* Bt, bool prune) {
#define UA_ARGS Qp, Kp, VT, lsrc, ldest, C, O, lse, lse2, reach, R, L, Lp, d, Zq, orow, s
  if (D == 256) return (dtype == 1 && Bt) ? fwd_tiles_256(UA_ARGS, Bt) : hipErrorInvalidValue;
#define UA_TILES variant, prune, Qp, Kp, VT, O, lse, lse2, reach, R, L, Lp, d, Zq, orow, s, Bt
  if (dtype == 1 && Bt) return D == 64 ? fwd_tiles<64>(UA_TILES) : fwd_tiles<128>(UA_TILES);
#undef UA_TILES
  if (dtype == 1) return D == 64 ? fused_v<bf16, 64>(variant, UA_ARGS) : fused_v<bf16, 128>(variant, UA_ARGS);
  return D == 64 ? fwd_split<64>(UA_ARGS) : fwd_split<128>(UA_ARGS);
#undef UA_ARGS
}

// chunked operator through the query-stationary kernel (chunk a multiple of 64; tiled working tensors)
template <class T, int D>
static hipError_t chunked2_t(const void* Qp, const void* Kp, const void* Vp, const void* VT, const float* lsrc, const float* ldest,
                             const float* C, const int* reach, void* out, void* denom, float* lse2, long o_sz,
                             long o_st, long o_sd, long o_si, int R, int L, int Lp, int d, int c, int nch, int Zq, hipStream_t s, int pair) {
  constexpr int NST = sizeof(T) == 2 ? 2 : 1, NW = 8;
  constexpr long VV = 16 / (long)sizeof(T);
  const int ovec = out && o_sd == 1 && d % VV == 0 && (uintptr_t)out % 16 == 0 && o_sz % VV == 0 && o_st % VV == 0 && o_si % VV == 0;
  ChunkOut<T> co{(T*)out, (T*)denom, o_sz, o_st, o_sd, o_si, c, nch, ovec};
  // two query blocks per workgroup once every CU gets at least four of the single ones
  const int n_blk = (Lp / 16 + NW - 1) / NW, gx = paired_items(n_blk, (long)n_blk * Zq >= 4L * device_cus(), pair);
  hipLaunchKernelGGL((k_fwd_fused2<T, D, NST, NW, true>), dim3(gx, Zq), dim3(64 * NW), 0, s, RowsOut{}, (const T*)Qp,
                     (const T*)Kp, (const T*)VT, lsrc, ldest, C, (T*)nullptr, (float*)nullptr, lse2, reach, R, L, Lp, d, co, (const _Float16*)nullptr);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (out && nch > 1) {
    const int vec = ovec;
    const int slabs = (std::min((nch - 1) * c, L) + kMaskedSlab - 1) / kMaskedSlab;
    hipLaunchKernelGGL((k_chunk_masked_out<T, D>), dim3(slabs, nch, Zq), dim3(256), 0, s, (const T*)Vp, co, R, L, Lp, d, vec);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  if (nch > 1) {
    hipLaunchKernelGGL((k_chunk_masked_denom<T>), dim3((Lp + 255) / 256, Zq), dim3(256), 0, s, (T*)denom, lse2, L, Lp, c, nch);
    e = hipGetLastError();
  }
  return e;
}
hipError_t launch_fwd_chunked2(int dtype, int D, const void* Qp, const void* Kp, const void* Vp, const void* VT, const float* lsrc,
                               const float* ldest, const float* C, const int* reach, void* out, void* denom,
                               float* lse2, long o_sz, long o_st, long o_sd, long o_si, int R, int L, int Lp, int d, int c, int nch,
                               int Zq, hipStream_t s, int pair) {
#define UA_ARGS Qp, Kp, Vp, VT, lsrc, ldest, C, reach, out, denom, lse2, o_sz, o_st, o_sd, o_si, R, L, Lp, d, c, nch, Zq, s, pair
  if (dtype == 1) return D == 64 ? chunked2_t<bf16, 64>(UA_ARGS) : chunked2_t<bf16, 128>(UA_ARGS);
  return D == 64 ? chunked2_t<float, 64>(UA_ARGS) : chunked2_t<float, 128>(UA_ARGS);
#undef UA_ARGS
}

template <class T, int D, int NW>
static hipError_t chunked_t(const void* Qp, const void* Kp, const void* VT, const float* lsrc, const float* ldest, void* out,
                            void* denom, float* lse2, long o_sz, long o_st, long o_sd, long o_si, int R, int L, int Lp,
                            int d, int c, int nch, int Zk, hipStream_t s) {
  const size_t lds = (64 * lds_stride<T>(D) + 32 * lds_stride<T>(32 * NW)) * sizeof(T) + (NW * 32 + D) * sizeof(float);
  allow_lds(k_fwd_chunked<T, D, NW>, lds);
  hipLaunchKernelGGL((k_fwd_chunked<T, D, NW>), dim3(nch, Zk), dim3(64 * NW), lds, s, (const T*)Qp, (const T*)Kp,
                     (const T*)VT, lsrc, ldest, (T*)out, (T*)denom, lse2, o_sz, o_st, o_sd, o_si, R, L, Lp,
                     d, c, nch);
  return hipGetLastError();
}
template <class T, int D>
static hipError_t chunked_nw(int NW, const void* Qp, const void* Kp, const void* VT, const float* lsrc, const float* ldest,
                             void* out, void* denom, float* lse2, long o_sz, long o_st, long o_sd, long o_si, int R, int L,
                             int Lp, int d, int c, int nch, int Zk, hipStream_t s) {
#define UA_ARGS Qp, Kp, VT, lsrc, ldest, out, denom, lse2, o_sz, o_st, o_sd, o_si, R, L, Lp, d, c, nch, Zk, s
  switch (NW) {
    case 1: return chunked_t<T, D, 1>(UA_ARGS);
    case 2: return chunked_t<T, D, 2>(UA_ARGS);
    case 4: return chunked_t<T, D, 4>(UA_ARGS);
    default: return chunked_t<T, D, 8>(UA_ARGS);
  }
#undef UA_ARGS
}
hipError_t launch_fwd_chunked(int dtype, int D, const void* Qp, const void* Kp, const void* VT, const float* lsrc,
                              const float* ldest, void* out, void* denom, float* lse2, long o_sz, long o_st, long o_sd,
                              long o_si, int R, int L, int Lp, int d, int c, int nch, int Zk, hipStream_t s) {
  int NW = c <= 32 ? 1 : c <= 64 ? 2 : c <= 128 ? 4 : 8;
#define UA_ARGS NW, Qp, Kp, VT, lsrc, ldest, out, denom, lse2, o_sz, o_st, o_sd, o_si, R, L, Lp, d, c, nch, Zk, s
  if (dtype == 1) return D == 64 ? chunked_nw<bf16, 64>(UA_ARGS) : chunked_nw<bf16, 128>(UA_ARGS);
  return D == 64 ? chunked_nw<float, 64>(UA_ARGS) : chunked_nw<float, 128>(UA_ARGS);
#undef UA_ARGS
}

}  // namespace ua
