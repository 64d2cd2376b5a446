// Layout kernels: bring user tensors (arbitrary strides, head dim d) into the padded,
// contiguous working layouts the matrix-core kernels read, plus small row reductions.
#pragma once
#include "ua_common.hpp"

namespace ua {

// offset of a row of a RowsView: its z part and its row part (the latter without divisions when row < inner)
__device__ __forceinline__ long rows_base(const RowsView& v, int z) {
  int i = z % v.N; z /= v.N;
  int r = z % v.R; z /= v.R;
  int h = z % v.H, b = z / v.H;
  return (long)b * v.sb + (long)h * v.sh + (long)r * v.sr + (long)i * v.sn;
}
__device__ __forceinline__ long rows_row(const RowsView& v, int row) {
  if (row < v.inner) return (long)row * v.si;
  return (long)(row / v.inner) * v.so + (long)(row % v.inner) * v.si;
}

// 32 rows of a tensor for pack_block: row `row0 + rr` of z at base(z) + the row part
struct PackSrc {
  RowsView x;
  int vec;      // every row start is 16-byte aligned and d is a multiple of the 16-byte vector (host-checked)
};

// One block of 32 rows of x (dtype T) -> nat and/or tr working tensors, zero padded (rows >= L, cols >= d).
//   tiled == 0: nat [Z][Lp][D] row-major, tr [Z][D][Lp] row-major       (chunked-mode kernels)
//   tiled != 0: both in tiles of 32 positions, k-group-major (nat_off / tr_off)   (fused kernels)
// tr stores position t at column perm16(t) (tr_mode 0), perm32(t) (1) or t (2) of its group of 32.
// norm2 (optional): [Z][Lp/32] receives the largest squared row norm of the block.
// DOT: `O` is a second tensor of the same shape, whose row-wise product with x goes to delta[z][t] (padded rows: 0).
template <class T, int D, bool DOT>
__device__ __forceinline__ void pack_block(float (*tile)[D + 1], const PackSrc& s, int z, int blk, T* __restrict__ nat,
                                           T* __restrict__ tr, int d, int L, int Lp, int tr_mode, int tiled,
                                           float* __restrict__ norm2, const PackSrc* O = nullptr, float* __restrict__ delta = nullptr) {
  constexpr int V = 16 / (int)sizeof(T), LPR = D / V;       // lanes per row of 16-byte vectors
  const int row0 = blk * 32, tid = threadIdx.x;
  const T* xp = reinterpret_cast<const T*>(s.x.p) + rows_base(s.x, z);
  const T* op = DOT ? reinterpret_cast<const T*>(O->x.p) + rows_base(O->x, z) : nullptr;
  const bool vec = s.vec && (!DOT || O->vec);
  if (vec) {
#pragma unroll
    for (int i = tid; i < 32 * LPR; i += 256) {
      const int rr = i / LPR, col = (i - rr * LPR) * V, row = row0 + rr;
      T v[V];
      float dot = 0.f;
      if (row < L && col < d) {
        *reinterpret_cast<uint4*>(v) = *reinterpret_cast<const uint4*>(xp + rows_row(s.x, row) + col);
        if constexpr (DOT) {
          T o[V];
          *reinterpret_cast<uint4*>(o) = *reinterpret_cast<const uint4*>(op + rows_row(O->x, row) + col);
#pragma unroll
          for (int e = 0; e < V; ++e) dot += (float)o[e] * (float)v[e];
        }
      } else {
#pragma unroll
        for (int e = 0; e < V; ++e) v[e] = cvt<T>(0.f);
      }
#pragma unroll
      for (int e = 0; e < V; ++e) tile[rr][col + e] = (float)v[e];
      if (nat && !tiled) *reinterpret_cast<uint4*>(nat + ((long)z * Lp + row) * D + col) = *reinterpret_cast<const uint4*>(v);
      if constexpr (DOT) {
#pragma unroll
        for (int m = LPR / 2; m >= 1; m >>= 1) dot += __shfl_xor(dot, m, 64);
        if ((tid & (LPR - 1)) == 0) delta[(long)z * Lp + row] = dot;
      }
    }
  } else {
    for (int i = tid; i < 32 * D; i += 256) {
      int rr = i / D, col = i - rr * D, row = row0 + rr;
      float val = 0.f;
      if (row < L && col < d) val = (float)xp[rows_row(s.x, row) + (long)col * s.x.sc];
      tile[rr][col] = val;
      if (nat && !tiled) nat[((long)z * Lp + row) * D + col] = cvt<T>(val);
    }
  }
  if (!tr && !(nat && tiled) && !norm2 && !DOT) return;
  __syncthreads();
  if (DOT && !vec) {
    const int rr = tid >> 3, row = row0 + rr;
    float dot = 0.f;
    if (row < L)
      for (int c = tid & 7; c < d; c += 8) dot += (float)op[rows_row(O->x, row) + (long)c * O->x.sc] * tile[rr][c];
#pragma unroll
    for (int m = 1; m <= 4; m <<= 1) dot += __shfl_xor(dot, m, 64);
    if ((tid & 7) == 0) delta[(long)z * Lp + row] = dot;
  }
  if (norm2) {
    // largest squared row norm of the block's (dtype-rounded) rows -> norm2[z][block]: 8 threads per row, then the
    // maximum over the block
    __shared__ float wmax[4];
    const int rr = tid >> 3;
    float s2 = 0.f;
    for (int c = tid & 7; c < D; c += 8) s2 += tile[rr][c] * tile[rr][c];
#pragma unroll
    for (int m = 1; m <= 4; m <<= 1) s2 += __shfl_xor(s2, m, 64);             // the 8 threads of a row
#pragma unroll
    for (int m = 8; m <= 32; m <<= 1) s2 = fmaxf(s2, __shfl_xor(s2, m, 64));   // the 8 rows of a wave
    if ((tid & 63) == 0) wmax[tid >> 6] = s2;
    __syncthreads();
    if (tid == 0) norm2[(long)z * (Lp / 32) + blk] = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
  }
  if (nat && tiled) {
    // one (k-group, row) cell of 8 elements per thread; consecutive threads write consecutive cells
    for (int i = tid; i < 4 * D; i += 256) {
      const int rr = i & 31, kg = i >> 5;
      T v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = cvt<T>(tile[rr][8 * kg + e]);
      T* dst = nat + nat_off<D>(z, Lp, row0 + rr, 8 * kg);
#pragma unroll
      for (int u = 0; u < 8 / V; ++u) reinterpret_cast<uint4*>(dst)[u] = reinterpret_cast<const uint4*>(v)[u];
    }
  }
  if (!tr) return;
  // perm16 and perm32 are bijections of 0..31: column p holds the position that maps onto it
  if (tiled) {
    for (int i = tid; i < 4 * D; i += 256) {
      const int dd = i % D, kg = i / D;
      T v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int p = 8 * kg + e;
        const int src = tr_mode == 0 ? perm16(p) : (tr_mode == 1 ? (((p >> 3) & 3) << 2 | ((p >> 2) & 1) << 4 | (p & 3)) : p);
        v[e] = cvt<T>(tile[src][dd]);
      }
      T* dst = tr + tr_off<D>(z, Lp, dd, blk, 8 * kg);
#pragma unroll
      for (int u = 0; u < 8 / V; ++u) reinterpret_cast<uint4*>(dst)[u] = reinterpret_cast<const uint4*>(v)[u];
    }
  } else {
    for (int i = tid; i < 32 * D; i += 256) {
      const int dd = i >> 5, rr = i & 31;
      const int src = tr_mode == 0 ? perm16(rr) : (tr_mode == 1 ? (((rr >> 3) & 3) << 2 | ((rr >> 2) & 1) << 4 | (rr & 3)) : rr);
      tr[((long)z * D + dd) * Lp + row0 + rr] = cvt<T>(tile[src][dd]);
    }
  }
}

// One tensor.  grid (Lp/32, Z).
// masked_nz (optional; chunked operator, z = zq*N + chunk, chunk size c): blocks of rows before their chunk are left
// untouched while *masked_nz is 0 (k_delta has found every such row of x to be zero, and no kernel reads them then).
template <class T, int D>
__global__ void __launch_bounds__(256) k_pack(RowsView x, T* __restrict__ nat, T* __restrict__ tr, int d, int L, int Lp,
                                              int tr_mode, int tiled, int vec, const int* __restrict__ masked_nz, int c) {
  __shared__ float tile[32][D + 1];
  const int z = blockIdx.y;
  if (masked_nz && (int)blockIdx.x * 32 + 32 <= (z % x.N) * c && *masked_nz == 0) return;
  pack_block<T, D, false>(tile, PackSrc{x, vec}, z, blockIdx.x, nat, tr, d, L, Lp, tr_mode, tiled, nullptr);
}

// Keys, values, queries and gates of a pass in one launch (as four launches each of them waits for the one before and the
// small ones cost a launch, 2-5 us each, whatever they hold).  Grid: Lp/32 blocks for every one of the Zk key heads, then
// the Zk value heads, then the Zq query heads; the key blocks also take the logarithms of their 32 positions' gates:
// lsrc / ldest [Zk][Lp] = log2(gate) / 3, kGatePad beyond L.  Tensors whose pointer is null are not written.
struct PackInputs {
  PackSrc K, V, Q;
  GateView g;
  void *Kp, *KT, *Vp, *VT, *Qp, *QT;
  float *lsrc, *ldest, *knorm2, *qnorm2;
  int Zk, d, L, Lp, tiled, mode, vmode;     // tr_mode of K and Q, and of V
};
template <class T, int D>
__global__ void __launch_bounds__(256) k_pack_inputs(PackInputs a) {
  __shared__ float tile[32][D + 1];
  const int nb = a.Lp >> 5, blk = blockIdx.x % nb, j = blockIdx.x / nb;
  if (j >= 2 * a.Zk) {
    pack_block<T, D, false>(tile, a.Q, j - 2 * a.Zk, blk, (T*)a.Qp, (T*)a.QT, a.d, a.L, a.Lp, a.mode, a.tiled, a.qnorm2);
  } else if (j >= a.Zk) {
    pack_block<T, D, false>(tile, a.V, j - a.Zk, blk, (T*)a.Vp, (T*)a.VT, a.d, a.L, a.Lp, a.vmode, a.tiled, nullptr);
  } else {
    if (threadIdx.x < 64) {
      const int t = 32 * blk + (threadIdx.x & 31), dest = threadIdx.x >> 5;
      float x = kGatePad;
      if (t < a.L) x = __builtin_amdgcn_logf(gate_at<T>(dest ? a.g.dest : a.g.src, gate_off(a.g, j, t), a.g.f32)) * (1.0f / 3.0f);
      (dest ? a.ldest : a.lsrc)[(long)j * a.Lp + t] = x;
    }
    pack_block<T, D, false>(tile, a.K, j, blk, (T*)a.Kp, (T*)a.KT, a.d, a.L, a.Lp, a.mode, a.tiled, a.knorm2);
  }
}

// Upstream gradient of the merged operator: dO -> tiled working tensors and delta[z][t] = dO . O in one pass over dO; lse
// (natural log, [Z][L]) is rewritten in log2 units into lse2 [Z][Lp] (also when a forward state holds lse2: the same bits
// with and without a state).  grid (Lp/32 * Z).
template <class T, int D>
__global__ void __launch_bounds__(256) k_pack_grad(PackSrc dO, PackSrc O, const float* __restrict__ lse, T* __restrict__ nat,
                                                   T* __restrict__ tr, float* __restrict__ delta, float* __restrict__ lse2, int d, int L, int Lp) {
  __shared__ float tile[32][D + 1];
  const int nb = Lp >> 5, blk = blockIdx.x % nb, z = blockIdx.x / nb;
  if (threadIdx.x < 32) {
    const int t = 32 * blk + threadIdx.x;
    lse2[(long)z * Lp + t] = t < L ? lse[(long)z * L + t] * kLog2e : 0.f;
  }
  pack_block<T, D, true>(tile, dO, z, blk, nat, tr, d, L, Lp, 1, 1, nullptr, &O, delta);
}

// delta[z][t] = sum_dd O[z][t][dd] * dO[z][t][dd] - sub[z][t]   (fp32; padded rows -> 0)
// O, dO, sub are views (sub optional, float); 16 lanes per row, 128 rows per block (grid (Lp/128, Z)).
// vec != 0: rows of O and dO start 16-byte aligned, have unit feature stride and d is a multiple of the vector.
// masked_nz (optional; chunked operator, z = zq*N + chunk, chunk size c): set to 1 when a row of dO or sub that lies
// before its chunk (t < chunk*c, a query that sees no key of the chunk) holds a non-zero.
template <class T>
__global__ void __launch_bounds__(256) k_delta(RowsView O, RowsView dO, RowsView sub, float* __restrict__ delta, int d, int L, int Lp, int vec,
                                               int* __restrict__ masked_nz, int c) {
  constexpr int V = 16 / (int)sizeof(T), IT = 8;
  const int z = blockIdx.y, sub16 = threadIdx.x & 15;
  const int t0 = blockIdx.x * (16 * IT) + (threadIdx.x >> 4);
  const int chunk_start = masked_nz ? (z % dO.N) * c : 0;
  const T* Oz = reinterpret_cast<const T*>(O.p) + rows_base(O, z);
  const T* Gz = reinterpret_cast<const T*>(dO.p) + rows_base(dO, z);
  const float* Sz = sub.p ? reinterpret_cast<const float*>(sub.p) + rows_base(sub, z) : nullptr;
  bool flag = false;
#pragma unroll
  for (int it = 0; it < IT; ++it) {
    const int t = t0 + 16 * it;
    float s = 0.f;
    bool nz = false;
    if (t < L) {
      const T* o = Oz + rows_row(O, t);
      const T* g = Gz + rows_row(dO, t);
      if (vec) {
        // a row before its chunk normally holds zeros: its product with O is then not needed
        const bool before_chunk = t < chunk_start;
        for (int cc = sub16 * V; cc < d; cc += 16 * V) {
          T a[V], b[V];
          *reinterpret_cast<uint4*>(b) = *reinterpret_cast<const uint4*>(g + cc);
          if (before_chunk) {
            bool any = false;
#pragma unroll
            for (int e = 0; e < V; ++e) any |= ((float)b[e] != 0.f);
            if (!any) continue;
          }
          *reinterpret_cast<uint4*>(a) = *reinterpret_cast<const uint4*>(o + cc);
#pragma unroll
          for (int e = 0; e < V; ++e) { s += (float)a[e] * (float)b[e]; nz |= ((float)b[e] != 0.f); }
        }
      } else {
        for (int cc = sub16; cc < d; cc += 16) {
          const float b = (float)g[(long)cc * dO.sc];
          s += (float)o[(long)cc * O.sc] * b;
          nz |= (b != 0.f);
        }
      }
    }
#pragma unroll
    for (int m = 8; m >= 1; m >>= 1) s += __shfl_xor(s, m, 64);
    if (sub16 == 0 && t < Lp) {
      if (Sz && t < L) {
        const float sv = Sz[rows_row(sub, t)];
        s -= sv;
        nz |= (sv != 0.f);
      }
      delta[(long)z * Lp + t] = s;
    }
    flag |= nz && t < chunk_start;
  }
  if (masked_nz && __any(flag)) {
    if ((threadIdx.x & 63) == 0 && *reinterpret_cast<volatile int*>(masked_nz) == 0) atomicOr(masked_nz, 1);
  }
}

// plain fill (kept as a kernel so that callers may capture the sequence in a HIP graph)
__global__ void __launch_bounds__(256) k_zero(float4* __restrict__ p, size_t n16) {
  for (size_t i = blockIdx.x * (size_t)256 + threadIdx.x; i < n16; i += (size_t)gridDim.x * 256) p[i] = make_float4(0.f, 0.f, 0.f, 0.f);
}

}  // namespace ua
