// LaplaceSubtraction on gfx950: pairwise L1 distance and its sign-weighted
// backward, on the vector ALU.
//
// Reference semantics (src/LaplaceSubtraction_cuda_kernel.cu):
//   forward  out[i,j] = cast(sum_c |f32(q[i,c]) - f32(k[c,j])|), c ascending      (:84-140)
//   dq       dq[i,c]  = cast(sum_j f32(g[i,j]) * sgn(f32(q[i,c]) - f32(k[c,j])))   (:183-266)
//   dk       dk[c,j]  = cast(-sum_i f32(g[i,j]) * sgn(f32(q[i,c]) - f32(k[c,j])))  (:309-392)
//   sgn(0) = 0 (:34-38); fp32 accumulation, fp64 for double (:17-19).
//
// Forward mapping: one wave = 64 consecutive query rows (one per lane) x JB key
// columns; the key tile sits in LDS and every lane reads the same address
// (broadcast), so each (c, j) step costs one subtract and one |.|-add per lane.
// For fp16 the subtract is v_fma_mix_f32 on the packed halves: no conversions.
//
// Backward mapping: one lane per channel c, one wave per run of query rows,
// key column held in registers, the grad_output row broadcast from LDS. dq is a
// lane-local sum over j; dk is a lane-local sum over the wave's rows, reduced
// across the workgroup's waves in LDS in a fixed order and across workgroups by
// a second small kernel (fixed order again), so results are deterministic. A
// kernel boundary rather than device-scope fences: with one L2 per XCD, an
// agent-scope release/acquire writes back / invalidates a whole L2.
#include <algorithm>

#include "lf_common.h"
#include "lf_internal.h"

namespace lfamd {

// ---------------------------------------------------------------------------
// Staged element type for the forward key tile.
// ---------------------------------------------------------------------------
template <typename T> struct StageOf { using type = float; };
template <> struct StageOf<f16s> { using type = uint16_t; };
template <> struct StageOf<double> { using type = double; };

__device__ __forceinline__ float stage_val(float v) { return v; }
__device__ __forceinline__ float stage_val(bf16s v) { return to_acc(v); }
__device__ __forceinline__ uint16_t stage_val(f16s v) { return v.bits; }
__device__ __forceinline__ double stage_val(double v) { return v; }

constexpr int kFwdKC = 64;  // minimum channels staged per LDS pass

// Query elements per 16-byte vector load in the forward.
template <typename T> struct QChunk { static constexpr int value = 16 / sizeof(T); };

// Forward launch flags.
constexpr int kFwdVecQ = 1;    // query rows start on 16 bytes and C % QChunk == 0
constexpr int kFwdVecOut = 2;  // output tile of whole rows starts on 16 bytes

// One wave = 64 query rows (one per lane) x JB key columns; one workgroup =
// W column blocks (one per wave) x `rowBlocks` consecutive 64-row blocks, so the
// staged key tile is reused for several row blocks. KC = channels staged per
// LDS pass (all of C when it fits, which is the common case).
// Waves per forward workgroup: wide column blocks need more registers.
__host__ __device__ constexpr int fwd_max_waves(int jb) { return jb >= 32 ? 8 : 16; }

template <typename T, int JB>
__global__ void __launch_bounds__(64 * fwd_max_waves(JB))
laplace_fwd_kernel(const T* __restrict__ query, const T* __restrict__ key, T* __restrict__ out,
                   int N, int M, int C, int colsPerGroup, int rowBlocks, int KC, int flags) {
  using S = typename StageOf<T>::type;
  using A = typename AccOf<T>::type;
  constexpr int SV = 16 / (int)sizeof(S);  // staged elements per 16-byte LDS read
  constexpr int JBP = round_up(JB, SV);
  constexpr int CK = QChunk<T>::value;
  constexpr bool kF16 = std::is_same<T, f16s>::value;

  const int W = blockDim.x >> 6;
  const int wave = uniform(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int bh = blockIdx.z;
  const int jg0 = blockIdx.y * colsPerGroup;
  const int ldsCols = W * JBP;
  const int nChunks = ceil_div(C, KC);
  const bool vecq = flags & kFwdVecQ;

  extern __shared__ __align__(16) unsigned char smem[];
  S* kt = reinterpret_cast<S*>(smem);                                          // [W][KC][JBP]
  T* ot = reinterpret_cast<T*>(smem + (size_t)KC * ldsCols * sizeof(S));      // [64][colsPerGroup]

  const T* kb = key + (size_t)bh * C * M;
  const S* kw = kt + (size_t)wave * KC * JBP;

  // Stages key channels [c0, c0 + KC) for this workgroup's columns. One
  // column per lane, so the index arithmetic is per column, not per element.
  auto stage = [&](int c0) {
    const int kc = min(KC, C - c0);
    for (int u = lane; u < ldsCols; u += 64) {
      const int wb = u / JBP, jj = u - wb * JBP;
      const int col = jg0 + wb * JB + jj;
      const bool ok = jj < JB && col < M;
      for (int cc = wave; cc < KC; cc += W)
        kt[((size_t)wb * KC + cc) * JBP + jj] = (ok && cc < kc) ? stage_val(kb[(size_t)(c0 + cc) * M + col]) : S(0);
    }
  };

  const int nrb = ceil_div(N, 64);
  const int rb0 = blockIdx.x * rowBlocks;
  for (int rbi = 0; rbi < rowBlocks && rb0 + rbi < nrb; ++rbi) {
    const int row0 = (rb0 + rbi) * 64;
    const int row = row0 + lane;
    const T* qrow = query + ((size_t)bh * N + (row < N ? row : N - 1)) * C;  // rows past N are never stored

    A acc[JB];
#pragma unroll
    for (int j = 0; j < JB; ++j) acc[j] = A(0);

    for (int ch = 0; ch < nChunks; ++ch) {
      const int c0 = ch * KC;
      const int kc = min(KC, C - c0);
      if (nChunks > 1 || rbi == 0) {
        __syncthreads();
        stage(c0);
        __syncthreads();
      }
      for (int cc = 0; cc < kc; cc += CK) {
        const int cg = c0 + cc;
        if constexpr (kF16) {
          uint32_t qh[4];
          if (vecq) {
            const uint4 v = *reinterpret_cast<const uint4*>(qrow + cg);
            qh[0] = v.x; qh[1] = v.y; qh[2] = v.z; qh[3] = v.w;
          } else {
#pragma unroll
            for (int p = 0; p < 4; ++p) {
              const uint32_t lo = (cg + 2 * p < C) ? qrow[cg + 2 * p].bits : 0u;
              const uint32_t hi = (cg + 2 * p + 1 < C) ? qrow[cg + 2 * p + 1].bits : 0u;
              qh[p] = lo | (hi << 16);
            }
          }
#pragma unroll
          for (int u = 0; u < CK; ++u) {
            uint32_t kwv[JBP / 2];
            const uint4* kr = reinterpret_cast<const uint4*>(kw + (cc + u) * JBP);
#pragma unroll
            for (int t = 0; t < JBP / 8; ++t) {
              const uint4 v = kr[t];
              kwv[4 * t] = v.x; kwv[4 * t + 1] = v.y; kwv[4 * t + 2] = v.z; kwv[4 * t + 3] = v.w;
            }
            const uint32_t qp = qh[u >> 1];
#pragma unroll
            for (int j = 0; j < JB; ++j) {
              const uint32_t kp = kwv[j >> 1];
              float d;
              if (u & 1) d = (j & 1) ? mix_sub_hh<1, 1>(qp, kp) : mix_sub_hh<1, 0>(qp, kp);
              else       d = (j & 1) ? mix_sub_hh<0, 1>(qp, kp) : mix_sub_hh<0, 0>(qp, kp);
              acc[j] += fabsf(d);
            }
          }
        } else {
          A qf[CK];
          if (vecq) {
            if constexpr (std::is_same<T, bf16s>::value) {
              const uint4 v = *reinterpret_cast<const uint4*>(qrow + cg);
              const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
              for (int p = 0; p < 4; ++p) {
                qf[2 * p] = __builtin_bit_cast(float, w[p] << 16);
                qf[2 * p + 1] = __builtin_bit_cast(float, w[p] & 0xffff0000u);
              }
            } else {
              const T* src = qrow + cg;
#pragma unroll
              for (int p = 0; p < CK; ++p) qf[p] = to_acc(src[p]);
            }
          } else {
#pragma unroll
            for (int p = 0; p < CK; ++p) qf[p] = (cg + p < C) ? to_acc(qrow[cg + p]) : A(0);
          }
#pragma unroll
          for (int u = 0; u < CK; ++u) {
            const S* kr = kw + (cc + u) * JBP;
            S kv[JBP];
#pragma unroll
            for (int t = 0; t < JBP; ++t) kv[t] = kr[t];
            const A qv = qf[u];
#pragma unroll
            for (int j = 0; j < JB; ++j) acc[j] += fabs(qv - (A)kv[j]);
          }
        }
      }
    }

    // Stage the 64 x colsPerGroup tile in LDS, then store it row-contiguously.
    if (rbi > 0) __syncthreads();  // previous block's stores have read ot
#pragma unroll
    for (int j = 0; j < JB; ++j) ot[lane * colsPerGroup + wave * JB + j] = from_acc<T>(acc[j]);
    __syncthreads();
    const int colsValid = min(colsPerGroup, M - jg0);
    const int rowsValid = min(64, N - row0);
    T* ob = out + ((size_t)bh * N + row0) * M + jg0;
    if (colsPerGroup == M) {
      // Whole rows: the tile is one contiguous range of rowsValid * M elements.
      const int total = rowsValid * M;
      int done = 0;
      if (flags & kFwdVecOut) {
        constexpr int VE = 16 / (int)sizeof(T);
        const int nv = total / VE;
        for (int e = threadIdx.x; e < nv; e += blockDim.x)
          reinterpret_cast<uint4*>(ob)[e] = reinterpret_cast<const uint4*>(ot)[e];
        done = nv * VE;
      }
      for (int e = done + threadIdx.x; e < total; e += blockDim.x) ob[e] = ot[e];
    } else {
      for (int r = wave; r < rowsValid; r += W)
        for (int cidx = lane; cidx < colsValid; cidx += 64) ob[(size_t)r * M + cidx] = ot[r * colsPerGroup + cidx];
    }
  }
}

// ---------------------------------------------------------------------------
// Forward with the key broadcast from LDS. Lane = query row, R rows per lane;
// a workgroup is the W = ceil(M / JB) waves that share one block of 64*R rows,
// wave w owning key columns [w*JB, w*JB + JB). The key is widened to fp32 once
// per workgroup into LDS; per channel a wave reads its JB key values as
// wave-wide broadcasts (ds_read_b128: one read feeds 8*R VALU instructions) and
// does |q - k| + acc as v_sub_f32 and v_add_f32 with an |.| modifier, both with
// VGPR operands only (full issue rate; an SGPR operand halves it on gfx950).
// The query is widened once per channel per row. Channels are summed in
// ascending order in fp32 (fp64 is not handled here), the reference's serial
// order, so results are bit-identical to it. The output tile of the 64*R rows
// is staged in LDS and written as one contiguous span. Requires C % 8 == 0 and a
// 16-byte aligned query (checked on the host).
// ---------------------------------------------------------------------------
template <typename T> __device__ __forceinline__ float elem_f32(const uint4& v, int e);
template <> __device__ __forceinline__ float elem_f32<f16s>(const uint4& v, int e) {
  const uint32_t w = (&v.x)[e >> 1];
  return (float)__builtin_bit_cast(_Float16, (uint16_t)(w >> (16 * (e & 1))));
}
template <> __device__ __forceinline__ float elem_f32<bf16s>(const uint4& v, int e) {
  const uint32_t w = (&v.x)[e >> 1];
  return __builtin_bit_cast(float, (e & 1) ? (w & 0xffff0000u) : (w << 16));
}
template <> __device__ __forceinline__ float elem_f32<float>(const uint4& v, int e) {
  return __builtin_bit_cast(float, (&v.x)[e]);
}

constexpr int kFbKC = 8;  // channels per query chunk of the broadcast forward

__host__ __device__ constexpr int fb_pitch(int jb) { return (jb + 3) & ~3; }

// Epilogue of the broadcast forward: the distance rounded to the element type,
// or the Laplacian kernel exp(-scale * distance) in fp32 (LaplacianFormer's
// K_xy; fp32 because the distance rounded to fp16 would move it by ~0.4 %).
enum FwdEpi { kEpiDist = 0, kEpiExp = 1 };
template <typename T, int EPI> struct FwdOut { using type = T; };
template <typename T> struct FwdOut<T, kEpiExp> { using type = float; };

// Channel sums of the broadcast forward for the first RR of a lane's R row sets
// (RR = 1 for a block of at most 64 rows: the second set would be idle lanes that
// still cost every instruction). acc[r][j] accumulates |q - k| over c ascending.
template <typename T, int JB, int R, int RR>
__device__ __forceinline__ void fb_sums(float (&acc)[R][JB], const uint4* qsm, const float* ksm, int rows,
                                        int wave, int lane, int KP, int QP, int C) {
  constexpr int JBS = fb_pitch(JB);
  constexpr int NG = JBS / 4;
  constexpr int EV = 16 / (int)sizeof(T);
  constexpr int NVC = kFbKC / EV;
  // Rows past the block's end read row 0 of the tile (their results are not stored).
  const uint4* qrow[RR];
#pragma unroll
  for (int r = 0; r < RR; ++r) qrow[r] = qsm + (r * 64 + lane < rows ? r * 64 + lane : 0) * QP;
  const float4* kw = reinterpret_cast<const float4*>(ksm + wave * JBS);
  const int KP4 = KP / 4;
  const int nChunks = C / kFbKC;
  // Key values one channel ahead and query vectors one chunk ahead of the
  // arithmetic; a compiler memory barrier per channel keeps it from hoisting a
  // whole chunk's reads (registers).
  uint4 qv[RR][NVC];
#pragma unroll
  for (int r = 0; r < RR; ++r)
#pragma unroll
    for (int v = 0; v < NVC; ++v) qv[r][v] = qrow[r][v];
  float4 kcur[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g) kcur[g] = kw[g];
  for (int kc = 0; kc < nChunks; ++kc) {
    uint4 qn[RR][NVC];
    const int kn = min(kc + 1, nChunks - 1);
#pragma unroll
    for (int r = 0; r < RR; ++r)
#pragma unroll
      for (int v = 0; v < NVC; ++v) qn[r][v] = qrow[r][kn * NVC + v];
#pragma unroll
    for (int cc = 0; cc < kFbKC; ++cc) {
      const int cnext = min(kc * kFbKC + cc + 1, C - 1);
      float4 knext[NG];
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        knext[g] = kw[cnext * KP4 + g];
        // Use the padding lane too, so the read stays one ds_read_b128 (a
        // narrower split, e.g. b96 + b32, costs more LDS cycles than b128).
        asm volatile("" ::"v"(knext[g].w));
      }
      float qf[RR];
#pragma unroll
      for (int r = 0; r < RR; ++r) qf[r] = elem_f32<T>(qv[r][cc / EV], cc % EV);
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const float k4[4] = {kcur[g].x, kcur[g].y, kcur[g].z, kcur[g].w};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          if (g * 4 + t < JB) {
#pragma unroll
            for (int r = 0; r < RR; ++r) acc[r][g * 4 + t] += fabsf(qf[r] - k4[t]);
          }
        }
      }
#pragma unroll
      for (int g = 0; g < NG; ++g) kcur[g] = knext[g];
      asm volatile("" ::: "memory");
    }
#pragma unroll
    for (int r = 0; r < RR; ++r)
#pragma unroll
      for (int v = 0; v < NVC; ++v) qv[r][v] = qn[r][v];
  }

}

template <typename T, int JB, int R, int EPI = kEpiDist>
__global__ void __launch_bounds__(1024)
laplace_fwd_bcast_kernel(const T* __restrict__ query, const T* __restrict__ key,
                         typename FwdOut<T, EPI>::type* __restrict__ out, int N, int Mg, int Mtot, int C,
                         float scale) {
  using O = typename FwdOut<T, EPI>::type;
  constexpr int JBS = fb_pitch(JB);
  constexpr int NG = JBS / 4;
  constexpr int EV = 16 / (int)sizeof(T);  // elements per 16-byte vector
  constexpr int NVC = kFbKC / EV;          // vectors per row per chunk
  const int W = blockDim.x >> 6;
  const int wave = uniform(threadIdx.x >> 6), lane = threadIdx.x & 63;
  // Workgroup -> (slice, row block): every slice's full blocks first, the
  // partial last blocks (N not a multiple of 64R) after all of them, so the
  // workgroups dispatched last, onto CUs that already hold their share, are
  // the short ones.
  // Column groups are the fastest grid index, so that the groups of one row
  // block run next to each other and share its query rows in L2.
  const int CG = (Mtot + Mg - 1) / Mg;
  const int cg = blockIdx.x % CG;
  const int nFull = N / (64 * R);
  const int BH = gridDim.y;
  const int id = blockIdx.y * (gridDim.x / CG) + blockIdx.x / CG;
  int bh, blk;
  if (id < BH * nFull) {
    bh = id / nFull;
    blk = id - bh * nFull;
  } else {
    bh = id - BH * nFull;
    blk = nFull;
  }
  const int i0 = blk * 64 * R;
  const int rows = min(64 * R, N - i0);
  // Column group cg: columns [cb0, cb0 + M) of the Mtot (the row stride
  // of key and output); one group covers all columns unless the tiles of all of
  // them would keep the workgroup to one per CU.
  const int cb0 = cg * Mg;
  const int M = min(Mg, Mtot - cb0);
  const int KP = W * JBS;              // key tile pitch (floats per channel)
  const int QV = C / EV;               // 16-byte vectors per query row
  const int QP = QV + 1;               // query tile pitch in vectors (padding: fewer bank conflicts)

  extern __shared__ __align__(16) unsigned char smem[];
  float* ksm = reinterpret_cast<float*>(smem);                  // [C][W*JBS] key, fp32
  uint4* qsm = reinterpret_cast<uint4*>(ksm + (size_t)C * KP);  // [64R][QP] query rows, raw
  O* otile = reinterpret_cast<O*>(qsm);                         // [64R][M] output (after the sums)

  // The block's query rows are one contiguous span: coalesced 16-byte copies.
  const uint4* qsrc = reinterpret_cast<const uint4*>(query + ((size_t)bh * N + i0) * C);
  for (int u = threadIdx.x; u < rows * QV; u += blockDim.x) {
    const int row = u / QV, v = u - row * QV;
    qsm[row * QP + v] = qsrc[u];
  }
  // Key tile, fp32, zero outside [0, M); channel c staged by wave c % W.
  const T* kb = key + (size_t)bh * C * Mtot + cb0;
  for (int c = wave; c < C; c += W) {
    for (int t = lane; t < KP; t += 64) {
      const int w = t / JBS, jj = t - w * JBS;
      const int col = w * JB + jj;
      ksm[c * KP + t] = (jj < JB && col < M) ? to_acc(kb[(size_t)c * Mtot + col]) : 0.0f;
    }
  }
  __syncthreads();

  float acc[R][JB];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int j = 0; j < JB; ++j) acc[r][j] = 0.0f;
  if (R > 1 && rows <= 64)
    fb_sums<T, JB, R, 1>(acc, qsm, ksm, rows, wave, lane, KP, QP, C);
  else
    fb_sums<T, JB, R, R>(acc, qsm, ksm, rows, wave, lane, KP, QP, C);

  __syncthreads();  // every wave is done with the query tile, which becomes the output tile
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int j = 0; j < JB; ++j) {
      const int col = wave * JB + j;
      if (col < M) {
        if constexpr (EPI == kEpiExp)
          otile[(r * 64 + lane) * M + col] = expf(-scale * acc[r][j]);
        else
          otile[(r * 64 + lane) * M + col] = from_acc<T>(acc[r][j]);
      }
    }
  __syncthreads();
  constexpr int OV = 16 / (int)sizeof(O);  // output elements per 16-byte vector
  O* dst = out + ((size_t)bh * N + i0) * Mtot + cb0;
  if (M != Mtot) {  // a column group: rows of M elements, Mtot apart
    if ((M % OV) == 0 && (reinterpret_cast<uintptr_t>(dst) & 15) == 0 && (Mtot % OV) == 0) {
      const int vr = M / OV;
      const uint4* src4 = reinterpret_cast<const uint4*>(otile);
      for (int t = threadIdx.x; t < rows * vr; t += blockDim.x) {
        const int r = t / vr;
        reinterpret_cast<uint4*>(dst + (size_t)r * Mtot)[t - r * vr] = src4[t];
      }
    } else {
      for (int t = threadIdx.x; t < rows * M; t += blockDim.x) {
        const int r = t / M;
        dst[(size_t)r * Mtot + (t - r * M)] = otile[t];
      }
    }
    return;
  }
  // Rows [i0, i0 + rows) are one contiguous span of rows*M elements.
  const int n = rows * M;
  int done = 0;
  if ((reinterpret_cast<uintptr_t>(dst) & 15) == 0) {
    const int nv = n / OV;
    const uint4* src4 = reinterpret_cast<const uint4*>(otile);
    uint4* dst4 = reinterpret_cast<uint4*>(dst);
    for (int t = threadIdx.x; t < nv; t += blockDim.x) dst4[t] = src4[t];
    done = nv * OV;
  }
  for (int t = done + threadIdx.x; t < n; t += blockDim.x) dst[t] = otile[t];
}

// ---------------------------------------------------------------------------
// Backward.
// ---------------------------------------------------------------------------
// sgn(q - k) with sgn(0) = 0. For fp16 inputs both operands are pre-scaled by
// 2^24, which makes every non-zero difference at least 1 in magnitude, so a
// clamp to [-1, 1] is the exact sign. For fp32/bf16 the difference is first
// scaled by 2^200 (ldexp; overflow to +-inf is fine) for the same effect.
template <typename T> struct SignOps {
  static __device__ __forceinline__ float scale(float v) { return v; }
  static __device__ __forceinline__ float sgn(float d) {
    return __builtin_amdgcn_fmed3f(ldexpf(d, 200), -1.0f, 1.0f);
  }
};
template <> struct SignOps<f16s> {
  static __device__ __forceinline__ float scale(float v) { return v * 16777216.0f; }
  static __device__ __forceinline__ float sgn(float d) {
    return __builtin_amdgcn_fmed3f(d, -1.0f, 1.0f);
  }
};
template <> struct SignOps<double> {
  static __device__ __forceinline__ double scale(double v) { return v; }
  static __device__ __forceinline__ double sgn(double d) {
    return (double)((d > 0.0) - (d < 0.0));
  }
};

constexpr int kBwdRB = 8;  // grad_output rows staged per LDS batch

// grad_output as staged in LDS: raw fp16 bits (consumed by v_fma_mix_f32),
// otherwise the accumulation type.
template <typename T> struct GStageOf { using type = typename AccOf<T>::type; };
template <> struct GStageOf<f16s> { using type = uint16_t; };
__device__ __forceinline__ float gstage(float v) { return v; }
__device__ __forceinline__ double gstage(double v) { return v; }
__device__ __forceinline__ float gstage(bf16s v) { return to_acc(v); }
__device__ __forceinline__ uint16_t gstage(f16s v) { return v.bits; }

template <typename T> constexpr int gstage_vec() { return 16 / (int)sizeof(typename GStageOf<T>::type); }

template <typename T, int JB, bool DQ, bool DK>
__global__ void __launch_bounds__(512)
laplace_bwd_kernel(const T* __restrict__ gout, const T* __restrict__ query,
                   const T* __restrict__ key, T* __restrict__ dq, T* __restrict__ dk,
                   typename AccOf<T>::type* __restrict__ partial, int N, int M, int C, int rowsPerWave) {
  using A = typename AccOf<T>::type;
  using SO = SignOps<T>;
  using GS = typename GStageOf<T>::type;
  constexpr bool kHalfG = std::is_same<T, f16s>::value;
  constexpr int GV = gstage_vec<T>();
  constexpr int JBP = round_up(JB, GV);

  const int W = blockDim.x >> 6;
  const int wave = uniform(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int bh = blockIdx.z;
  const int cb = blockIdx.y;
  const int x = blockIdx.x;
  const int nx = gridDim.x;
  const int slice = bh * gridDim.y + cb;
  const int c = cb * 64 + lane;
  const bool cval = c < C;
  const int rowBeg = (x * W + wave) * rowsPerWave;
  const int rowEnd = min(N, rowBeg + rowsPerWave);
  const bool multiJ = M > JB;

  extern __shared__ __align__(16) unsigned char smem[];
  GS* gsm = reinterpret_cast<GS*>(smem);               // [W][kBwdRB][JBP]  grad_output rows
  A* qsm = reinterpret_cast<A*>(gsm + (size_t)W * kBwdRB * JBP);  // [W][kBwdRB][64] scaled query values
  A* ksm = qsm + (size_t)W * kBwdRB * 64;              // [JB][64]          scaled key tile
  A* red = ksm + JB * 64;                              // [JB][64]          (DK)
  A* dqp = red + (DK ? JB * 64 : 0);                   // [W][rowsPerWave][64] (DQ && multiJ)

  const T* qb = query + (size_t)bh * N * C;
  const T* gb = gout + (size_t)bh * N * M;
  const T* kb = key + (size_t)bh * C * M;
  GS* gw = gsm + (size_t)wave * kBwdRB * JBP;
  A* qw = qsm + (size_t)wave * kBwdRB * 64;

  for (int jb0 = 0; jb0 < M; jb0 += JB) {
    const bool lastJ = jb0 + JB >= M;
    // Key tile [64 channels][JB columns] staged through LDS with coalesced loads,
    // then each lane keeps its channel's JB scaled values in registers.
    __syncthreads();  // previous j-block's readers of ksm are done
    for (int t = threadIdx.x; t < 64 * JB; t += blockDim.x) {
      const int cl = t / JB, j = t - cl * JB;
      const int cc = cb * 64 + cl, col = jb0 + j;
      ksm[j * 64 + cl] = (cc < C && col < M) ? SO::scale(to_acc(kb[(size_t)cc * M + col])) : A(0);
    }
    __syncthreads();
    A kreg[JB];
    A dka[JB];
#pragma unroll
    for (int j = 0; j < JB; ++j) {
      kreg[j] = ksm[j * 64 + lane];
      dka[j] = A(0);
    }

    // Software pipeline: the next batch's grad_output elements and query values
    // are loaded into registers while the current batch is computed from LDS.
    constexpr int NSTG = ceil_div(kBwdRB * JBP, 64);
    T gpre[NSTG];
    T qpre[kBwdRB];
    auto fetch = [&](int rb) {
      const int nr = min(kBwdRB, rowEnd - rb);
#pragma unroll
      for (int s = 0; s < NSTG; ++s) {
        const int e = lane + 64 * s;
        const int r = e / JBP, jj = e - r * JBP;
        const int col = jb0 + jj;
        gpre[s] = (r < nr && jj < JB && col < M) ? gb[(size_t)(rb + r) * M + col] : T{};
      }
#pragma unroll
      for (int r = 0; r < kBwdRB; ++r) qpre[r] = (r < nr && cval) ? qb[(size_t)(rb + r) * C + c] : T{};
    };
    if (rowBeg < rowEnd) fetch(rowBeg);

    for (int rb = rowBeg; rb < rowEnd; rb += kBwdRB) {
      const int nr = min(kBwdRB, rowEnd - rb);
#pragma unroll
      for (int s = 0; s < NSTG; ++s) {
        const int e = lane + 64 * s;
        if (e < kBwdRB * JBP) gw[e] = gstage(gpre[s]);
      }
#pragma unroll
      for (int r = 0; r < kBwdRB; ++r) qw[r * 64 + lane] = SO::scale(to_acc(qpre[r]));
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      if (rb + kBwdRB < rowEnd) fetch(rb + kBwdRB);

      for (int r = 0; r < nr; ++r) {
        const int i = rb + r;
        const A qv = qw[r * 64 + lane];
        A dqa = A(0);
        if (DQ && multiJ && jb0 > 0) dqa = dqp[((size_t)wave * rowsPerWave + (i - rowBeg)) * 64 + lane];
        const GS* gr = gw + r * JBP;
        if constexpr (kHalfG) {
          // 8 halves per 16-byte broadcast read; v_fma_mix_f32 widens them in place.
#pragma unroll
          for (int j0 = 0; j0 < JBP; j0 += 8) {
            const uint4 v = *reinterpret_cast<const uint4*>(gr + j0);
            const uint32_t gw4[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int t = 0; t < 8; ++t) {
              const int j = j0 + t;
              if (j < JB) {
                const float s = SO::sgn(qv - kreg[j]);
                const uint32_t gp = gw4[t >> 1];
                if (t & 1) {
                  if (DQ) dqa = mix_fma_fh<1>(s, gp, dqa);
                  if (DK) dka[j] = mix_fms_fh<1>(s, gp, dka[j]);
                } else {
                  if (DQ) dqa = mix_fma_fh<0>(s, gp, dqa);
                  if (DK) dka[j] = mix_fms_fh<0>(s, gp, dka[j]);
                }
              }
            }
          }
        } else {
#pragma unroll
          for (int j0 = 0; j0 < JBP; j0 += GV) {
            A gv[GV];
#pragma unroll
            for (int t = 0; t < GV; ++t) gv[t] = gr[j0 + t];
#pragma unroll
            for (int t = 0; t < GV; ++t) {
              const int j = j0 + t;
              if (j < JB) {
                const A s = SO::sgn(qv - kreg[j]);
                if (DQ) dqa = fma(s, gv[t], dqa);
                if (DK) dka[j] = fma(s, -gv[t], dka[j]);
              }
            }
          }
        }
        if (DQ) {
          if (lastJ) {
            if (cval) dq[((size_t)bh * N + i) * C + c] = from_acc<T>(dqa);
          } else {
            dqp[((size_t)wave * rowsPerWave + (i - rowBeg)) * 64 + lane] = dqa;
          }
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }

    if (DK) {
      // Fold the waves' partial sums in wave order (deterministic).
      for (int w = 0; w < W; ++w) {
        if (wave == w) {
#pragma unroll
          for (int j = 0; j < JB; ++j)
            red[j * 64 + lane] = (w == 0 ? A(0) : red[j * 64 + lane]) + dka[j];
        }
        __syncthreads();
      }
      // partial[slice][x][c_local][M]
      A* pb = partial + ((size_t)slice * nx + x) * 64 * M;
      for (int t = threadIdx.x; t < 64 * JB; t += blockDim.x) {
        const int cl = t / JB, j = t - cl * JB;
        const int col = jb0 + j;
        if (col < M) pb[(size_t)cl * M + col] = red[j * 64 + cl];
      }
      __syncthreads();
    }
  }

}

// ---------------------------------------------------------------------------
// Backward with every key column in registers (M in {16, 32, 49} for fp16,
// {16, 49} for fp32 / bf16), every per-triple instruction at the full VALU rate.
//
// With q' = 2^24 q and k' = 2^24 k (exact for fp16 values, whose nonzero
// differences are at least 2^-24), d = q' - k' is 0 or at least 1 in magnitude,
// so y = clamp(d/2 + 1/2) is exactly (sgn(q - k) + 1) / 2 and sgn = 2y - 1:
//   grad_query[i,c] = sum_j (2 g_ij) y_ijc - sum_j g_ij
//   grad_key[c,j]   = sum_i g_ij - sum_i (2 g_ij) y_ijc
// Per triple: v_sub, v_fma+clamp, two v_fma, all with VGPR operands (an SGPR
// operand, v_med3 or v_fma_mix would issue at half rate on gfx950). fp32 and
// bf16 scale the difference twice by 2^100 instead (every nonzero fp32
// difference is at least 2^-149, so |d| 2^200 >= 2^51; overflow to +-inf clamps
// correctly): one v_mul more per triple.
//
// Lane = channel, key' and the grad_key sums of the MC columns in registers.
// Each wave owns a row range and stages its grad rows, scaled by 2, in a private
// LDS batch of RB rows; every lane reads them as wave-wide broadcasts (one
// ds_read_b128 feeds 16 VALU instructions). The row sums sum_j g_ij and column
// sums sum_i g_ij come from the same batch. No cross-wave synchronisation until
// the final, wave-ordered grad_key reduction. Requires N*MC even and a 4-byte
// aligned grad_output (checked on the host).
// ---------------------------------------------------------------------------
constexpr int kBcRB = 8;  // grad rows per LDS batch
constexpr int kBcBufs = 4;  // LDS accumulators of the workgroup grad_key reduction

// fp32 steps y = (sgn(q - k) + 1)/2 of the two backward kernels below. A workgroup whose
// keys are all below 2^103 scales keys and queries by 2^24: exact, a key cannot overflow,
// and a query that does is an infinity on its own side of every key. A nonzero scaled
// difference is then at least 2^-125 and one FMA by 2^126 takes it past the clamp: a
// subtraction and a clamped FMA. With larger keys (infinities, NaN) the plain difference
// is scaled twice by 2^100 (>= 2^-149 becomes >= 2^51), one instruction more.
// Both loops are compiled where a kernel computes one gradient of a plain grad_output
// (fp32, 32 slices, N = 3136, M = 49, C = 64: grad_query 40 -> 33 us); with both
// gradients the second loop's registers spill (55 -> 93 us with it), and those keep the
// unscaled step alone.
constexpr float kStepKeyMax = 0x1p103f, kStepPre = 0x1p24f, kStepFast = 0x1p126f, kStepSlow = 0x1p100f;

// f(column, channel) over a 64-channel tile of MC columns, consecutive lanes on consecutive
// columns (contiguous in the key's layout), 64 / MC channels per wave and pass, so no division. The loop
// stays short, since what a call of a few rows pays for here is fetching its instructions once (with t / MC
// and t % MC of one flat loop, one row, fp32, M = 49, C = 64, grad_key: 19.7 us, now 11.3; before that loop
// 13.8. Flat for M = 16 and 32 alone: fp16 grad_query, 2048 slices of 9 rows, M = 32, 36.7 against 23 us).
template <int MC, typename F> __device__ __forceinline__ void each_tile_column(int W, int wave, int lane, F f) {
  constexpr int CP = 64 / MC;
  static_assert(CP == 1 || CP * MC == 64, "whole channels per pass");
  asm volatile("" : "+v"(lane));  // the lane's place is formed anew, not held in registers through the row loop
  const int j = CP == 1 ? lane : lane % MC;
  if (j < MC)
#pragma unroll 4
    for (int cl = wave * CP + (CP == 1 ? 0 : lane / MC); cl < 64; cl += W * CP) f(j, cl);
}

// Floats of the key tile [mc][65], whole 16-byte groups.
__host__ __device__ constexpr int bcast_key_floats(int mc) { return (mc * 65 + 3) & ~3; }

// Workgroup sum of the per-wave grad_key partials v[MC] (lane = channel), in a
// fixed order: wave w adds into LDS accumulator w % kBcBufs in rounds of
// increasing w / kBcBufs, then the accumulators are summed 0, 1, ... and the
// result goes to out(column, channel, sum), consecutive threads on consecutive
// channels, or with `cols` on consecutive columns (the pitch of 65 keeps both walks of
// the LDS and both stores coalesced). Every read of a round is issued before its
// writes. Needs kBcBufs * bcast_key_floats(MC) floats of LDS at `red`.
template <int MC, typename Out>
__device__ __forceinline__ void bcast_reduce_dk(const float (&v)[MC], float* red, int W, int wave, int lane,
                                                bool cols, Out out) {
  constexpr int BF = bcast_key_floats(MC);
  const int nb = min(W, kBcBufs);
  float* buf = red + (wave % nb) * BF;
  __syncthreads();  // every wave is done with the LDS it used before
  for (int round = 0; round * nb < W; ++round) {
    if (wave / nb == round) {
      if (round == 0) {
#pragma unroll
        for (int j = 0; j < MC; ++j) buf[j * 65 + lane] = v[j];
      } else {
        float pv[MC];
#pragma unroll
        for (int j = 0; j < MC; ++j) pv[j] = buf[j * 65 + lane];
#pragma unroll
        for (int j = 0; j < MC; ++j) buf[j * 65 + lane] = pv[j] + v[j];
      }
    }
    __syncthreads();
  }
  auto sum = [&](int j, int cl) {
    float s = red[j * 65 + cl];
    for (int b = 1; b < nb; ++b) s += red[b * BF + j * 65 + cl];
    return s;
  };
  if (cols)
    each_tile_column<MC>(W, wave, lane, [&](int j, int cl) { out(j, cl, sum(j, cl)); });
  else
    for (int j = wave; j < MC; j += W) out(j, lane, sum(j, lane));
}

__host__ __device__ constexpr int bcast_max_waves(int mc) { return mc <= 16 ? 16 : 12; }
// Row pitch (floats) of a staged grad row: whole 16-byte groups, an even number
// of them (the row loop keeps two groups in flight in a two-slot ring).
__host__ __device__ constexpr int bcast_pitch(int mc) { return (mc + 7) & ~7; }

// Where the backward's grad_output comes from: its elements, or (LaplacianFormer's
// kernel K = exp(-s * dist)) the gradient of K in fp32 together with K, from which
// the distance's gradient g = -s * gK * K is formed while a batch is staged.
enum BwdGrad { kGradF16 = 0, kGradKernel = 1 };

// Whether a backward kernel compiles both fp32 step loops (kStepFast).
template <typename T, bool DQ, bool DK, int GSRC>
constexpr bool two_step_loops() { return sizeof(T) == 4 && !(DQ && DK) && GSRC == kGradF16; }

// fp32 grad_query alone, a row per wave: where the slices outnumber the CUs it counts that two
// workgroups fit one, 128 registers at M = 49 (both step loops took 134), 64 at M = 16 (300 slices of 100
// rows, C = 64: 9.7 us, 11.2 with the 73 that both loops took). 64 registers hold one loop only: TWO says
// whether both are compiled (launch_bcast_bwd_rpw).
template <typename T, int MC, bool DQ, bool DK, int GSRC, int RPW>
constexpr bool bcast_paired() { return two_step_loops<T, DQ, DK, GSRC>() && !DK && RPW == 1; }

// The kernel-gradient backward's rows: up to three row sets (a layer's K_mm, K_qm and
// K_km share one key) taken as one concatenation, set i ending at row (column-block
// kernel: row batch) end[i]; unused sets are empty. One launch and one grad_key
// reduction replace one of each per set, and the waves' shares stay even whatever the
// sets' lengths.
struct RowSources {
  const float* gk[3];
  const float* kv[3];
  const void* q[3];
  void* dq[3];
  int len[3];
  int end[3];
};

// A batch of rows: set s, first row `row` of it, nr rows.
struct RowBatch {
  int s, row, nr;
};

// (A select per use, not an indexed load: the set is uniform and the struct stays in
// the kernel's arguments.)
template <typename P>
__device__ __forceinline__ P pick3(const P (&a)[3], int s) {
  return s == 0 ? a[0] : s == 1 ? a[1] : a[2];
}

// RPW = 2 (C <= 32): a wave's halves take two rows at once, lane (h, c) channel c of
// row 2i + h, where one row would leave half the lanes idle; the halves' grad_key sums
// are added at the end. (M = 49 with grad_key: up to 13 registers spill in this form, 11 to 13 with
// both gradients of a kernel gradient, 3 of that one's and 2 of fp32 grad_key's with RPW = 1.)
template <typename T, int MC, bool DQ, bool DK, int GSRC = kGradF16, int RPW = 1, bool TWO = true>
__global__ void __launch_bounds__(64 * bcast_max_waves(MC),
                                  (bcast_paired<T, MC, DQ, DK, GSRC, RPW>() ? (MC > 16 ? 4 : TWO ? 7 : 8) : 1))
laplace_bwd_bcast_kernel(const T* __restrict__ gout, RowSources src, float gscale, const T* __restrict__ query,
                         const T* __restrict__ key, T* __restrict__ dq, T* __restrict__ dk,
                         float* __restrict__ partial, int N, int C, int rowsPerWave) {
  constexpr int RB = kBcRB;
  constexpr int MP = bcast_pitch(MC);            // LDS row pitch (floats)
  constexpr bool kF16 = std::is_same<T, f16s>::value;
  // 16-bit inputs take the ordered-pattern step (tmap16): y = clamp(T(q) + (1/2 - T(k))).
  constexpr bool k16 = sizeof(T) == 2;
  constexpr bool kTwo = TWO && two_step_loops<T, DQ, DK, GSRC>();
  constexpr int EPW = sizeof(T) == 2 ? 2 : 1;    // grad elements per 32-bit word
  constexpr int GD = GSRC == kGradF16 ? RB * MC / EPW : RB * MC;  // grad words of a full batch
  constexpr int NL = (GD + 63) / 64;             // words per lane per batch
  const int W = blockDim.x >> 6;
  const int wave = uniform(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int bh = blockIdx.z, cb = blockIdx.y, x = blockIdx.x, nx = gridDim.x;
  const int slice = bh * gridDim.y + cb;
  const int hr = RPW == 2 ? lane >> 5 : 0, ln = RPW == 2 ? lane & 31 : lane;  // row of a pair, channel of the block
  const int c = cb * 64 + ln;
  const bool cval = c < C;
  const int rowBeg = uniform((x * W + wave) * rowsPerWave);
  const int rowEnd = uniform(min(GSRC == kGradKernel ? src.end[2] : N, rowBeg + rowsPerWave));

  extern __shared__ __align__(16) unsigned char smem[];
  float* ksm = reinterpret_cast<float*>(smem);             // [MC][65] key tile, then grad_key sums
  // This wave's batch: [RB][MP] 2g, [RB] -sum_j g, [MP] column sums, [RB / RPW][64] query.
  float* gsm = ksm + bcast_key_floats(MC) + wave * (RB * MP + RB + MP + RB / RPW * 64);
  float* gneg = gsm + RB * MP;
  float* hsm = gneg + RB;
  float* qsm = hsm + MP;

  const uint32_t* gw = reinterpret_cast<const uint32_t*>(gout + (size_t)bh * N * MC);
  const T* kb = key + (size_t)bh * C * MC;

  uint32_t gpre[NL];
  float kpre[GSRC == kGradKernel ? NL : 1];
  const float gscale2 = -2.0f * gscale;  // 2 * (-s * gK) * K == (-2s * gK) * K exactly
  int kwords = 0;                        // valid words of the fetched kernel-gradient batch
  T qpre[RB / RPW];
  // The batch at row `pos` of the concatenation: it ends with its set. (N is the only
  // set of a plain grad_output.)
  auto locate = [&](int pos) {
    RowBatch b{0, pos, min(RB, rowEnd - pos)};
    if constexpr (GSRC == kGradKernel) {
      b.s = (pos >= src.end[0]) + (pos >= src.end[1]);
      b.nr = min(b.nr, pick3(src.end, b.s) - pos);
      if (b.s) b.row = pos - (b.s == 1 ? src.end[0] : src.end[1]);
    }
    return b;
  };
  auto row_of = [&](const RowBatch& b) { return (size_t)bh * (GSRC == kGradKernel ? pick3(src.len, b.s) : N) + b.row; };
  auto fetch = [&](const RowBatch& b) {
    const size_t row = row_of(b);
    const T* qr = (GSRC == kGradKernel ? static_cast<const T*>(pick3(src.q, b.s)) : query) + row * C;
    if constexpr (GSRC == kGradF16) {
      const int words = b.nr * MC / EPW;
      const uint32_t* gs = gw + (size_t)b.row * MC / EPW;
#pragma unroll
      for (int t = 0; t < NL; ++t) {
        const int e = lane + 64 * t;
        gpre[t] = e < words ? gs[e] : 0u;
      }
    } else {
      // Branch-free: lanes past the batch re-read its last element (nr >= 1, so
      // words >= MC >= 1) and are zeroed when the batch is staged.
      const int words = b.nr * MC;
      const float* gs = pick3(src.gk, b.s) + row * MC;
      const float* ks = pick3(src.kv, b.s) + row * MC;
#pragma unroll
      for (int t = 0; t < NL; ++t) {
        const int e = min(lane + 64 * t, words - 1);
        gpre[t] = __builtin_bit_cast(uint32_t, gs[e]);
        kpre[t] = ks[e];
      }
      kwords = words;
    }
#pragma unroll
    for (int i = 0; i < RB / RPW; ++i) {
      const int r = RPW * i + hr;
      qpre[i] = (cval && r < b.nr) ? qr[(size_t)r * C + c] : T{};
    }
  };
  // The first batch's loads are in flight while the key tile is staged.
  RowBatch next{};
  if (rowBeg < rowEnd) {
    next = locate(rowBeg);
    fetch(next);
  }

  // Key tile (contiguous reads; the pitch of 65 spreads the stores over the banks): 16-bit
  // keys as the step terms 1/2 - T(k), fp32 keys as values.
  bool big = false;
  each_tile_column<MC>(W, wave, lane, [&](int j, int cl) {
    const int cc = cb * 64 + cl;
    const T kv = kb[(size_t)min(cc, C - 1) * MC + j];
    float v;
    if constexpr (k16) v = 0.5f - tmap16(kv.bits);
    else v = to_acc(kv);
    if constexpr (kTwo) big |= !(fabsf(v) < kStepKeyMax);
    ksm[j * 65 + cl] = cc < C ? v : 0.0f;
  });
  bool fast = false;  // (workgroup-uniform)
  if constexpr (kTwo) fast = !__syncthreads_or(big);
  else __syncthreads();
  const float pre = kTwo && fast ? kStepPre : 1.0f;
  float kreg[MC], dka[MC];
#pragma unroll
  for (int j = 0; j < MC; ++j) {
    kreg[j] = ksm[j * 65 + ln] * pre;
    if (DK) dka[j] = 0.0f;
  }
  float hsum = 0.0f;  // lane j < MC: sum over this wave's rows of g[i][j]
  const uint32_t dcol = (uint32_t)(hr * C + c);  // the lane's element of a stored row (pair)
  // (A VGPR operand: an SGPR one would halve the issue rate.)
  float scl = kTwo && fast ? kStepFast : kStepSlow;
  asm volatile("" : "+v"(scl));

  auto batches = [&](auto fastc) {
    for (int pos = rowBeg; pos < rowEnd;) {
      const RowBatch cur = next;
      const int nr = uniform(cur.nr);
      pos += nr;
      // Stage this batch: 2g as fp32, row-major [RB][MP] (exact for fp16 g; for the
      // kernel gradient g = -s * gK * K, rounded once, then doubled exactly).
      if constexpr (GSRC == kGradF16 && EPW == 2) {
#pragma unroll
        for (int t = 0; t < NL; ++t) {
          const int e = 2 * (lane + 64 * t);
          if (e < RB * MC) {
            const int r0 = e / MC, j0 = e - r0 * MC;
            const int r1 = (e + 1) / MC, j1 = e + 1 - r1 * MC;
            float lo, hi;
            if constexpr (kF16) {
              lo = (float)__builtin_bit_cast(_Float16, (uint16_t)(gpre[t] & 0xffffu));
              hi = (float)__builtin_bit_cast(_Float16, (uint16_t)(gpre[t] >> 16));
            } else {  // bf16
              lo = __builtin_bit_cast(float, gpre[t] << 16);
              hi = __builtin_bit_cast(float, gpre[t] & 0xffff0000u);
            }
            gsm[r0 * MP + j0] = 2.0f * lo;
            gsm[r1 * MP + j1] = 2.0f * hi;
          }
        }
      } else if constexpr (GSRC == kGradF16) {  // fp32: one element per word
#pragma unroll
        for (int t = 0; t < NL; ++t) {
          const int e = lane + 64 * t;
          if (e < RB * MC) {
            const int r = e / MC, j = e - r * MC;
            gsm[r * MP + j] = 2.0f * __builtin_bit_cast(float, gpre[t]);
          }
        }
      } else {
#pragma unroll
        for (int t = 0; t < NL; ++t) {
          const int e = lane + 64 * t;
          if (e < RB * MC) {
            const int r = e / MC, j = e - r * MC;
            const float v = (gscale2 * __builtin_bit_cast(float, gpre[t])) * kpre[t];
            gsm[r * MP + j] = e < kwords ? v : 0.0f;
          }
        }
      }
#pragma unroll
      for (int i = 0; i < RB / RPW; ++i) {
        if constexpr (k16) qsm[i * 64 + lane] = tmap16(qpre[i].bits);
        else qsm[i * 64 + lane] = to_acc(qpre[i]) * pre;
      }
      wave_sync();
      // Row sums (lane r) for grad_query and column sums (lane j) for grad_key.
      // Rows past nr are zero in the batch. All reads of a sum are issued before
      // the additions, so no chain of dependent LDS round trips.
      if (DQ) {
        const float4* rowp = reinterpret_cast<const float4*>(gsm + min(lane, RB - 1) * MP);
        // (Half the row at a time: a whole row's registers would spill some of the columns' at M = 49 and
        // cost a wave per SIMD at M = 32.)
        constexpr int NH = 2, HQ = MP / 4 / NH;
        float sum = 0.0f;
#pragma unroll
        for (int h = 0; h < NH; ++h) {
          float4 v[HQ];
#pragma unroll
          for (int jq = 0; jq < HQ; ++jq) v[jq] = rowp[h * HQ + jq];
#pragma unroll
          for (int jq = 0; jq < HQ; ++jq) {
            const float e[4] = {v[jq].x, v[jq].y, v[jq].z, v[jq].w};
#pragma unroll
            for (int t = 0; t < 4; ++t)
              if ((h * HQ + jq) * 4 + t < MC) sum += e[t];
          }
          asm volatile("" : "+v"(sum)::"memory");
        }
        if (lane < RB) gneg[lane] = -0.5f * sum;
      }
      if (DK) {
        float hv[RB];
#pragma unroll
        for (int r = 0; r < RB; ++r) hv[r] = gsm[r * MP + min(lane, MC - 1)];
#pragma unroll
        for (int r = 0; r < RB; ++r) hsum += hv[r];
      }
      wave_sync();
      if (pos < rowEnd) {
        next = locate(pos);
        fetch(next);
      }
      T* dqr = (GSRC == kGradKernel ? static_cast<T*>(pick3(src.dq, cur.s)) : dq) + row_of(cur) * C;

      // Row loop, software-pipelined two broadcast reads ahead (LDS latency under
      // load exceeds one column group's VALU time); the next row's query value,
      // initial sum and first two grad groups are read during the current row's
      // last groups. The scheduling barriers keep the compiler from computing
      // every column's step up front (MC more registers).
      constexpr int NQ = MP / 4;
      static_assert(NQ >= 2 && NQ % 2 == 0, "two groups in flight, slots aligned at every row start");
      // (Row pair i of a batch is rows RPW i + hr; rows past nr are zero there.)
      const float* gh = gsm + hr * MP;
      float qn = qsm[lane];
      float accn = DQ ? gneg[hr] : 0.0f;
      float4 gq[2] = {reinterpret_cast<const float4*>(gh)[0], reinterpret_cast<const float4*>(gh)[1]};
#pragma unroll 1
      for (int i = 0; i * RPW < nr; ++i) {
        const int in = min(i + 1, RB / RPW - 1);
        const float4* g4 = reinterpret_cast<const float4*>(gh + RPW * i * MP);
        const float4* g4n = reinterpret_cast<const float4*>(gh + RPW * in * MP);
        const float qv = qn;
        // grad_query of the row as four independent partial sums (columns j = t
        // mod 4), combined once at the end: a single chain of MC dependent FMAs
        // would stall a wave on every column.
        float acc[4] = {accn, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int jq = 0; jq < NQ; ++jq) {
          const float4 gv = gq[jq & 1];
          if (jq + 2 < NQ) gq[jq & 1] = g4[jq + 2];
          else gq[jq & 1] = g4n[jq + 2 - NQ];
          if (jq == NQ - 1) {
            qn = qsm[in * 64 + lane];
            if (DQ) accn = gneg[RPW * in + hr];
          }
          const float gg[4] = {gv.x, gv.y, gv.z, gv.w};
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const int j = jq * 4 + t;
            if (j < MC) {
              float y;
              if constexpr (k16) {
                y = __builtin_amdgcn_fmed3f(qv + kreg[j], 0.0f, 1.0f);  // one clamped add
              } else if constexpr (decltype(fastc)::value) {
                y = __builtin_amdgcn_fmed3f(__builtin_fmaf(qv - kreg[j], scl, 0.5f), 0.0f, 1.0f);
              } else {
                const float e = (qv - kreg[j]) * scl;
                y = __builtin_amdgcn_fmed3f(__builtin_fmaf(e, scl, 0.5f), 0.0f, 1.0f);
              }
              if (DQ) acc[t] = fmaf(gg[t], y, acc[t]);
              if (DK) {
                dka[j] = fmaf(gg[t], y, dka[j]);
                asm volatile("" : "+v"(dka[j]));  // update in place, not after the row
              }
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        if (DQ) {
          float total = (acc[0] + acc[1]) + (acc[2] + acc[3]);
          // Materialise the sum here: sunk into the store's branch, the
          // accumulation would keep every column's step value live.
          asm volatile("" : "+v"(total));
          if (cval && (RPW == 1 || RPW * i + hr < nr)) (dqr + (size_t)(RPW * i) * C)[dcol] = from_acc<T>(total);
        }
      }
      wave_sync();
    }
  };
  if constexpr (kTwo) {
    if (fast) batches(std::true_type{});
    else batches(std::false_type{});
  } else {
    batches(std::false_type{});
  }

  if (DK) {
    // This wave's grad_key partial: column sums of g minus the accumulated 2g*step.
    if (lane < MC) hsm[lane] = 0.5f * hsum;
    wave_sync();
#pragma unroll
    for (int j = 0; j < MC; ++j) {
      if constexpr (RPW == 2) dka[j] += __shfl_xor(dka[j], 32);
      dka[j] = hsm[j] - dka[j];
    }
    // The slice's only workgroup stores grad_key itself; else the reduction kernel sums
    // the workgroups' partials ([MC][64]) in order.
    const bool only = nx == 1;
    float* pout = partial + ((size_t)slice * nx + x) * 64 * MC;
    T* dkb = dk + ((size_t)bh * C + cb * 64) * MC;
    const int cn = C - cb * 64;
    bcast_reduce_dk<MC>(dka, reinterpret_cast<float*>(smem), W, wave, lane, only, [&](int j, int cl, float v) {
      if (!only) pout[j * 64 + cl] = v;
      else if (cl < cn) dkb[cl * MC + j] = from_acc<T>(v);
    });
  }
}

// ---------------------------------------------------------------------------
// Backward for 17 <= M <= 256 columns in CB = ceil(M / 32) blocks of 32, fp16 /
// bf16 / fp32 (the last block zero-padded when M is not a multiple of 32).
//
// A workgroup is RG row groups of CB waves; wave (g, b) of a group takes the
// 32 columns [32b, 32b + 32) of every row batch (RB rows) of its group, with
// its columns' key values and grad_key sums in registers, as the kernel above does
// for all columns. A row's grad_query is the sum of the CB waves'
// column-block partials: each wave leaves its partials in LDS (double-buffered
// by batch parity), and after one workgroup barrier per batch each wave of the
// group sums RB/CB of the batch's rows in column-block order (deterministic).
// grad_key: the RG groups' sums in group order, then the workgroup partials
// summed over the slice by the reduction kernel.
//
// Step y = (sgn(q - k) + 1)/2 at the full VALU rate: 16-bit operands through their
// ordered patterns (tmap16), one clamped add; fp32 in two or three instructions
// (kStepFast, kStepSlow).
// ---------------------------------------------------------------------------
constexpr int kMbMC = 32;  // columns per wave
constexpr int kMbRB = 8;   // rows per batch

// LOOP: a batch's rows go through a loop, only those there are, with the one fp32 step; otherwise
// the batch is unrolled (below). mb_row_loop says which.
template <typename T, int CB, bool DQ, bool DK, int GSRC = kGradF16, bool LOOP = false>
__global__ void __launch_bounds__(1024)
laplace_bwd_mb_kernel(const T* __restrict__ gout, const T* __restrict__ query, const T* __restrict__ key,
                      T* __restrict__ dq, float* __restrict__ partial, int N, int C, int rowsPerWG, int Mt,
                      RowSources src, float gscale) {
  // M = CB * 32 columns in registers and LDS; the tensors have Mt <= M columns (the
  // last block is partial when Mt is not a multiple of 32: its columns from Mt on
  // have zero grad and key, so they add nothing and are not stored).
  constexpr int MC = kMbMC, RB = kMbRB, M = CB * MC;
  constexpr int MP = MC;                       // LDS row pitch of a staged batch (floats)
  // 16-bit inputs take the ordered-pattern step (tmap16): y = clamp(T(q) + (1/2 - T(k))).
  constexpr bool k16 = std::is_same<T, f16s>::value || std::is_same<T, bf16s>::value;
  constexpr bool kTwo = !LOOP && two_step_loops<T, DQ, DK, GSRC>();
  // Grad elements per fetched 32-bit word: 2 for 16-bit grads, 1 for fp32 grads and
  // for the kernel-gradient source (fp32 gK and K, g = -s * gK * K formed at staging).
  constexpr int EPW = GSRC == kGradKernel ? 1 : (4 / (int)sizeof(T) > 0 ? 4 / (int)sizeof(T) : 1);
  constexpr int GW = RB * MC / EPW;            // grad words of a batch (this wave's columns)
  constexpr int NL = (GW + 63) / 64;           // words per lane
  static_assert(GW % 64 == 0, "whole words per lane");
  const int W = blockDim.x >> 6;
  const int RG = W / CB;
  const int wave = uniform(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int cbk = wave % CB, grp = wave / CB;
  const int bh = blockIdx.z, chb = blockIdx.y, x = blockIdx.x, nx = gridDim.x;
  const int slice = bh * gridDim.y + chb;
  const int c = chb * 64 + lane;
  const bool cval = c < C;
  const int cq = min(c, C - 1);
  // Batches of RB rows, each of one row set (the sets' ends in src count batches).
  const int b0 = x * (rowsPerWG / RB);
  const int nb = max(0, min((GSRC == kGradKernel ? src.end[2] : (N + RB - 1) / RB) - b0, rowsPerWG / RB));
  const int rounds = (nb + RG - 1) / RG;        // batch t goes to group t % RG

  extern __shared__ __align__(16) unsigned char smem[];
  float* big = reinterpret_cast<float*>(smem);  // key tile [M][64] at the start, then the
                                                // grad_query partials [2][W][RB][64]
  const int bigFloats = max(M * 64, 2 * W * RB * 64);
  float* gsm = big + bigFloats + wave * (RB * MP + RB + RB * 64);  // this wave: [RB][MP] 2g,
  float* gneg = gsm + RB * MP;                                      // [RB] -sum_j g,
  float* qsm = gneg + RB;                                           // [RB][64] query values

  auto locate = [&](int t) {
    RowBatch b{0, (b0 + t) * RB, 0};
    int len = N;
    if constexpr (GSRC == kGradKernel) {
      b.s = (b0 + t >= src.end[0]) + (b0 + t >= src.end[1]);
      if (b.s) b.row -= RB * (b.s == 1 ? src.end[0] : src.end[1]);
      len = pick3(src.len, b.s);
    }
    b.nr = min(RB, len - b.row);
    return b;
  };
  auto row_of = [&](const RowBatch& b) { return (size_t)bh * (GSRC == kGradKernel ? pick3(src.len, b.s) : N) + b.row; };
  const T* kb = key + (size_t)bh * C * Mt;

  // Next batch of this group: this wave's 32 columns of RB rows (clamped to the
  // last valid row; rows past the batch are zeroed at staging) and RB query values.
  uint32_t gpre[NL];
  float kpre[GSRC == kGradKernel ? NL : 1];
  const float gscale2 = -2.0f * gscale;  // 2 * (-s * gK) * K == (-2s * gK) * K exactly
  T qpre[RB];
  int fnr = 0;
  auto fetch = [&](int t) {
    const RowBatch b = locate(t);
    const int nr = b.nr;
    const size_t row = row_of(b);
#pragma unroll
    for (int s = 0; s < NL; ++s) {
      const int w = lane + 64 * s;               // word of the batch block
      const int r = min(w / (MC / EPW), nr - 1), jw = w - (w / (MC / EPW)) * (MC / EPW);
      const int col = cbk * MC + jw * EPW;
      if constexpr (GSRC == kGradKernel) {
        const size_t o = (row + r) * Mt + min(col, Mt - 1);
        gpre[s] = col < Mt ? __builtin_bit_cast(uint32_t, pick3(src.gk, b.s)[o]) : 0u;
        kpre[s] = col < Mt ? pick3(src.kv, b.s)[o] : 0.0f;
        continue;
      }
      const T* rowp = gout + (row + r) * Mt;
      if constexpr (EPW == 2) {
        if (Mt & 1) {  // odd row length: rows do not start on 4-byte words, two 16-bit loads
          const uint32_t lo = col < Mt ? rowp[min(col, Mt - 1)].bits : 0u;
          const uint32_t hi = col + 1 < Mt ? rowp[min(col + 1, Mt - 1)].bits : 0u;
          gpre[s] = lo | (hi << 16);
          continue;
        }
      }
      // Even row length (or fp32): a word is all in or all out of the row.
      gpre[s] = col < Mt ? *reinterpret_cast<const uint32_t*>(rowp + min(col, Mt - EPW)) : 0u;
    }
#pragma unroll
    for (int r = 0; r < RB; ++r)
      qpre[r] = (GSRC == kGradKernel ? static_cast<const T*>(pick3(src.q, b.s)) : query)[(row + min(r, nr - 1)) * C + cq];
    fnr = nr;
  };
  int t0 = grp;  // this group's first batch
  if (t0 < nb) fetch(t0);

  // Key tile (global [C][M], coalesced over j): 16-bit keys as the step terms
  // 1/2 - T(k) (see tmap16), fp32 keys as values. Columns past Mt have zero grad.
  bool huge = false;
  for (int t = threadIdx.x; t < 64 * M; t += blockDim.x) {
    const int cl = t / M, j = t - cl * M;
    const int cc = chb * 64 + cl;
    const bool in = cc < C && j < Mt;
    const T kv = kb[(size_t)min(cc, C - 1) * Mt + min(j, Mt - 1)];
    if constexpr (k16)
      big[j * 64 + cl] = in ? 0.5f - tmap16(kv.bits) : 0.0f;
    else {
      if constexpr (kTwo) huge |= !(fabsf(to_acc(kv)) < kStepKeyMax);
      big[j * 64 + cl] = in ? to_acc(kv) : 0.0f;
    }
  }
  bool fast = false;  // (workgroup-uniform)
  if constexpr (kTwo) fast = !__syncthreads_or(huge);
  else __syncthreads();
  const float pre = kTwo && fast ? kStepPre : 1.0f;
  float kreg[MC], dka[MC];
#pragma unroll
  for (int j = 0; j < MC; ++j) {
    kreg[j] = big[(cbk * MC + j) * 64 + lane] * pre;
    if (DK) dka[j] = 0.0f;
  }
  __syncthreads();  // the key tile's LDS becomes the partial buffers
  float scl = kTwo && fast ? kStepFast : kStepSlow;
  asm volatile("" : "+v"(scl));  // VGPR operand: an SGPR one would halve the issue rate
  float hsum = 0.0f;  // lane j < MC: sum over this wave's rows of 2 g[i][j]

  auto batches = [&](auto fastc) {
    for (int round = 0; round < rounds; ++round) {
      const int t = round * RG + grp;
      const bool have = t < nb;                          // uniform per wave
      const int nr = have ? fnr : 0;
      float* dqp = big + ((round & 1) * W + wave) * RB * 64;  // this wave's partials of this batch
      if (have) {
        // Stage: 2g as fp32 [RB][MP], rows past nr zero.
#pragma unroll
        for (int s = 0; s < NL; ++s) {
          const int w = lane + 64 * s;
          const int r = w / (MC / EPW), jw = w - r * (MC / EPW);
          const bool ok = r < nr;
          if constexpr (EPW == 2) {
            const float lo = std::is_same<T, f16s>::value
                                 ? (float)__builtin_bit_cast(_Float16, (uint16_t)(gpre[s] & 0xffffu))
                                 : __builtin_bit_cast(float, gpre[s] << 16);
            const float hi = std::is_same<T, f16s>::value
                                 ? (float)__builtin_bit_cast(_Float16, (uint16_t)(gpre[s] >> 16))
                                 : __builtin_bit_cast(float, gpre[s] & 0xffff0000u);
            gsm[r * MP + 2 * jw] = ok ? 2.0f * lo : 0.0f;
            gsm[r * MP + 2 * jw + 1] = ok ? 2.0f * hi : 0.0f;
          } else if constexpr (GSRC == kGradKernel) {
            gsm[r * MP + jw] = ok ? (gscale2 * __builtin_bit_cast(float, gpre[s])) * kpre[s] : 0.0f;
          } else {
            gsm[r * MP + jw] = ok ? 2.0f * __builtin_bit_cast(float, gpre[s]) : 0.0f;
          }
        }
#pragma unroll
        for (int r = 0; r < RB; ++r) {
          if constexpr (k16)
            qsm[r * 64 + lane] = tmap16(qpre[r].bits);
          else
            qsm[r * 64 + lane] = to_acc(qpre[r]) * pre;
        }
        wave_sync();
        if (DQ) {
          const float4* rowp = reinterpret_cast<const float4*>(gsm + min(lane, RB - 1) * MP);
          float4 v[MP / 4];
#pragma unroll
          for (int jq = 0; jq < MP / 4; ++jq) v[jq] = rowp[jq];
          float sum = 0.0f;
#pragma unroll
          for (int jq = 0; jq < MP / 4; ++jq) sum += (v[jq].x + v[jq].y) + (v[jq].z + v[jq].w);
          if (lane < RB) gneg[lane] = -0.5f * sum;
        }
        if (DK) {
          float hv[RB];
#pragma unroll
          for (int r = 0; r < RB; ++r) hv[r] = gsm[r * MP + min(lane, MC - 1)];
#pragma unroll
          for (int r = 0; r < RB; ++r) hsum += hv[r];
        }
        wave_sync();
        if (t + RG < nb) fetch(t + RG);

        // Row loop as in the register-column kernel above (grad values two 16-byte groups
        // ahead, four partial sums per row, grad_key sums updated in place), unrolled over
        // the whole batch so that every LDS address is an immediate (rows past nr have zero
        // grad and are not stored). That leaves the registers to fit: a spilled one is
        // reloaded behind the next batch's loads, whose latency it then waits for. bf16,
        // 128 slices, N = 4096, M = 256, C = 64, both gradients: 798 -> 660 us (1.3 ns per
        // VALU instruction and SIMD, 1.0 to 1.35 being the rate of four waves of the loop's
        // adds and FMAs alone); three or four groups ahead spill 6 to 12 registers and take
        // 750 to 800 us; half waves on 16 columns x 2 channels each, which halve the LDS
        // reads, spill 2 and take 699 us, and gain 1 to 3 % where only one gradient is asked.
        constexpr int NQ = MP / 4, NG = RB * NQ, LA = 2;
        const float4* g4 = reinterpret_cast<const float4*>(gsm);
        float qn = qsm[lane];
        float accn = DQ ? gneg[0] : 0.0f;
        float4 gq[LA];
#pragma unroll
        for (int u = 0; u < LA; ++u) gq[u] = g4[u];
        auto columns = [&](auto jc, float4 gv, float qv, float (&acc)[4]) {
          const float gg[4] = {gv.x, gv.y, gv.z, gv.w};
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int j = decltype(jc)::value * 4 + u;
            float y;
            if constexpr (k16) {
              y = __builtin_amdgcn_fmed3f(qv + kreg[j], 0.0f, 1.0f);  // one clamped add
            } else if constexpr (decltype(fastc)::value) {
              y = __builtin_amdgcn_fmed3f(__builtin_fmaf(qv - kreg[j], scl, 0.5f), 0.0f, 1.0f);
            } else {
              const float e = (qv - kreg[j]) * scl;
              y = __builtin_amdgcn_fmed3f(__builtin_fmaf(e, scl, 0.5f), 0.0f, 1.0f);
            }
            if (DQ) acc[u] = fmaf(gg[u], y, acc[u]);
            if (DK) {
              dka[j] = fmaf(gg[u], y, dka[j]);
              asm volatile("" : "+v"(dka[j]));  // update in place, not after the row
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        };
        auto store_row = [&](int r, const float (&acc)[4]) {
          if (DQ) {
            float total = (acc[0] + acc[1]) + (acc[2] + acc[3]);
            asm volatile("" : "+v"(total));
            dqp[r * 64 + lane] = total;
          }
        };
        if constexpr (LOOP) {
#pragma unroll 1
          for (int r = 0; r < nr; ++r) {
            const int rn = min(r + 1, RB - 1);
            const float4* gr = g4 + r * NQ;
            const float4* gn = g4 + rn * NQ;
            const float qv = qn;
            float acc[4] = {accn, 0.0f, 0.0f, 0.0f};
            unrolled<NQ>([&](auto jc) {
              constexpr int jq = jc.value;
              const float4 gv = gq[jq % LA];
              gq[jq % LA] = jq + LA < NQ ? gr[jq + LA] : gn[jq + LA - NQ];
              if constexpr (jq == NQ - 1) {
                qn = qsm[rn * 64 + lane];
                if (DQ) accn = gneg[rn];
              }
              columns(jc, gv, qv, acc);
            });
            store_row(r, acc);
          }
        } else {
          unrolled<RB>([&](auto rc) {
            constexpr int r = rc.value;
            const float qv = qn;
            float acc[4] = {accn, 0.0f, 0.0f, 0.0f};
            unrolled<NQ>([&](auto jc) {
              constexpr int jq = jc.value, at = r * NQ + jq;
              const float4 gv = gq[at % LA];
              if constexpr (at + LA < NG) gq[at % LA] = g4[at + LA];
              if constexpr (jq == NQ - 1 && r + 1 < RB) {
                qn = qsm[(r + 1) * 64 + lane];
                if (DQ) accn = gneg[r + 1];
              }
              columns(jc, gv, qv, acc);
            });
            store_row(r, acc);
          });
        }
      }
      if (DQ) {
        // Every wave of the workgroup has written this batch's partials (and is
        // done reading the partials of two batches ago, in the other buffer).
        __syncthreads();
        if (have) {
          const RowBatch b = locate(t);
          T* dqr = (GSRC == kGradKernel ? static_cast<T*>(pick3(src.dq, b.s)) : dq) + row_of(b) * C;
          const float* gp = big + ((round & 1) * W + grp * CB) * RB * 64;  // the group's CB waves
          for (int r = cbk; r < nr; r += CB) {
            float sv = 0.0f;
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) sv += gp[(cb * RB + r) * 64 + lane];
            if (cval) dqr[(size_t)r * C + c] = from_acc<T>(sv);
          }
        }
      }
      if (have) wave_sync();
    }
  };
  if constexpr (kTwo) {
    if (fast) batches(std::true_type{});
    else batches(std::false_type{});
  } else {
    batches(std::false_type{});
  }

  if (DK) {
    // This wave's grad_key partial for its 32 columns, then the RG groups' sums in
    // group order into red[M][64], written out as the workgroup's partial.
    if (lane < MC) gsm[lane] = 0.5f * hsum;
    wave_sync();
#pragma unroll
    for (int j = 0; j < MC; ++j) dka[j] = gsm[j] - dka[j];
    __syncthreads();  // every wave is done with the partial buffers
    float* red = big;
    for (int g = 0; g < RG; ++g) {
      if (grp == g) {
#pragma unroll
        for (int j = 0; j < MC; ++j) {
          float* p = &red[(cbk * MC + j) * 64 + lane];
          *p = g == 0 ? dka[j] : *p + dka[j];
        }
      }
      __syncthreads();
    }
    float* out = partial + ((size_t)slice * nx + x) * 64 * Mt;
    for (int tt = threadIdx.x; tt < 64 * Mt; tt += blockDim.x) out[tt] = red[tt];
  }
}

// grad_key = sum over the workgroups of a slice of their partial sums, in
// workgroup order (deterministic). One thread per (channel, column).
template <typename T>
__global__ void __launch_bounds__(256)
laplace_dk_reduce_kernel(const typename AccOf<T>::type* __restrict__ partial, T* __restrict__ dk,
                         int nx, int M, int C) {
  using A = typename AccOf<T>::type;
  const int bh = blockIdx.z, cb = blockIdx.y;
  const int slice = bh * gridDim.y + cb;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 64 * M) return;
  const int cl = t / M, j = t - cl * M;
  const int cc = cb * 64 + cl;
  if (cc >= C) return;
  const A* pb = partial + (size_t)slice * nx * 64 * M + t;
  A s = A(0);
#pragma unroll 8
  for (int x = 0; x < nx; ++x) s += pb[(size_t)x * 64 * M];
  dk[((size_t)bh * C + cc) * M + j] = from_acc<T>(s);
}

// Same sum over column-major partials ([M][64] per workgroup, channel fastest).
template <typename T = f16s>
__global__ void __launch_bounds__(256)
laplace_dk_reduce_cm_kernel(const float* __restrict__ partial, T* __restrict__ dk, int nx, int M, int C) {
  const int bh = blockIdx.z, cb = blockIdx.y;
  const int slice = bh * gridDim.y + cb;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 64 * M) return;
  const int j = t >> 6, cl = t & 63;
  const int cc = cb * 64 + cl;
  if (cc >= C) return;
  const float* pb = partial + (size_t)slice * nx * 64 * M + t;
  float s = 0.0f;
#pragma unroll 8
  for (int x = 0; x < nx; ++x) s += pb[(size_t)x * 64 * M];
  dk[((size_t)bh * C + cc) * M + j] = from_acc<T>(s);
}

// ---------------------------------------------------------------------------
// Legacy reduce forward: one workgroup of bd = min(C, 256) threads per output,
// arithmetic in the element type, halving-tree fold (reference :399-447).
// ---------------------------------------------------------------------------
template <typename T> struct NativeOf { using type = float; };
template <> struct NativeOf<f16s> { using type = _Float16; };
template <> struct NativeOf<double> { using type = double; };

template <typename T> __device__ __forceinline__ typename NativeOf<T>::type to_native(T v);
template <> __device__ __forceinline__ float to_native<float>(float v) { return v; }
template <> __device__ __forceinline__ double to_native<double>(double v) { return v; }
template <> __device__ __forceinline__ _Float16 to_native<f16s>(f16s v) {
  return __builtin_bit_cast(_Float16, v.bits);
}
template <> __device__ __forceinline__ float to_native<bf16s>(bf16s v) { return to_acc(v); }

// One rounding to the element type after each native operation (bf16 is
// emulated in fp32 and rounded back; fp32 has enough precision for that to
// equal a direct bf16 operation).
template <typename T> __device__ __forceinline__ typename NativeOf<T>::type round_native(typename NativeOf<T>::type v) { return v; }
template <> __device__ __forceinline__ float round_native<bf16s>(float v) { return to_acc(from_acc<bf16s>(v)); }

template <typename T>
__global__ void __launch_bounds__(256)
laplace_reduce_fwd_kernel(const T* __restrict__ query, const T* __restrict__ key, T* __restrict__ out,
                          int64_t total, int N, int M, int C) {
  using Nt = typename NativeOf<T>::type;
  __shared__ Nt sdata[256];
  const int bd = blockDim.x;
  for (int64_t idx = blockIdx.x; idx < total; idx += gridDim.x) {
    const int64_t bh = idx / ((int64_t)N * M);
    const int64_t rem = idx - bh * N * M;
    const int p = (int)(rem / M), qj = (int)(rem - (int64_t)p * M);
    const T* qr = query + (bh * N + p) * C;
    const T* kc = key + bh * C * M + qj;
    Nt s = Nt(0);
    for (int c = threadIdx.x; c < C; c += bd) {
      Nt diff = round_native<T>(to_native(qr[c]) - to_native(kc[(int64_t)c * M]));
      s = round_native<T>(s + (diff >= Nt(0) ? diff : -diff));
    }
    sdata[threadIdx.x] = s;
    __syncthreads();
    for (int stride = bd / 2; stride > 0; stride >>= 1) {
      if ((int)threadIdx.x < stride) sdata[threadIdx.x] = round_native<T>(sdata[threadIdx.x] + sdata[threadIdx.x + stride]);
      __syncthreads();
    }
    if (threadIdx.x == 0) {
      if constexpr (std::is_same<T, f16s>::value) out[idx] = f16s{__builtin_bit_cast(uint16_t, sdata[0])};
      else if constexpr (std::is_same<T, bf16s>::value) out[idx] = from_acc<bf16s>(sdata[0]);
      else out[idx] = sdata[0];
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Host side.
// ---------------------------------------------------------------------------
namespace {

struct Dims {
  int64_t B, H, N, M, C;
  int64_t BH() const { return B * H; }
};

int check_dims(const Dims& d, const char* who) {
  if (d.B < 0 || d.H < 0 || d.N < 0 || d.M < 0 || d.C < 0)
    return fail(LFAMD_ERR_ARG, "%s: negative size", who);
  if (d.N > INT32_MAX / 2 || d.M > INT32_MAX / 2 || d.C > INT32_MAX / 2 || d.BH() > 65535)
    return fail(LFAMD_ERR_UNSUPPORTED, "%s: sizes too large (B*H must be <= 65535)", who);
  return LFAMD_OK;
}

bool empty(const Dims& d) { return d.BH() == 0 || d.N == 0 || d.M == 0; }

// ---- forward ----
template <typename T> constexpr int stage_bytes() { return (int)sizeof(typename StageOf<T>::type); }

template <typename T, int JB>
int launch_fwd_jb(const T* q, const T* k, T* o, const Dims& d, hipStream_t st) {
  constexpr int SV = 16 / stage_bytes<T>();
  constexpr int JBP = round_up(JB, SV);
  constexpr int CK = QChunk<T>::value;
  const int M = (int)d.M, N = (int)d.N, C = (int)d.C;
  const size_t ldsBudget = 64 * 1024;
  int W = std::min(fwd_max_waves(JB), ceil_div(M, JB));
  // Channels staged per pass: all of C (rounded to the query chunk) when it fits.
  auto lds = [&](int w, int kc) {
    return (size_t)kc * w * JBP * stage_bytes<T>() + (size_t)64 * w * JB * sizeof(T);
  };
  while (W > 1 && lds(W, kFwdKC) > ldsBudget) --W;
  int KC = round_up(C, CK);
  while (KC > kFwdKC && lds(W, KC) > ldsBudget) KC = std::max(kFwdKC, round_up(KC / 2, CK));
  const int cols = W * JB;
  const int colGroups = ceil_div(M, cols);
  const int nrb = ceil_div(N, 64);
  // Row blocks per workgroup: reuse the staged key tile while keeping ~6 waves per SIMD.
  const int64_t target = 6LL * 4 * num_cus();
  const int64_t waves1 = (int64_t)nrb * colGroups * d.BH() * W;
  const int rowBlocks = (int)std::max<int64_t>(1, std::min<int64_t>(nrb, waves1 / target));
  dim3 grid(ceil_div(nrb, rowBlocks), colGroups, (unsigned)d.BH());
  dim3 block(64 * W);
  int flags = 0;
  if (C % CK == 0 && (reinterpret_cast<uintptr_t>(q) & 15) == 0) flags |= kFwdVecQ;
  // Whole-row tiles start at ((bh*N + row0) * M) elements: 16-byte aligned for every
  // tile when the base is and 64*M*sizeof(T) and N*M*sizeof(T) are multiples of 16.
  if (cols == M && (reinterpret_cast<uintptr_t>(o) & 15) == 0 && (64 * (size_t)M * sizeof(T)) % 16 == 0 &&
      ((size_t)N * M * sizeof(T)) % 16 == 0)
    flags |= kFwdVecOut;
  hipLaunchKernelGGL((laplace_fwd_kernel<T, JB>), grid, block, lds(W, KC), st, q, k, o, N, M, C, cols, rowBlocks,
                     KC, flags);
  return check_launch("laplace forward");
}

// Column block: the candidate with the least padding, ties to the larger block.
int pick_fwd_jb(int64_t M) {
  const int cands[4] = {7, 8, 16, 32};
  int best = 32;
  int64_t bestPad = INT64_MAX;
  for (int jb : cands) {
    const int64_t pad = ceil_div((int)M, jb) * (int64_t)jb - M;
    if (pad < bestPad || (pad == bestPad && jb > best)) { bestPad = pad; best = jb; }
  }
  return best;
}

// Column block: the least padding W*JB - M with W = ceil(M/JB) <= 16 waves,
// ties to the block count nearest 8 waves.
int pick_fb_jb(int64_t M) {
  int best = 16, bestWaste = 1 << 30, bestDist = 1 << 30;
  for (int jb : {4, 7, 8, 16}) {
    const int w = ceil_div((int)M, jb);
    if (w > 16) continue;
    const int waste = w * jb - (int)M, dist = std::abs(w - 8);
    if (waste < bestWaste || (waste == bestWaste && dist < bestDist)) {
      best = jb;
      bestWaste = waste;
      bestDist = dist;
    }
  }
  return best;
}

constexpr int kFbR = 2;  // query rows per lane of the broadcast forward

template <typename T> constexpr int dtype_of();
template <> constexpr int dtype_of<float>() { return LFAMD_F32; }
template <> constexpr int dtype_of<f16s>() { return LFAMD_F16; }
template <> constexpr int dtype_of<bf16s>() { return LFAMD_BF16; }
template <> constexpr int dtype_of<double>() { return LFAMD_F64; }

// LDS of the broadcast forward: fp32 key tile [C][W*JBS], then the query tile
// [64R][C/EV + 1] 16-byte vectors, which the output tile [64R][M] (elements of
// out_bytes) reuses.
size_t fb_lds_bytes_g(int dtype, const Dims& d, size_t out_bytes, int mg) {
  const int jb = pick_fb_jb(d.M);
  const int W = ceil_div(mg, jb);
  const size_t es = dtype_size(dtype);
  const size_t qtile = (size_t)64 * kFbR * (d.C * es / 16 + 1) * 16;
  const size_t otile = (size_t)64 * kFbR * mg * out_bytes;
  return (size_t)W * d.C * fb_pitch(jb) * 4 + std::max(qtile, otile);
}

// Columns per workgroup: all M, or half of them (a multiple of the per-wave
// block) when the tiles of all M would leave room for only one workgroup per CU
// and there are row blocks for several rounds of the chip, or when all M do not
// fit one workgroup's LDS at all (fp32 output at M = 256). Config 4 (bf16,
// M = 256, 4096 row blocks): 662 -> 560 us; with a single round of row blocks
// the split measured slower (31 -> 34 us at 256 blocks), so it is not taken there.
int fb_group_cols(int dtype, const Dims& d, size_t out_bytes) {
  const int jb = pick_fb_jb(d.M);
  const int half = ceil_div(ceil_div((int)d.M, 2), jb) * jb;
  const int64_t blocks = (int64_t)ceil_div((int)d.N, 64 * kFbR) * d.BH();
  const size_t full = fb_lds_bytes_g(dtype, d, out_bytes, (int)d.M), lim = (size_t)max_lds_bytes();
  if (half < d.M && (full > lim || (2 * full > lim && blocks >= 4 * (int64_t)num_cus()))) return half;
  return (int)d.M;
}

size_t fb_lds_bytes(int dtype, const Dims& d, size_t out_bytes) {
  return fb_lds_bytes_g(dtype, d, out_bytes, fb_group_cols(dtype, d, out_bytes));
}

// Broadcast forward: a non-fp64 type, C % 8 == 0, 16-byte aligned query,
// M <= 256 and the key and output tiles within the LDS of one workgroup.
bool fwd_bcast_ok(int dtype, const Dims& d, const void* q, size_t out_bytes) {
  if (dtype == LFAMD_F64 || d.C % kFbKC != 0 || d.M > 256) return false;
  if ((reinterpret_cast<uintptr_t>(q) & 15) != 0) return false;
  return fb_lds_bytes(dtype, d, out_bytes) <= (size_t)max_lds_bytes();
}

template <typename T, int JB, int EPI>
int launch_fwd_bcast_jb(const void* q, const void* k, void* o, const Dims& d, float scale, hipStream_t st) {
  using O = typename FwdOut<T, EPI>::type;
  const int mg = fb_group_cols(dtype_of<T>(), d, sizeof(O));
  const int W = ceil_div(mg, JB);
  const size_t lds = fb_lds_bytes_g(dtype_of<T>(), d, sizeof(O), mg);
  auto kern = laplace_fwd_bcast_kernel<T, JB, kFbR, EPI>;
  if (lds > 65536)
    if (int s = set_dyn_lds(reinterpret_cast<const void*>(kern), lds, "laplace forward")) return s;
  dim3 grid(ceil_div((int)d.N, 64 * kFbR) * ceil_div((int)d.M, mg), (unsigned)d.BH());
  hipLaunchKernelGGL(kern, grid, dim3(64 * W), lds, st, static_cast<const T*>(q), static_cast<const T*>(k),
                     static_cast<O*>(o), (int)d.N, mg, (int)d.M, (int)d.C, scale);
  return check_launch("laplace forward");
}

template <typename T, int EPI = kEpiDist>
int launch_fwd_bcast(const void* q, const void* k, void* o, const Dims& d, hipStream_t st, float scale = 0.0f) {
  switch (pick_fb_jb(d.M)) {
    case 4: return launch_fwd_bcast_jb<T, 4, EPI>(q, k, o, d, scale, st);
    case 7: return launch_fwd_bcast_jb<T, 7, EPI>(q, k, o, d, scale, st);
    case 8: return launch_fwd_bcast_jb<T, 8, EPI>(q, k, o, d, scale, st);
    default: return launch_fwd_bcast_jb<T, 16, EPI>(q, k, o, d, scale, st);
  }
}

template <typename T>
int launch_fwd(const void* q, const void* k, void* o, const Dims& d, hipStream_t st) {
  const T* qq = static_cast<const T*>(q);
  const T* kk = static_cast<const T*>(k);
  T* oo = static_cast<T*>(o);
  switch (pick_fwd_jb(d.M)) {
    case 7: return launch_fwd_jb<T, 7>(qq, kk, oo, d, st);
    case 8: return launch_fwd_jb<T, 8>(qq, kk, oo, d, st);
    case 16: return launch_fwd_jb<T, 16>(qq, kk, oo, d, st);
    default: return launch_fwd_jb<T, 32>(qq, kk, oo, d, st);
  }
}

// ---- backward ----
struct BwdPlan {
  int JB;           // key columns per register block
  int W;            // waves per workgroup
  int nx;           // workgroups per (bh, channel block) slice
  int rowsPerWave;
  int ncb;          // channel blocks of 64
  size_t lds;
  size_t partialElems;
};

int pick_bwd_jb(int64_t M) {
  if (M <= 16) return 16;
  if (M <= 32) return 32;
  if (M == 49) return 49;
  return 64;
}

BwdPlan plan_bwd(const Dims& d, bool dq, bool dkey, size_t accBytes, size_t gBytes) {
  BwdPlan p{};
  p.JB = pick_bwd_jb(d.M);
  p.ncb = ceil_div((int)d.C, 64);
  const int GV = 16 / (int)gBytes;
  const int JBP = round_up(p.JB, GV);
  const bool multiJ = d.M > p.JB;
  const int64_t slices = d.BH() * p.ncb;
  const int N = (int)std::max<int64_t>(d.N, 1);
  // One round of resident waves: 2 per SIMD (the kernel may use up to 256
  // registers), at least 8 rows per wave.
  const int target = 8 * num_cus();
  int64_t wps = std::max<int64_t>(1, ceil_div(target, (int)std::min<int64_t>(slices, target)));
  wps = std::min<int64_t>(wps, ceil_div(N, 8));
  int rows = ceil_div(N, (int)wps);
  if (dq && multiJ) rows = std::min(rows, 64);
  wps = ceil_div(N, rows);
  const size_t budget = 96 * 1024;
  auto lds = [&](int w) {
    size_t b = (size_t)w * kBwdRB * (JBP * gBytes + 64 * accBytes) + (size_t)p.JB * 64 * accBytes;
    if (dkey) b += (size_t)p.JB * 64 * accBytes;
    if (dq && multiJ) b += (size_t)w * rows * 64 * accBytes;
    return b;
  };
  int W = (int)std::min<int64_t>(8, wps);
  while (W > 1 && lds(W) > budget) --W;
  p.W = W;
  p.nx = ceil_div((int)wps, W);
  p.rowsPerWave = ceil_div(N, p.nx * W);
  if (dq && multiJ) p.rowsPerWave = std::min(p.rowsPerWave, rows);
  p.lds = lds(W);
  p.partialElems = dkey ? (size_t)slices * p.nx * 64 * (size_t)d.M : 0;
  return p;
}

// Plan of the register-resident-column backward: 3 waves per SIMD resident (4 for M <= 16).
struct BcPlan {
  int W, nx, rowsPerWave, ncb;
  size_t lds, partialElems;
};

// (M = 64 runs faster on the column-block kernel below: 57 vs 62 us at B=32 N=3136.)
// fp32 / bf16 with M = 32 (a column block) run the column-block kernel.
bool bcast_bwd_ok(int dtype, const Dims& d, const void* g) {
  if (dtype == LFAMD_F16) {
    if (!(d.M == 16 || d.M == 32 || d.M == 49)) return false;
  } else if (dtype == LFAMD_F32 || dtype == LFAMD_BF16) {
    if (!(d.M == 16 || d.M == 49)) return false;
  } else {
    return false;
  }
  if (dtype != LFAMD_F32 && (d.N * d.M) % 2 != 0) return false;
  return (reinterpret_cast<uintptr_t>(g) & 3) == 0;
}

BcPlan plan_bcast(const Dims& d, bool dkey) {
  BcPlan p{};
  p.ncb = ceil_div((int)d.C, 64);
  const int64_t slices = d.BH() * p.ncb;
  const int N = (int)std::max<int64_t>(d.N, 1);
  const int wmax = bcast_max_waves((int)d.M);
  const int target = wmax * num_cus();
  int64_t wps = std::max<int64_t>(1, ceil_div(target, (int)std::min<int64_t>(slices, target)));
  wps = std::min<int64_t>(wps, ceil_div(N, 8));
  const int W = (int)std::min<int64_t>(wmax, wps);
  p.W = W;
  p.nx = ceil_div((int)wps, W);
  p.rowsPerWave = round_up(ceil_div(N, p.nx * W), 2);
  const int mp = bcast_pitch((int)d.M);
  const int rpw = d.C <= 32 ? 2 : 1;
  p.lds = ((size_t)bcast_key_floats((int)d.M) + (size_t)W * (kBcRB * mp + kBcRB + mp + kBcRB / rpw * 64)) * 4;
  if (dkey) p.lds = std::max(p.lds, (size_t)std::min(W, kBcBufs) * bcast_key_floats((int)d.M) * 4);
  p.partialElems = dkey ? (size_t)slices * p.nx * 64 * (size_t)d.M : 0;
  return p;
}

// Kernel-gradient source of the backward (LaplacianFormer's K = exp(-s * dist)).
struct KernGrad {
  RowSources src = {};
  float scale = 0.0f;
};

template <typename T, int MC, bool DQ, bool DK, int GSRC, int RPW>
int launch_bcast_bwd_rpw(const void* g, const void* q, const void* k, void* dq, void* dk, void* ws, const Dims& d,
                         const BcPlan& p, hipStream_t st, const KernGrad& kg) {
  dim3 grid(p.nx, p.ncb, (unsigned)d.BH());
  auto kern = laplace_bwd_bcast_kernel<T, MC, DQ, DK, GSRC, RPW>;
  // M = 16 with one batch of rows per wave: one step loop, in registers that two workgroups share (bcast_paired;
  // 64 slices of 50 rows 5.5 against 5.7 us). More rows: both loops (24 slices of 3000 rows, C = 64: 17.8
  // against 20.5 us).
  if constexpr (MC == 16 && bcast_paired<T, MC, DQ, DK, GSRC, RPW>())
    if (p.rowsPerWave <= kBcRB) kern = laplace_bwd_bcast_kernel<T, MC, DQ, DK, GSRC, RPW, false>;
  hipLaunchKernelGGL(kern, grid, dim3(64 * p.W), p.lds, st,
                     static_cast<const T*>(g), kg.src, kg.scale, static_cast<const T*>(q),
                     static_cast<const T*>(k), static_cast<T*>(dq), static_cast<T*>(dk),
                     static_cast<float*>(ws), (int)d.N, (int)d.C, p.rowsPerWave);
  return check_launch("laplace backward");
}

template <typename T, int MC, bool DQ, bool DK, int GSRC>
int launch_bcast_bwd_mc(const void* g, const void* q, const void* k, void* dq, void* dk, void* ws, const Dims& d,
                        const BcPlan& p, hipStream_t st, const KernGrad& kg) {
  int s = d.C <= 32 ? launch_bcast_bwd_rpw<T, MC, DQ, DK, GSRC, 2>(g, q, k, dq, dk, ws, d, p, st, kg)
                    : launch_bcast_bwd_rpw<T, MC, DQ, DK, GSRC, 1>(g, q, k, dq, dk, ws, d, p, st, kg);
  if (s || !DK || p.nx == 1) return s;
  dim3 rgrid(ceil_div(64 * MC, 256), p.ncb, (unsigned)d.BH());
  hipLaunchKernelGGL(laplace_dk_reduce_cm_kernel<T>, rgrid, dim3(256), 0, st, static_cast<const float*>(ws),
                     static_cast<T*>(dk), p.nx, MC, (int)d.C);
  return check_launch("laplace backward_key reduction");
}

template <typename T, bool DQ, bool DK, int GSRC>
int launch_bcast_bwd_t(const void* g, const void* q, const void* k, void* dq, void* dk, void* ws, const Dims& d,
                       const BcPlan& p, hipStream_t st, const KernGrad& kg) {
  if constexpr (std::is_same<T, f16s>::value)
    if (d.M == 32) return launch_bcast_bwd_mc<T, 32, DQ, DK, GSRC>(g, q, k, dq, dk, ws, d, p, st, kg);
  if (d.M == 16) return launch_bcast_bwd_mc<T, 16, DQ, DK, GSRC>(g, q, k, dq, dk, ws, d, p, st, kg);
  return launch_bcast_bwd_mc<T, 49, DQ, DK, GSRC>(g, q, k, dq, dk, ws, d, p, st, kg);
}

template <bool DQ, bool DK, int GSRC = kGradF16>
int launch_bcast_bwd(int dtype, const void* g, const void* q, const void* k, void* dq, void* dk, void* ws,
                     const Dims& d, const BcPlan& p, hipStream_t st, const KernGrad& kg = {}) {
  if (dtype == LFAMD_F32) return launch_bcast_bwd_t<float, DQ, DK, GSRC>(g, q, k, dq, dk, ws, d, p, st, kg);
  if (dtype == LFAMD_BF16) return launch_bcast_bwd_t<bf16s, DQ, DK, GSRC>(g, q, k, dq, dk, ws, d, p, st, kg);
  return launch_bcast_bwd_t<f16s, DQ, DK, GSRC>(g, q, k, dq, dk, ws, d, p, st, kg);
}

// ---- backward for 17 <= M <= 256 in column blocks of 32 (fp16 / bf16 / fp32) ----
struct MbPlan {
  int CB, RG, W, nx, ncb, rowsPerWG;
  size_t lds, partialElems;
};

// Any 17 <= M <= 256; a last column block of fewer than 32 columns is
// zero-padded. (16-bit grad rows of odd length are fetched element by element.)
bool mb_bwd_ok(int dtype, const Dims& d, const void* g) {
  if (!(dtype == LFAMD_F16 || dtype == LFAMD_BF16 || dtype == LFAMD_F32)) return false;
  if (d.M < 17 || d.M > 8 * kMbMC) return false;
  // Word loads need 4-byte rows; odd 16-bit rows are read element by element.
  const bool elementwise = dtype != LFAMD_F32 && d.M % 2 != 0;
  return (reinterpret_cast<uintptr_t>(g) & (elementwise ? 1 : 3)) == 0;
}

MbPlan plan_mb(const Dims& d, bool dkey) {
  MbPlan p{};
  p.ncb = ceil_div((int)d.C, 64);
  p.CB = ceil_div((int)d.M, kMbMC);
  p.RG = std::max(1, 16 / p.CB);
  p.W = p.CB * p.RG;
  const int64_t slices = d.BH() * p.ncb;
  const int N = (int)std::max<int64_t>(d.N, 1);
  // One workgroup per CU when the slices allow it, each with at least one batch per row group.
  int nx = (int)std::max<int64_t>(1, ceil_div(num_cus(), (int)std::min<int64_t>(slices, num_cus())));
  nx = std::min(nx, std::max(1, N / (kMbRB * p.RG)));
  p.rowsPerWG = round_up(ceil_div(N, nx), kMbRB);
  p.nx = ceil_div(N, p.rowsPerWG);
  const size_t bigFloats = std::max<size_t>((size_t)p.CB * kMbMC * 64, (size_t)2 * p.W * kMbRB * 64);
  p.lds = (bigFloats + (size_t)p.W * (kMbRB * kMbMC + kMbRB + kMbRB * 64)) * 4;
  p.partialElems = dkey ? (size_t)slices * p.nx * 64 * (size_t)d.M : 0;
  return p;
}

// Rows through a loop (LOOP) instead of an unrolled batch of eight, which computes a short
// batch's missing rows too (on zero grad) and whose instructions a few rows do not pay back:
//   up to 6 rows (fp32 grad_query, one row, M = 32: 4.6 us against 6.4 unrolled; five rows 6.1
//   against 6.8);
//   where three waves or more per SIMD have rows, so that issue slots count, and
//   - one gradient, and the short batch is a round of its own with more than a quarter of all rounds'
//     rows missing (bf16 grad_query: 4 of 17 rows, M = 196, 14.7 against 15.6; 256 of 130 rows, M = 17, 11.3
//     against 12.0; M = 64, three rounds, is the faster unrolled), or
//   - the missing rows are more than 8 % of the rows (bf16 grad_query, 2048 slices of 9 rows, M = 196,
//     C = 64: 90 against 98 us); within two rounds 2 % for grad_key and 3 % for grad_query of 16-bit
//     types (256 x 100 rows, M = 17: 1.016 against 1.05 of the time before the unrolled batch; in more
//     rounds 300 x 100 rows, M = 196, take 71 us looped and 67 unrolled); 15 % for one fp32 gradient,
//     whose loop has the slower step only (64 of 50 rows, M = 100, 17.1 looped against 15.9), 50 % for
//     both of a kernel gradient, whose loop spills (fp16, 64 of 50 rows, M = 64, 18.2 looped against 17.4).
// Full batches are faster unrolled at any count (fp32 grad_query, 300 slices of 64 rows, M = 64:
// 0.9 of the loop's time). Several workgroups per slice: only the last can have a short batch.
bool mb_row_loop(const Dims& d, const MbPlan& p, bool f32, bool dq, bool dk, int gsrc) {
  if (p.nx > 1 || d.N < 1) return false;
  if (d.N <= 6) return true;
  const int64_t batches = (d.N + kMbRB - 1) / kMbRB, rounds = (batches + p.RG - 1) / p.RG;
  if (batches * p.CB < 12) return false;
  const int64_t missing = batches * kMbRB - d.N;
  if (!(dq && dk) && (batches - 1) % p.RG == 0 && 4 * missing > kMbRB * rounds) return true;
  const int percent = gsrc == kGradKernel ? 50 : f32 && !(dq && dk) ? 15 : (dq && dk) || rounds > 2 ? 8 : dq ? 3 : 2;
  return 100 * missing > percent * d.N;
}

template <typename T, int CB, bool DQ, bool DK, int GSRC = kGradF16>
int launch_mb_cb(const void* g, const void* q, const void* k, void* dq, void* dk, void* ws, const Dims& d,
                 const MbPlan& p, hipStream_t st, const KernGrad& kg = {}) {
  auto kern = mb_row_loop(d, p, sizeof(T) == 4, DQ, DK, GSRC) ? laplace_bwd_mb_kernel<T, CB, DQ, DK, GSRC, true> : laplace_bwd_mb_kernel<T, CB, DQ, DK, GSRC>;
  if (p.lds > 65536)
    if (int s = set_dyn_lds(reinterpret_cast<const void*>(kern), p.lds, "laplace backward")) return s;
  dim3 grid(p.nx, p.ncb, (unsigned)d.BH());
  hipLaunchKernelGGL(kern, grid, dim3(64 * p.W), p.lds, st, static_cast<const T*>(g), static_cast<const T*>(q),
                     static_cast<const T*>(k), static_cast<T*>(dq), static_cast<float*>(ws), (int)d.N, (int)d.C,
                     p.rowsPerWG, (int)d.M, kg.src, kg.scale);
  int s = check_launch("laplace backward");
  if (s || !DK) return s;
  dim3 rgrid(ceil_div(64 * (int)d.M, 256), p.ncb, (unsigned)d.BH());
  hipLaunchKernelGGL(laplace_dk_reduce_cm_kernel<T>, rgrid, dim3(256), 0, st, static_cast<const float*>(ws),
                     static_cast<T*>(dk), p.nx, (int)d.M, (int)d.C);
  return check_launch("laplace backward_key reduction");
}

template <typename T, bool DQ, bool DK, int GSRC = kGradF16>
int launch_mb_t(const void* g, const void* q, const void* k, void* dq, void* dk, void* ws, const Dims& d,
                const MbPlan& p, hipStream_t st, const KernGrad& kg = {}) {
  switch (p.CB) {
    case 1: return launch_mb_cb<T, 1, DQ, DK, GSRC>(g, q, k, dq, dk, ws, d, p, st, kg);
    case 2: return launch_mb_cb<T, 2, DQ, DK, GSRC>(g, q, k, dq, dk, ws, d, p, st, kg);
    case 3: return launch_mb_cb<T, 3, DQ, DK, GSRC>(g, q, k, dq, dk, ws, d, p, st, kg);
    case 4: return launch_mb_cb<T, 4, DQ, DK, GSRC>(g, q, k, dq, dk, ws, d, p, st, kg);
    case 5: return launch_mb_cb<T, 5, DQ, DK, GSRC>(g, q, k, dq, dk, ws, d, p, st, kg);
    case 6: return launch_mb_cb<T, 6, DQ, DK, GSRC>(g, q, k, dq, dk, ws, d, p, st, kg);
    case 7: return launch_mb_cb<T, 7, DQ, DK, GSRC>(g, q, k, dq, dk, ws, d, p, st, kg);
    default: return launch_mb_cb<T, 8, DQ, DK, GSRC>(g, q, k, dq, dk, ws, d, p, st, kg);
  }
}

template <bool DQ, bool DK, int GSRC = kGradF16>
int launch_mb(int dtype, const void* g, const void* q, const void* k, void* dq, void* dk, void* ws,
              const Dims& d, const MbPlan& p, hipStream_t st, const KernGrad& kg = {}) {
  switch (dtype) {
    case LFAMD_F16: return launch_mb_t<f16s, DQ, DK, GSRC>(g, q, k, dq, dk, ws, d, p, st, kg);
    case LFAMD_BF16: return launch_mb_t<bf16s, DQ, DK, GSRC>(g, q, k, dq, dk, ws, d, p, st, kg);
    default: return launch_mb_t<float, DQ, DK, GSRC>(g, q, k, dq, dk, ws, d, p, st, kg);
  }
}

// lfamd_laplace_kernel_backward_rows replaced, for bf16 / fp32 layers (M <= 64), three
// times {g = -s gK K as an elementwise pass, casts, backward, reduction} by one launch:
// B=2 H=2 14x14 d=32 fp32 layer step 198 -> 136 us, B=64 H=4 14x14 d=32 bf16 259 -> 148 us
// (the three backwards 24 us each with half their lanes idle at d = 32).
// The fused kernel-gradient backward: M in {16, 49} (fp16: 32 too) on the
// register-resident-column kernel, any other 17 <= M <= 256 on the column-block
// kernel (the former spills at M = 64: 94 us there against 87 us composed).
bool kernel_bwd_bcast(int dtype, const Dims& d) { return d.M == 16 || d.M == 49 || (d.M == 32 && dtype == LFAMD_F16); }
bool kernel_bwd_shape(int dtype, const Dims& d) {
  return kernel_bwd_bcast(dtype, d) || (d.M >= 17 && d.M <= 8 * kMbMC);
}
bool kernel_bwd_ok(int dtype, const Dims& d) { return dtype == LFAMD_F16 && kernel_bwd_shape(dtype, d); }

// The row sets of a kernel-gradient backward; `unit` is what the sets' ends count
// (rows, or the column-block kernel's row batches). d.N is their total.
KernGrad kern_grad(int nsrc, const float* const* gk, const float* const* kv, const void* const* q, void* const* dq,
                   const int64_t* lens, int unit, float scale) {
  KernGrad kg;
  int end = 0;
  for (int i = 0; i < 3; ++i) {
    if (i < nsrc) {
      kg.src.gk[i] = gk[i];
      kg.src.kv[i] = kv[i];
      kg.src.q[i] = q[i];
      kg.src.dq[i] = dq[i];
      kg.src.len[i] = (int)lens[i];
      end += ceil_div((int)lens[i], unit);
    }
    kg.src.end[i] = end;
  }
  kg.scale = scale;
  return kg;
}

template <typename T, int JB, bool DQ, bool DK>
int launch_bwd_jb(const T* g, const T* q, const T* k, T* dq, T* dk, void* ws, const Dims& d,
                  const BwdPlan& p, hipStream_t st) {
  using A = typename AccOf<T>::type;
  dim3 grid(p.nx, p.ncb, (unsigned)d.BH());
  dim3 block(64 * p.W);
  hipLaunchKernelGGL((laplace_bwd_kernel<T, JB, DQ, DK>), grid, block, p.lds, st, g, q, k, dq, dk,
                     static_cast<A*>(ws), (int)d.N, (int)d.M, (int)d.C, p.rowsPerWave);
  int s = check_launch("laplace backward");
  if (s || !DK) return s;
  dim3 rgrid(ceil_div(64 * (int)d.M, 256), p.ncb, (unsigned)d.BH());
  hipLaunchKernelGGL(laplace_dk_reduce_kernel<T>, rgrid, dim3(256), 0, st, static_cast<const A*>(ws), dk,
                     p.nx, (int)d.M, (int)d.C);
  return check_launch("laplace backward_key reduction");
}

template <typename T, bool DQ, bool DK>
int launch_bwd_t(const void* g, const void* q, const void* k, void* dq, void* dk, void* ws,
                 const Dims& d, const BwdPlan& p, hipStream_t st) {
  auto G = static_cast<const T*>(g);
  auto Q = static_cast<const T*>(q);
  auto K = static_cast<const T*>(k);
  auto DQp = static_cast<T*>(dq);
  auto DKp = static_cast<T*>(dk);
  switch (p.JB) {
    case 16: return launch_bwd_jb<T, 16, DQ, DK>(G, Q, K, DQp, DKp, ws, d, p, st);
    case 32: return launch_bwd_jb<T, 32, DQ, DK>(G, Q, K, DQp, DKp, ws, d, p, st);
    case 49: return launch_bwd_jb<T, 49, DQ, DK>(G, Q, K, DQp, DKp, ws, d, p, st);
    default: return launch_bwd_jb<T, 64, DQ, DK>(G, Q, K, DQp, DKp, ws, d, p, st);
  }
}

template <bool DQ, bool DK>
int launch_bwd(int dtype, const void* g, const void* q, const void* k, void* dq, void* dk, void* ws,
               const Dims& d, const BwdPlan& p, hipStream_t st) {
  switch (dtype) {
    case LFAMD_F32: return launch_bwd_t<float, DQ, DK>(g, q, k, dq, dk, ws, d, p, st);
    case LFAMD_F16: return launch_bwd_t<f16s, DQ, DK>(g, q, k, dq, dk, ws, d, p, st);
    case LFAMD_BF16: return launch_bwd_t<bf16s, DQ, DK>(g, q, k, dq, dk, ws, d, p, st);
    default: return launch_bwd_t<double, DQ, DK>(g, q, k, dq, dk, ws, d, p, st);
  }
}

// Fills `n` elements of `p` with zero (used when the reduction length is 0).
template <typename T>
__global__ void fill_zero_kernel(T* __restrict__ p, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    p[i] = T{};
}

int zero_fill(void* p, int64_t bytes, hipStream_t st) {
  if (bytes <= 0) return LFAMD_OK;
  const int64_t words = bytes / 2;  // every element type is a multiple of 2 bytes
  const int blocks = (int)std::min<int64_t>(1024, (words + 255) / 256);
  hipLaunchKernelGGL(fill_zero_kernel<uint16_t>, dim3(blocks), dim3(256), 0, st, static_cast<uint16_t*>(p), words);
  return check_launch("zero fill");
}

int bwd_common(int dtype, const void* g, const void* q, const void* k, void* dq, void* dk,
               const Dims& d, void* ws, size_t wsBytes, void* stream, bool doDq, bool doDk,
               const char* who) {
  if (!valid_dtype(dtype)) return fail(LFAMD_ERR_DTYPE, "%s: unsupported dtype %d", who, dtype);
  int s = check_dims(d, who);
  if (s) return s;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const size_t es = dtype_size(dtype);
  if (d.BH() == 0 || d.C == 0) return ok();
  if (d.M == 0 || d.N == 0) {
    // Empty reduction: the gradients are zero (the output is empty when N or M is 0).
    if (doDq && (s = zero_fill(dq, d.BH() * d.N * d.C * (int64_t)es, st))) return s;
    if (doDk && (s = zero_fill(dk, d.BH() * d.C * d.M * (int64_t)es, st))) return s;
    return ok();
  }
  if (!g || !q || !k || (doDq && !dq) || (doDk && !dk)) return fail(LFAMD_ERR_ARG, "%s: null pointer", who);
  const size_t acc = dtype == LFAMD_F64 ? 8 : 4;
  if (doDk && ws && (reinterpret_cast<uintptr_t>(ws) & (acc - 1)))
    return fail(LFAMD_ERR_ARG, "%s: workspace not %zu-byte aligned", who, acc);
  if (b2_ok(dtype, d.BH(), d.N, d.M, d.C) && (reinterpret_cast<uintptr_t>(q) & 3) == 0)
    return b2_launch(dtype, g, q, k, doDq ? dq : nullptr, doDk ? dk : nullptr, ws, wsBytes, d.BH(), d.N, d.M, d.C,
                     st, who);
  if (bcast_bwd_ok(dtype, d, g)) {
    const BcPlan sp = plan_bcast(d, doDk);
    if (doDk && (!ws || wsBytes < sp.partialElems * 4))
      return fail(LFAMD_ERR_ARG, "%s: workspace of %zu bytes needed, %zu given", who, sp.partialElems * 4, wsBytes);
    if (doDq && doDk) return launch_bcast_bwd<true, true>(dtype, g, q, k, dq, dk, ws, d, sp, st);
    if (doDq) return launch_bcast_bwd<true, false>(dtype, g, q, k, dq, dk, ws, d, sp, st);
    return launch_bcast_bwd<false, true>(dtype, g, q, k, dq, dk, ws, d, sp, st);
  }
  if (mb_bwd_ok(dtype, d, g)) {
    const MbPlan mp = plan_mb(d, doDk);
    if (doDk && (!ws || wsBytes < mp.partialElems * 4))
      return fail(LFAMD_ERR_ARG, "%s: workspace of %zu bytes needed, %zu given", who, mp.partialElems * 4, wsBytes);
    if (doDq && doDk) return launch_mb<true, true>(dtype, g, q, k, dq, dk, ws, d, mp, st);
    if (doDq) return launch_mb<true, false>(dtype, g, q, k, dq, dk, ws, d, mp, st);
    return launch_mb<false, true>(dtype, g, q, k, dq, dk, ws, d, mp, st);
  }
  const BwdPlan p = plan_bwd(d, doDq, doDk, acc, dtype == LFAMD_F16 ? 2 : acc);
  if (doDk) {
    const size_t need = p.partialElems * acc;
    if (!ws || wsBytes < need)
      return fail(LFAMD_ERR_ARG, "%s: workspace of %zu bytes needed, %zu given", who, need, wsBytes);
  }
  if (doDq && doDk) return launch_bwd<true, true>(dtype, g, q, k, dq, dk, ws, d, p, st);
  if (doDq) return launch_bwd<true, false>(dtype, g, q, k, dq, dk, ws, d, p, st);
  return launch_bwd<false, true>(dtype, g, q, k, dq, dk, ws, d, p, st);
}

}  // namespace
}  // namespace lfamd

using namespace lfamd;

extern "C" {

int lfamd_laplace_forward(int dtype, const void* query, const void* key, void* output,
                          int64_t batch, int64_t heads, int64_t q_len, int64_t k_len,
                          int64_t channels, void* stream) {
  if (!valid_dtype(dtype)) return fail(LFAMD_ERR_DTYPE, "laplace forward: unsupported dtype %d", dtype);
  const Dims d{batch, heads, q_len, k_len, channels};
  int s = check_dims(d, "laplace forward");
  if (s) return s;
  if (empty(d)) return ok();
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (d.C == 0) return zero_fill(output, d.BH() * d.N * d.M * (int64_t)dtype_size(dtype), st);
  if (!query || !key || !output) return fail(LFAMD_ERR_ARG, "laplace forward: null pointer");
  if (f2_ok(dtype, d.BH(), d.N, d.M, d.C, query))
    return f2_launch(dtype, false, query, key, output, d.BH(), d.N, d.C, 0.0f, st);
  if (f3_ok(dtype, d.BH(), d.N, d.M, d.C, query, output))
    return f3_launch(dtype, query, key, output, d.BH(), d.N, d.M, d.C, st);
  if (fwd_bcast_ok(dtype, d, query, dtype_size(dtype))) {
    switch (dtype) {
      case LFAMD_F32: return launch_fwd_bcast<float>(query, key, output, d, st);
      case LFAMD_F16: return launch_fwd_bcast<f16s>(query, key, output, d, st);
      default: return launch_fwd_bcast<bf16s>(query, key, output, d, st);
    }
  }
  switch (dtype) {
    case LFAMD_F32: return launch_fwd<float>(query, key, output, d, st);
    case LFAMD_F16: return launch_fwd<f16s>(query, key, output, d, st);
    case LFAMD_BF16: return launch_fwd<bf16s>(query, key, output, d, st);
    default: return launch_fwd<double>(query, key, output, d, st);
  }
}

int lfamd_laplace_backward_query(int dtype, const void* grad_output, const void* query,
                                 const void* key, void* grad_query, int64_t batch,
                                 int64_t heads, int64_t q_len, int64_t k_len,
                                 int64_t channels, void* stream) {
  return bwd_common(dtype, grad_output, query, key, grad_query, nullptr,
                    Dims{batch, heads, q_len, k_len, channels}, nullptr, 0, stream, true, false,
                    "laplace backward_query");
}

size_t lfamd_laplace_backward_workspace_size(int dtype, int64_t batch, int64_t heads,
                                             int64_t q_len, int64_t k_len, int64_t channels) {
  const Dims d{batch, heads, q_len, k_len, channels};
  if (!valid_dtype(dtype) || check_dims(d, "workspace") || d.BH() == 0 || d.N == 0 || d.M == 0 || d.C == 0)
    return 0;
  const size_t acc = dtype == LFAMD_F64 ? 8 : 4;
  // Any of the backward paths may run (which one also depends on pointer alignment).
  size_t bytes = plan_bwd(d, true, true, acc, dtype == LFAMD_F16 ? 2 : acc).partialElems * acc;
  if (dtype != LFAMD_F64) bytes = std::max(bytes, plan_bcast(d, true).partialElems * 4);
  if (dtype != LFAMD_F64 && d.M >= 17 && d.M <= 8 * kMbMC)
    bytes = std::max(bytes, plan_mb(d, true).partialElems * 4);
  if (b2_ok(dtype, d.BH(), d.N, d.M, d.C)) bytes = std::max(bytes, b2_workspace_elems(d.BH(), d.N, d.M, d.C) * 4);
  return bytes;
}

int lfamd_laplace_backward_key(int dtype, const void* grad_output, const void* query,
                               const void* key, void* grad_key, int64_t batch,
                               int64_t heads, int64_t q_len, int64_t k_len,
                               int64_t channels, void* workspace, size_t workspace_bytes,
                               void* stream) {
  return bwd_common(dtype, grad_output, query, key, nullptr, grad_key,
                    Dims{batch, heads, q_len, k_len, channels}, workspace, workspace_bytes, stream,
                    false, true, "laplace backward_key");
}

int lfamd_laplace_backward(int dtype, const void* grad_output, const void* query,
                           const void* key, void* grad_query, void* grad_key,
                           int64_t batch, int64_t heads, int64_t q_len, int64_t k_len,
                           int64_t channels, void* workspace, size_t workspace_bytes,
                           void* stream) {
  return bwd_common(dtype, grad_output, query, key, grad_query, grad_key,
                    Dims{batch, heads, q_len, k_len, channels}, workspace, workspace_bytes, stream,
                    true, true, "laplace backward");
}

int lfamd_laplace_kernel_forward(int dtype, const void* query, const void* key, float* output,
                                 int64_t batch, int64_t heads, int64_t q_len, int64_t k_len,
                                 int64_t channels, float scale, void* stream) {
  if (!valid_dtype(dtype)) return fail(LFAMD_ERR_DTYPE, "laplace kernel forward: unsupported dtype %d", dtype);
  const Dims d{batch, heads, q_len, k_len, channels};
  int s = check_dims(d, "laplace kernel forward");
  if (s) return s;
  if (empty(d)) return ok();
  if (d.C == 0 || !fwd_bcast_ok(dtype, d, query, sizeof(float)))
    return fail(LFAMD_ERR_UNSUPPORTED, "laplace kernel forward: no fused path for dtype %d, M=%lld, C=%lld",
                dtype, (long long)d.M, (long long)d.C);
  if (!query || !key || !output) return fail(LFAMD_ERR_ARG, "laplace kernel forward: null pointer");
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (f2_ok(dtype, d.BH(), d.N, d.M, d.C, query))
    return f2_launch(dtype, true, query, key, output, d.BH(), d.N, d.C, scale, st);
  switch (dtype) {
    case LFAMD_F32: return launch_fwd_bcast<float, kEpiExp>(query, key, output, d, st, scale);
    case LFAMD_F16: return launch_fwd_bcast<f16s, kEpiExp>(query, key, output, d, st, scale);
    default: return launch_fwd_bcast<bf16s, kEpiExp>(query, key, output, d, st, scale);
  }
}

int lfamd_laplace_kernel_forward_multi(int dtype, int num_sources, const void* const* queries,
                                       const int64_t* q_lens, const void* key, float* const* outputs,
                                       int64_t batch, int64_t heads, int64_t k_len, int64_t channels,
                                       float scale, void* stream) {
  const char* who = "laplace kernel forward (several sources)";
  if (!valid_dtype(dtype)) return fail(LFAMD_ERR_DTYPE, "%s: unsupported dtype %d", who, dtype);
  if (num_sources < 1 || num_sources > 3 || !queries || !q_lens || !outputs)
    return fail(LFAMD_ERR_ARG, "%s: 1 to 3 sources with their arrays expected", who);
  for (int i = 0; i < num_sources; ++i)
    if (q_lens[i] < 1 || !queries[i] || !outputs[i]) return fail(LFAMD_ERR_ARG, "%s: source %d empty or null", who, i);
  const Dims d{batch, heads, 1, k_len, channels};
  int s = check_dims(d, who);
  if (s) return s;
  if (d.BH() == 0) return ok();
  if (!key) return fail(LFAMD_ERR_ARG, "%s: null pointer", who);
  for (int i = 0; i < num_sources; ++i)
    if (!f2_ok(dtype, d.BH(), q_lens[i], d.M, d.C, queries[i]))
      return fail(LFAMD_ERR_UNSUPPORTED, "%s: no single-launch path (dtype %d, M=%lld, C=%lld, source %d)", who,
                  dtype, (long long)d.M, (long long)d.C, i);
  return f2_launch_multi(dtype, num_sources, queries, q_lens, key, outputs, d.BH(), d.C, scale,
                         static_cast<hipStream_t>(stream));
}

namespace {
// The segmented fused-kernel backward applies: fp16, M = 49, C % 64 == 0,
// 1 to 3 sources of at least one row, 4-byte aligned queries.
int multi_bwd_check(int dtype, int nsrc, const int64_t* q_lens, const void* const* queries, const Dims& d,
                    const char* who) {
  if (nsrc < 1 || nsrc > 3 || !q_lens) return fail(LFAMD_ERR_ARG, "%s: 1 to 3 sources expected", who);
  for (int i = 0; i < nsrc; ++i)
    if (q_lens[i] < 1) return fail(LFAMD_ERR_ARG, "%s: source %d has no rows", who, i);
  if (dtype != LFAMD_F16 || d.M != 49 || d.C <= 0 || d.C % 64 != 0 || d.BH() < 1 || d.C / 64 > 65535)
    return fail(LFAMD_ERR_UNSUPPORTED, "%s: no single-launch path (dtype %d, M=%lld, C=%lld)", who, dtype,
                (long long)d.M, (long long)d.C);
  // The kernel holds row counts and its linear workgroup id in 32-bit ints.
  for (int i = 0; i < nsrc; ++i)
    if (q_lens[i] > INT32_MAX / 2)
      return fail(LFAMD_ERR_UNSUPPORTED, "%s: source %d has %lld rows (at most %d)", who, i, (long long)q_lens[i],
                  INT32_MAX / 2);
  if (b2_multi_workgroups(nsrc, q_lens, d.BH(), d.C) > INT32_MAX)
    return fail(LFAMD_ERR_UNSUPPORTED, "%s: too many workgroups for one launch", who);
  if (queries)
    for (int i = 0; i < nsrc; ++i)
      if (reinterpret_cast<uintptr_t>(queries[i]) & 3)
        return fail(LFAMD_ERR_UNSUPPORTED, "%s: query %d not 4-byte aligned", who, i);
  return LFAMD_OK;
}
}  // namespace

size_t lfamd_laplace_kernel_backward_multi_workspace_size(int dtype, int num_sources, const int64_t* q_lens,
                                                          int64_t batch, int64_t heads, int64_t k_len,
                                                          int64_t channels) {
  const Dims d{batch, heads, 1, k_len, channels};
  if (check_dims(d, "laplace kernel backward (several sources)") ||
      multi_bwd_check(dtype, num_sources, q_lens, nullptr, d, "laplace kernel backward (several sources)"))
    return 0;
  return b2_workspace_elems_multi(num_sources, q_lens, d.BH(), d.C) * 4;
}

int lfamd_laplace_kernel_backward_multi(int dtype, int num_sources, const float* const* grad_kernels,
                                        const float* const* kernels, const void* const* queries,
                                        const int64_t* q_lens, const void* key, void* const* grad_queries,
                                        void* grad_key, int64_t batch, int64_t heads, int64_t k_len,
                                        int64_t channels, float scale, void* workspace, size_t workspace_bytes,
                                        void* stream) {
  const char* who = "laplace kernel backward (several sources)";
  if (!valid_dtype(dtype)) return fail(LFAMD_ERR_DTYPE, "%s: unsupported dtype %d", who, dtype);
  const Dims d{batch, heads, 1, k_len, channels};
  int s = check_dims(d, who);
  if (s) return s;
  if (!grad_kernels || !kernels || !queries || !grad_queries || !key || !grad_key)
    return fail(LFAMD_ERR_ARG, "%s: null pointer", who);
  if ((s = multi_bwd_check(dtype, num_sources, q_lens, queries, d, who))) return s;
  for (int i = 0; i < num_sources; ++i)
    if (!grad_kernels[i] || !kernels[i] || !grad_queries[i]) return fail(LFAMD_ERR_ARG, "%s: null pointer", who);
  return b2_launch_multi(num_sources, grad_kernels, kernels, queries, grad_queries, q_lens, key, grad_key, workspace,
                         workspace_bytes, d.BH(), d.C, scale, static_cast<hipStream_t>(stream), who);
}

int lfamd_laplace_kernel_backward(int dtype, const float* grad_kernel, const float* kernel,
                                  const void* query, const void* key, void* grad_query, void* grad_key,
                                  int64_t batch, int64_t heads, int64_t q_len, int64_t k_len,
                                  int64_t channels, float scale, void* workspace,
                                  size_t workspace_bytes, void* stream) {
  const char* who = "laplace kernel backward";
  if (!valid_dtype(dtype)) return fail(LFAMD_ERR_DTYPE, "%s: unsupported dtype %d", who, dtype);
  const Dims d{batch, heads, q_len, k_len, channels};
  int s = check_dims(d, who);
  if (s) return s;
  const bool doDq = grad_query != nullptr, doDk = grad_key != nullptr;
  if (d.BH() == 0 || d.C == 0 || !(doDq || doDk)) return ok();
  if (d.N == 0 || !kernel_bwd_ok(dtype, d))
    return fail(LFAMD_ERR_UNSUPPORTED, "%s: no fused path for dtype %d, N=%lld, M=%lld", who, dtype,
                (long long)d.N, (long long)d.M);
  if (!grad_kernel || !kernel || !query || !key) return fail(LFAMD_ERR_ARG, "%s: null pointer", who);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (b2_ok(dtype, d.BH(), d.N, d.M, d.C) && (reinterpret_cast<uintptr_t>(query) & 3) == 0)
    return b2_launch(dtype, nullptr, query, key, grad_query, grad_key, workspace, workspace_bytes, d.BH(), d.N, d.M,
                     d.C, st, who, B2Grad{grad_kernel, kernel, scale});
  const bool bcast = kernel_bwd_bcast(dtype, d);
  const KernGrad kg = kern_grad(1, &grad_kernel, &kernel, &query, &grad_query, &q_len, bcast ? 1 : kMbRB, scale);
  if (!bcast) {
    const MbPlan mp = plan_mb(d, doDk);
    if (doDk && (!workspace || workspace_bytes < mp.partialElems * 4))
      return fail(LFAMD_ERR_ARG, "%s: workspace of %zu bytes needed, %zu given", who, mp.partialElems * 4,
                  workspace_bytes);
    if (doDq && doDk)
      return launch_mb<true, true, kGradKernel>(dtype, nullptr, query, key, grad_query, grad_key, workspace, d, mp, st, kg);
    if (doDq)
      return launch_mb<true, false, kGradKernel>(dtype, nullptr, query, key, grad_query, nullptr, workspace, d, mp, st, kg);
    return launch_mb<false, true, kGradKernel>(dtype, nullptr, query, key, nullptr, grad_key, workspace, d, mp, st, kg);
  }
  const BcPlan sp = plan_bcast(d, doDk);
  if (doDk && (!workspace || workspace_bytes < sp.partialElems * 4))
    return fail(LFAMD_ERR_ARG, "%s: workspace of %zu bytes needed, %zu given", who, sp.partialElems * 4,
                workspace_bytes);
  if (doDq && doDk)
    return launch_bcast_bwd<true, true, kGradKernel>(dtype, nullptr, query, key, grad_query, grad_key, workspace, d, sp, st, kg);
  if (doDq)
    return launch_bcast_bwd<true, false, kGradKernel>(dtype, nullptr, query, key, grad_query, nullptr, workspace, d, sp, st, kg);
  return launch_bcast_bwd<false, true, kGradKernel>(dtype, nullptr, query, key, nullptr, grad_key, workspace, d, sp, st, kg);
}

namespace {
// The row sets' total as one row count: the plans' rows, padded to whole row batches per
// set where the column-block kernel takes them.
int rows_bwd_dims(int dtype, int nsrc, const int64_t* lens, Dims& d, const char* who) {
  if (nsrc < 1 || nsrc > 3 || !lens) return fail(LFAMD_ERR_ARG, "%s: 1 to 3 sources expected", who);
  int64_t rows = 0;
  for (int i = 0; i < nsrc; ++i) {
    if (lens[i] < 1) return fail(LFAMD_ERR_ARG, "%s: source %d has no rows", who, i);
    if (lens[i] > INT32_MAX / 8)
      return fail(LFAMD_ERR_UNSUPPORTED, "%s: source %d has %lld rows (at most %d)", who, i, (long long)lens[i],
                  INT32_MAX / 8);
    rows += kernel_bwd_bcast(dtype, d) ? lens[i] : round_up((int)lens[i], kMbRB);
  }
  d.N = rows;
  if (dtype == LFAMD_F64 || !kernel_bwd_shape(dtype, d) || d.C < 1 || d.BH() < 1 || d.BH() > 65535 ||
      ceil_div((int)d.C, 64) > 65535)
    return fail(LFAMD_ERR_UNSUPPORTED, "%s: no fused path for dtype %d, M=%lld, C=%lld", who, dtype, (long long)d.M,
                (long long)d.C);
  return LFAMD_OK;
}

// The register-column kernel's partial sums; 16 bytes, for a size that is not 0, where a
// slice's only workgroup stores grad_key itself and none are written.
size_t rows_bwd_bytes(const BcPlan& p) { return p.nx == 1 ? 16 : p.partialElems * 4; }
}  // namespace

size_t lfamd_laplace_kernel_backward_rows_workspace_size(int dtype, int num_sources, const int64_t* q_lens,
                                                         int64_t batch, int64_t heads, int64_t k_len,
                                                         int64_t channels) {
  const char* who = "laplace kernel backward (row sets)";
  Dims d{batch, heads, 1, k_len, channels};
  if (!valid_dtype(dtype) || check_dims(d, who) || rows_bwd_dims(dtype, num_sources, q_lens, d, who)) return 0;
  return kernel_bwd_bcast(dtype, d) ? rows_bwd_bytes(plan_bcast(d, true)) : plan_mb(d, true).partialElems * 4;
}

int lfamd_laplace_kernel_backward_rows(int dtype, int num_sources, const float* const* grad_kernels,
                                       const float* const* kernels, const void* const* queries,
                                       const int64_t* q_lens, const void* key, void* const* grad_queries,
                                       void* grad_key, int64_t batch, int64_t heads, int64_t k_len,
                                       int64_t channels, float scale, void* workspace, size_t workspace_bytes,
                                       void* stream) {
  const char* who = "laplace kernel backward (row sets)";
  if (!valid_dtype(dtype)) return fail(LFAMD_ERR_DTYPE, "%s: unsupported dtype %d", who, dtype);
  Dims d{batch, heads, 1, k_len, channels};
  int s = check_dims(d, who);
  if (s || (s = rows_bwd_dims(dtype, num_sources, q_lens, d, who))) return s;
  if (!grad_kernels || !kernels || !queries || !grad_queries || !key || !grad_key)
    return fail(LFAMD_ERR_ARG, "%s: null pointer", who);
  for (int i = 0; i < num_sources; ++i)
    if (!grad_kernels[i] || !kernels[i] || !queries[i] || !grad_queries[i])
      return fail(LFAMD_ERR_ARG, "%s: null pointer", who);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const bool bcast = kernel_bwd_bcast(dtype, d);
  const KernGrad kg = kern_grad(num_sources, grad_kernels, kernels, queries, grad_queries, q_lens,
                                bcast ? 1 : kMbRB, scale);
  const BcPlan bp = bcast ? plan_bcast(d, true) : BcPlan{};
  const MbPlan mp = bcast ? MbPlan{} : plan_mb(d, true);
  const size_t need = bcast ? rows_bwd_bytes(bp) : mp.partialElems * 4;
  if (!workspace || workspace_bytes < need)
    return fail(LFAMD_ERR_ARG, "%s: workspace of %zu bytes needed, %zu given", who, need, workspace_bytes);
  return bcast ? launch_bcast_bwd<true, true, kGradKernel>(dtype, nullptr, nullptr, key, nullptr, grad_key, workspace,
                                                           d, bp, st, kg)
               : launch_mb<true, true, kGradKernel>(dtype, nullptr, nullptr, key, nullptr, grad_key, workspace, d, mp,
                                                    st, kg);
}

int lfamd_laplace_reduce_forward(int dtype, const void* query, const void* key,
                                 void* output, int64_t batch, int64_t heads,
                                 int64_t q_len, int64_t k_len, int64_t channels,
                                 void* stream) {
  if (!valid_dtype(dtype)) return fail(LFAMD_ERR_DTYPE, "laplace reduce_forward: unsupported dtype %d", dtype);
  const Dims d{batch, heads, q_len, k_len, channels};
  int s = check_dims(d, "laplace reduce_forward");
  if (s) return s;
  if (empty(d)) return ok();
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (d.C == 0) return zero_fill(output, d.BH() * d.N * d.M * (int64_t)dtype_size(dtype), st);
  if (!query || !key || !output) return fail(LFAMD_ERR_ARG, "laplace reduce_forward: null pointer");
  const int64_t total = d.BH() * d.N * d.M;
  const int bd = (int)std::min<int64_t>(d.C, 256);
  const unsigned blocks = (unsigned)std::min<int64_t>(total, 1 << 20);
#define LFAMD_REDUCE(T)                                                                        \
  hipLaunchKernelGGL(laplace_reduce_fwd_kernel<T>, dim3(blocks), dim3(bd), 0, st,              \
                     static_cast<const T*>(query), static_cast<const T*>(key), static_cast<T*>(output), \
                     total, (int)d.N, (int)d.M, (int)d.C)
  switch (dtype) {
    case LFAMD_F32: LFAMD_REDUCE(float); break;
    case LFAMD_F16: LFAMD_REDUCE(f16s); break;
    case LFAMD_BF16: LFAMD_REDUCE(bf16s); break;
    default: LFAMD_REDUCE(double); break;
  }
#undef LFAMD_REDUCE
  return check_launch("laplace reduce_forward");
}

}  // extern "C"
