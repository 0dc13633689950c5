// NewtonInverse products on the bf16 matrix cores, to fp32 accuracy.
//
// Every fp32 operand is held as x = p1 + p2 + p3, three bf16 pieces of 8
// significant bits each (p1 = x rounded to bf16, p2 the rest rounded, p3 what is
// left): exactly for 0 and 2^-110 <= |x| < 3.39e38 (above, p1 rounds to infinity).
// Below, p3 ends at bf16's smallest subnormal, 2^-133, which the matrix instructions
// keep: x is held to within 2^-134. So the operands are scaled by powers of two where
// a caller's can be out of that range. A product takes the six piece products of
// weight 2^-16 and more (p1q1, p1q2, p2q1, p1q3, p2q2, p3q1), accumulated in fp32
// by v_mfma_f32_16x16x32_bf16; the three left out add up to less than 2^-24 |x| |y|,
// under the rounding of one fp32 product. Six of these instructions do the work
// of eight v_mfma_f32_16x16x4_f32 in 96 cycles instead of 256.
#pragma once

#include <type_traits>
#include <utility>

#include "lf_common.h"
#include "mix_common.h"

namespace lfamd {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// Two values' leading bf16 pieces (nearest even), packed (x0 in the low half).
__device__ __forceinline__ uint32_t bf16_pair(float x0, float x1) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{x0, x1}, bf16x2));
}

// x0, x1 as three packed pairs of pieces.
__device__ __forceinline__ void split_pair(float x0, float x1, uint32_t (&h)[3]) {
#pragma unroll
  for (int pc = 0; pc < 3; ++pc) {
    h[pc] = bf16_pair(x0, x1);
    if (pc < 2) {
      x0 -= __builtin_bit_cast(float, h[pc] << 16);
      x1 -= __builtin_bit_cast(float, h[pc] & 0xffff0000u);
    }
  }
}

// Four consecutive k of an operand: per piece two packed pairs.
__device__ __forceinline__ void split_quad(const float (&x)[4], uint2 (&h)[3]) {
  uint32_t a[3], b[3];
  split_pair(x[0], x[1], a);
  split_pair(x[2], x[3], b);
#pragma unroll
  for (int pc = 0; pc < 3; ++pc) h[pc] = uint2{a[pc], b[pc]};
}

// The accumulator layout of a 16 x 16 tile D (lane (i, g) = (lane % 16, lane / 16)
// holds D[4g + r][i], r < 4) is half of the B operand of a product over D's rows:
// in the k order k = 32u + 4g + r (r < 4), 32u + 16 + 4g + r, lane (i, g) of the B
// operand Y(32u.., 16 columns) holds Y[k][i], i.e. its own accumulators of tiles 2u
// and 2u + 1. So a product's columns pass into the next product in registers.
// The A operand X (16 rows, 32 k) in the same order: lane (l, g) holds X[l][k].
// quad_transpose turns the pieces of D[4g + r][i] into those of an A operand over
// D's columns: lane (i, g), a = i % 4, q = i / 4, gets D[4g + a][4q + r], r < 4,
// which is lane (l, g') = (4g + a, q) of the operand (half u's low or high).
__device__ __forceinline__ uint2 quad_transpose(uint2 d, int lane) {
  const bool up = lane & 2;
  const uint32_t ox = (uint32_t)__builtin_amdgcn_mov_dpp((int)d.x, 0x4e, 0xf, 0xf, true);  // lane ^ 2
  const uint32_t oy = (uint32_t)__builtin_amdgcn_mov_dpp((int)d.y, 0x4e, 0xf, 0xf, true);
  const uint32_t lo = up ? oy : d.x;   // columns 0/1 of the quad, rows 2A and 2A + 1 (A = a / 2)
  const uint32_t hi = up ? d.y : ox;   // columns 2/3
  const uint32_t nl = (uint32_t)__builtin_amdgcn_mov_dpp((int)lo, 0xb1, 0xf, 0xf, true);  // lane ^ 1
  const uint32_t nh = (uint32_t)__builtin_amdgcn_mov_dpp((int)hi, 0xb1, 0xf, 0xf, true);
  // Even lanes: {own low, neighbour's low}; odd lanes: {neighbour's high, own high}.
  const uint32_t sel = lane & 1 ? 0x03020706u : 0x05040100u;  // bytes 0-3: own, 4-7: neighbour
  return uint2{__builtin_amdgcn_perm(nl, lo, sel), __builtin_amdgcn_perm(nh, hi, sel)};
}

// The forward kernels iterate on P / 2 and 2V, whose products are those of P and V exactly: a
// finite P then never rounds to an infinite first piece. (Small entries need nothing: P has
// 0.01 on its diagonal, and a finite alpha means row sums between 2^-64 and 2^64, so 2^-134 is
// far under the rounding of P and V by norm.)
constexpr float kHalfP = 0.5f;
__device__ __forceinline__ float twice_v0(float alpha, float p) { return 2.0f * (alpha * p); }

template <int NT> struct ChainLayout {
  static constexpr int NP = 16 * NT;
  static constexpr int KS = (NT + 1) / 2;        // 32-k steps
  static constexpr int LS = NP + 4;              // pitch of the staged P (floats)
  static constexpr int OPS = NT * KS * 3 * 64;   // 16-byte words of one matrix's A operands
  static constexpr int LDS = 2 * OPS * 16;
  static_assert(NP * LS <= OPS * 4, "the staged P fits one operand buffer");
};

// NewtonInverse forward of one matrix with 16 (NT - 1) < n <= 16 NT on NT waves, the
// reference's V <- 2V - V(PV). Wave w owns columns 16w .. 16w + 15 of V, T = PV and
// U = VT through the whole iteration, in registers (V in fp32 and as the B operand's
// pieces; T straight from PV's accumulators into VT's B operand). P's A operand
// stays in registers too (every wave all of P); what the waves exchange is V's A
// operand, through two LDS buffers with one barrier per iteration. Bound by the
// matrix instructions and the splitting of T and V between them (their issue slots
// add up on a SIMD unless they alternate in one wave, hence the scheduling groups):
// 1024 x 64^2, 12 iterations, 70.0 us against 101.5 with fp32 matrix instructions,
// 32 x 64^2, 10 iterations, 18.9 against 24.4; 1024 x 32^2 16.4 against 18.9, 1024 x
// 48^2 40 against 54.6. `sm`: LDS bytes. Other waves of a larger workgroup must not
// call this.
template <typename T, int NT>
__device__ __forceinline__ void newton_fwd_chain_body(const T* __restrict__ Mg, T* __restrict__ Og, int n, int iters,
                                                      unsigned char* sm, float* red) {
  using L = ChainLayout<NT>;
  constexpr int NP = L::NP, KS = L::KS, LS = L::LS;
  const int w = uniform(threadIdx.x >> 6), lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  uint4* buf = reinterpret_cast<uint4*>(sm);
  float* Ps = reinterpret_cast<float*>(sm + L::OPS * 16);  // in buffer 1 until V1's operands go there

  // P = f32(mat) + 0.01 I, zero outside n x n.
  constexpr int PER = NP * NP / (64 * NT);
  float pv[PER];
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int e = threadIdx.x + q * 64 * NT, i = e / NP, j = e - i * NP;
    pv[q] = (i < n && j < n) ? to_acc(Mg[i * n + j]) + (i == j ? 0.01f : 0.f) : 0.f;
  }
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int e = threadIdx.x + q * 64 * NT, i = e / NP, j = e - i * NP;
    Ps[i * LS + j] = pv[q];
  }
  __syncthreads();

  // Wave w splits row tile w of P (kept in fp32 for V0 = alpha P below).
  auto op = [&](int b, int t, int u, int pc) { return buf + b * L::OPS + ((t * KS + u) * 3 + pc) * 64; };
  float xr[KS][8];
#pragma unroll
  for (int u = 0; u < KS; ++u)
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      float4 v{0.f, 0.f, 0.f, 0.f};
      if (2 * u + hf < NT) v = *reinterpret_cast<const float4*>(&Ps[(16 * w + li) * LS + 32 * u + 16 * hf + 4 * lg]);
      xr[u][4 * hf] = v.x; xr[u][4 * hf + 1] = v.y; xr[u][4 * hf + 2] = v.z; xr[u][4 * hf + 3] = v.w;
    }
  auto put_rows = [&](auto f) {
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      uint2 h0[3], h1[3];
      const float a[4] = {f(xr[u][0]), f(xr[u][1]), f(xr[u][2]), f(xr[u][3])};
      const float b[4] = {f(xr[u][4]), f(xr[u][5]), f(xr[u][6]), f(xr[u][7])};
      split_quad(a, h0);
      split_quad(b, h1);
#pragma unroll
      for (int pc = 0; pc < 3; ++pc) op(0, w, u, pc)[lane] = uint4{h0[pc].x, h0[pc].y, h1[pc].x, h1[pc].y};
    }
  };
  put_rows([](float p) { return kHalfP * p; });
  // alpha = 1.8 / (max_i sum_j P_ij)^2, row sums in ascending j, one thread per row.
  float row = -1e30f;
  if ((int)threadIdx.x < n) {
    float s = 0.f;
#pragma unroll
    for (int q = 0; q < NP / 4; ++q) {
      const float4 v = *reinterpret_cast<const float4*>(&Ps[threadIdx.x * LS + 4 * q]);
      s = (((s + v.x) + v.y) + v.z) + v.w;
    }
    row = s;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) row = fmaxf(row, __shfl_xor(row, off));
  if (lane == 0) red[w] = row;
  __syncthreads();
  float mx = red[0];
#pragma unroll
  for (int k = 1; k < NT; ++k) mx = fmaxf(mx, red[k]);
  const float alpha = 1.8f / (mx * mx);
  uint4 pa[NT][KS][3];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int u = 0; u < KS; ++u)
#pragma unroll
      for (int pc = 0; pc < 3; ++pc) pa[t][u][pc] = op(0, t, u, pc)[lane];
  float vf[NT][4];
  uint2 vh[2 * KS][3];  // the pieces of tiles 2u, 2u + 1: the B operand of step u
#pragma unroll
  for (int t = 0; t < 2 * KS; ++t) {
    if (t < NT) {
#pragma unroll
      for (int r = 0; r < 4; ++r) vf[t][r] = twice_v0(alpha, Ps[(16 * t + 4 * lg + r) * LS + 16 * w + li]);
      split_quad(vf[t], vh[t]);
    } else {
#pragma unroll
      for (int pc = 0; pc < 3; ++pc) vh[t][pc] = uint2{0u, 0u};
    }
  }
  __syncthreads();  // P's operands are in registers
  put_rows([=](float p) { return twice_v0(alpha, p); });

  // Where this wave's tile (t, w) goes in V's A operand: row tile t, step w / 2,
  // half w % 2, operand lane (4 lg + li % 4, li / 4).
  const int olane = (4 * lg + (li & 3)) + 16 * (li >> 2);
  uint2 th[2 * KS][3];
  v4f ua[2 * KS];  // U's tiles
  // V = 2V - U on tile t, and its pieces (own B operand; V's A operand in buffer b).
  auto update = [&](int t, int b) {
#pragma unroll
    for (int r = 0; r < 4; ++r) vf[t][r] = 2.0f * vf[t][r] - ua[t][r];
    split_quad(vf[t], vh[t]);
#pragma unroll
    for (int pc = 0; pc < 3; ++pc) {
      const uint2 v = quad_transpose(vh[t][pc], lane);
      uint4* d = op(b, t, w >> 1, pc) + olane;
      if (NT % 2 && w == NT - 1)  // no odd neighbour: the step's second half is zero padding
        *d = uint4{v.x, v.y, 0u, 0u};
      else
        reinterpret_cast<uint2*>(d)[w & 1] = v;
    }
  };
  auto yop = [&](const uint2 (&h)[2 * KS][3], int u, uint4 (&y)[3]) {
#pragma unroll
    for (int pc = 0; pc < 3; ++pc) y[pc] = uint4{h[2 * u][pc].x, h[2 * u][pc].y, h[2 * u + 1][pc].x, h[2 * u + 1][pc].y};
  };
  // One step of the products for tiles t0 .. t1 - 1, interleaved over the tiles.
  auto step = [&](auto&& x, const uint4 (&y)[3], v4f (&acc)[2 * KS], int t0, int t1, bool first) {
#pragma unroll
    for (int t = 0; t < 2 * KS; ++t)
#pragma unroll
      for (int s = 2; s >= 0; --s)
#pragma unroll
        for (int i = 0; i <= s; ++i)
          if (t >= t0 && t < t1) {
            const v4f c = first && s == 2 && i == 0 ? v4f{0.f, 0.f, 0.f, 0.f} : acc[t];
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x(t, i)),
                                                             __builtin_bit_cast(bf16x8, y[s - i]), c, 0, 0, 0);
          }
  };
  // Interleaves the region's matrix instructions with its VALU work, n to one.
  auto mix = [&](auto count, auto valu) {
#pragma unroll
    for (int k = 0; k < decltype(count)::value; ++k) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, decltype(valu)::value, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  using std::integral_constant;
  // The last two tiles of an update run beside the next iteration's first products
  // (which read the other tiles only). V = 2V - V gives them their start.
#pragma unroll
  for (int t = 0; t < NT; ++t) ua[t] = v4f{vf[t][0], vf[t][1], vf[t][2], vf[t][3]};
#pragma unroll 1
  for (int it = 0; it < iters; ++it) {
    const int cur = it & 1;
    uint4 y[3];
    v4f ta[2 * KS];
    auto px = [&](int t, int i, int u) { return pa[t < NT ? t : 0][u][i]; };
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (KS == 2) {
      // T = P V
      yop(vh, 0, y);
      step([&](int t, int i) { return px(t, i, 0); }, y, ta, 0, NT, true);
#pragma unroll
      for (int t = 2; t < NT; ++t) update(t, cur);
      mix(integral_constant<int, 6 * NT>{}, integral_constant<int, 4>{});
      yop(vh, 1, y);
      step([&](int t, int i) { return px(t, i, 1); }, y, ta, 0, 2, false);
      step([&](int t, int i) { return px(t, i, 1); }, y, ta, 2, NT, false);
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const float a[4] = {ta[t][0], ta[t][1], ta[t][2], ta[t][3]};
        split_quad(a, th[t]);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 12, 0);
#pragma unroll
      for (int k = 0; k < 6 * (NT - 2); ++k) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
      }
      __syncthreads();  // V's operands are complete; the other buffer is free
      __builtin_amdgcn_sched_barrier(0);
      // U = V T
      uint4 x[NT][3];
      auto fetch = [&](int u) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int pc = 0; pc < 3; ++pc) x[t][pc] = op(cur, t, u, pc)[lane];
      };
      auto vx = [&](int t, int i) { return x[t < NT ? t : 0][i]; };
      fetch(0);
      yop(th, 0, y);
      step(vx, y, ua, 0, NT, true);
#pragma unroll
      for (int t = 2; t < 4; ++t) {
        float a[4] = {0.f, 0.f, 0.f, 0.f};
        if (t < NT)
#pragma unroll
          for (int r = 0; r < 4; ++r) a[r] = ta[t][r];
        split_quad(a, th[t]);
      }
      fetch(1);
      mix(integral_constant<int, 6 * NT>{}, integral_constant<int, 3>{});
      yop(th, 1, y);
      step(vx, y, ua, 0, 2, false);
      step(vx, y, ua, 2, NT, false);
      update(0, cur ^ 1);
      update(1, cur ^ 1);
      __builtin_amdgcn_sched_group_barrier(0x008, 12, 0);
      mix(integral_constant<int, 6 * (NT - 2)>{}, integral_constant<int, 8>{});
    } else {
      yop(vh, 0, y);
      step([&](int t, int i) { return px(t, i, 0); }, y, ta, 0, NT, true);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const float a[4] = {ta[t][0], ta[t][1], ta[t][2], ta[t][3]};
        split_quad(a, th[t]);
      }
      __syncthreads();
      uint4 x[NT][3];
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int pc = 0; pc < 3; ++pc) x[t][pc] = op(cur, t, 0, pc)[lane];
      yop(th, 0, y);
      step([&](int t, int i) { return x[t < NT ? t : 0][i]; }, y, ua, 0, NT, true);
#pragma unroll
      for (int t = 0; t < NT; ++t) update(t, cur ^ 1);
    }
  }
  if constexpr (KS == 2)
#pragma unroll
    for (int t = 2; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) vf[t][r] = 2.0f * vf[t][r] - ua[t][r];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 16 * t + 4 * lg + r, j = 16 * w + li;
      if (i < n && j < n) Og[i * n + j] = from_acc<T>(kHalfP * vf[t][r]);
    }
}


// ---------------------------------------------------------------------------
// 32 x 32 tiles (v_mfma_f32_32x32x16_bf16: 32 cycles, of which an in-order wave
// can fill 28 with other instructions; the 16 x 16 x 32 form takes 20 and leaves
// little of them). Lane (i, h) = (lane % 32, lane / 32) holds D[8(r/4) + 4h + r%4][i],
// r < 16, of a tile. In the k order of its registers a tile is the B operand of two
// 16-k steps (registers 0-7 and 8-15): step s's dword 2 c3 + c1 of lane (i, h) holds
// k = 16s + 8 c3 + 4h + 2 c1 and k + 1. An A operand's lane (l, h) holds X[l][k] at
// the same k; it is stored at slot (l ^ (2h + 8 (s % 2))) + 32h of its 64 16-byte
// slots, so that the transposing 4-byte writes of store_rows fall on 64 banks.
// ---------------------------------------------------------------------------
typedef float v16f __attribute__((ext_vector_type(16)));

__device__ __forceinline__ int op_slot(int lane, int s) {
  const int l = lane & 31, h = lane >> 5;
  return (l ^ (2 * h + 8 * (s & 1))) + 32 * h;
}

// Registers r0 .. r0 + 7 of a tile as the pieces of one step's operand. Piece by
// piece over all eight values: a VALU result is ready after two issue slots, so a
// pair's own chain of six would run at half rate.
__device__ __forceinline__ void split8r(const float (&x)[8], uint4 (&h)[3]) {
  float y[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) y[e] = x[e];
#pragma unroll
  for (int pc = 0; pc < 3; ++pc) {
    uint32_t d[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) d[e] = bf16_pair(y[2 * e], y[2 * e + 1]);
    h[pc] = uint4{d[0], d[1], d[2], d[3]};
    if (pc == 2) break;
    float lo[4], hi[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) lo[e] = __builtin_bit_cast(float, d[e] << 16);
#pragma unroll
    for (int e = 0; e < 4; ++e) hi[e] = __builtin_bit_cast(float, d[e] & 0xffff0000u);
#pragma unroll
    for (int e = 0; e < 4; ++e) y[2 * e] -= lo[e];
#pragma unroll
    for (int e = 0; e < 4; ++e) y[2 * e + 1] -= hi[e];
  }
}

__device__ __forceinline__ v16f mfma_split32(const uint4 (&x)[3], const uint4 (&y)[3], v16f acc) {
#pragma unroll
  for (int s = 2; s >= 0; --s)
#pragma unroll
    for (int i = 0; i <= s; ++i)
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, x[i]),
                                                    __builtin_bit_cast(bf16x8, y[s - i]), acc, 0, 0, 0);
  return acc;
}

// Writes tile pieces (steps e = 0, 1 of the B operand) transposed into the A operand
// of row tile t (base of its first block `ops`, KS steps of 3 pieces) at this wave's
// columns 32w .. 32w + 31 (steps 2w, 2w + 1).
struct RowStore {
  uint32_t sel;
  int off[2][2];  // [b & 1][row pair j] byte offsets
  __device__ __forceinline__ RowStore(int w, int lane) {
    const int c0 = lane & 1, c1 = (lane >> 1) & 1, c2 = (lane >> 2) & 1, c3 = (lane >> 3) & 1, c4 = (lane >> 4) & 1;
    const int h = lane >> 5;
    sel = c0 ? 0x03020706u : 0x05040100u;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        off[b][j] = ((2 * w + c4) * 3 * 64 + 8 * (b ^ c4) + 4 * h + 2 * (j ^ c2) + c0 + 32 * c2) * 16 + 4 * (2 * c3 + c1);
  }
  // One of six stages (step e, piece pc) of storing a tile.
  __device__ __forceinline__ void stage(int k, unsigned char* ops, const uint4 (&hh)[2][3]) const {
    const int e = k / 3, pc = k % 3;
    const uint32_t d[4] = {hh[e][pc].x, hh[e][pc].y, hh[e][pc].z, hh[e][pc].w};
    uint32_t n[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) n[q] = (uint32_t)__builtin_amdgcn_mov_dpp((int)d[q], 0xb1, 0xf, 0xf, true);  // lane ^ 1
#pragma unroll
    for (int q = 0; q < 4; ++q)  // rows 8 (2e + q / 2) + 4h + 2 (q % 2) + {0, 1}
      *reinterpret_cast<uint32_t*>(ops + off[q >> 1][q & 1] + 256 * e + 1024 * pc) = __builtin_amdgcn_perm(n[q], d[q], sel);
  }
};

struct TileLayout {
  static constexpr int NR = 2, KS = 4, NP = 64;
  static constexpr int LS = NP + 4;
  static constexpr int OPS = NR * KS * 3 * 1024;  // bytes of one matrix's A operands
  static constexpr int PS = NP * LS * 4;          // bytes of the staged fp32 P
  static constexpr int LDS = OPS > PS ? OPS : PS;
};

// NewtonInverse forward for 48 < n <= 64 on two waves of 32 columns each, for batches
// that fill the chip. A workgroup is two matrices (a wave on each SIMD:
// two-wave workgroups were placed on the same two SIMDs, 5460 against 4290 cycles
// per iteration at two matrices per CU), and with two workgroups per CU one wave's
// barriers run under another's products. P's A operand stays in registers, V's in
// one LDS buffer. The matrix cores bound it: they are busy 97 % of an iteration at
// four matrices per CU, at the 1.7-1.9 GHz that the chip then runs (1024 x 64^2, 12
// iterations: 59.5 us, against 70.0 on newton_fwd_chain_body).
template <typename T>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
newton_fwd_tile_kernel(const T* __restrict__ mat, T* __restrict__ out, int64_t bh, int n, int iters) {
  using L = TileLayout;
  constexpr int NR = L::NR, KS = L::KS, NP = L::NP, LS = L::LS;
  extern __shared__ __align__(16) unsigned char tile_all[];
  const int wv = uniform(threadIdx.x >> 6), w = wv % NR, lane = threadIdx.x & 63, li = lane & 31, lh = lane >> 5;
  unsigned char* tile_sm = tile_all + (wv / NR) * L::LDS;
  float* Ps = reinterpret_cast<float*>(tile_sm);
  // (An odd batch's last workgroup computes its matrix twice and stores it once.)
  const int64_t m0 = (int64_t)blockIdx.x * 2 + wv / NR;
  const int64_t m = m0 < bh ? m0 : bh - 1;
  const T* Mg = mat + (size_t)m * n * n;
  T* Og = out + (size_t)m * n * n;
  const int tid = threadIdx.x & (64 * NR - 1);
  if (std::is_same<T, float>::value && n == NP && (reinterpret_cast<uintptr_t>(mat) & 15) == 0) {
    constexpr int PER = NP * NP / 4 / (64 * NR);
    float4 v[PER];
#pragma unroll
    for (int q = 0; q < PER; ++q) v[q] = reinterpret_cast<const float4*>(Mg)[tid + 64 * NR * q];
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int e = tid + 64 * NR * q, i = e / (NP / 4), j = 4 * (e % (NP / 4));
      if (i - j == 0) v[q].x += 0.01f;
      if (i - j == 1) v[q].y += 0.01f;
      if (i - j == 2) v[q].z += 0.01f;
      if (i - j == 3) v[q].w += 0.01f;
      *reinterpret_cast<float4*>(&Ps[i * LS + j]) = v[q];
    }
  } else {
#pragma unroll 16
    for (int e = tid; e < NP * NP; e += 64 * NR) {
      const int i = e / NP, j = e - i * NP;
      Ps[i * LS + j] = (i < n && j < n) ? to_acc(Mg[i * n + j]) + (i == j ? 0.01f : 0.f) : 0.f;
    }
  }
  __syncthreads();
  uint4 pa[NR][KS][3];
#pragma unroll
  for (int t = 0; t < NR; ++t)
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const float4 a = *reinterpret_cast<const float4*>(&Ps[(32 * t + li) * LS + 16 * s + 4 * lh]);
      const float4 b = *reinterpret_cast<const float4*>(&Ps[(32 * t + li) * LS + 16 * s + 8 + 4 * lh]);
      const float x[8] = {kHalfP * a.x, kHalfP * a.y, kHalfP * a.z, kHalfP * a.w,
                          kHalfP * b.x, kHalfP * b.y, kHalfP * b.z, kHalfP * b.w};
      split8r(x, pa[t][s]);
    }
  // alpha: every wave forms all rows' sums (ascending j, one lane per row).
  float mx = -1e30f;
#pragma unroll
  for (int t = 0; t < NR; t += 2) {
    float sum = 0.f;
#pragma unroll
    for (int q = 0; q < NP / 4; ++q) {
      const float4 v = *reinterpret_cast<const float4*>(&Ps[(32 * t + lane) * LS + 4 * q]);
      sum = (((sum + v.x) + v.y) + v.z) + v.w;
    }
    if (32 * t + lane < n) mx = fmaxf(mx, sum);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
  const float alpha = 1.8f / (mx * mx);
  float vf[NR][16];
  v16f ua[NR];
#pragma unroll
  for (int t = 0; t < NR; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      vf[t][r] = twice_v0(alpha, Ps[(32 * t + 8 * (r >> 2) + 4 * lh + (r & 3)) * LS + 32 * w + li]);
      ua[t][r] = vf[t][r];  // the first update: V = 2V - V
    }
  __syncthreads();
  const RowStore rs(w, lane);
  const int slot[2] = {op_slot(lane, 0) * 16, op_slot(lane, 1) * 16};
  uint4 vh[NR][2][3], th[NR][2][3];
  auto ops = [&](int t) { return tile_sm + t * KS * 3 * 1024; };
  auto store = [&](int t) {
#pragma unroll
    for (int k = 0; k < 6; ++k) rs.stage(k, ops(t), vh[t]);
  };
  auto split_tile = [&](const auto& a, uint4 (&h)[2][3]) {
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const float x[8] = {a[8 * e], a[8 * e + 1], a[8 * e + 2], a[8 * e + 3],
                          a[8 * e + 4], a[8 * e + 5], a[8 * e + 6], a[8 * e + 7]};
      split8r(x, h[e]);
    }
  };
  auto update = [&](int t) {
#pragma unroll
    for (int r = 0; r < 16; ++r) vf[t][r] = 2.0f * vf[t][r] - ua[t][r];
    split_tile(vf[t], vh[t]);
  };
  const v16f zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  // Row tile t of P V or V T over the steps of k tile kt.
  auto pv = [&](v16f& acc, int t, int kt) {
#pragma unroll
    for (int s = 2 * kt; s < 2 * kt + 2; ++s) acc = mfma_split32(pa[t][s], vh[kt][s & 1], acc);
  };
  auto vt = [&](v16f& acc, int t, int kt) {
#pragma unroll
    for (int s = 2 * kt; s < 2 * kt + 2; ++s) {
      uint4 x[3];
#pragma unroll
      for (int pc = 0; pc < 3; ++pc)
        x[pc] = *reinterpret_cast<const uint4*>(ops(t) + (s * 3 + pc) * 1024 + slot[s & 1]);
      acc = mfma_split32(x, th[kt][s & 1], acc);
    }
  };
  // A SIMD does not fill one wave's back-to-back matrix instructions with another's
  // VALU work: each region's splitting goes between its products, VALU per MFMA.
  auto mix = [&](auto mfmas, auto valu) {
#pragma unroll
    for (int k = 0; k < decltype(mfmas)::value; ++k) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, decltype(valu)::value, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  using std::integral_constant;
  update(0);
#pragma unroll 1
  for (int it = 0; it < iters; ++it) {
    v16f ta[2] = {zero, zero};
    __builtin_amdgcn_sched_barrier(0);
    pv(ta[0], 0, 0);  // T = P V
    pv(ta[1], 1, 0);
    store(0);
    update(1);
    mix(integral_constant<int, 24>{}, integral_constant<int, 7>{});
    pv(ta[0], 0, 1);
    store(1);
    mix(integral_constant<int, 12>{}, integral_constant<int, 5>{});
    pv(ta[1], 1, 1);
    split_tile(ta[0], th[0]);
    mix(integral_constant<int, 12>{}, integral_constant<int, 8>{});
    __syncthreads();  // V's operands are complete
    ua[0] = zero;
    ua[1] = zero;
    vt(ua[0], 0, 0);  // U = V T
    vt(ua[1], 1, 0);
    split_tile(ta[1], th[1]);
    mix(integral_constant<int, 24>{}, integral_constant<int, 4>{});
    vt(ua[0], 0, 1);
    __builtin_amdgcn_sched_barrier(0);
    vt(ua[1], 1, 1);
    update(0);
    mix(integral_constant<int, 12>{}, integral_constant<int, 9>{});
    __syncthreads();  // and read
  }
  // (tile 0's last update is done)
#pragma unroll
  for (int r = 0; r < 16; ++r) ua[0][r] = vf[0][r];
#pragma unroll
  for (int t = 0; t < NR; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int i = 32 * t + 8 * (r >> 2) + 4 * lh + (r & 3), j = 32 * w + li;
      if (i < n && j < n && m0 < bh) Og[i * n + j] = from_acc<T>(kHalfP * (2.0f * vf[t][r] - ua[t][r]));
    }
}


// Product j (0 .. 5) of one step's piece products, smallest first.
__device__ __forceinline__ v16f mfma_piece(const uint4 (&x)[3], const uint4 (&y)[3], int j, bool first, v16f acc) {
  constexpr int xi[6] = {0, 1, 2, 0, 1, 0}, yi[6] = {2, 1, 0, 1, 0, 0};
  const v16f zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, x[xi[j]]),
                                                 __builtin_bit_cast(bf16x8, y[yi[j]]), first ? zero : acc, 0, 0, 0);
}

// A tile's 16 registers split into the two steps' pieces in 16 stages of four to six
// VALU instructions, to be issued between matrix instructions: four stages for each
// four registers.
struct SplitTask {
  float y[4], z[4];
  static __device__ __forceinline__ void open(const uint4& h, int c, float (&z)[4]) {
    const uint32_t d0 = c == 0 ? h.x : h.z, d1 = c == 0 ? h.y : h.w;
    z[0] = __builtin_bit_cast(float, d0 << 16);
    z[1] = __builtin_bit_cast(float, d0 & 0xffff0000u);
    z[2] = __builtin_bit_cast(float, d1 << 16);
    z[3] = __builtin_bit_cast(float, d1 & 0xffff0000u);
  }
  template <typename A> static __device__ __forceinline__ float at(const A& a, int r) {
    if constexpr (std::is_invocable_v<A, int>) return a(r);
    else return a[r];
  }
  // V's four values of registers 4q .. 4q + 3 back from their pieces (exactly: the sum
  // of the last two is V less the first), in two stages.
  __device__ __forceinline__ void rebuild(int k, int q, const uint4 (&h)[2][3]) {
    const int e = q / 2, c = q % 2;
    if (k == 0) {
      open(h[e][2], c, y);
      open(h[e][1], c, z);
    } else {
      open(h[e][0], c, z);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] += z[i];
  }
  template <typename A> __device__ __forceinline__ void stage(int k, const A& a, uint4 (&h)[2][3]) {
    const int q = k / 4, e = q / 2, c = q % 2;  // registers 4q .. 4q + 3: dwords 2c, 2c + 1 of step e
    auto put = [&](int pc) {
      const uint32_t d0 = bf16_pair(y[0], y[1]), d1 = bf16_pair(y[2], y[3]);
      if (c == 0) {
        h[e][pc].x = d0;
        h[e][pc].y = d1;
      } else {
        h[e][pc].z = d0;
        h[e][pc].w = d1;
      }
    };
    if (k % 4 == 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) y[i] = at(a, 4 * q + i);
      put(0);
    } else if (k % 4 == 1) {
      open(h[e][0], c, z);
#pragma unroll
      for (int i = 0; i < 4; ++i) y[i] -= z[i];
    } else if (k % 4 == 2) {
      put(1);
      open(h[e][1], c, z);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) y[i] -= z[i];
      put(2);
    }
  }
};

template <int NR, int KS> struct WideLayout {
  static constexpr int NP = 32 * NR;
  static constexpr int LS = NP + 4;
  static constexpr int VSTEP = 2 * NR;                // steps stored per row tile (the update writes whole tiles)
  static constexpr int VOPS = NR * VSTEP * 3 * 1024;  // V's A operand (the staged fp32 P before it)
  static constexpr int POPS = NR * KS * 2 * 1024;     // P's first two pieces
  // Steps whose third piece is in LDS too, as far as 160 KB go (the others': registers).
  static constexpr int ROOM = (160 * 1024 - VOPS - POPS) / 1024;
  static constexpr int P3 = ROOM < NR * KS ? ROOM : NR * KS;
  static constexpr int LDS = VOPS + POPS + P3 * 1024;
  static_assert(NP * LS * 4 <= VOPS, "the staged P fits V's operand");
};

// NewtonInverse forward for 32 (NR - 1) < n <= 32 NR, 16 (KS - 1) < n <= 16 KS,
// NR = 3 or 4: one workgroup of NR waves per matrix and CU, wave w owning columns
// 32w .. 32w + 31 as in newton_fwd_tile_kernel. V's A operand is in LDS, with P's
// first two pieces and what fits of its third; the rest of that is in registers.
// Everything but the products is cut into stages that go between the matrix
// instructions, since each SIMD has one wave: beside the products of row tile t run
// the split of T's tile t - 1 (or V's update) and the storing of V's tile t. 512 x 100^2, 10 iterations: 168 us against 272 with fp32
// matrix instructions, 64 x 100^2 82 against 130, 1024 x 128^2, 12 iterations, 647
// against 997 (NR = 4 spills P's third pieces, 38 registers at KS = 7, the n = 100 above
// among them, and 185 at KS = 8: 384 are allowed, 256 and 128 accumulation ones).
template <typename T, int NR, int KS>
__global__ void __launch_bounds__(64 * NR) __attribute__((amdgpu_waves_per_eu(1, 1), amdgpu_num_vgpr(192)))
newton_fwd_wide_kernel(const T* __restrict__ mat, T* __restrict__ out, int n, int iters) {
  using L = WideLayout<NR, KS>;
  constexpr int NP = L::NP, LS = L::LS;
  extern __shared__ __align__(16) unsigned char wide_sm[];
  float* Ps = reinterpret_cast<float*>(wide_sm);
  const int w = uniform(threadIdx.x >> 6), lane = threadIdx.x & 63, li = lane & 31, lh = lane >> 5;
  const T* Mg = mat + (size_t)blockIdx.x * n * n;
  T* Og = out + (size_t)blockIdx.x * n * n;
  {
    // Row i by wave i mod NR, a column (of 64) per lane; every load in flight before the first store.
    constexpr int RW = NP / NR, CW = (NP + 63) / 64;
    T v[RW][CW];
#pragma unroll
    for (int q = 0; q < RW; ++q)
#pragma unroll
      for (int c = 0; c < CW; ++c) {
        const int i = NR * q + w, j = 64 * c + lane;
        v[q][c] = Mg[(i < n ? i : n - 1) * n + (j < n ? j : n - 1)];
      }
#pragma unroll
    for (int q = 0; q < RW; ++q)
#pragma unroll
      for (int c = 0; c < CW; ++c) {
        const int i = NR * q + w, j = 64 * c + lane;
        const float p = to_acc(v[q][c]) + (i == j ? 0.01f : 0.f);
        if (NP % 64 == 0 || j < NP) Ps[i * LS + j] = i < n && j < n ? p : 0.f;
      }
  }
  __syncthreads();
  // alpha: every wave forms all rows' sums (ascending j, one lane per row).
  float mx = -1e30f;
#pragma unroll 1
  for (int t = 0; t < NP; t += 64) {
    const int row = t + lane;
    float sum = 0.f;
#pragma unroll 8
    for (int q = 0; q < NP / 4; ++q) {
      const float4 v = *reinterpret_cast<const float4*>(&Ps[(row < NP ? row : NP - 1) * LS + 4 * q]);
      sum = (((sum + v.x) + v.y) + v.z) + v.w;
    }
    if (row < n) mx = fmaxf(mx, sum);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
  const float alpha = 1.8f / (mx * mx);

  const int slot[2] = {op_slot(lane, 0) * 16, op_slot(lane, 1) * 16};
  auto pop = [&](int t, int s, int pc) { return wide_sm + L::VOPS + ((t * KS + s) * 2 + pc) * 1024 + slot[s & 1]; };
  auto pop3 = [&](int i) { return wide_sm + L::VOPS + L::POPS + i * 1024 + slot[i % KS & 1]; };
  auto vop = [&](int t, int s, int pc) { return wide_sm + ((t * L::VSTEP + s) * 3 + pc) * 1024 + slot[s & 1]; };
  // P's pieces: every wave splits all of P for the third ones it keeps, wave w stores row tile w.
  constexpr int NREG = NR * KS - L::P3;
  uint4 p3[NREG > 0 ? NREG : 1];
#pragma unroll
  for (int i = 0; i < NR * KS; ++i) {
    const int t = i / KS, s = i % KS;
    const float4 a = *reinterpret_cast<const float4*>(&Ps[(32 * t + li) * LS + 16 * s + 4 * lh]);
    const float4 b = *reinterpret_cast<const float4*>(&Ps[(32 * t + li) * LS + 16 * s + 8 + 4 * lh]);
    const float x[8] = {kHalfP * a.x, kHalfP * a.y, kHalfP * a.z, kHalfP * a.w,
                        kHalfP * b.x, kHalfP * b.y, kHalfP * b.z, kHalfP * b.w};
    uint4 h[3];
    split8r(x, h);
    if (i >= L::P3) p3[i >= L::P3 ? i - L::P3 : 0] = h[2];
    if (t == w) {
      *reinterpret_cast<uint4*>(pop(t, s, 0)) = h[0];
      *reinterpret_cast<uint4*>(pop(t, s, 1)) = h[1];
      if (i < L::P3) *reinterpret_cast<uint4*>(pop3(i)) = h[2];
    }
  }
  // V itself is held in its pieces alone (their sum is exact): the B operand vh.
  uint4 vh[NR][2][3], th[NR][2][3];
  v16f acc[2];  // row tile t's sums in acc[t % 2]
  SplitTask sp;
#pragma unroll
  for (int t = 0; t < NR; ++t) {
    float v0[16];
#pragma unroll
    for (int r = 0; r < 16; ++r)
      v0[r] = twice_v0(alpha, Ps[(32 * t + 8 * (r >> 2) + 4 * lh + (r & 3)) * LS + 32 * w + li]);
#pragma unroll
    for (int k = 0; k < 16; ++k) sp.stage(k, v0, vh[t]);
    if (t == NR - 1)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[t & 1][r] = v0[r];  // the first update: V = 2V - V
  }
  __syncthreads();
  const RowStore rs(w, lane);
  auto fence = [] { __builtin_amdgcn_sched_barrier(0); };
  // V = 2V - U on tile t and its pieces, in 24 stages.
  float u4[4];
  auto update = [&](int k, int t) {
    const int q = k / 6, p = k % 6;
    if (p < 2) {
      sp.rebuild(p, q, vh[t]);
    } else {
      if (p == 2)
#pragma unroll
        for (int i = 0; i < 4; ++i) u4[i] = 2.0f * sp.y[i] - acc[t & 1][4 * q + i];
      sp.stage(4 * q + p - 2, [&](int r) { return u4[r & 3]; }, vh[t]);
    }
  };
  constexpr int M0 = 12 * (NR - 1);  // products of a row tile before its last k tile
  constexpr int MT = 6 * KS;         // products of a row tile
  static_assert(M0 >= 24 && MT >= 27, "the stages fit beside the products");
#pragma unroll 1
  for (int it = 0; it < iters; ++it) {
    uint4 x[2][3];
    // T = P V
    unrolled<NR>([&](auto tc) {
      constexpr int t = decltype(tc)::value;
      // Tile 0 must not use the accumulator that the last update reads.
      constexpr int b = NR % 2 ? (t & 1) ^ 1 : t & 1;
      auto load = [&](int s) {
#pragma unroll
        for (int pc = 0; pc < 2; ++pc) x[s & 1][pc] = *reinterpret_cast<const uint4*>(pop(t, s, pc));
        const int i = t * KS + s;
        x[s & 1][2] = i < L::P3 ? *reinterpret_cast<const uint4*>(pop3(i)) : p3[i < L::P3 ? 0 : i - L::P3];
      };
      load(0);
      unrolled<MT>([&](auto mc) {
        constexpr int m = decltype(mc)::value, s = m / 6;
        if constexpr (m % 6 == 0) {
          if constexpr (s + 1 < KS) load(s + 1);
          fence();
        }
        acc[b] = mfma_piece(x[s & 1], vh[s >> 1][s & 1], m % 6, m == 0, acc[b]);
        if constexpr (t == 0) {
          if constexpr (m < 24) update(m, NR - 1);
          if constexpr (m >= M0 - 6 && m < M0) rs.stage(m - (M0 - 6), wide_sm, vh[0]);
        } else {
          if constexpr (m >= 3 && m < 19) sp.stage(m - 3, acc[b ^ 1], th[t - 1]);
          if constexpr (m >= 19 && m < 25) rs.stage(m - 19, wide_sm + t * L::VSTEP * 3 * 1024, vh[t]);
        }
        fence();
      });
    });
    __syncthreads();  // V's operand is complete
    // U = V T, V = 2V - U
    unrolled<NR>([&](auto tc) {
      constexpr int t = decltype(tc)::value, b = t & 1;
      auto load = [&](int s) {
#pragma unroll
        for (int pc = 0; pc < 3; ++pc) x[s & 1][pc] = *reinterpret_cast<const uint4*>(vop(t, s, pc));
      };
      load(0);
      unrolled<MT>([&](auto mc) {
        constexpr int m = decltype(mc)::value, s = m / 6;
        if constexpr (m % 6 == 0) {
          if constexpr (s + 1 < KS) load(s + 1);
          fence();
        }
        // (T's last tile is in acc[1]: see above.)
        acc[b] = mfma_piece(x[s & 1], th[s >> 1][s & 1], m % 6, m == 0, acc[b]);
        if constexpr (t == 0) {
          if constexpr (m >= 3 && m < 19) sp.stage(m - 3, acc[1], th[NR - 1]);
        } else if constexpr (m >= 3 && m < 27) {
          update(m - 3, t - 1);
        }
        fence();
      });
    });
    __syncthreads();  // V's operand is read
  }
#pragma unroll
  for (int t = 0; t < NR; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      if (r % 4 == 0) {
        sp.rebuild(0, r / 4, vh[t]);
        sp.rebuild(1, r / 4, vh[t]);
      }
      // (The last tile's last update is still to be done.)
      const float v = t == NR - 1 ? 2.0f * sp.y[r % 4] - acc[t & 1][r] : sp.y[r % 4];
      const int i = 32 * t + 8 * (r >> 2) + 4 * lh + (r & 3), j = 32 * w + li;
      if (i < n && j < n) Og[i * n + j] = from_acc<T>(kHalfP * v);
    }
}


// ---------------------------------------------------------------------------
// Batched D = f(op(X) op(Y)) over NP x NP fp32 matrices (row-major, matrix stride
// NP * NP), op = transpose when TX / TY, on bf16 pieces. MODE 0: D = XY; 1: D = 2E - XY;
// 2: D = -XY. SCALED multiplies the result by the matrix's alpha (from the init
// kernel's row sums). One TM x TN output tile per workgroup of 2 x 2 waves. Grid: tiles
// x matrices, flattened so that all tiles of a matrix share blockIdx.x mod 8 (workgroups
// are dealt to the 8 XCDs round robin, so a matrix's tiles share one L2).
//
// The backward's operands (TX: S = V^T G, TY: -S V^T) are a caller's tensors of any
// magnitude. Its workgroups follow the largest entry of both panels while staging them;
// where one is outside [2^-86, 2^126), out of the pieces' range or near its lower end, they run
// again with the panels scaled by powers of two to [1, 2) and take the exponents back at
// the store. 128 x 256^2: 70.4 us for both products against 69.3 without the check (scaling
// every operand behind a pass for the maxima: 79).
//
// Both operands are staged 32 k at a time, split on the way into their pieces in MFMA
// operand order (two buffers, one barrier per 32 k, global loads two stages ahead):
// each element is split once per tile that reads it, 4 VALU instructions to an MFMA,
// and the stages of that go between the matrix instructions.
//
// Staging by rows (op(X)[i][k] with k contiguous): a lane has four k of one row.
// By columns (k strided): a lane has four k of JB = T / 32 neighbouring rows or
// columns of the operand. Either way four k of one row are 8 bytes of an operand slot;
// the slot of row l is permuted so that a half wave's 32 writes fall on 64 banks.
// ---------------------------------------------------------------------------
constexpr int kGmK = 32;  // k per stage

// Slot (of 64 16-byte ones) of row l, half h of step s in row tile `tile`.
template <int T, bool COLS> __device__ __forceinline__ int gm_slot(int l, int h, int s, int tile) {
  if constexpr (!COLS) return (l ^ (4 * h + 8 * s)) + 32 * h;
  else if constexpr (T == 128) return (((l & 3) * 8 + (l >> 2)) ^ (8 * (tile & 1))) + 32 * h;
  else return ((l & 1) * 16 + (l >> 1)) + 32 * h;
}

// One operand's staging of a workgroup: T rows (or columns) x 32 k per stage.
template <int T, bool COLS> struct GmStage {
  static constexpr int Q = T / 32;  // quads (four k of one row) per thread
  using Regs = float4[COLS ? 4 : Q];  // COLS: row k of the quad, Q columns (x, y for T = 64)
  int goff, loff[Q];
  __device__ __forceinline__ GmStage(int tid, int NP) {
    const int w = tid >> 6, lane = tid & 63;
    if constexpr (!COLS) {
      const int f = tid & 7, row = tid >> 3;  // 32 rows a pass
      goff = row * NP + 4 * f;
      const int s = f >> 2, c3 = (f >> 1) & 1, h = f & 1;
#pragma unroll
      for (int q = 0; q < Q; ++q) loff[q] = (q * 2 + s) * 3072 + gm_slot<T, COLS>(row, h, s, q) * 16 + 8 * c3;
    } else {
      const int jq = (lane & 15) + 16 * (w & 1), c3 = (lane >> 4) & 1, h = lane >> 5, s = w >> 1;
      goff = (16 * s + 8 * c3 + 4 * h) * NP + Q * jq;
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int j = Q * jq + q;
        loff[q] = ((j >> 5) * 2 + s) * 3072 + gm_slot<T, COLS>(j & 31, h, s, j >> 5) * 16 + 8 * c3;
      }
    }
  }
  // Stage k0 of the operand whose rows (COLS: columns) start at `base`.
  __device__ __forceinline__ void load(Regs& r, const float* __restrict__ base, int NP, int k0) const {
    if constexpr (!COLS) {
#pragma unroll
      for (int q = 0; q < Q; ++q) r[q] = *reinterpret_cast<const float4*>(base + (unsigned)(goff + 32 * q * NP + k0));
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float* p = base + (unsigned)(goff + (k0 + k) * NP);
        if constexpr (Q == 4) {
          r[k] = *reinterpret_cast<const float4*>(p);
        } else {
          const float2 v = *reinterpret_cast<const float2*>(p);
          r[k].x = v.x;
          r[k].y = v.y;
        }
      }
    }
  }
  static __device__ __forceinline__ float at(const Regs& r, int q, int k) {
    if constexpr (!COLS) return k == 0 ? r[q].x : k == 1 ? r[q].y : k == 2 ? r[q].z : r[q].w;
    else return q == 0 ? r[k].x : q == 1 ? r[k].y : q == 2 ? r[k].z : r[k].w;
  }
};

// max(m, |a|, |b|) in one instruction (fmaxf would first quiet what was loaded).
__device__ __forceinline__ float max3_abs(float m, float a, float b) {
  float r;
  asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(r) : "v"(m), "v"(a), "v"(b));
  return r;
}

template <int TM, int TN> constexpr int gm_lds() { return 2 * (TM + TN) * kGmK * 3 * 2; }

template <int TM, int TN, bool TX, bool TY, int MODE, bool SCALED>
__global__ void __launch_bounds__(256)
newton_gemm_kernel(const float* __restrict__ X, const float* __restrict__ Y, const float* __restrict__ E,
                   const float* __restrict__ rowsum, float* __restrict__ D, int NP, int K, int nMat) {
  constexpr int RT = TM / 64, CT = TN / 64;  // 32 x 32 tiles per wave
  extern __shared__ __align__(16) unsigned char gm_sm[];
  constexpr int ABYTES = TM * kGmK * 6, BUF = (TM + TN) * kGmK * 6;
  const int ntm = NP / TM, ntn = NP / TN, tiles = ntm * ntn;
  const int id = blockIdx.x, hi = id >> 3;  // id = (m % 8) + 8 (t + tiles (m / 8))
  const int t = hi % tiles, m = hi / tiles * 8 + (id & 7);
  if (m >= nMat) return;  // whole workgroup
  const int ti = t / ntn, tj = t - ti * ntn;
  const size_t mo = (size_t)m * NP * NP;
  const int tid = threadIdx.x, wave = uniform(tid >> 6), lane = tid & 63, li = lane & 31, lh = lane >> 5;
  const int wr = wave >> 1, wc = wave & 1;
  GmStage<TM, TX> sa(tid, NP);
  GmStage<TN, !TY> sb(tid, NP);
  const float* Xb = X + mo + (TX ? (size_t)ti * TM : (size_t)ti * TM * NP);
  const float* Yb = Y + mo + (TY ? (size_t)tj * TN * NP : (size_t)tj * TN);
  struct Set {
    typename GmStage<TM, TX>::Regs a;
    typename GmStage<TN, !TY>::Regs b;
  } rg;
  auto gload = [&](Set& r, int kc) {
    sa.load(r.a, Xb, NP, kc * kGmK);
    sb.load(r.b, Yb, NP, kc * kGmK);
  };
  constexpr bool RANGE = TX || TY;
  __shared__ int pflag[RANGE ? 4 : 1];
  float scaleA = 1.0f, scaleB = 1.0f, maxA = 0.f, maxB = 0.f;  // of the panels
  int expo = 0;
  // Quad q (A's, then B's) of the staged registers, in four stages, the last one stored to buffer
  // b; scaled or, at first, followed for the largest entries.
  constexpr int QA = GmStage<TM, TX>::Q, QB = GmStage<TN, !TY>::Q, QS = QA + QB;
  uint32_t d0[3], d1[3];
  float y[4];
  auto stage = [&](auto scaled, const Set& rs, int i, int b) {
    const int q = i / 4;
    auto put = [&](int pc) {
      d0[pc] = bf16_pair(y[0], y[1]);
      d1[pc] = bf16_pair(y[2], y[3]);
    };
    auto drop = [&](int pc) {
      y[0] -= __builtin_bit_cast(float, d0[pc] << 16);
      y[1] -= __builtin_bit_cast(float, d0[pc] & 0xffff0000u);
      y[2] -= __builtin_bit_cast(float, d1[pc] << 16);
      y[3] -= __builtin_bit_cast(float, d1[pc] & 0xffff0000u);
    };
    if (i % 4 == 0) {
#pragma unroll
      for (int k = 0; k < 4; ++k) y[k] = q < QA ? sa.at(rs.a, q < QA ? q : 0, k) : sb.at(rs.b, q < QA ? 0 : q - QA, k);
      if constexpr (decltype(scaled)::value) {
#pragma unroll
        for (int k = 0; k < 4; ++k) y[k] *= q < QA ? scaleA : scaleB;
      } else if constexpr (RANGE) {
        float& mx = q < QA ? maxA : maxB;
        mx = max3_abs(mx, y[0], y[1]);
        mx = max3_abs(mx, y[2], y[3]);
      }
      put(0);
    } else if (i % 4 == 1) {
      drop(0);
    } else if (i % 4 == 2) {
      put(1);
      drop(1);
    } else {
      put(2);
      unsigned char* p = gm_sm + b * BUF + (q < QA ? sa.loff[q < QA ? q : 0] : ABYTES + sb.loff[q < QA ? 0 : q - QA]);
#pragma unroll
      for (int pc = 0; pc < 3; ++pc) *reinterpret_cast<uint2*>(p + 1024 * pc) = uint2{d0[pc], d1[pc]};
    }
  };
  const int nk = K / kGmK;
  v16f acc[RT][CT];
  float alpha = 1.0f;
  auto product = [&](auto scaled) {
    gload(rg, 0);
#pragma unroll
    for (int i = 0; i < 4 * QS; ++i) stage(scaled, rg, i, 0);
    gload(rg, nk > 1 ? 1 : 0);
    if constexpr (SCALED) {
      __shared__ float red[4];
      float v = -3.4e38f;
      for (int i = tid; i < NP; i += 256) v = fmaxf(v, rowsum[(size_t)m * NP + i]);
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off));
      if (lane == 0) red[wave] = v;
      __syncthreads();
      const float mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
      alpha = 1.8f / (mx * mx);
    } else {
      __syncthreads();
    }
    int aoff[2][RT], boff[2][CT];  // this lane's slots, per step
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int r = 0; r < RT; ++r) aoff[s][r] = ((wr * RT + r) * 2 + s) * 3072 + gm_slot<TM, TX>(li, lh, s, wr * RT + r) * 16;
#pragma unroll
      for (int c = 0; c < CT; ++c)
        boff[s][c] = ABYTES + ((wc * CT + c) * 2 + s) * 3072 + gm_slot<TN, !TY>(li, lh, s, wc * CT + c) * 16;
    }
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int q = 0; q < 16; ++q) acc[r][c][q] = 0.f;
    constexpr int MC = 12 * RT * CT;  // products per stage
    // Stage kc: the products from buffer kc % 2, between them the next stage's splitting,
    // at the end the loads of the one after.
#pragma unroll 1
    for (int kc = 0; kc < nk; ++kc) {
      const unsigned char* buf = gm_sm + (kc & 1) * BUF;
      uint4 xa[2][RT][3], xb[2][CT][3];
      auto fetch = [&](int s) {
#pragma unroll
        for (int pc = 0; pc < 3; ++pc) {
#pragma unroll
          for (int r = 0; r < RT; ++r) xa[s][r][pc] = *reinterpret_cast<const uint4*>(buf + aoff[s][r] + 1024 * pc);
#pragma unroll
          for (int c = 0; c < CT; ++c) xb[s][c][pc] = *reinterpret_cast<const uint4*>(buf + boff[s][c] + 1024 * pc);
        }
      };
      fetch(0);
      fetch(1);  // (spread over the first step's products instead, 1076 against 982 us at 128 x 256^2)
      __builtin_amdgcn_sched_barrier(0);
      unrolled<MC>([&](auto mc) {
        constexpr int mm = decltype(mc)::value, s = mm / (MC / 2), e = mm % (MC / 2), r = e / 6 / CT, c = e / 6 % CT;
        acc[r][c] = mfma_piece(xa[s][r], xb[s][c], e % 6, false, acc[r][c]);
        // (After the last stage's products nobody reads the other buffer.)
        constexpr int PER = (4 * QS + MC - 5) / (MC - 4);  // stages per product, done before the last products
        if constexpr (mm >= 2) {
#pragma unroll
          for (int k = 0; k < PER; ++k)
            if ((mm - 2) * PER + k < 4 * QS) stage(scaled, rg, (mm - 2) * PER + k, (kc + 1) & 1);
        }
        if constexpr (mm == MC - 1)
          if (kc + 2 < nk) gload(rg, kc + 2);
        __builtin_amdgcn_sched_barrier(0);
      });
      __syncthreads();
    }
  };
  product(std::false_type{});
  if constexpr (RANGE) {
    // In range: each panel has an entry of 2^-86 or more (or zeros alone) and none of 2^126 or more.
    const int flags = (__any(maxA >= 0x1p-86f) ? 1 : 0) | (__any(maxB >= 0x1p-86f) ? 2 : 0) |
                      (__any(maxA > 0.f) ? 4 : 0) | (__any(maxB > 0.f) ? 8 : 0) |
                      (__any(!(maxA < 0x1p126f && maxB < 0x1p126f)) ? 16 : 0);
    if (lane == 0) pflag[wave] = flags;
    __syncthreads();
    const int all = uniform(pflag[0] | pflag[1] | pflag[2] | pflag[3]);
    if ((all & 16) || (all & 5) == 4 || (all & 10) == 8) {
      auto exponent = [&](float v) {  // of the panel's largest entry, where 2^-e is normal
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off));
        __syncthreads();
        if (lane == 0) pflag[wave] = (int)(__builtin_bit_cast(uint32_t, v) >> 23) - 127;
        __syncthreads();
        return uniform(min(max(max(max(pflag[0], pflag[1]), max(pflag[2], pflag[3])), -126), 126));
      };
      const int ea = exponent(maxA), eb = exponent(maxB);
      scaleA = __builtin_bit_cast(float, (uint32_t)(127 - ea) << 23);
      scaleB = __builtin_bit_cast(float, (uint32_t)(127 - eb) << 23);
      expo = ea + eb;
      product(std::true_type{});
    }
  }

  float* Dm = D + mo;
  const float* Em = MODE == 1 ? E + mo : nullptr;
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      const int i0 = ti * TM + 32 * (wr * RT + r) + 4 * lh, j = tj * TN + 32 * (wc * CT + c) + li;
      float ev[16];
      if constexpr (MODE == 1)
#pragma unroll
        for (int q = 0; q < 16; ++q) ev[q] = Em[(unsigned)((i0 + 8 * (q >> 2) + (q & 3)) * NP + j)];
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        float v = acc[r][c][q];
        if (MODE == 1) v = 2.0f * ev[q] - v;
        if (MODE == 2) v = -v;
        if constexpr (RANGE) v = __builtin_amdgcn_ldexpf(v, expo);
        if (SCALED) v = alpha * v;
        Dm[(unsigned)((i0 + 8 * (q >> 2) + (q & 3)) * NP + j)] = v;
      }
    }
}

}  // namespace lfamd
