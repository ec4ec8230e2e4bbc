// q8_hal.hip — the HAL Q8 lane: int8 codes + f32 per-block scales with the activation quantized
// on the device (the semantics of fcuda_q8_matmul_f32, internal/compute/cuda_backend.h:104-111,
// whose CPU reference is cpuBackend.MatMul / BatchedMatMul on Q8_0,
// internal/compute/cpuref.go:113-191).
//
// Every result here is bit-identical to the CPU reference, not just within a tolerance:
//   * quantizeVecQ8 (cpuref.go:505-527): d = amax/127, inv = 1/d, code = q8round(x*inv), with
//     IEEE-rounded single operations and q8round's truncate-then-round-half-away rule
//     (internal/model/quant.go:89-104);
//   * MatMul = qdot8scalar (cpuref.go:532-548): per block the exact int32 dot, then
//     acc = acc + (f32(isum) * dw) * dx in block order. The int32 dot is exact in any order;
//     one lane owns a row's running sum and adds the blocks' terms in order;
//   * BatchedMatMul = qgemm8cell (cpuref.go:553-577, lanes = 16): per block 16 pair products
//     p_k = w[2k]x[2k] + w[2k+1]x[2k+1], acc_k += f32(p_k) * (dw * dx), then the fixed pairwise
//     tree. One thread owns a lane sum of a (row, token) cell from its first block to its last.
// The reference is Go on amd64, which never fuses multiply-add, so this file is built with
// -ffp-contract=off (fak_amd/build.py): by default hipcc contracts a*b - c into one fma even when
// written with __fmul_rn/__fsub_rn, which turned q8round of a product that rounds to 43.5 into 43
// instead of 44.
#include "kernels.hpp"
#include "q8round.hpp"

namespace fhip {
namespace {

typedef _Float16 hal_h2 __attribute__((ext_vector_type(2)));

// One thread per (row, block): quantizeVecQ8 of X[rows][in] into codes [rows][in] and
// scales [rows][in / block].
__global__ void q8_quantize_kernel(const float *__restrict__ X, int8_t *__restrict__ codes,
                                   float *__restrict__ scales, int rows, int in, int block) {
  const int nblk = in / block;
  const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= (long long)rows * nblk) return;
  const int row = (int)(id / nblk), b = (int)(id - (long long)row * nblk);
  const float *xb = X + (size_t)row * in + (size_t)b * block;
  int8_t *qb = codes + (size_t)row * in + (size_t)b * block;
  float amax = 0.f;
  for (int i = 0; i < block; ++i) {
    const float a = fabsf(xb[i]);
    if (a > amax) amax = a;
  }
  const float d = __fdiv_rn(amax, 127.f);
  scales[id] = d;
  if (d == 0.f) {
    for (int i = 0; i < block; ++i) qb[i] = 0;
    return;
  }
  const float inv = __fdiv_rn(1.f, d);
  for (int i = 0; i < block; ++i) qb[i] = (int8_t)q8round(__fmul_rn(xb[i], inv));
}

// One token, blocks of 32 codes, 16-byte aligned operands (a row is then whole 16-byte units).
// What bounds it is the codes' stream from HBM and the two latencies around it, so:
//   * one launch: each workgroup quantizes the activation into LDS itself (eight lanes per block;
//     its loads go out before the first codes' loads, the arithmetic runs under them), where a
//     separate quantize launch of one thread per block cost more than the whole product;
//   * a wave owns kHalRows rows and reads them coalesced, 16 bytes per lane, up to 4 kHalRows
//     loads in flight; two neighbouring lanes hold a block, so its int32 dot is four v_dot4 and
//     one exchange;
//   * the terms (f32(isum) * dw) * dx of all blocks are made in parallel and parked in LDS, and
//     one lane per row adds them in block order: the reference's chain, bit for bit, at the
//     latency of the additions alone.
// 3584 x 3584: 63 -> 6.4 us per call; the four-lanes-per-row kernel below (any block) walked a
// row with one dependent load per block.
constexpr int kHalRows = 4;                 // rows per wave
constexpr int kHalWG = 4 * kHalRows;        // rows per workgroup of four waves
__host__ __device__ inline int hal_term_stride(int nblk) { return nblk | 1; }  // odd: no bank conflicts
inline size_t hal_gemv_lds(int in) {
  const int nblk = in / 32;
  return (size_t)in + (size_t)nblk * 4 + (size_t)kHalWG * hal_term_stride(nblk) * 4;
}

__global__ __launch_bounds__(256) void q8_hal_gemv32_kernel(const uint8_t *__restrict__ codes,
                                                            const float *__restrict__ wscale,
                                                            const float *__restrict__ X,
                                                            float *__restrict__ Y, int out, int in) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nblk = in / 32, nu = in / 16, nx = in / 4, ts = hal_term_stride(nblk);
  uint8_t *qx = smem;
  float *dx = reinterpret_cast<float *>(smem + in);
  float *terms = dx + nblk;
  const int row0 = blockIdx.x * kHalWG + kHalRows * wave;

  constexpr int XI = 4, J = 4;
  const float4 *X4 = reinterpret_cast<const float4 *>(X);
  float4 xv[XI];
#pragma unroll
  for (int i = 0; i < XI; ++i) xv[i] = X4[min(tid + 256 * i, nx - 1)];
  // Codes and scales of pass j0: unit lane + 64 (j0 + j) of each row (clamped; repeats unused).
  uint4 w[kHalRows][J];
  float sc[kHalRows][J];
  auto load = [&](int j0) {
#pragma unroll
    for (int r = 0; r < kHalRows; ++r) {
      const int row = min(row0 + r, out - 1);
#pragma unroll
      for (int j = 0; j < J; ++j) {
        const int u = min(lane + 64 * (j0 + j), nu - 1);
        w[r][j] = ld_stream(codes + (size_t)row * in + 16 * (size_t)u);
        sc[r][j] = wscale[(size_t)row * nblk + (u >> 1)];
      }
    }
  };
  load(0);
  // quantizeVecQ8 of four values: lanes 8k .. 8k + 7 hold a block (in / 4 is a multiple of 8, so
  // a block's lanes are valid together).
  auto quantize = [&](int v, const float4 x) {
    float amax = fmaxf(fmaxf(fmaxf(fmaxf(0.f, fabsf(x.x)), fabsf(x.y)), fabsf(x.z)), fabsf(x.w));
    amax = fmaxf(amax, __shfl_xor(amax, 1));
    amax = fmaxf(amax, __shfl_xor(amax, 2));
    amax = fmaxf(amax, __shfl_xor(amax, 4));
    const float d = __fdiv_rn(amax, 127.f);
    uint32_t q = 0;
    if (d != 0.f) {
      const float inv = __fdiv_rn(1.f, d);
      q = (uint32_t)(q8round(__fmul_rn(x.x, inv)) & 255) |
          (uint32_t)(q8round(__fmul_rn(x.y, inv)) & 255) << 8 |
          (uint32_t)(q8round(__fmul_rn(x.z, inv)) & 255) << 16 |
          (uint32_t)q8round(__fmul_rn(x.w, inv)) << 24;
    }
    if (v < nx) {
      *reinterpret_cast<uint32_t *>(qx + 4 * v) = q;
      if ((v & 7) == 0) dx[v >> 3] = d;
    }
  };
#pragma unroll
  for (int i = 0; i < XI; ++i) quantize(tid + 256 * i, xv[i]);
  for (int v = tid + 256 * XI; v - tid < nx; v += 256) quantize(v, X4[min(v, nx - 1)]);
  __syncthreads();

  for (int j0 = 0; 64 * j0 < nu; j0 += J) {
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int u = lane + 64 * (j0 + j), uc = min(u, nu - 1), b = uc >> 1;
      const uint4 x = *reinterpret_cast<const uint4 *>(qx + 16 * uc);
      const float xd = dx[b];
#pragma unroll
      for (int r = 0; r < kHalRows; ++r) {
        int isum = __builtin_amdgcn_sdot4((int)w[r][j].x, (int)x.x, 0, false);
        isum = __builtin_amdgcn_sdot4((int)w[r][j].y, (int)x.y, isum, false);
        isum = __builtin_amdgcn_sdot4((int)w[r][j].z, (int)x.z, isum, false);
        isum = __builtin_amdgcn_sdot4((int)w[r][j].w, (int)x.w, isum, false);
        isum += __shfl_xor(isum, 1);
        if (u < nu && (lane & 1) == 0)
          terms[(kHalRows * wave + r) * ts + b] = __fmul_rn(__fmul_rn((float)isum, sc[r][j]), xd);
      }
    }
    if (64 * (j0 + J) < nu) load(j0 + J);
  }
  __syncthreads();
  if (tid >= kHalWG) return;
  const float *t = terms + tid * ts;
  float acc = 0.f;
  int b = 0;
  for (; b + 16 <= nblk; b += 16) {
    float v[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) v[k] = t[b + k];
#pragma unroll
    for (int k = 0; k < 16; ++k) acc = __fadd_rn(acc, v[k]);
  }
  for (; b < nblk; ++b) acc = __fadd_rn(acc, t[b]);
  const int row = blockIdx.x * kHalWG + tid;
  if (row < out) Y[row] = acc;
}

// MatMul of any block size: a wave owns 16 rows; the 4 lanes of a row each form the int32 dot of 8
// bytes of the current block, the quad sum is exact, and the row's first lane accumulates
// acc = acc + (f32(isum) * dw) * dx in block order.
__global__ __launch_bounds__(256) void q8_hal_gemv_kernel(
    const int8_t *__restrict__ codes, const float *__restrict__ wscale,
    const int8_t *__restrict__ qx, const float *__restrict__ dx, float *__restrict__ Y, int out,
    int in, int block) {
  const int lane = threadIdx.x & 63;
  const int row = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 16 + (lane >> 2);
  const int q = lane & 3;
  const int nblk = in / block;
  const bool valid = row < out;
  const int8_t *wr = codes + (size_t)(valid ? row : 0) * in;
  const float *ws = wscale + (size_t)(valid ? row : 0) * nblk;
  float acc = 0.f;
  for (int b = 0; b < nblk; ++b) {
    int isum = 0;
    // this lane's dwords of the block: 4 * (q + 4 j), j = 0.. (block / 16 of them)
    for (int o = 4 * q; o < block; o += 16) {
      const int w4 = *reinterpret_cast<const int *>(wr + (size_t)b * block + o);
      const int x4 = *reinterpret_cast<const int *>(qx + (size_t)b * block + o);
      isum = __builtin_amdgcn_sdot4(w4, x4, isum, false);
    }
    isum += __shfl_xor(isum, 1);
    isum += __shfl_xor(isum, 2);
    acc = __fadd_rn(acc, __fmul_rn(__fmul_rn((float)isum, ws[b]), dx[b]));
  }
  if (valid && q == 0) Y[row] = acc;
}

// BatchedMatMul: one thread per (row o, token t), t fastest. Pair products come from sdot4 on
// the dword with the other pair's bytes masked to zero.
__global__ __launch_bounds__(256) void q8_hal_gemm_kernel(
    const int8_t *__restrict__ codes, const float *__restrict__ wscale,
    const int8_t *__restrict__ qx, const float *__restrict__ dx, float *__restrict__ Y, int out,
    int in, int P, int block) {
  const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= (long long)out * P) return;
  const int o = (int)(id / P), t = (int)(id - (long long)o * P);
  const int nblk = in / block;
  const int8_t *wr = codes + (size_t)o * in;
  const int8_t *xr = qx + (size_t)t * in;
  const float *ws = wscale + (size_t)o * nblk;
  const float *xs = dx + (size_t)t * nblk;
  float acc[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) acc[k] = 0.f;
  for (int b = 0; b < nblk; ++b) {
    const int *w4 = reinterpret_cast<const int *>(wr + (size_t)b * block);
    const int *x4 = reinterpret_cast<const int *>(xr + (size_t)b * block);
    const float s = __fmul_rn(ws[b], xs[b]);
#pragma unroll
    for (int j = 0; j < 8; ++j) {  // dword j holds pairs 2j (bytes 0-1) and 2j + 1 (bytes 2-3)
      const int w = w4[j], x = x4[j];
      const int p0 = __builtin_amdgcn_sdot4(w & 0x0000FFFF, x, 0, false);
      const int p1 = __builtin_amdgcn_sdot4(w & (int)0xFFFF0000u, x, 0, false);
      acc[2 * j] = __fadd_rn(acc[2 * j], __fmul_rn((float)p0, s));
      acc[2 * j + 1] = __fadd_rn(acc[2 * j + 1], __fmul_rn((float)p1, s));
    }
  }
#pragma unroll
  for (int k = 0; k < 8; ++k) acc[k] = __fadd_rn(acc[k], acc[k + 8]);
#pragma unroll
  for (int k = 0; k < 4; ++k) acc[k] = __fadd_rn(acc[k], acc[k + 4]);
  acc[0] = __fadd_rn(acc[0], acc[2]);
  acc[1] = __fadd_rn(acc[1], acc[3]);
  Y[(size_t)t * out + o] = __fadd_rn(acc[0], acc[1]);
}

// Batched activations for q8_hal_gemm32_kernel: quantizeVecQ8 of each 32-value block, the codes
// as f16 (exact), the scales as q8_quantize_kernel writes them. Eight lanes per block, each four
// values (rows are whole blocks, so a block's lanes are valid together).
__global__ __launch_bounds__(256) void q8_hal_xprep_kernel(const float4 *__restrict__ X,
                                                           uint2 *__restrict__ xh,
                                                           float *__restrict__ dx, long long n) {
  const long long id = (long long)blockIdx.x * 256 + threadIdx.x;
  const float4 x = X[id < n ? id : n - 1];
  float amax = fmaxf(fmaxf(fmaxf(fmaxf(0.f, fabsf(x.x)), fabsf(x.y)), fabsf(x.z)), fabsf(x.w));
  amax = fmaxf(amax, __shfl_xor(amax, 1));
  amax = fmaxf(amax, __shfl_xor(amax, 2));
  amax = fmaxf(amax, __shfl_xor(amax, 4));
  const float d = __fdiv_rn(amax, 127.f);
  hal_h2 lo = {(_Float16)0.f, (_Float16)0.f}, hi = lo;
  if (d != 0.f) {
    const float inv = __fdiv_rn(1.f, d);
    lo = {(_Float16)q8round(__fmul_rn(x.x, inv)), (_Float16)q8round(__fmul_rn(x.y, inv))};
    hi = {(_Float16)q8round(__fmul_rn(x.z, inv)), (_Float16)q8round(__fmul_rn(x.w, inv))};
  }
  if (id >= n) return;
  xh[id] = make_uint2(__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi));
  if ((id & 7) == 0) dx[id >> 3] = d;
}

// BatchedMatMul on 32-code blocks with 16-byte aligned rows. The 16 lane sums of a cell take, per
// block and lane, a pair product, one rounded multiply by the block's scale and one rounded add,
// none of which may be merged (the results are the CPU's bits): it is VALU-bound at three
// instructions per pair, and everything else is kept off that path:
//   * codes are f16 in LDS, so a pair product is one v_dot2_f32_f16 (integers below 2^24: exact),
//     not two masked v_dot4 and a conversion; weights are converted once per workgroup while
//     staged, activations once per call by q8_hal_xprep_kernel;
//   * a thread owns RP rows x TP tokens, so each 16-byte LDS read feeds several cells;
//   * four threads share a cell, each with four of its lane sums, so that a few tokens still fill
//     the chip (with one thread per cell 3584 x 3584 at 64 tokens took 111 us, 63 so); the
//     reference's tree (k with k + 8, k + 4, k + 2, k + 1) pairs whole threads first, then the
//     sums within one.
// Chunks of CH blocks, double-buffered: the next chunk's loads are in flight under the products.
// The pad puts the 16 lanes of an LDS read phase on different banks.
// us per call before (one thread per cell, every operand read from global memory) and now:
// 3584 x 3584 at 2 / 16 / 64 tokens 59 / 63 / 204 and 13.6 / 28.5 / 63; 18944 x 3584 61 / 240 / 930
// and 30 / 73 / 239; 3584 x 18944 246 / 259 / 1118 and 48 / 124 / 296.
template <int RT, int TT, int RP, int TP, int CH>
__global__ __launch_bounds__(256) void q8_hal_gemm32_kernel(
    const uint8_t *__restrict__ codes, const float *__restrict__ wscale,
    const u32x4 *__restrict__ xh, const float *__restrict__ dx, float *__restrict__ Y, int out,
    int in, int P) {
  constexpr int Q = 4;                        // threads per cell, four lane sums each
  constexpr int kStr = (CH * 64 + 64) / 16;   // LDS row stride, 16-byte units
  constexpr int TL = TT / TP, RL = RT / RP;                // threads along tokens and rows
  static_assert(TL * RL * Q == 256, "one workgroup is 256 threads");
  constexpr int WU = (RT * CH * 2 + 255) / 256, XU = (TT * CH * 4 + 255) / 256;
  __shared__ u32x4 wl[2][RT * kStr], xl[2][TT * kStr];
  __shared__ float wsl[2][RT * CH], xsl[2][TT * CH];
  const int tid = threadIdx.x;
  const int q = tid % Q, ti = (tid / Q) % TL, ri = tid / (Q * TL);
  const int nblk = in / 32;
  const int r0 = blockIdx.x * RT, t0 = blockIdx.y * TT;

  u32x4 wr[WU], xr[XU];
  constexpr int WS = (RT * CH + 255) / 256, XS = (TT * CH + 255) / 256;
  float wsr[WS], xsr[XS];
  auto load = [&](int b0) {
#pragma unroll
    for (int k = 0; k < WU; ++k) {  // unit: row, 16 codes
      const int u = min(tid + 256 * k, RT * CH * 2 - 1);
      const int row = min(r0 + u / (CH * 2), out - 1), c = min(2 * b0 + u % (CH * 2), 2 * nblk - 1);
      wr[k] = *reinterpret_cast<const u32x4 *>(codes + (size_t)row * in + 16 * (size_t)c);
    }
#pragma unroll
    for (int k = 0; k < XU; ++k) {  // unit: token, 8 f16 codes
      const int u = min(tid + 256 * k, TT * CH * 4 - 1);
      const int t = min(t0 + u / (CH * 4), P - 1), c = min(4 * b0 + u % (CH * 4), 4 * nblk - 1);
      xr[k] = xh[(size_t)t * (in / 8) + c];
    }
    const int sb = min(b0 + tid % CH, nblk - 1);
#pragma unroll
    for (int k = 0; k < WS; ++k)
      wsr[k] = wscale[(size_t)min(r0 + min((tid + 256 * k) / CH, RT - 1), out - 1) * nblk + sb];
#pragma unroll
    for (int k = 0; k < XS; ++k)
      xsr[k] = dx[(size_t)min(t0 + min((tid + 256 * k) / CH, TT - 1), P - 1) * nblk + sb];
  };
  // Two codes of a dword (bytes by the selector) as f16: 1024 + (b ^ 0x80) - 1152, exact.
  auto pair = [](uint32_t w, uint32_t sel) {
    const hal_h2 k1152 = {(_Float16)1152.f, (_Float16)1152.f};
    const uint32_t m = __builtin_amdgcn_perm(0x64646464u, w ^ 0x80808080u, sel);
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(hal_h2, m) - k1152);
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int k = 0; k < WU; ++k) {
      const int u = tid + 256 * k;
      if (u < RT * CH * 2) {
        u32x4 *d = &wl[buf][(u / (CH * 2)) * kStr + 2 * (u % (CH * 2))];
        d[0] = u32x4{pair(wr[k].x, 0x04010400u), pair(wr[k].x, 0x04030402u),
                          pair(wr[k].y, 0x04010400u), pair(wr[k].y, 0x04030402u)};
        d[1] = u32x4{pair(wr[k].z, 0x04010400u), pair(wr[k].z, 0x04030402u),
                          pair(wr[k].w, 0x04010400u), pair(wr[k].w, 0x04030402u)};
      }
    }
#pragma unroll
    for (int k = 0; k < XU; ++k) {
      const int u = tid + 256 * k;
      if (u < TT * CH * 4) xl[buf][(u / (CH * 4)) * kStr + u % (CH * 4)] = xr[k];
    }
#pragma unroll
    for (int k = 0; k < WS; ++k)
      if (tid + 256 * k < RT * CH) wsl[buf][tid + 256 * k] = wsr[k];
#pragma unroll
    for (int k = 0; k < XS; ++k)
      if (tid + 256 * k < TT * CH) xsl[buf][tid + 256 * k] = xsr[k];
  };

  float acc[RP][TP][4];
#pragma unroll
  for (int i = 0; i < RP; ++i)
#pragma unroll
    for (int j = 0; j < TP; ++j)
#pragma unroll
      for (int k = 0; k < 4; ++k) acc[i][j][k] = 0.f;

  load(0);
  store(0);
  __syncthreads();
  for (int b0 = 0, buf = 0; b0 < nblk; b0 += CH, buf ^= 1) {
    const bool more = b0 + CH < nblk;
    if (more) load(b0 + CH);
    const int nb = min(CH, nblk - b0);
    for (int b = 0; b < nb; ++b) {
      float s[RP][TP];
#pragma unroll
      for (int i = 0; i < RP; ++i)
#pragma unroll
        for (int j = 0; j < TP; ++j)
          s[i][j] = __fmul_rn(wsl[buf][(ri + RL * i) * CH + b], xsl[buf][(ti + TL * j) * CH + b]);
      u32x4 wv[RP], xv[TP];
#pragma unroll
      for (int i = 0; i < RP; ++i) wv[i] = wl[buf][(ri + RL * i) * kStr + 4 * b + q];
#pragma unroll
      for (int j = 0; j < TP; ++j) xv[j] = xl[buf][(ti + TL * j) * kStr + 4 * b + q];
#pragma unroll
      for (int i = 0; i < RP; ++i)
#pragma unroll
        for (int j = 0; j < TP; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float p = __builtin_amdgcn_fdot2(__builtin_bit_cast(hal_h2, (uint32_t)wv[i][e]),
                                                   __builtin_bit_cast(hal_h2, (uint32_t)xv[j][e]), 0.f, false);
            acc[i][j][e] = __fadd_rn(acc[i][j][e], __fmul_rn(p, s[i][j]));
          }
    }
    if (more) store(buf ^ 1);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < RP; ++i)
#pragma unroll
    for (int j = 0; j < TP; ++j) {
      float *a = acc[i][j];
#pragma unroll
      for (int k = 0; k < 4; ++k) a[k] = __fadd_rn(a[k], __shfl_xor(a[k], 2));
#pragma unroll
      for (int k = 0; k < 4; ++k) a[k] = __fadd_rn(a[k], __shfl_xor(a[k], 1));
      const float y = __fadd_rn(__fadd_rn(a[0], a[2]), __fadd_rn(a[1], a[3]));
      const int row = r0 + ri + RL * i, t = t0 + ti + TL * j;
      if (q == 0 && row < out && t < P) Y[(size_t)t * out + row] = y;
    }
}

template <int RT, int TT, int RP, int TP, int CH>
void launch_hal_gemm(const int8_t *codes, const float *ws, const void *xh, const float *dx, float *Y,
                     int out, int in, int P) {
  q8_hal_gemm32_kernel<RT, TT, RP, TP, CH><<<dim3(ceil_div(out, RT), ceil_div(P, TT)), 256, 0, stream()>>>(
      (const uint8_t *)codes, ws, (const u32x4 *)xh, dx, Y, out, in, P);
}

int launch_quantize(const float *X, int8_t *codes, float *scales, int rows, int in, int block) {
  const long long n = (long long)rows * (in / block);
  if (n == 0) return FHIP_OK;
  const int bs = 256;
  q8_quantize_kernel<<<(unsigned)((n + bs - 1) / bs), bs, 0, stream()>>>(X, codes, scales, rows,
                                                                         in, block);
  FHIP_CHECK_LAUNCH("q8_quantize_kernel");
  return FHIP_OK;
}

bool aligned4(const void *p) { return ((uintptr_t)p & 3) == 0; }

}  // namespace
}  // namespace fhip

using namespace fhip;

extern "C" int fhip_q8_quantize_f32(const float *dX, int8_t *dCodes, float *dScales, int rows,
                                    int in, int block) {
  clear_error();
  if (rows < 0 || in < 0 || block <= 0 || in % block)
    return fail(FHIP_EINVAL, "fhip_q8_quantize_f32: need rows >= 0 and in a multiple of block "
                             "(rows=%d in=%d block=%d)", rows, in, block);
  if ((!dX || !dCodes || !dScales) && rows > 0 && in > 0)
    return fail(FHIP_EINVAL, "fhip_q8_quantize_f32: null pointer");
  if (rows > 0 && in > 0) {
    untag_range(dCodes, (size_t)rows * in);
    untag_range(dScales, (size_t)rows * (in / block) * 4);
  }
  return launch_quantize(dX, dCodes, dScales, rows, in, block);
}

extern "C" int fhip_q8_matmul_f32(const int8_t *dCodes, const float *dScales, const float *dX,
                                  float *dY, int out, int in, int P, int block) {
  clear_error();
  if (out < 0 || in <= 0 || P < 0 || block <= 0 || in % block || block % 4)
    return fail(FHIP_EINVAL, "fhip_q8_matmul_f32: need in a positive multiple of block and "
                             "block a multiple of 4 (out=%d in=%d P=%d block=%d)",
                out, in, P, block);
  if (P > 1 && block < 32)
    return fail(FHIP_EINVAL, "fhip_q8_matmul_f32: the batched (P > 1) lane reads 16 pairs per "
                             "block and needs block >= 32 (block=%d)", block);
  if (out == 0 || P == 0) return FHIP_OK;
  if (!dCodes || !dScales || !dX || !dY)
    return fail(FHIP_EINVAL, "fhip_q8_matmul_f32: null pointer");
  if (!aligned4(dCodes)) return fail(FHIP_EINVAL, "fhip_q8_matmul_f32: dCodes must be 4-byte aligned");
  untag_range(dY, (size_t)P * out * 4);
  const int nblk = in / block;
  // A row of 32-code blocks whose start is 16-byte aligned is whole 16-byte units; other blocks
  // and alignments, and rows whose terms do not fit in LDS, take the general kernels.
  const bool units = block == 32 && (((uintptr_t)dCodes | (uintptr_t)dX) & 15) == 0;
  // The one-token kernel's workgroups read X while others write Y: an output over the input (which
  // the general kernels, quantizing X first, allow) takes those.
  const bool apart = (uintptr_t)(dX + in) <= (uintptr_t)dY || (uintptr_t)(dY + out) <= (uintptr_t)dX;
  if (P == 1 && units && apart && hal_gemv_lds(in) <= (size_t)lds_limit()) {
    q8_hal_gemv32_kernel<<<ceil_div(out, kHalWG), 256, hal_gemv_lds(in), stream()>>>(
        (const uint8_t *)dCodes, dScales, dX, dY, out, in);
    FHIP_CHECK_LAUNCH("q8_hal_gemv32_kernel");
    return FHIP_OK;
  }
  if (P > 1 && units && ceil_div(P, 4) <= 65535) {
    const size_t xb = ((size_t)P * in * 2 + 255) & ~(size_t)255;
    unsigned char *wsp = (unsigned char *)workspace(xb + (size_t)P * nblk * 4);
    if (!wsp) return FHIP_ENOMEM;
    float *xs = (float *)(wsp + xb);
    const long long n4 = (long long)P * in / 4;
    q8_hal_xprep_kernel<<<(unsigned)((n4 + 255) / 256), 256, 0, stream()>>>((const float4 *)dX, (uint2 *)wsp,
                                                                           xs, n4);
    FHIP_CHECK_LAUNCH("q8_hal_xprep_kernel");
    // Up to eight tokens 16 x 4 tiles, the cells spread over the most threads; above, 2 x 2 cells per
    // thread, whose LDS reads are shared (us, 16 x 4 / 16 x 16 tiles, 3584 x 3584, 18944 x 3584, 3584
    // x 18944: 8 tokens 16.9 / 28.8, 51.6 / 72.5, 64 / 124; 16 tokens 26.6 / 28.5, 91 / 73, 109 /
    // 124; 64 tokens 72.9 / 63.0, 332 / 239, 328 / 296).
    if (P <= 8)
      launch_hal_gemm<16, 4, 1, 1, 16>(dCodes, dScales, wsp, xs, dY, out, in, P);
    else
      launch_hal_gemm<16, 16, 2, 2, 8>(dCodes, dScales, wsp, xs, dY, out, in, P);
    FHIP_CHECK_LAUNCH("q8_hal_gemm32_kernel");
    return FHIP_OK;
  }
  // activation codes and scales in the library workspace (calls on one library are serialized)
  const size_t qbytes = ((size_t)P * in + 255) & ~(size_t)255;
  unsigned char *ws = (unsigned char *)workspace(qbytes + (size_t)P * nblk * 4);
  if (!ws) return FHIP_ENOMEM;
  int8_t *qx = reinterpret_cast<int8_t *>(ws);
  float *dx = reinterpret_cast<float *>(ws + qbytes);
  if (int rc = launch_quantize(dX, qx, dx, P, in, block)) return rc;
  if (P == 1) {
    const int waves = ceil_div(out, 16);
    q8_hal_gemv_kernel<<<ceil_div(waves, 4), 256, 0, stream()>>>(dCodes, dScales, qx, dx, dY,
                                                                 out, in, block);
    FHIP_CHECK_LAUNCH("q8_hal_gemv_kernel");
    return FHIP_OK;
  }
  const long long n = (long long)out * P;
  q8_hal_gemm_kernel<<<(unsigned)((n + 255) / 256), 256, 0, stream()>>>(dCodes, dScales, qx, dx,
                                                                        dY, out, in, P, block);
  FHIP_CHECK_LAUNCH("q8_hal_gemm_kernel");
  return FHIP_OK;
}
