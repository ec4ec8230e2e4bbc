// q8_0_gemm.hip — GGUF Q8_0 matmul for more than a few tokens (prefill) on the 32x32x16 f16 MFMA:
//   Y[t][o] = sum_b d_{o,b} * sum_{k in b} code_{o,k} X[t][k],   b the 32-weight blocks.
//
// The int8 codes are exact f16 operands and X enters as two f16 operands per value, hi = f16(v)
// and lo = f16(v - hi) with v = x 2^-k, so a product carries ~22 bits of x; the f32 sum of a block
// (four MFMAs) is scaled by the block's f16 d in f32. 2^k is a power of two per (token, K range of
// a workgroup) that puts the range's largest magnitude in [2^13, 2^14); the range's result is
// multiplied back by it (exact). A range with a block whose largest magnitude that would put under 1
// (2^13 and more below the range's) has a scale per block instead, applied to the block's sum: f16
// would hold too few bits of its values, or none, and they are all there is where the weights of the
// larger blocks are zero. (Where every token has such blocks: 18944 x 3584 at 32 / 512 tokens 34 / 380 us.)
// A range holding a NaN or an infinity gets the scale NaN, which reaches every output of that token.
//
// Three launches: the operands of X once per call (q8_gemm_xprep_kernel), the GEMM, and, when K is
// split, the ordered sum of the ranges. us per call against slices of 16 tokens on the GEMV: 3584 x
// 3584 at 32 / 128 / 512 tokens 36 / 146 / 562 -> 15.1 / 21.3 / 47, 18944 x 3584 144 / 576 / 2278 ->
// 24.5 / 60 / 181. Up to 32 tokens the weights' stream bounds it (18944 x 3584: 68.6 MB, 14.4 us at
// a large copy's rate); at 512 the MFMAs, two per product (95 us at a large f16 matmul's rate), whose
// operand reads keep the LDS at its peak: a wave of 32 rows reads one operand unit per MFMA.
#include <type_traits>

#include "kernels.hpp"

namespace fhip {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));

// Operand units of one 32-token tile and block: [K16 slice s][hi, lo][64 lanes] x 16 B, lane l =
// 8 f16 of token l % 32 at K = 32 b + 16 s + 8 (l / 32) + j. xa[(tile * nb2 + b) * 256 + ...], nb2
// the blocks padded to pairs (zeros).
constexpr int kBlkUnits = 4 * 64;

// One workgroup per (padded token, K range): the range's largest magnitude, then the conversion.
// UPT > 0: each thread keeps its UPT 8-value units in registers (ranges of up to 256 UPT units);
// UPT = 0 reads the range twice. The 32 tokens of an operand tile run on one XCD (workgroups go to
// the 8 XCDs round-robin), so one L2 assembles each 512-byte run of a unit.
template <int UPT>
__global__ __launch_bounds__(256) void q8_gemm_xprep_kernel(const float *__restrict__ X, int M, int K,
                                                            int npairs, int SK, uint4 *__restrict__ xa,
                                                            float *__restrict__ tscale,
                                                            float *__restrict__ bscale) {
  __shared__ uint32_t wmax[4], wmin[4];
  const int tokens = gridDim.x;
  int t = blockIdx.x;
  if (t < (tokens & ~255)) {
    const int x = t & 7, slot = t >> 3;
    t = 32 * (8 * (slot >> 5) + x) + (slot & 31);
  }
  const int sp = blockIdx.y, tid = threadIdx.x;
  const int u0 = 8 * (int)((long long)sp * npairs / SK), u1 = 8 * (int)((long long)(sp + 1) * npairs / SK);
  const int nu = min(u1, K / 8);  // units with values; up to u1 the padding block's zeros
  const bool valid = t < M;
  const float4 *row = reinterpret_cast<const float4 *>(X + (size_t)(valid ? t : 0) * K);
  uint32_t m = 0, mn = ~0u;  // largest magnitude, and smallest of a block's that are not zero
  // Largest magnitude of a block: its four units are four neighbouring threads'.
  auto block_max = [](const float4 a, const float4 b) {
    uint32_t w = max(absmax4_bits(a.x, a.y, a.z, a.w), absmax4_bits(b.x, b.y, b.z, b.w));
    w = max(w, lane_xor<1>(w));
    return max(w, lane_xor<2>(w));
  };
  auto see = [&](const uint32_t w) {
    m = max(m, w);
    mn = min(mn, w - 1);  // zero last
  };
  auto real = [&](int u) { return u < nu ? u : nu - 4 + (u & 3); };  // repeats do not change either
  float4 reg[UPT > 0 ? UPT : 1][2];
  if (UPT > 0) {
#pragma unroll
    for (int j = 0; j < UPT; ++j) {
      const int u = real(u0 + tid + 256 * j);
      reg[j][0] = row[2 * u];
      reg[j][1] = row[2 * u + 1];
    }
#pragma unroll
    for (int j = 0; j < UPT; ++j) see(block_max(reg[j][0], reg[j][1]));
  } else {
    for (int u = u0 + tid; u < nu; u += 256) see(block_max(row[2 * u], row[2 * u + 1]));
  }
  m = max(m, group_mirror<8>(m));  // groups of four lanes hold the same values
  mn = min(mn, group_mirror<8>(mn));
  m = max(m, group_mirror<16>(m));
  mn = min(mn, group_mirror<16>(mn));
#pragma unroll
  for (int o = 16; o <= 32; o <<= 1) {
    m = max(m, (uint32_t)__shfl_xor((int)m, o));
    mn = min(mn, (uint32_t)__shfl_xor((int)mn, o));
  }
  if ((tid & 63) == 0) {
    wmax[tid >> 6] = m;
    wmin[tid >> 6] = mn;
  }
  __syncthreads();
  m = valid ? max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3])) : 0u;
  mn = min(min(wmin[0], wmin[1]), min(wmin[2], wmin[3])) + 1;
  const bool finite = m < 0x7F800000u;
  // The exponent that puts w in [2^13, 2^14), at least -126: 2^k stays normal, and the bits of
  // magnitudes below 2^-112 all fit in the operands.
  auto exponent = [](uint32_t w) {
    int e = 0;
    (void)frexpf(__uint_as_float(w), &e);
    return max(e - 14, -126);
  };
  const int k = finite && m ? exponent(m) : 0;
  const bool fine = finite && m && (m >> 23) > (mn >> 23) + 13;
  // -1: the scales are the blocks'
  if (tid == 0) tscale[(size_t)sp * tokens + t] = !finite ? __builtin_nanf("") : fine ? -1.f : ldexpf(1.f, k);
  const int tt = t >> 5, lt = t & 31, nb2 = 2 * npairs;
  auto put = [&](int u, const float4 a, const float4 b) {
    const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    const bool live = valid && finite && u < nu;
    int kb = k;
    if (fine) {  // uniform over the workgroup
      const uint32_t w = u < nu ? block_max(a, b) : 0u;
      kb = w ? exponent(w) : 0;
      if ((u & 3) == 0) bscale[((size_t)tt * nb2 + (u >> 2)) * 32 + lt] = ldexpf(1.f, kb);
    }
    f16x8 hi, lo;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float s = live ? ldexpf(v[j], -kb) : 0.f;
      hi[j] = (_Float16)s;
      lo[j] = (_Float16)(s - (float)hi[j]);
    }
    uint4 *d = xa + ((size_t)tt * nb2 + (u >> 2)) * kBlkUnits + ((u >> 1) & 1) * 128 + 32 * (u & 1) + lt;
    d[0] = __builtin_bit_cast(uint4, hi);
    d[64] = __builtin_bit_cast(uint4, lo);
  };
  if (UPT > 0) {
#pragma unroll
    for (int j = 0; j < UPT; ++j) {
      const int u = u0 + tid + 256 * j;
      if (u < u1) put(u, reg[j][0], reg[j][1]);
    }
  } else {
    for (int u = u0 + tid; u < u1; u += 256) put(u, row[2 * real(u)], row[2 * real(u) + 1]);
  }
}

// Waits on this wave's loads, then a bare workgroup barrier (see q4k_gemm32.hip).
#define FHIP_LDS_BARRIER_Q8(imm)     \
  do {                               \
    __builtin_amdgcn_s_waitcnt(imm); \
    asm volatile("" ::: "memory");   \
    __builtin_amdgcn_s_barrier();    \
    asm volatile("" ::: "memory");   \
  } while (0)
constexpr int wait_vm_q8(int n) { return 0x0070 | (n & 15) | ((n >> 4) << 14); }

constexpr int kRows = 128;            // rows per workgroup: 32 per wave
constexpr int kWUnits = 2 * 64 + 16;  // a wave's share of a pair: two tiles' codes, 64 scale dwords
constexpr int kWLoads = 3;
// Loads a wave may leave pending at the end of a stage: those of the last stage issued.
constexpr int q8_wait(int TT) { return 2 * TT + kWLoads; }

// Workgroup = four waves x 32 rows x TT 32-token tiles over one K range. A stage is a pair of blocks
// (64 values): 8 KB of operands per token tile, shared by the waves, and each wave's two records,
// all by direct-to-LDS loads issued two stages ahead into three buffers, so no load returns to a
// register and the one wait per stage is a fixed count. The pair gives a wave 2 TT independent chains
// of four MFMAs between barriers (with one block per stage the chain's latency set the time: 3584 x
// 18944 at 17 tokens in one K range: 181 us against 145).
// The wave count is what the LDS allows; stated, it puts the block results that the VALU scales in VGPRs
// (512 tokens of 18944 x 3584 198 -> 181 us, 17 of 3584 x 18944 25.4 -> 23.8; the compiler had taken AGPRs).
template <int TT>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(TT == 1 ? 3 : 2, TT == 1 ? 3 : 2))) void q8_gemm_kernel(const uint8_t *__restrict__ W,
                                                      const uint4 *__restrict__ xa,
                                                      const float *__restrict__ tscale,
                                                      const float *__restrict__ bscale,
                                                      float *__restrict__ Y, float *__restrict__ part,
                                                      int N, int M, int npairs, int ntiles, int MTG,
                                                      int tokens, int SK) {
  constexpr int kTU = 2 * kBlkUnits, kAU = TT * kTU;  // operand units of a stage: per tile, all
  // Named arrays: the compiler tracks direct-to-LDS loads per object.
  __shared__ u32x4 A0[kAU], A1[kAU], A2[kAU];
  __shared__ u32x4 W0[4 * kWUnits], W1[4 * kWUnits], W2[4 * kWUnits];
  __shared__ __align__(16) float ts[32 * TT];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kap = lane >> 5, rho = lane & 31, r16 = rho & 15;
  const int sp = blockIdx.x % SK, task = blockIdx.x / SK, mg = task % MTG, ng = task / MTG;
  const int p0 = (int)((long long)sp * npairs / SK), p1 = (int)((long long)(sp + 1) * npairs / SK);
  const int np = p1 - p0;
  const int tile0 = 8 * ng + 2 * wave;  // this wave's two 16-row tiles (clamped to the last)
  auto abuf = [&](int k) -> u32x4 * { return k == 0 ? A0 : k == 1 ? A1 : A2; };
  auto wbuf = [&](int k) -> u32x4 * { return k == 0 ? W0 : k == 1 ? W1 : W2; };
  const int wu = wave * kWUnits;  // this wave's units of a pair's buffer
  // This lane's codes of K16 slice 0, and its scale dword (opaque indices: see lds_load16).
  const uint32_t cu = in_reg(wu + 64 * (rho >> 4) + 16 * kap + r16), su = in_reg(4 * (wu + 128) + rho);
  const int off16 = 16 * lane;
  // Scales: lane l takes row l % 16 of tile (l / 16) % 2; lanes 32.. repeat them into the padding.
  const int offs = (lane & 16 ? (min(tile0 + 1, ntiles - 1) - min(tile0, ntiles - 1)) * npairs * kQ8Record : 0) +
                   4 * (lane & 15);
  const void *ra = xa + (size_t)TT * mg * npairs * kTU;
  const void *rw0 = W + (size_t)min(tile0, ntiles - 1) * npairs * kQ8Record;
  const void *rw1 = W + (size_t)min(tile0 + 1, ntiles - 1) * npairs * kQ8Record;
  auto load = [&](int p, u32x4 *wd, u32x4 *ad) {  // wave w loads units 2 w and 2 w + 1 (of 8) of each token tile
    const int pc = p0 + min(p, np - 1), so = pc * kQ8Record;
    lds_load16(rw0, wd + wu, off16, so + kQ8Hdr);
    lds_load16(rw1, wd + (wu + 64), off16, so + kQ8Hdr);
    lds_load4(rw0, wd + (wu + 128), offs, so);
#pragma unroll
    for (int i = 0; i < TT; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        lds_load16(ra, ad + i * kTU + (2 * wave + j) * 64, off16,
                   (pc + i * npairs) * kTU * 16 + (2 * wave + j) * 1024);
  };

  f32x16 acc[TT];
#pragma unroll
  for (int i = 0; i < TT; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[i][e] = 0.f;
  load(0, W0, A0);
  load(1, W1, A1);
  const float tsl = tscale[(size_t)sp * tokens + 32 * TT * mg + (tid & (32 * TT - 1))];
  if (tid < 32 * TT) ts[tid] = tsl;
  FHIP_LDS_BARRIER_Q8(wait_vm_q8(0));

  const uint32_t k1152 = in_reg(0x64806480u), k64 = in_reg(0x64646464u);
  const uint32_t al = in_reg(lane);
  auto ranges = [&](auto fine) {  // fine: with block scales
    for (int pb = 0; pb < np; pb += 3) {
#pragma unroll
      for (int u = 0; u < 3; ++u) {
        load(pb + u + 2, wbuf((u + 2) % 3), abuf((u + 2) % 3));
        if (pb + u < np) {
          const u32x4 *Wb = wbuf(u), *Ab = abuf(u);
          const u32x4 cq[2] = {Wb[cu], Wb[cu + 32]};  // K16 slice q of both blocks
          const uint32_t sc = reinterpret_cast<const uint32_t *>(Wb)[su];
          f32x16 tmp[2][TT];
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            f16x8 b[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              // Codes 16 q + 8 kap .. + 8 of row rho, block h: 1024 + (code ^ 0x80) - 1152, exact.
              const uint32_t x0 = cq[q][2 * h] ^ 0x80808080u, x1 = cq[q][2 * h + 1] ^ 0x80808080u;
              auto pair = [&](uint32_t x, uint32_t sel) {
                return __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2, __builtin_amdgcn_perm(k64, x, sel)) -
                                                        __builtin_bit_cast(h2, k1152));
              };
              b[h] = __builtin_bit_cast(f16x8, u32x4{pair(x0, 0x04010400u), pair(x0, 0x04030402u),
                                                     pair(x1, 0x04010400u), pair(x1, 0x04030402u)});
            }
#pragma unroll
            for (int hl = 0; hl < 2; ++hl)
#pragma unroll
              for (int i = 0; i < TT; ++i)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                  const f16x8 a = __builtin_bit_cast(f16x8, Ab[i * kTU + h * kBlkUnits + (2 * q + hl) * 64 + al]);
                  f32x16 c = tmp[h][i];
                  if (q == 0 && hl == 0)
#pragma unroll
                    for (int e = 0; e < 16; ++e) c[e] = 0.f;
                  tmp[h][i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b[h], c, 0, 0, 0);
                }
          }
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const float d = (float)__builtin_bit_cast(_Float16, (uint16_t)(h ? sc >> 16 : sc & 0xffffu));
            if constexpr (decltype(fine)::value) {
#pragma unroll
              for (int i = 0; i < TT; ++i)
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                  const int tl = 8 * a + 4 * kap;
                  const float4 b4 = *reinterpret_cast<const float4 *>(
                      bscale + ((size_t)(TT * mg + i) * 2 * npairs + 2 * (p0 + pb + u) + h) * 32 + tl);
                  const float bs[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
                  for (int e = 0; e < 4; ++e)
                    tmp[h][i][4 * a + e] *= ts[32 * i + tl + e] < 0.f ? bs[e] : 1.f;
                }
            }
#pragma unroll
            for (int i = 0; i < TT; ++i)
#pragma unroll
              for (int e = 0; e < 16; ++e) acc[i][e] = fmaf(d, tmp[h][i][e], acc[i][e]);
          }
        }
        FHIP_LDS_BARRIER_Q8(wait_vm_q8(q8_wait(TT)));
      }
    }
  };
  // A loop of its own: the test within it cost every call (0.8 us of 22 at 128 tokens of 3584 x 3584).
  if (__builtin_amdgcn_ballot_w64(tsl < 0.f) != 0)
    ranges(std::true_type{});
  else
    ranges(std::false_type{});
  __builtin_amdgcn_s_waitcnt(wait_vm_q8(0));  // no direct-to-LDS load may outlive the workgroup

  const int o = kRows * ng + 32 * wave + rho;
  if (o >= N) return;
#pragma unroll
  for (int i = 0; i < TT; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int tl = 32 * i + 8 * (e >> 2) + 4 * kap + (e & 3), tok = 32 * TT * mg + tl;
      if (tok >= M) continue;
      const float v = acc[i][e] * fabsf(ts[tl]);
      if (SK == 1)
        Y[(size_t)tok * N + o] = v;
      else
        part[((size_t)sp * M + tok) * N + o] = v;
    }
}
#undef FHIP_LDS_BARRIER_Q8

}  // namespace

// Y of up to kQ8GemmTokens tokens (longer calls come in slices of that, which bounds the scratch).
int q8_0_gemm(const void *Wv, const float *X, float *Y, int N, int K, int M) {
  const int npairs = q8_groups(K), ntiles = q4k_tiles(N);
  const int cus = cu_count() > 0 ? cu_count() : 256;
  // Two token tiles per workgroup share each dequantized weight, but halve the grid: taken for many
  // tokens of a matrix large enough to fill the chip all the same (us, one / two tiles: 512 tokens
  // 18944 x 3584 204 / 196, 3584 x 18944 239 / 212, 8192 x 2048 55 / 52, 2048 x 2048 22.7 / 27.2; 128
  // tokens 3584 x 3584 21.2 / 26.3).
  const int TT = M > 128 && (long long)N * K >= 8 << 20 ? 2 : 1;
  const int MTG = ceil_div(M, 32 * TT), tokens = 32 * TT * MTG;
  const int tasks = MTG * ceil_div(N, kRows);
  // K ranges: about 7/4 workgroups per CU, each of at least three pairs of blocks (3584 x 3584 at 17
  // tokens, 28 tasks: 4 / 7 / 14 ranges 14.7 / 13.2 / 13.6 us; at 128, 112 tasks: 2 / 4 / 7 ranges
  // 24.0 / 22.4 / 25.7).
  int SK = 7 * cus / 4 / tasks;
  if (SK > npairs / 3) SK = npairs / 3;
  if (SK < 1) SK = 1;
  const size_t xb = (size_t)tokens * npairs * 64 * 4;
  const size_t tb = ((size_t)SK * tokens * 4 + 255) & ~(size_t)255;
  const size_t bb = (size_t)tokens * npairs * 2 * 4;  // block scales
  const size_t pb = SK > 1 ? (size_t)SK * M * N * 4 : 0;
  unsigned char *ws = (unsigned char *)workspace(xb + tb + bb + pb);
  if (!ws) return FHIP_ENOMEM;
  if (int rc = check_disjoint("q8_0_gemm", X, (size_t)M * K * 4, ws, xb + tb + bb + pb)) return rc;
  uint4 *xa = (uint4 *)ws;
  float *ts = (float *)(ws + xb), *bs = (float *)(ws + xb + tb), *part = (float *)(ws + xb + tb + bb);
  const dim3 pg(tokens, SK);
  const int units = 8 * ceil_div(npairs, SK);
  if (units <= 256)
    q8_gemm_xprep_kernel<1><<<pg, 256, 0, stream()>>>(X, M, K, npairs, SK, xa, ts, bs);
  else if (units <= 512)
    q8_gemm_xprep_kernel<2><<<pg, 256, 0, stream()>>>(X, M, K, npairs, SK, xa, ts, bs);
  else if (units <= 1024)
    q8_gemm_xprep_kernel<4><<<pg, 256, 0, stream()>>>(X, M, K, npairs, SK, xa, ts, bs);
  else
    q8_gemm_xprep_kernel<0><<<pg, 256, 0, stream()>>>(X, M, K, npairs, SK, xa, ts, bs);
  FHIP_CHECK_LAUNCH("q8_gemm_xprep_kernel");
  const uint8_t *W = (const uint8_t *)Wv;
  if (TT == 1)
    q8_gemm_kernel<1><<<tasks * SK, 256, 0, stream()>>>(W, xa, ts, bs, Y, part, N, M, npairs, ntiles, MTG, tokens, SK);
  else
    q8_gemm_kernel<2><<<tasks * SK, 256, 0, stream()>>>(W, xa, ts, bs, Y, part, N, M, npairs, ntiles, MTG, tokens, SK);
  FHIP_CHECK_LAUNCH("q8_gemm_kernel");
  return SK > 1 ? sum_ranges(part, Y, SK, M * N) : FHIP_OK;
}

}  // namespace fhip
