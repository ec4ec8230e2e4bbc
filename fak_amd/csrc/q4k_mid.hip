// q4k_mid.hip — Q4_K matmul for a few tokens to a few tens (speculative verify on small matrices,
// short prompts) on the 32x32x16 f16 MFMA.
//
// The arithmetic is that of q4k_gemv16.hip: weight operands are the exact integers sc_s * n, each
// super-block's f32 result is scaled by the row's d, the min term is one more MFMA over the sub-block
// sums, and activations are scaled by a power of two per (token, K range) that puts the range's
// largest magnitude in [2^13, 2^14). Up to 16 tokens the 32 operand rows are the f16 of each value and
// the f16 of its remainder (~22 bits); above, 32 tokens in f16.
//
// The data path is another: the operands are made once per call (mid_xprep_kernel), not by every
// workgroup, and every workgroup streams them and its weight records to LDS by direct loads two
// stages ahead, so no load returns to a register and nothing but the MFMAs' own operands is converted
// in the loop. What bounds it: a workgroup's super-block takes about 1.15 us (its 37 KB through the
// direct loads, and a wave's own chain of unpack and MFMA), so time is the longest range, plus the
// launches before and after it. us per call against the kernels it replaced (q4k_gemv16.hip up to 16
// tokens and its 32-token form up to 32, the prefill GEMM for more): 4096 x 4096 at 5 / 16 / 32 / 64 /
// 128 tokens 14.3 / 14.7 / 14.8 / 22.1 / 23.8 -> 11.4 / 11.9 / 13.3 / 16.4 / 19.8; 4096 x 11008 at 32 /
// 64 27.6 / 30.5 -> 16.7 / 24.6; 18944 x 3584 28.6 / 31.7 -> 21.6 / 27.9; 25600 x 5120 40.2 / 46.8 ->
// 29.8 / 38.6.
#include <type_traits>

#include "kernels.hpp"

namespace fhip {
namespace {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
__device__ __forceinline__ h2 as_h2(uint32_t u) { return __builtin_bit_cast(h2, u); }
__device__ __forceinline__ uint32_t as_u(h2 v) { return __builtin_bit_cast(uint32_t, v); }

// Operand units of one 32-row tile and super-block: 16 K16 slices [64 lanes] x 16 B, lane l = 8 f16 of
// operand row l % 32 at K = 256 b + 16 s + 8 (l / 32) + perm8(j); then the unit of sub-block sums:
// lane l < 32, element j = S / 32 of row l and sub-block perm8(j), lanes 32.. zero.
constexpr int kSbUnits = 17;

// One workgroup per (padded token, K range): the range's largest magnitude, then the operands. UPT > 0:
// each thread keeps its UPT 8-value units in registers (ranges of up to 256 UPT units); UPT = 0 reads
// the range twice.
template <bool HL, int UPT>
__global__ __launch_bounds__(256) void mid_xprep_kernel(const float *__restrict__ X, int M, int K, int nblk,
                                                        int SK, u32x4 *__restrict__ xa,
                                                        float *__restrict__ tscale) {
  __shared__ uint32_t wmax[4];
  const int tokens = gridDim.x, t = blockIdx.x, sp = blockIdx.y, tid = threadIdx.x;
  const int u0 = 32 * (sp * nblk / SK), u1 = 32 * ((sp + 1) * nblk / SK);
  const bool valid = t < M;
  const float4 *row = reinterpret_cast<const float4 *>(X + (size_t)(valid ? t : 0) * K);
  uint32_t m = 0;
  float4 reg[UPT > 0 ? UPT : 1][2];
  auto see = [&](const float4 v) { m = max(m, absmax4_bits(v.x, v.y, v.z, v.w)); };
  if (UPT > 0) {
#pragma unroll
    for (int j = 0; j < UPT; ++j) {
      const int u = min(u0 + tid + 256 * j, u1 - 1);
      reg[j][0] = row[2 * u];
      reg[j][1] = row[2 * u + 1];
    }
#pragma unroll
    for (int j = 0; j < UPT; ++j) {
      see(reg[j][0]);
      see(reg[j][1]);
    }
  } else {
    for (int u = u0 + tid; u < u1; u += 256) {
      see(row[2 * u]);
      see(row[2 * u + 1]);
    }
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, o));
  if ((tid & 63) == 0) wmax[tid >> 6] = m;
  __syncthreads();
  m = valid ? max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3])) : 0u;
  const bool finite = m < 0x7F800000u;
  int e = 0;
  (void)frexpf(__uint_as_float(m), &e);
  const int k = finite ? e - 14 : 0;
  if (tid == 0) tscale[(size_t)sp * tokens + t] = !finite ? __builtin_nanf("") : m ? ldexpf(1.f, k) : 1.f;
  constexpr int TPT = HL ? 16 : 32;  // tokens per operand tile
  const int tile = t / TPT, r = t % TPT;
  auto put = [&](int u, const float4 a, const float4 c) {
    const float v[8] = {a.x, a.y, a.z, a.w, c.x, c.y, c.z, c.w};
    const bool live = valid && finite;
    float s[8], sum = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      s[j] = live ? ldexpf(v[j], -k) : 0.f;
      sum += s[j];
    }
    f16x8 hi, lo;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      hi[j] = (_Float16)s[perm8(j)];
      lo[j] = (_Float16)(s[perm8(j)] - (float)hi[j]);
    }
    const int b = u >> 5, q = u & 31;
    u32x4 *d = xa + ((size_t)tile * nblk + b) * (kSbUnits * 64);
    d[(q >> 1) * 64 + 32 * (q & 1) + r] = __builtin_bit_cast(u32x4, hi);
    if (HL) d[(q >> 1) * 64 + 32 * (q & 1) + 16 + r] = __builtin_bit_cast(u32x4, lo);
    // Sub-block sums: four neighbouring threads, added in pairs (units of a sub-block in one wave).
    sum += __shfl_xor(sum, 1);
    sum += __shfl_xor(sum, 2);
    if ((q & 3) == 0) {
      const float S = sum * 0.03125f;
      const _Float16 Sh = (_Float16)S;
      _Float16 *su = reinterpret_cast<_Float16 *>(d + 16 * 64);
      su[8 * r + perm8(q >> 2)] = Sh;
      if (HL) su[8 * (16 + r) + perm8(q >> 2)] = (_Float16)(S - (float)Sh);
    }
    if (q == 0) {
      d[16 * 64 + 32 + r] = u32x4{0u, 0u, 0u, 0u};
      if (HL) d[16 * 64 + 48 + r] = u32x4{0u, 0u, 0u, 0u};
    }
  };
  if (UPT > 0) {
#pragma unroll
    for (int j = 0; j < UPT; ++j) {
      const int u = u0 + tid + 256 * j;
      if (u < u1) put(u, reg[j][0], reg[j][1]);
    }
  } else {
    for (int u = u0 + tid; u < u1; u += 256) put(u, row[2 * u], row[2 * u + 1]);
  }
}

#define FHIP_LDS_BARRIER_MID(imm)    \
  do {                               \
    __builtin_amdgcn_s_waitcnt(imm); \
    asm volatile("" ::: "memory");   \
    __builtin_amdgcn_s_barrier();    \
    asm volatile("" ::: "memory");   \
  } while (0)
constexpr int wait_vm_mid(int n) { return 0x0070 | (n & 15) | ((n >> 4) << 14); }

// Workgroup = NW waves x 32 rows x TT operand tiles over one K range. A stage is half a super-block:
// 8 operand units per tile, shared by the waves, and each wave's two record parts; three buffers, each
// stage loaded two ahead. The super-block's headers and sum units come with its first half.
template <int TT, bool HL, int NW>
__global__ __launch_bounds__(64 * NW) void q4k_mid_kernel(const uint8_t *__restrict__ W,
                                                          const u32x4 *__restrict__ xa,
                                                          const float *__restrict__ tscale,
                                                          float *__restrict__ Y, float *__restrict__ part,
                                                          int N, int M, int nblk, int ntiles, int MTG,
                                                          int tokens, int SK) {
  constexpr int kAU = TT * 8 * 64, kWW = 2 * 64;  // operand units of a stage; a wave's record units
  constexpr int kSU = kAU + NW * kWW;             // one stage: operands, then each wave's records
  constexpr int kHU = NW * 64 + TT * 64;          // per super-block: headers (32 + 32 repeats), S units
  __shared__ u32x4 S0[kSU], S1[kSU], S2[kSU];
  __shared__ u32x4 H0[kHU], H1[kHU], H2[kHU];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kap = lane >> 5, rho = lane & 31, r16 = rho & 15;
  const int sp = blockIdx.x % SK, task = blockIdx.x / SK, mg = task % MTG, ng = task / MTG;
  const int b0 = sp * nblk / SK, b1 = (sp + 1) * nblk / SK, nb = b1 - b0;
  const int tile0 = 2 * NW * ng + 2 * wave;
  const int t0c = min(tile0, ntiles - 1), t1c = min(tile0 + 1, ntiles - 1);
  auto sbuf = [&](int k) -> u32x4 * { return k == 0 ? S0 : k == 1 ? S1 : S2; };
  auto hbuf = [&](int k) -> u32x4 * { return k == 0 ? H0 : k == 1 ? H1 : H2; };
  const int off16 = 16 * lane;
  const int offh = (lane & 16 ? (t1c - t0c) * nblk * kQ4kRecord : 0) + 16 * (lane & 15);
  const void *ra = xa + (size_t)TT * mg * nblk * (kSbUnits * 64);
  const void *rw0 = W + (size_t)t0c * nblk * kQ4kRecord;
  const void *rw1 = W + (size_t)t1c * nblk * kQ4kRecord;
  constexpr int kAL = 8 * TT / NW;  // operand loads per wave and stage
  // Stage s: half hh = s & 1 of super-block s / 2 of the range.
  auto load = [&](int b, int hh, u32x4 *sd, u32x4 *hd) {
    const int bc = b0 + min(b, nb - 1), so = bc * kQ4kRecord;
    if (hh == 0) {
      lds_load16(rw0, hd + wave * 64, offh, so);
      lds_load16(ra, hd + (NW * 64 + (wave % TT) * 64), off16, (((wave % TT) * nblk + bc) * kSbUnits + 16) * 1024);
    }
    lds_load16(rw0, sd + (kAU + wave * kWW), off16, so + kQ4kHdr + 1024 * hh);
    lds_load16(rw1, sd + (kAU + wave * kWW + 64), off16, so + kQ4kHdr + 1024 * hh);
#pragma unroll
    for (int j = 0; j < kAL; ++j) {
      const int un = kAL * wave + j, i = un >> 3, q = un & 7;  // token tile, slice of the half
      lds_load16(ra, sd + un * 64, off16, ((i * nblk + bc) * kSbUnits + 8 * hh + q) * 1024);
    }
  };
  f32x16 acc[TT], tmp[TT][2];
#pragma unroll
  for (int i = 0; i < TT; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[i][e] = 0.f;
  load(0, 0, S0, H0);
  load(0, 1, S1, nullptr);
  FHIP_LDS_BARRIER_MID(wait_vm_mid(0));

  const uint32_t al = in_reg(lane);
  const uint32_t wl = in_reg(kAU + wave * kWW + 64 * (rho >> 4) + 16 * kap + r16), hl = in_reg(wave * 64 + (rho & 31));
  const uint32_t kLo = in_reg(0x000F000Fu), kHi = in_reg(0x00F000F0u);
  const uint32_t kMagic = in_reg(0x64006400u), kB02 = in_reg(0x00FF00FFu);
  const h2 k1024 = {(_Float16)1024.f, (_Float16)1024.f}, kN1024 = -k1024;
  const h2 k16th = {(_Float16)0.0625f, (_Float16)0.0625f}, k32 = {(_Float16)32.f, (_Float16)32.f};
  constexpr int kEven = 4 + kAL, kOdd = 2 + kAL;  // loads of an even / odd stage
  for (int bb = 0; bb < nb; bb += 3) {
#pragma unroll
    for (int u = 0; u < 6; ++u) {
      const int b = bb + u / 2, hh = u & 1;
      load(b + 1, hh, sbuf((u + 2) % 3), hbuf((u / 2 + 1) % 3));
      if (b < nb) {
        const u32x4 *Sb = sbuf(u % 3), *Hb = hbuf(u / 2);
        // the super-block's scales (read again at each half: cheaper than held registers)
        const u32x4 hd = Hb[hl];
        const uint32_t sc4 = hh == 0 ? hd[1] & 0x3F3F3F3Fu : (hd[3] & 0x0F0F0F0Fu) | ((hd[1] >> 2) & 0x30303030u);
        const h2 ep = as_h2((sc4 & kB02) | kMagic) - k1024;         // sub-blocks 4 hh, 4 hh + 2
        const h2 op = as_h2(((sc4 >> 8) & kB02) | kMagic) - k1024;  // 4 hh + 1, 4 hh + 3
        const u32x4 nb0 = Sb[wl], nb1 = Sb[wl + 32];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const _Float16 sa = c ? ep.y : ep.x, sb = c ? op.y : op.x;
          const h2 SL = {sa, sa}, SH = h2{sb, sb} * k16th;
          const h2 NL = SL * kN1024, NH = SH * kN1024;
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const u32x4 q = h ? nb1 : nb0;
            const uint32_t x0 = c ? q[2] : q[0], x1 = c ? q[3] : q[1];
            const uint32_t y0 = x0 >> 8, y1 = x1 >> 8;
            u32x4 lw, hw;
            lw[0] = as_u(__builtin_elementwise_fma(as_h2((x0 & kLo) | kMagic), SL, NL));
            lw[1] = as_u(__builtin_elementwise_fma(as_h2((y0 & kLo) | kMagic), SL, NL));
            lw[2] = as_u(__builtin_elementwise_fma(as_h2((x1 & kLo) | kMagic), SL, NL));
            lw[3] = as_u(__builtin_elementwise_fma(as_h2((y1 & kLo) | kMagic), SL, NL));
            hw[0] = as_u(__builtin_elementwise_fma(as_h2((x0 & kHi) | kMagic), SH, NH));
            hw[1] = as_u(__builtin_elementwise_fma(as_h2((y0 & kHi) | kMagic), SH, NH));
            hw[2] = as_u(__builtin_elementwise_fma(as_h2((x1 & kHi) | kMagic), SH, NH));
            hw[3] = as_u(__builtin_elementwise_fma(as_h2((y1 & kHi) | kMagic), SH, NH));
#pragma unroll
            for (int hi = 0; hi < 2; ++hi)
#pragma unroll
              for (int i = 0; i < TT; ++i) {
                const f16x8 a = __builtin_bit_cast(f16x8, Sb[(i * 8 + 4 * c + 2 * hi + h) * 64 + al]);
                f32x16 z = tmp[i][hi];
                if (hh == 0 && c == 0 && h == 0)
#pragma unroll
                  for (int e = 0; e < 16; ++e) z[e] = 0.f;
                tmp[i][hi] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, __builtin_bit_cast(f16x8, hi ? hw : lw), z, 0, 0, 0);
              }
          }
        }
        if (hh == 1) {
          const float d = (float)__builtin_bit_cast(_Float16, (uint16_t)(hd[0] & 0xffffu));
          const float dm = (float)__builtin_bit_cast(_Float16, (uint16_t)(hd[0] >> 16));
          const uint32_t mnl = hd[2] & 0x3F3F3F3Fu;
          const uint32_t mnh = ((hd[3] >> 4) & 0x0F0F0F0Fu) | ((hd[2] >> 2) & 0x30303030u);
          u32x4 mw;
          mw[0] = as_u((as_h2((mnl & kB02) | kMagic) - k1024) * k32);
          mw[1] = as_u((as_h2(((mnl >> 8) & kB02) | kMagic) - k1024) * k32);
          mw[2] = as_u((as_h2((mnh & kB02) | kMagic) - k1024) * k32);
          mw[3] = as_u((as_h2(((mnh >> 8) & kB02) | kMagic) - k1024) * k32);
#pragma unroll
          for (int i = 0; i < TT; ++i) {
            f32x16 mt;
#pragma unroll
            for (int e = 0; e < 16; ++e) mt[e] = 0.f;
            mt = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, Hb[(NW + i) * 64 + al]),
                                                        __builtin_bit_cast(f16x8, mw), mt, 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 16; ++e)
              acc[i][e] = fmaf(d, tmp[i][0][e] + tmp[i][1][e], fmaf(-dm, mt[e], acc[i][e]));
          }
        }
      }
      if (hh == 0)
        FHIP_LDS_BARRIER_MID(wait_vm_mid(kEven));
      else
        FHIP_LDS_BARRIER_MID(wait_vm_mid(kOdd));
    }
  }
  __builtin_amdgcn_s_waitcnt(wait_vm_mid(0));

  const int o = 32 * NW * ng + 32 * wave + rho;
  if (o >= N) return;
  constexpr int TPT = HL ? 16 : 32, NV = HL ? 8 : 16;
  float4 sc[TT][NV / 4];  // every scale before the first store: a store would wait for a load after it
#pragma unroll
  for (int i = 0; i < TT; ++i)
#pragma unroll
    for (int a = 0; a < NV / 4; ++a)
      sc[i][a] = *reinterpret_cast<const float4 *>(tscale + (size_t)sp * tokens + TPT * (TT * mg + i) + 8 * a + 4 * kap);
#pragma unroll
  for (int i = 0; i < TT; ++i)
#pragma unroll
    for (int e = 0; e < NV; ++e) {
      const int tok = TPT * (TT * mg + i) + 8 * (e >> 2) + 4 * kap + (e & 3);
      if (tok >= M) continue;
      const float v = (HL ? acc[i][e] + acc[i][(e + 8) & 15] : acc[i][e]) *
                      ((e & 3) == 0 ? sc[i][e >> 2].x : (e & 3) == 1 ? sc[i][e >> 2].y : (e & 3) == 2 ? sc[i][e >> 2].z : sc[i][e >> 2].w);
      if (SK == 1)
        Y[(size_t)tok * N + o] = v;
      else
        part[((size_t)sp * M + tok) * N + o] = v;
    }
}
#undef FHIP_LDS_BARRIER_MID

}  // namespace

namespace {

struct MidPlan {
  bool hl;
  int TT, NW, MTG, tokens, tasks, SK;
  size_t xb, tb, pb;  // operands, token scales, K-range partial results
  float cost;
};

// The K split with the lowest estimated time (us): the longest range's super-blocks at the pace of one
// workgroup per CU (t1), or of two (t2, where two fit), in as many rounds as the grid takes, and for a
// split the launch that adds the ranges and its traffic. Fitted to sweeps of the range count at ten
// shapes from 1536 x 1024 to 5120 x 25600; the choice is the best or within 4% of it at each.
MidPlan plan_mid(int N, int K, int M, int TT, int NW) {
  MidPlan p{};
  const int nblk = K / 256, cus = cu_count() > 0 ? cu_count() : 256;
  p.hl = M <= 16;
  p.TT = TT;
  p.NW = NW;
  p.MTG = p.hl ? 1 : ceil_div(M, 32 * TT);
  p.tokens = p.hl ? 16 : 32 * TT * p.MTG;
  p.tasks = p.MTG * ceil_div(N, 32 * NW);
  const float t1 = TT == 2 ? 2.0f : 1.15f, t2 = 1.9f;
  const int fit = NW == 8 ? 1 : 2;  // workgroups per CU
  for (int sk = 1; sk <= nblk && sk <= 32; ++sk) {
    const long long wgs = (long long)p.tasks * sk;
    const float pace = wgs <= cus || fit == 1 ? t1 : t2;
    const float rounds = wgs <= cus ? 1.f : (float)((wgs + fit * cus - 1) / (fit * cus));
    const float c = rounds * ceil_div(nblk, sk) * pace +
                    (sk > 1 ? 2.2f + 8.f * sk * (float)M * (float)N / 3.5e6f : 0.f);
    if (sk == 1 || c < p.cost) {
      p.cost = c;
      p.SK = sk;
    }
  }
  p.xb = (size_t)(p.hl ? 1 : TT * p.MTG) * nblk * kSbUnits * 1024;
  p.tb = ((size_t)p.SK * p.tokens * 4 + 255) & ~(size_t)255;
  p.pb = p.SK > 1 ? (size_t)p.SK * M * N * 4 : 0;
  return p;
}

// One operand tile and four waves per workgroup, or (above 32 tokens) two tiles and eight waves, which
// halve the operand traffic of a large matrix: 64 tokens of 18944 x 3584 32.2 / 28.3 us, of 3584 x 3584
// 14.8 / 18.6.
MidPlan plan_mid(int N, int K, int M) {
  const MidPlan p = plan_mid(N, K, M, 1, 4);
  if (M <= 32) return p;
  const MidPlan q = plan_mid(N, K, M, 2, 8);
  return q.cost < p.cost ? q : p;
}

}  // namespace

// Which calls take this kernel (us, before / here). Up to 16 tokens matrices of up to 36 M weights
// (3584 x 3584 at 8 tokens 17.8 / 10.6, 8192 x 4096 14.6 / 13.4, 4096 x 8192 15.0 / 13.4; larger ones
// mostly lose: 11008 x 4096 15.2 / 15.8, 25600 x 5120 23.9 / 27); 17..64 tokens all (8192 x 4096 at 32,
// the closest, 17.4 / 16.1); 65..128 small matrices (4096 x 4096 at 128 tokens 24.0 / 20.7, 8192 x 4096
// at 65 23.7 / 25.2). Rows long enough to make the operands large keep the other kernels.
bool q4k_mid_takes(int N, int K, int M) {
  const long long w = (long long)N * K;
  if (M < 5 || K > 262144) return false;
  if (M <= 16) return w <= 36000000;
  if (M <= 64) return true;
  return M <= 128 && w <= 20000000;
}

size_t q4k_mid_ws_bytes(int N, int K, int M) {
  const MidPlan p = plan_mid(N, K, M);
  return p.xb + p.tb + p.pb;
}

int q4k_mid(const void *Wv, const float *X, float *Y, int N, int K, int M) {
  const MidPlan p = plan_mid(N, K, M);
  const int nblk = K / 256, ntiles = q4k_tiles(N), SK = p.SK, MTG = p.MTG, tokens = p.tokens;
  const size_t xb = p.xb, tb = p.tb, pb = p.pb;
  unsigned char *ws = (unsigned char *)workspace(xb + tb + pb);
  if (!ws) return FHIP_ENOMEM;
  if (int rc = check_disjoint("q4k_mid", X, (size_t)M * K * 4, ws, xb + tb + pb)) return rc;
  u32x4 *xa = (u32x4 *)ws;
  float *ts = (float *)(ws + xb), *part = (float *)(ws + xb + tb);
  const dim3 pg(tokens, SK);
  const int units = 32 * ceil_div(nblk, SK);
  auto prep = [&](auto hl) {
    constexpr bool H = decltype(hl)::value;
    if (units <= 256)
      mid_xprep_kernel<H, 1><<<pg, 256, 0, stream()>>>(X, M, K, nblk, SK, xa, ts);
    else if (units <= 512)
      mid_xprep_kernel<H, 2><<<pg, 256, 0, stream()>>>(X, M, K, nblk, SK, xa, ts);
    else
      mid_xprep_kernel<H, 0><<<pg, 256, 0, stream()>>>(X, M, K, nblk, SK, xa, ts);
  };
  if (p.hl)
    prep(std::true_type{});
  else
    prep(std::false_type{});
  FHIP_CHECK_LAUNCH("mid_xprep_kernel");
  const uint8_t *W = (const uint8_t *)Wv;
  auto run = [&](auto kern) {
    kern<<<p.tasks * SK, 64 * p.NW, 0, stream()>>>(W, xa, ts, Y, part, N, M, nblk, ntiles, MTG, tokens, SK);
  };
  if (p.hl)
    run(q4k_mid_kernel<1, true, 4>);
  else if (p.TT == 1)
    run(q4k_mid_kernel<1, false, 4>);
  else
    run(q4k_mid_kernel<2, false, 8>);
  FHIP_CHECK_LAUNCH("q4k_mid_kernel");
  return SK > 1 ? sum_ranges(part, Y, SK, M * N) : FHIP_OK;
}

}  // namespace fhip
