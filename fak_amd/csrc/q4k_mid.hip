// q4k_mid.hip — Q4_K and Q6_K matmul for a few tokens to a few tens (speculative verify, short prompts;
// up to 128 on small matrices) on the 32x32x16 f16 MFMA.
//
// The arithmetic is that of q4k_gemv16.hip: weight operands are exact (Q4_K the integers sc_s * n, Q6_K
// sc_g (q - 32) / 4 as two operands), each super-block's f32 result is scaled by the row's d, Q4_K's min
// term is one more MFMA over the sub-block sums, and activations are scaled by a power of two per
// (token, K range) that puts the range's largest magnitude in [2^13, 2^14). Up to 16 tokens the 32
// operand rows are the f16 of each value and the f16 of its remainder (~22 bits); above, 32 tokens in
// f16. A range with a super-block whose largest magnitude lies 2^13 and more below the range's has a scale
// per super-block instead (up to 32 tokens), applied to the super-block's sum: the range's would leave such
// values too few bits, or none, and they are all there is where the weights of the larger ones are zero.
//
// The data path is another: the operands are made once per call (mid_xprep_kernel), not by every
// workgroup, and every workgroup streams them and its weight records to LDS by direct loads two
// stages ahead, so no load returns to a register and nothing but the MFMAs' own operands is converted
// in the loop. What bounds it: a workgroup's super-block takes about 1.15 us (Q6_K 1.6: a wave's own
// chain of LDS reads, unpack and MFMAs; its 37 (44) KB of direct loads hide behind it), two on a CU
// 1.7 (2.5), near the memory's pace; so time is the longest range, plus the launches before and after it.
// us per call with cold weights (9 to 16 copies in turn) against the kernels it replaced (q4k_gemv16.hip, up
// to 16 tokens and its former 32-token form up to 32, the prefill GEMM for more):
//   Q4_K 3584 x 3584 at 8 / 16 / 32 / 64 tokens   18.1 / 18.5 / 18.2 / 22.4 -> 12.0 / 12.8 / 14.1 / 15.7
//        18944 x 3584                             20.7 / 21.8 / 30.6 / 34.1 -> 20.4 / 21.7 / 23.2 / 31.1
//        8192 x 11008                             31.2 / 33.4 / 42.5 / 41.0 -> 22.5 / 24.3 / 25.7 / 34.8
//   Q6_K 3584 x 3584 at 2 / 16 / 32 / 64          18.1 / 18.7 / 21.3 / 26.0 -> 12.9 / 13.5 / 14.8 / 17.0
//        18944 x 3584                             29.0 / 32.0 / 36.6 / 38.8 -> 24.0 / 27.8 / 29.2 / 36.8
//        5120 x 25600                             42.5 / 47.7 / 55.8 / 60.9 -> 36.3 / 40.7 / 41.4 / 54.1
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
                                                        float *__restrict__ tscale,
                                                        float *__restrict__ bscale) {
  __shared__ uint32_t wmax[4], wmin[4];
  const int tokens = gridDim.x, t = blockIdx.x, sp = blockIdx.y, tid = threadIdx.x;
  const int u0 = 32 * (sp * nblk / SK), u1 = 32 * ((sp + 1) * nblk / SK);
  const bool valid = t < M;
  const float4 *row = reinterpret_cast<const float4 *>(X + (size_t)(valid ? t : 0) * K);
  uint32_t m = 0, mn = ~0u;  // largest magnitude, and smallest of a super-block's that are not zero
  float4 reg[UPT > 0 ? UPT : 1][2];
  // Largest magnitude of a super-block: its 32 units are half a wave's.
  auto block_max = [](const float4 a, const float4 c) {
    uint32_t w = max(absmax4_bits(a.x, a.y, a.z, a.w), absmax4_bits(c.x, c.y, c.z, c.w));
    w = max(w, lane_xor<1>(w));
    w = max(w, lane_xor<2>(w));
    w = max(w, group_mirror<8>(w));
    w = max(w, group_mirror<16>(w));
    return max(w, (uint32_t)__shfl_xor((int)w, 16));
  };
  auto see = [&](const uint32_t w) {
    m = max(m, w);
    mn = min(mn, w - 1);  // zero last
  };
  auto real = [&](int u) { return u < u1 ? u : u1 - 32 + (u & 31); };  // repeats do not change either
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
    for (int u = u0 + tid; u < u1; u += 256) see(block_max(row[2 * u], row[2 * u + 1]));
  }
  m = max(m, (uint32_t)__shfl_xor((int)m, 32));
  mn = min(mn, (uint32_t)__shfl_xor((int)mn, 32));
  if ((tid & 63) == 0) {
    wmax[tid >> 6] = m;
    wmin[tid >> 6] = mn;
  }
  __syncthreads();
  m = valid ? max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3])) : 0u;
  mn = min(min(wmin[0], wmin[1]), min(wmin[2], wmin[3])) + 1;
  const bool finite = m < 0x7F800000u;
  // The exponent that puts w in [2^13, 2^14), at least -126: 2^k stays normal, and the bits of magnitudes
  // below 2^-112 all fit in the operands.
  auto exponent = [](uint32_t w) {
    int e = 0;
    (void)frexpf(__uint_as_float(w), &e);
    return max(e - 14, -126);
  };
  const int k = finite && m ? exponent(m) : 0;
  const bool fine = bscale && finite && m && (m >> 23) > (mn >> 23) + 13;
  // -1: the scales are the super-blocks'
  if (tid == 0) tscale[(size_t)sp * tokens + t] = !finite ? __builtin_nanf("") : fine ? -1.f : ldexpf(1.f, k);
  constexpr int TPT = HL ? 16 : 32;  // tokens per operand tile
  const int tile = t / TPT, r = t % TPT;
  auto put = [&](int u, const float4 a, const float4 c) {
    const float v[8] = {a.x, a.y, a.z, a.w, c.x, c.y, c.z, c.w};
    const bool live = valid && finite;
    const int b = u >> 5, q = u & 31;
    int kb = k;
    if (fine) {  // uniform over the workgroup
      const uint32_t w = block_max(a, c);
      kb = w ? exponent(w) : 0;
      if (q == 0) bscale[((size_t)tile * nblk + b) * TPT + r] = ldexpf(1.f, kb);
    }
    float s[8], sum = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      s[j] = live ? ldexpf(v[j], -kb) : 0.f;
      sum += s[j];
    }
    f16x8 hi, lo;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      hi[j] = (_Float16)s[perm8(j)];
      lo[j] = (_Float16)(s[perm8(j)] - (float)hi[j]);
    }
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
// The wave count is what the LDS allows; stated, it keeps the super-block results that the VALU scales in
// VGPRs (the compiler had taken AGPRs for one operand tile).
template <int FMT, int TT, bool HL, int NW>  // FMT 0: Q4_K, 1: Q6_K
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2, 2))) void quant_mid_kernel(const uint8_t *__restrict__ W,
                                                            const u32x4 *__restrict__ xa,
                                                            const float *__restrict__ tscale,
                                                            const float *__restrict__ bscale,
                                                            float *__restrict__ Y, float *__restrict__ part,
                                                            int N, int M, int nblk, int ntiles, int MTG,
                                                            int tokens, int SK) {
  constexpr int kRec = FMT == 0 ? kQ4kRecord : kQ6kRecord, kWL = FMT == 0 ? 2 : 3;  // record loads per stage
  constexpr int kAU = TT * 8 * 64, kWW = kWL * 64;  // operand units of a stage; a wave's record units
  constexpr int kSU = kAU + NW * kWW;             // one stage: operands, then each wave's records
  constexpr int kHU = NW * 64 + (FMT == 0 ? TT * 64 : 0);  // per super-block: headers, Q4_K S units
  __shared__ u32x4 S0[kSU], S1[kSU], S2[kSU];
  __shared__ u32x4 H0[kHU], H1[kHU], H2[kHU];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kap = lane >> 5, rho = lane & 31, r16 = rho & 15;
  // Workgroups go to the 8 XCDs in turn; each XCD takes a contiguous run of (range, rows, tokens), so its
  // L2 holds the operands of one or two ranges and a record read for one token group serves the next.
  const int x = blockIdx.x & 7, per = gridDim.x >> 3, id = x * per + min(x, (int)(gridDim.x & 7)) + (blockIdx.x >> 3);
  const int tasks = gridDim.x / SK, sp = id / tasks, task = id - sp * tasks, mg = task % MTG, ng = task / MTG;
  const int b0 = sp * nblk / SK, b1 = (sp + 1) * nblk / SK, nb = b1 - b0;
  const int tile0 = 2 * NW * ng + 2 * wave;
  const int t0c = min(tile0, ntiles - 1), t1c = min(tile0 + 1, ntiles - 1);
  auto sbuf = [&](int k) -> u32x4 * { return k == 0 ? S0 : k == 1 ? S1 : S2; };
  auto hbuf = [&](int k) -> u32x4 * { return k == 0 ? H0 : k == 1 ? H1 : H2; };
  const int off16 = 16 * lane;
  // Header loads of the 32 rows (tiles t0c, t1c): Q4_K lane l row l % 32's 16 bytes; Q6_K lane l < 32 the
  // row's scales, lanes 32..35 the rows' d, the rest repeat them.
  const int dt = (t1c - t0c) * nblk * kRec;
  const int offh = FMT == 0 || lane < 32 ? (lane & 16 ? dt : 0) + 16 * (lane & 15)
                                         : (lane & 2 ? dt : 0) + kQ6kD + 16 * (lane & 1);
  const int offq = (lane & 32 ? dt : 0) + 16 * (lane & 31);  // Q6_K: both tiles' qh
  const void *ra = xa + (size_t)TT * mg * nblk * (kSbUnits * 64);
  const void *rw0 = W + (size_t)t0c * nblk * kRec;
  const void *rw1 = W + (size_t)t1c * nblk * kRec;
  constexpr int kAL = 8 * TT / NW;  // operand loads per wave and stage
  // Stage s: half hh = s & 1 of super-block s / 2 of the range.
  auto load = [&](int b, int hh, u32x4 *sd, u32x4 *hd) {
    const int bc = b0 + min(b, nb - 1), so = bc * kRec;
    if (hh == 0) {
      lds_load16(rw0, hd + wave * 64, offh, so);
      if (FMT == 0)
        lds_load16(ra, hd + (NW * 64 + (wave % TT) * 64), off16, (((wave % TT) * nblk + bc) * kSbUnits + 16) * 1024);
    }
    constexpr int kQ = FMT == 0 ? kQ4kHdr : kQ6kQl;
    lds_load16(rw0, sd + (kAU + wave * kWW), off16, so + kQ + 1024 * hh);
    lds_load16(rw1, sd + (kAU + wave * kWW + 64), off16, so + kQ + 1024 * hh);
    if (FMT == 1) lds_load16(rw0, sd + (kAU + wave * kWW + 128), offq, so + kQ6kQh + 512 * hh);
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
  constexpr int TPT = HL ? 16 : 32, NV = HL ? 8 : 16;  // tokens per operand tile, of them a lane's
  const float tsl = TT == 1 ? tscale[(size_t)sp * tokens + TPT * mg + (lane & (TPT - 1))] : 0.f;
  load(0, 0, S0, H0);
  load(0, 1, S1, nullptr);
  FHIP_LDS_BARRIER_MID(wait_vm_mid(0));

  const uint32_t al = in_reg(lane);
  const uint32_t wl = in_reg(kAU + wave * kWW + 64 * (rho >> 4) + 16 * kap + r16), hl = in_reg(wave * 64 + (rho & 31));
  const uint32_t kLo = in_reg(0x000F000Fu), kHi = in_reg(0x00F000F0u);
  const uint32_t kMagic = in_reg(0x64006400u), kB02 = in_reg(0x00FF00FFu);
  const h2 k1024 = {(_Float16)1024.f, (_Float16)1024.f}, kN1024 = -k1024;
  const h2 k16th = {(_Float16)0.0625f, (_Float16)0.0625f}, k32 = {(_Float16)32.f, (_Float16)32.f};
  constexpr int kEven = (FMT == 0 ? 2 : 1) + kWL + kAL, kOdd = kWL + kAL;  // loads of an even / odd stage
  // Q6_K: this lane's 8 ql bytes of (tile, group h), qh bytes and d, in units of 8 and 2 bytes.
  const uint32_t ql = FMT == 1 ? in_reg(2 * (kAU + wave * kWW + 64 * (rho >> 4) + r16) + kap) : 0u;
  const uint32_t qq = FMT == 1 ? in_reg(2 * (kAU + wave * kWW + 128 + 32 * (rho >> 4) + r16) + kap) : 0u;
  const uint32_t dl = FMT == 1 ? in_reg(8 * (wave * 64 + 32 + 2 * (rho >> 4)) + r16) : 0u;
  const uint32_t k80 = FMT == 1 ? in_reg(0x80808080u) : 0u;
  const uint32_t kB6 = FMT == 1 ? in_reg(0x00C000C0u) : 0u, kB8 = FMT == 1 ? in_reg(0x03000300u) : 0u;
  const h2 k1152 = {(_Float16)1152.f, (_Float16)1152.f}, k4th = {(_Float16)0.25f, (_Float16)0.25f};
  const h2 k64th = k16th * k4th, kTb = {(_Float16)0.0625f, (_Float16)0.015625f};  // b under 2^6, 2^8
  const h2 kOb = {(_Float16)-72.f, (_Float16)-24.f};  // -(1024 + 2 2^6) / 16, -(1024 + 2 2^8) / 64
  auto range = [&](auto fine) {  // fine: with super-block scales
    for (int bb = 0; bb < nb; bb += 3) {
#pragma unroll
      for (int u = 0; u < 6; ++u) {
        const int b = bb + u / 2, hh = u & 1;
        load(b + 1, hh, sbuf((u + 2) % 3), hbuf((u / 2 + 1) % 3));
        if (b < nb) {
          const u32x4 *Sb = sbuf(u % 3), *Hb = hbuf(u / 2);
          float bs[NV];  // this super-block's scales, 1 for tokens whose range has one scale
          if constexpr (decltype(fine)::value) {
            if (hh == 1) {
#pragma unroll
              for (int a = 0; a < NV / 4; ++a) {
                const int r = 8 * a + 4 * kap;
                const float4 s4 = *reinterpret_cast<const float4 *>(
                    bscale + ((size_t)mg * nblk + b0 + b) * TPT + r);
                const float4 t4 = *reinterpret_cast<const float4 *>(tscale + (size_t)sp * tokens + TPT * mg + r);
                bs[4 * a] = t4.x < 0.f ? s4.x : 1.f;
                bs[4 * a + 1] = t4.y < 0.f ? s4.y : 1.f;
                bs[4 * a + 2] = t4.z < 0.f ? s4.z : 1.f;
                bs[4 * a + 3] = t4.w < 0.f ? s4.w : 1.f;
              }
            }
          }
          if constexpr (FMT == 0) {
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
                for (int e = 0; e < 16; ++e) {
                  if constexpr (decltype(fine)::value)
                    acc[i][e] = fmaf(d, (tmp[i][0][e] + tmp[i][1][e]) * bs[e % NV], fmaf(-dm, mt[e] * bs[e % NV], acc[i][e]));
                  else
                    acc[i][e] = fmaf(d, tmp[i][0][e] + tmp[i][1][e], fmaf(-dm, mt[e], acc[i][e]));
                }
              }
            }
          } else {
            // Q6_K: group g = K16 slice g. With q = n + 16 b (nibble n, qh field b), sc_g (q - 32) / 4 is the
            // sum of two operands that f16 holds exactly, sc_g n / 4 (up to 480) and 4 sc_g (b - 2) (up to
            // 1024), each one fma of the field under the exponent of 1024 (n 2^(4 c), b 2^(6 + 2 hi)). Both
            // feed one chain, whose running sum is that of the whole weights: with a chain each the error
            // against 64 bits is 4% larger.
            const uint2 *Q = reinterpret_cast<const uint2 *>(Sb);
            const u32x4 hd = Hb[hl];
#pragma unroll
            for (int c = 0; c < 2; ++c) {
              const uint32_t sw = hd[2 * hh + c] ^ k80;
#pragma unroll
              for (int h = 0; h < 2; ++h) {
                const h2 P = as_h2(((h ? sw >> 8 : sw) & kB02) | kMagic) - k1152;  // scales of hi = 0, 1
                const h2 SP = P * (c ? k64th : k4th), NP = SP * kN1024, TP = P * kTb, OP = P * kOb;
                const uint2 qa = Q[ql + 32 * h], qb = Q[ql + 64 + 32 * h], qh = Q[qq + 32 * h];
#pragma unroll
                for (int hi = 0; hi < 2; ++hi) {
                  const _Float16 s = hi ? SP.y : SP.x, n = hi ? NP.y : NP.x, t = hi ? TP.y : TP.x, o = hi ? OP.y : OP.x;
                  const h2 S = {s, s}, N0 = {n, n}, T = {t, t}, O = {o, o};
                  const uint32_t mn = c ? kHi : kLo, mb = hi ? kB8 : kB6;
                  u32x4 vn, vb;
#pragma unroll
                  for (int m = 0; m < 2; ++m) {
                    const uint32_t x = hi ? (m ? qb.y : qb.x) : (m ? qa.y : qa.x), b4 = m ? qh.y : qh.x;
                    const uint32_t be = b4 << (c ? 2 : 6), bo = b4 >> (c ? 6 : 2);
                    vn[2 * m] = as_u(__builtin_elementwise_fma(as_h2((x & mn) | kMagic), S, N0));
                    vn[2 * m + 1] = as_u(__builtin_elementwise_fma(as_h2(((x >> 8) & mn) | kMagic), S, N0));
                    vb[2 * m] = as_u(__builtin_elementwise_fma(as_h2((be & mb) | kMagic), T, O));
                    vb[2 * m + 1] = as_u(__builtin_elementwise_fma(as_h2((bo & mb) | kMagic), T, O));
                  }
#pragma unroll
                  for (int i = 0; i < TT; ++i) {
                    const f16x8 a = __builtin_bit_cast(f16x8, Sb[(i * 8 + 4 * c + 2 * hi + h) * 64 + al]);
                    f32x16 z = tmp[i][hi];
                    if (hh == 0 && c == 0 && h == 0)
#pragma unroll
                      for (int e = 0; e < 16; ++e) z[e] = 0.f;
                    z = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, __builtin_bit_cast(f16x8, vn), z, 0, 0, 0);
                    tmp[i][hi] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, __builtin_bit_cast(f16x8, vb), z, 0, 0, 0);
                  }
                }
              }
            }
            if (hh == 1) {
              const float d = 4.f * (float)reinterpret_cast<const _Float16 *>(Hb)[dl];
#pragma unroll
              for (int i = 0; i < TT; ++i)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                  if constexpr (decltype(fine)::value)
                    acc[i][e] = fmaf(d, (tmp[i][0][e] + tmp[i][1][e]) * bs[e % NV], acc[i][e]);
                  else
                    acc[i][e] = fmaf(d, tmp[i][0][e] + tmp[i][1][e], acc[i][e]);
                }
            }
          }
        }
        if (hh == 0)
          FHIP_LDS_BARRIER_MID(wait_vm_mid(kEven));
        else
          FHIP_LDS_BARRIER_MID(wait_vm_mid(kOdd));
      }
    }
  };
  // In a loop of its own; two operand tiles have none (more than 32 tokens).
  if (TT == 1 && __builtin_amdgcn_ballot_w64(tsl < 0.f) != 0)
    range(std::integral_constant<bool, TT == 1>{});
  else
    range(std::false_type{});
  __builtin_amdgcn_s_waitcnt(wait_vm_mid(0));

  const int o = 32 * NW * ng + 32 * wave + rho;
  if (o >= N) return;
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
                      fabsf((e & 3) == 0 ? sc[i][e >> 2].x : (e & 3) == 1 ? sc[i][e >> 2].y : (e & 3) == 2 ? sc[i][e >> 2].z : sc[i][e >> 2].w);
      if (SK == 1)
        Y[(size_t)tok * N + o] = v;
      else
        part[((size_t)sp * M + tok) * N + o] = v;
    }
}
#undef FHIP_LDS_BARRIER_MID

}  // namespace

namespace {

constexpr int kF16Row = 262144;  // rows longer than this take hi and lo operands up to 32 tokens
constexpr int kMidRanges = 64;  // what sum_ranges reads at once
// Operands (at most 36 MB, by mid_takes) and partial results together stay well inside the 64 MiB of the
// no-allocation entry, whatever the shape. (Longer rows come from Q6_K only, which has no such entry.)
constexpr size_t kMidScratch = (size_t)48 << 20;

struct MidPlan {
  bool hl;
  int TT, NW, MTG, tokens, tasks, SK;
  size_t xb, tb, bb, pb;  // operands, token scales, super-block scales, K-range partial results
  float cost;
};

// The K split with the lowest estimated time (us): the super-blocks of a range (between the mean and the
// longest) at the pace of one workgroup per CU, or of two where the grid gives a CU two and they fit, in
// as many rounds as the grid takes, and for a split the launch that adds the ranges and its traffic.
// Fitted to sweeps of the range count at 75 shapes from 500 x 1024 to 25600 x 5120 and 2..128 tokens:
// the choice is within 1.5% of the best there on average, 10% at the worst.
struct MidPace {
  float one, two, wide, longest, start, launch, range, traffic;
};
constexpr MidPace kMidPace[2] = {{1.13f, 1.68f, 2.15f, 0.61f, 0.4f, 1.9f, 0.06f, 7.4f / 3.5e6f},
                                 {1.52f, 2.53f, 3.67f, 0.87f, 1.3f, 1.9f, 0.07f, 6.0f / 3.5e6f}};
MidPlan plan_mid(int fmt, int N, int K, int M, int TT, int NW) {
  MidPlan p{};
  const int nblk = K / 256, cus = cu_count() > 0 ? cu_count() : 256;
  p.hl = M <= 16 || K > kF16Row;
  p.TT = TT;
  p.NW = NW;
  p.MTG = p.hl ? ceil_div(M, 16) : ceil_div(M, 32 * TT);
  p.tokens = p.hl ? 16 * p.MTG : 32 * TT * p.MTG;
  p.tasks = p.MTG * ceil_div(N, 32 * NW);
  const MidPace &m = kMidPace[fmt];
  const int fit = NW == 8 ? 1 : 2;  // workgroups per CU
  p.xb = (size_t)TT * p.MTG * nblk * kSbUnits * 1024;
  for (int sk = 1; sk <= nblk && sk <= kMidRanges; ++sk) {
    if (sk > 1 && K <= kF16Row && p.xb + (size_t)sk * M * N * 4 > kMidScratch) break;
    const long long wgs = (long long)p.tasks * sk;
    const float pace = fit == 1 ? m.wide : wgs <= cus ? m.one : m.two;
    const float rounds = wgs <= cus ? 1.f : (float)((wgs + fit * cus - 1) / (fit * cus));
    const float len = m.longest * ceil_div(nblk, sk) + (1.f - m.longest) * nblk / sk;
    const float c = rounds * (len * pace + m.start) +
                    (sk > 1 ? m.launch + m.range * sk + m.traffic * sk * (float)M * (float)N : 0.f);
    if (sk == 1 || c < p.cost) {
      p.cost = c;
      p.SK = sk;
    }
    if (rounds > 3.f) break;  // more ranges only add rounds
  }
  p.tb = ((size_t)p.SK * p.tokens * 4 + 255) & ~(size_t)255;
  p.bb = M <= 32 ? ((size_t)p.tokens * nblk * 4 + 255) & ~(size_t)255 : 0;
  p.pb = p.SK > 1 ? (size_t)p.SK * M * N * 4 : 0;
  return p;
}

// One operand tile and four waves per workgroup, or (above 32 tokens) two tiles and eight waves, which
// halve the operand traffic of a large matrix: 64 tokens of 18944 x 3584 32.2 / 28.3 us, of 3584 x 3584
// 14.8 / 18.6.
MidPlan plan_mid(int fmt, int N, int K, int M) {
  const MidPlan p = plan_mid(fmt, N, K, M, 1, 4);
  if (M <= 32) return p;
  const MidPlan q = plan_mid(fmt, N, K, M, 2, 8);
  return q.cost < p.cost ? q : p;
}

}  // namespace

namespace {
// Up to 16 tokens: all but few rows of more than 96 super-blocks, where the workgroups of
// q4k_gemv16.hip already fill the chip and need no launch before them. (us, that kernel / this, 16
// tokens: Q6_K 1000 x 25600 17.6 / 18.3, 3584 x 25600 32.8 / 26.9; 8 tokens of Q4_K 2560 x 25600 17.8 /
// 18.4, 3584 x 25600 22.7 / 20.1.) 17..64: all. 65..128: matrices of up to w128 weights, whose prefill
// GEMM runs too few tiles. Rows long enough to make the operands large keep the other kernels.
bool mid_takes(int N, int K, int M, long long w128) {
  if (K > kF16Row) return false;
  if (M <= 16) return K <= 24576 || N >= 3072;
  return M <= 64 || (M <= 128 && K <= 131072 && (long long)N * K <= w128);
}
}  // namespace

// Besides, up to 16 tokens of Q4_K: matrices of more than 100 M weights are as fast without the operand
// launch (25600 x 5120 at 8 tokens 23.9 / 24.2), and so are ones that q4k_gemv16.hip divides into equal
// ranges of one workgroup per CU (11008 x 5120 15.6 / 16.4). 65..128 tokens (us, GEMM / this): 24 M
// weights (11008 x 2048 at 128 24.1 / 21.8), on long rows 70 M, as the GEMM's ranges there are short
// (1536 x 25600 36.8 / 32.0, 3584 x 18944 43.6 / 39.7), not on many short rows (18944 x 1024 17.7 / 18.2).
bool q4k_mid_takes(int N, int K, int M) {
  const long long w = (long long)N * K;
  const int nblk = K / 256;
  if (M < 5 || (M > 64 && N > 12288)) return false;
  if (M <= 16 && w > 100000000) return false;
  if (M <= 16 && w > 50000000 && nblk % 4 == 0 && (long long)ceil_div(N, 256) * (nblk / 4) <= cu_count()) return false;
  return mid_takes(N, K, M, K > 10240 ? 70000000 : 24000000);
}

// 65..128 tokens: 8192 x 2048 at 128 25.8 / 20.6, 1536 x 8192 20.8 / 17.9.
// 17..32 tokens of more than a few rows of kF16Row to 2^20 values, whose two groups of 16 tokens read the
// records through one L2 (us, q4k_gemv16.hip / this at 24 tokens: 3584 x 262400 524 / 377, 1000 x 262400
// 156 / 132, 2000 x 524288 593 / 450; 40 x 262400 36.9 / 66.9, as 64 ranges leave it few workgroups).
// Rows of two super-blocks are one launch of q4k_gemv16.hip (3000 x 512 at 8 / 24 tokens 8.5 / 8.7, this 9.4 /
// 9.8; of one super-block 8.4 / 8.8, this 7.9 / 8.6).
bool q6k_mid_takes(int N, int K, int M) {
  if (K > kF16Row) return M > 16 && M <= 32 && N >= 512 && K <= 4 * kF16Row;
  if (K == 512 && M <= 32) return false;
  return M >= 2 && mid_takes(N, K, M, 1 << 24);
}

size_t mid_ws_bytes(int fmt, int N, int K, int M) {
  const MidPlan p = plan_mid(fmt, N, K, M);
  return p.xb + p.tb + p.bb + p.pb;
}

namespace {
template <int FMT>
int launch_mid(const void *Wv, const float *X, float *Y, int N, int K, int M) {
  const MidPlan p = plan_mid(FMT, N, K, M);
  const int nblk = K / 256, ntiles = q4k_tiles(N), SK = p.SK, MTG = p.MTG, tokens = p.tokens;
  const size_t xb = p.xb, tb = p.tb, bb = p.bb, bytes = xb + tb + bb + p.pb;
  unsigned char *ws = (unsigned char *)workspace(bytes);
  if (!ws) return FHIP_ENOMEM;
  if (int rc = check_disjoint("quant_mid", X, (size_t)M * K * 4, ws, bytes)) return rc;
  u32x4 *xa = (u32x4 *)ws;
  float *ts = (float *)(ws + xb), *bs = bb ? (float *)(ws + xb + tb) : nullptr, *part = (float *)(ws + xb + tb + bb);
  const dim3 pg(tokens, SK);
  const int units = 32 * ceil_div(nblk, SK);
  auto prep = [&](auto hl) {
    constexpr bool H = decltype(hl)::value;
    if (units <= 256)
      mid_xprep_kernel<H, 1><<<pg, 256, 0, stream()>>>(X, M, K, nblk, SK, xa, ts, bs);
    else if (units <= 512)
      mid_xprep_kernel<H, 2><<<pg, 256, 0, stream()>>>(X, M, K, nblk, SK, xa, ts, bs);
    else
      mid_xprep_kernel<H, 0><<<pg, 256, 0, stream()>>>(X, M, K, nblk, SK, xa, ts, bs);
  };
  if (p.hl)
    prep(std::true_type{});
  else
    prep(std::false_type{});
  FHIP_CHECK_LAUNCH("mid_xprep_kernel");
  const uint8_t *W = (const uint8_t *)Wv;
  auto run = [&](auto kern) {
    kern<<<p.tasks * SK, 64 * p.NW, 0, stream()>>>(W, xa, ts, bs, Y, part, N, M, nblk, ntiles, MTG, tokens, SK);
  };
  if (p.hl)
    run(quant_mid_kernel<FMT, 1, true, 4>);
  else if (p.TT == 1)
    run(quant_mid_kernel<FMT, 1, false, 4>);
  else
    run(quant_mid_kernel<FMT, 2, false, 8>);
  FHIP_CHECK_LAUNCH("quant_mid_kernel");
  return SK > 1 ? sum_ranges(part, Y, SK, M * N) : FHIP_OK;
}
}  // namespace

int q4k_mid(const void *W, const float *X, float *Y, int N, int K, int M) {
  return launch_mid<0>(W, X, Y, N, K, M);
}

int q6k_mid(const void *W, const float *X, float *Y, int N, int K, int M) {
  return launch_mid<1>(W, X, Y, N, K, M);
}

}  // namespace fhip
