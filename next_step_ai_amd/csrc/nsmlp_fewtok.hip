// Few-token products over NF4 rows on v_mfma_f32_16x16x32_f16: the sparse MLP
// of up to 32 tokens over the union of their blocks (a short prefill chunk, a
// batch of sequences decoded together).
//
// With few tokens the product is bound by the weight stream, as a decode is:
// every union block is read once for all tokens, and a 16-token MFMA tile
// costs the same whether one or sixteen of its rows are used.  So no token
// lists and no gathered token tiles: each wave keeps all the call's tokens of
// its own K range in registers (the MFMA A operand) and streams weight rows
// past them (the B operand), as the one-token kernels do with v_dot2.
//
//   k_ft_list  the union's block ids in ascending order and each block's
//              token mask, by one workgroup in LDS;
//   k_ft_gu    gate and up of every union block for every token: a wave holds
//              NCH chunks of 128 columns of NT x 16 tokens (NT NCH = 8: 128
//              VGPRs) and streams tiles of 16 weight rows through a register
//              pipeline of 8 chunk loads (8 KB a wave, 64 KB a CU); the column
//              waves' sums meet in LDS, and act = fp16(silu(g) u) is formed at
//              the end, zero for the tokens that did not select the block;
//   k_ft_down  the same with K = the union's blocks: a wave holds the
//              activations of its 4 NCH blocks and streams output rows past
//              them; fp32 partial sums per group of waves;
//   k_ft_fin   the partial sums in group order + bias, rounded once.
//
// Weights go into the MFMAs as their fp16 code values (exact products, fp32
// sums); the absmax multiplies the fp32 result of its own 64 columns
// (gate/up) or of its block (down), as in the decode kernels.  For that an
// MFMA's 32 K slots have to lie in one absmax block, while a lane loads 16
// packed bytes (32 columns) at once: the lane groups' dwords are exchanged
// with v_permlane32_swap / v_permlane16_swap, 2 (4) VALU operations per 16
// bytes, instead of narrower loads.
//
// Every sum is taken in a fixed order.
//
// At hidden 16384 and 8 tokens (1092 of 1664 blocks, 894 MB) gate/up and down
// take about 240 us, 3.7 TB/s: two waves a SIMD (the tokens' registers) leave
// the lookups' and MFMAs' latency partly open, not the weight stream.
#include <mutex>

#include "nsmlp_replut.h"

namespace nsmlp {

namespace {

constexpr int kFtThreads = 512;
constexpr int kFtWaves = 8;
constexpr int kFtLutWords = kRepLutBytes / 4;
constexpr float kFtRange = 8388608.0f;  // 2^23, the range of the grouped down's partial products

typedef unsigned u32x2v_t __attribute__((ext_vector_type(2)));

// Exchanges lanes 32..63 of a with lanes 0..31 of b.
__device__ __forceinline__ void swap32(uint32_t& a, uint32_t& b) {
  const u32x2v_t r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}
// Exchanges lanes 16..31 of a with 0..15 of b, and 48..63 of a with 32..47 of b.
__device__ __forceinline__ void swap16(uint32_t& a, uint32_t& b) {
  const u32x2v_t r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}
// The values of v in lane groups 0..3 (16 lanes each), each in every group.
__device__ __forceinline__ void group_values(float v, float (&o)[4]) {
  uint32_t a = __float_as_uint(v), b = a;
  swap16(a, b);  // groups 0 0 2 2 | 1 1 3 3
  uint32_t c = a, d = b;
  swap32(a, c);  // 0 0 0 0 | 2 2 2 2
  swap32(b, d);  // 1 1 1 1 | 3 3 3 3
  o[0] = __uint_as_float(a);
  o[1] = __uint_as_float(b);
  o[2] = __uint_as_float(c);
  o[3] = __uint_as_float(d);
}
__device__ __forceinline__ uint32_t ft_lane(uint32_t v, int lane) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, lane);
}
// 8 codes of a packed dword as fp16, in element order.
__device__ __forceinline__ half8_t ft_codes8(uint32_t v, uint32_t (&ad)[4]) {
  NSMLP_SET_BYTE1(ad[0], v, "BYTE_0");
  NSMLP_SET_BYTE1(ad[1], v, "BYTE_1");
  NSMLP_SET_BYTE1(ad[2], v, "BYTE_2");
  NSMLP_SET_BYTE1(ad[3], v, "BYTE_3");
  return as_h8(make_uint4(lds_ld_u32(ad[0]), lds_ld_u32(ad[1]), lds_ld_u32(ad[2]), lds_ld_u32(ad[3])));
}

// Groups the union's chunks are split over (each group's waves hold them all
// between them, its workgroups share the output rows): the count from the
// fewest that hold them on whose busiest wave has the least to stream, the
// smaller of equals (fewer partial sums).
constexpr int kFtGroupsTried = 12;
__host__ __device__ inline int ft_groups_min(int nu, int NT) {
  const int nch = 6 / NT, chunks = (nu + 3) / 4;
  const int cg = (chunks + 8 * nch - 1) / (8 * nch);
  return cg > 0 ? cg : 1;
}
__host__ __device__ inline int ft_down_groups(int nu, int H, int wgs, int NT) {
  const int chunks = (nu + 3) / 4, nrg = H / (64 / NT), lo = ft_groups_min(nu, NT);
  int best = lo, cost = 0x7FFFFFFF;
  for (int cg = lo; cg < lo + kFtGroupsTried && cg <= wgs; ++cg) {
    const int wpc = wgs / cg;
    const int c = ((chunks + 8 * cg - 1) / (8 * cg) + 1) * ((nrg + wpc - 1) / wpc);
    if (c < cost) {
      cost = c;
      best = cg;
    }
  }
  return best;
}

// ------------------------------------------------------------ union list --
constexpr int kFtMaxNB = 4096;
constexpr int kFtMaxTok = 32;

__global__ void __launch_bounds__(1024) k_ft_list(FewTokArgs p) {
  __shared__ uint32_t mask[kFtMaxNB];
  __shared__ int wsum[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int NB = p.d.NB;
  for (int i = tid; i < NB; i += 1024) mask[i] = 0;
  __syncthreads();
  bool bad = false;
  for (int i = tid; i < p.M * p.k; i += 1024) {
    const int t = i / p.k, b = p.sel[i];
    if (b < 0 || b >= NB)
      bad = true;
    else
      atomicOr(&mask[b], 1u << t);
  }
  if (bad) atomicOr(p.d.status, NSMLP_STATUS_BLOCK_UNAVAILABLE);
  __syncthreads();
  const int per = (NB + 1023) / 1024, b0 = tid * per;  // at most 4 consecutive blocks a thread
  int cnt = 0;
  for (int i = 0; i < per; ++i) {
    const int b = b0 + i;
    cnt += b < NB && mask[b] != 0;
  }
  const int incl = (int)wave_incl_scan((unsigned)cnt, lane);
  if (lane == kWave - 1) wsum[wave] = incl;
  __syncthreads();
  int pos = incl - cnt;
  for (int w = 0; w < 16; ++w) pos += w < wave ? wsum[w] : 0;
  if (tid == 1023) {
    p.nu[0] = pos + cnt;
    p.nu[1] = ft_down_groups(pos + cnt, p.d.H, p.wgs, p.NT);
  }
  for (int i = 0; i < per; ++i) {
    const int b = b0 + i;
    if (b < NB && mask[b] != 0) {
      p.ublk[pos] = b;
      p.umask[pos++] = mask[b];
    }
  }
}

// ----------------------------------------------------------------- gate/up --
// Chunks of 128 columns: lane (j, g) of a wave loads the 16 packed bytes of
// columns 32 g .. 32 g + 31 of row j (64 bytes of each of 16 rows per load).
// After swap32 of dwords 0, 2 and 1, 3 the dwords are the B fragments of four
// MFMAs, two per 64-column half: K slots 8 g .. 8 g + 7 of fragment s are the
// chunk's columns 64 (s / 2) + 32 (g % 2) + 16 (g / 2) + 8 (s % 2) .. + 7.
// Absmax: lane (j, g) reads those of row j and halves 4 q + g; group_values
// hands each to all four groups.
template <int NT, int NCH>
struct FtGeo {
  static constexpr int SU = (NCH + 1) / 2;  // chunks of a tile's first unit (the second has NCH - SU)
  static constexpr int PD = 8 / (SU == 3 ? 4 : SU);  // units in flight: 8 chunk loads (6 for SU = 3)
  static constexpr int RB = PD / 2;                  // tiles per loop body
  static constexpr int NH = (2 * SU + 3) / 4;        // absmax values a lane loads per unit
  static constexpr int kSlots = NT == 1 ? 64 : 30;   // tile sums held in LDS
  static constexpr int kCombWords = 2 * kFtWaves * NT * 256;  // the waves' sums, two buffers
  static constexpr int kC2Word = kFtLutWords, kCombWord = kC2Word + 512, kSlotWord = kCombWord + kCombWords;
  static constexpr size_t kLds = (size_t)(kSlotWord + kSlots * NT * 256) * 4;
  static_assert(kLds <= 160 * 1024, "LDS");
};

template <bool DQ, int NT, int NCH>
__global__ void __launch_bounds__(kFtThreads, 2) k_ft_gu(FewTokArgs p) {
  using G = FtGeo<NT, NCH>;
  constexpr int SU = G::SU, PD = G::PD, RB = G::RB, NH = G::NH;
  extern __shared__ __attribute__((aligned(16))) uint32_t lds[];  // no static LDS: the table is at LDS address 0
  const DecodeArgs& d = p.d;
  float* c2 = reinterpret_cast<float*>(lds + G::kC2Word);
  float4_t* comb = reinterpret_cast<float4_t*>(lds + G::kCombWord);
  float4_t* slots = reinterpret_cast<float4_t*>(lds + G::kSlotWord);
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 15, g = lane >> 4;
  const int H = d.H, M = p.M, p_a2 = p.gu_a2bytes;
  const int CW = p.gu_cw, RW = kFtWaves / CW, CGS = p.gu_cgs, chunks = H >> 7;
  const int cw = wave & (CW - 1), rw = wave / CW;
  const int nu = p.nu[0];
  // pairs: (union block, 16-row half), each a gate and an up tile
  const int p_lo = (int)(blockIdx.x * (2u * (unsigned)nu) / gridDim.x);
  const int p_hi = (int)((blockIdx.x + 1) * (2u * (unsigned)nu) / gridDim.x);
  {
    LutCodes codes;
    lut_codes_load(d.code, d.code_up, tid, codes);
    lut_store(lds, codes, tid);
    if constexpr (DQ) c2[tid] = tid < 256 ? d.gate.code2[tid] : d.up.code2[tid - 256];
  }
  lds_barrier();
  const rsrc_t rx = make_rsrc(p.x, M * H * 2);
  // What issue needs of the kernel arguments, kept in SGPRs (opaque to the
  // compiler, which otherwise loads the fields again for every tile: a scalar
  // load's round trip each, waited for together with the LDS reads).
  auto bytes_of = [](const auto* q) { return reinterpret_cast<uint64_t>(q); };
  auto pick = [](bool c, auto a, auto b) { return c ? a : b; };  // by value: a conditional over the variables selects an address
  uint64_t w_g = bytes_of(d.gate.packed), w_u = bytes_of(d.up.packed), w_hg = bytes_of(d.host_gate.packed),
           w_hu = bytes_of(d.host_up.packed);
  uint64_t a_g = DQ ? bytes_of(d.gate.qabsmax) : bytes_of(d.gate.absmax);
  uint64_t a_u = DQ ? bytes_of(d.up.qabsmax) : bytes_of(d.up.absmax);
  uint64_t a_hg = DQ ? bytes_of(d.host_gate.qabsmax) : bytes_of(d.host_gate.absmax);
  uint64_t a_hu = DQ ? bytes_of(d.host_up.qabsmax) : bytes_of(d.host_up.absmax);
  uint64_t s_g = bytes_of(d.gate.absmax2), s_u = bytes_of(d.up.absmax2);
  uint32_t rs = (uint32_t)d.gate.row_stride, A = (uint32_t)d.gate.abs_row_stride;
  uint32_t qsh = (uint32_t)d.qbs_shift, dsh = (uint32_t)d.dq_shift;
  float off_g = d.gate.offset, off_u = d.up.offset;
  asm volatile(""
               : "+s"(w_g), "+s"(w_u), "+s"(w_hg), "+s"(w_hu), "+s"(a_g), "+s"(a_u), "+s"(a_hg), "+s"(a_hu), "+s"(s_g),
                 "+s"(s_u), "+s"(rs), "+s"(A), "+s"(qsh), "+s"(dsh), "+s"(off_g), "+s"(off_u));

  struct Stage {
    uint4 w[SU];
    uint32_t qa[NH];
    float am[NH];
  };
  for (int pb = p_lo; pb < p_hi; pb += G::kSlots / 2) {
    const int np = min(p_hi - pb, G::kSlots / 2), ntl = 2 * np;
    const int R = (ntl + RW - 1) / RW, VT = R * CGS;
    // lane i: block reference of pair i (slot, or the block id with bit 30 for
    // a host copy; bit 31: unavailable)
    uint32_t enc_v = 0x80000000u, bid_v = 0;
    if (lane < np) {
      const int b = p.ublk[(pb + lane) >> 1];
      const BlockRef br = resolve_id(d, b);
      enc_v = !br.ok ? 0x80000000u : br.dev ? (uint32_t)br.q : (0x40000000u | (uint32_t)br.q);
      bid_v = (uint32_t)b;
      if (!br.ok && wave == 0) atomicOr(d.status, NSMLP_STATUS_BLOCK_UNAVAILABLE);
    }
    int icg = 0, ir = 0;  // column group and round of the next tile to issue
    auto issue = [&](Stage& st, auto unit) {
      constexpr int U = decltype(unit)::value;
      const int t = ir * RW + rw;
      const bool live = icg < CGS && t < ntl;
      const int lp = live ? t >> 1 : 0;
      const uint32_t enc = ft_lane(enc_v, lp);
      const bool up = (t & 1) != 0, dev = (enc & 0x40000000u) == 0;
      const bool ok = live && (enc & 0x80000000u) == 0;
      const uint32_t q = ok ? enc & 0x3FFFFFFFu : 0u;
      const uint32_t h16 = (uint32_t)((pb + lp) & 1) * 16u;
      const int chb = (icg * CW + cw) * NCH;
      const uint64_t base = pick(up, pick(dev, w_u, w_hu), pick(dev, w_g, w_hg)) + (uint64_t)q * (32u * rs) + h16 * rs;
      const rsrc_t rp = make_rsrc(reinterpret_cast<const void*>(base), ok ? 16 * (int)rs : 0);
      // columns past the last chunk read the next row (or zeros past the
      // tile): their tokens are zero
      const uint32_t voff = (uint32_t)j * rs + (uint32_t)(chb * 64) + 16u * (uint32_t)g;
      constexpr int c0 = U == 0 ? 0 : SU, c1 = U == 0 ? SU : NCH;
#pragma unroll
      for (int c = c0; c < c1; ++c) st.w[c - c0] = buf_ld16(rp, voff + 64u * (uint32_t)c, 0);
      {
        const uint64_t ab = pick(up, pick(dev, a_u, a_hu), pick(dev, a_g, a_hg)) + (uint64_t)q * (32u * A * (DQ ? 1u : 4u));
        const rsrc_t ra = make_rsrc(reinterpret_cast<const void*>(ab), ok ? (int)(32u * A * (DQ ? 1u : 4u)) : 0);
        const rsrc_t r2 = make_rsrc(reinterpret_cast<const void*>(pick(up, s_u, s_g)), ok ? p_a2 : 0);
        const uint32_t r = h16 + (uint32_t)j, bid = ft_lane(bid_v, lp);
        const uint32_t f0 = (32u * bid + r) * A;
#pragma unroll
        for (int i = 0; i < (2 * (c1 - c0) + 3) / 4; ++i) {
          const uint32_t e = (uint32_t)(128 * chb + 64 * (2 * c0 + 4 * i + g)) >> qsh;
          if constexpr (DQ) {
            st.qa[i] = buf_ldu8(ra, ((r >> 1) * A + e) * 2u + (r & 1u), 0);
            st.am[i] = buf_ldfc(r2, ((f0 + e) >> dsh) * 4u, 0);
          } else {
            st.qa[i] = 0;
            st.am[i] = buf_ldf(ra, (r * A + e) * 4u, 0);
          }
        }
      }
      if constexpr (U == 1) {
        if (++ir == R) {
          ir = 0;
          ++icg;
        }
      }
    };
    half8_t x[NCH][4][NT];
    auto load_x = [&](int cg) {
      const int chb = (cg * CW + cw) * NCH;
#pragma unroll
      for (int c = 0; c < NCH; ++c)
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int n = 0; n < NT; ++n) {
            const int t = 16 * n + j;
            const uint32_t col = (uint32_t)(128 * (chb + c) + 64 * (s >> 1) + 32 * (g & 1) + 16 * (g >> 1) + 8 * (s & 1));
            x[c][s][n] = as_h8(buf_ld16c(rx, t < M && chb + c < chunks ? ((uint32_t)t * (uint32_t)H + col) * 2u : kOffNone, 0));
          }
    };
    using U0 = std::integral_constant<int, 0>;
    using U1 = std::integral_constant<int, 1>;
    load_x(0);
    Stage st[PD];
#pragma unroll
    for (int i = 0; i < PD; i += 2) {
      issue(st[i], U0{});
      issue(st[i + 1], U1{});
    }
    sched_fence();

    uint32_t ad[4];
    int cg = 0, r = 0;
    for (int v0 = 0; v0 < VT; v0 += RB) {
#pragma unroll
      for (int i = 0; i < RB; ++i) {
        if (v0 + i < VT) {  // uniform over the workgroup
          if (r == 0 && v0 + i > 0) load_x(cg);
          const int t = r * RW + rw;
          const int mych = min(chunks - (cg * CW + cw) * NCH, NCH);
          const bool ok = t < ntl && (ft_lane(enc_v, t < ntl ? t >> 1 : 0) & 0x80000000u) == 0;
#pragma unroll
          for (int m = 0; m < 4; ++m) ad[m] = ((t & 1) ? 128u : 0u) + (uint32_t)(lane & 31) * 4u;
          float4_t acc[NT];
#pragma unroll
          for (int n = 0; n < NT; ++n) acc[n] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
          auto unit = [&](Stage& su, auto uc) {
            constexpr int U = decltype(uc)::value;
            constexpr int c0 = U == 0 ? 0 : SU, c1 = U == 0 ? SU : NCH;
#pragma unroll
            for (int cp = c0; cp < c1; cp += 2) {  // two chunks: four halves, one absmax load of the lane
              constexpr int kPair = 2;
              float4_t cc[2 * kPair][NT];
#pragma unroll
              for (int c = cp; c < cp + 2 && c < c1; ++c) {
                uint4 w = su.w[c - c0];
                swap32(w.x, w.z);
                swap32(w.y, w.w);
                const uint32_t dw[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                  const half8_t b = ft_codes8(dw[s], ad);
                  float4_t(&o)[NT] = cc[2 * (c - cp) + (s >> 1)];
#pragma unroll
                  for (int n = 0; n < NT; ++n)
                    o[n] = mfma16(x[c][s][n], b, (s & 1) ? o[n] : float4_t{0.0f, 0.0f, 0.0f, 0.0f});
                }
              }
              // the halves' absmax, every one in all lane groups
              const int q = (cp - c0) / 2;
              float a = su.am[q];
              if constexpr (DQ) a = dq_absmax(c2[((t & 1) ? 256 : 0) + su.qa[q]], a, pick((t & 1) != 0, off_u, off_g));
              a = ok && 2 * cp + g < 2 * mych ? a : 0.0f;
              float am[4];
              group_values(a, am);
              mfma_drain();
#pragma unroll
              for (int hb = 0; hb < 4 && cp + hb / 2 < c1; ++hb)
#pragma unroll
                for (int n = 0; n < NT; ++n)
#pragma unroll
                  for (int e = 0; e < 4; ++e) acc[n][e] = __builtin_fmaf(cc[hb][n][e], am[hb], acc[n][e]);
#pragma unroll
              for (int n = 0; n < NT; ++n) asm volatile("" : "+v"(acc[n]));  // summed here, not at its use
            }
          };
          unit(st[2 * i], U0{});
          issue(st[2 * i], U0{});
          sched_fence();
          unit(st[2 * i + 1], U1{});
          issue(st[2 * i + 1], U1{});
          sched_fence();
          // the column waves' sums: one wave per (row wave, token tile), a
          // different one each round, adds them in column order
          const int par = (v0 + i) & 1;
#pragma unroll
          for (int n = 0; n < NT; ++n) comb[((par * kFtWaves + wave) * NT + n) * 64 + lane] = acc[n];
          lds_barrier();
          for (int job = (wave - (v0 + i)) & 7; job < RW * NT; job += kFtWaves) {
            const int n = job % NT, rwj = job / NT, tj = r * RW + rwj;
            if (tj < ntl) {
              float4_t y = comb[((par * kFtWaves + rwj * CW) * NT + n) * 64 + lane];
              for (int c = 1; c < CW; ++c) y += comb[((par * kFtWaves + rwj * CW + c) * NT + n) * 64 + lane];
              float4_t* sl = slots + (tj * NT + n) * 64 + lane;
              *sl = cg == 0 ? y : *sl + y;
            }
          }
          if (++r == R) {
            r = 0;
            ++cg;
          }
        }
      }
    }
    lds_barrier();
    // act of (pair, token, row): element e of lane 16 g + j of token tile n is
    // token 16 n + 4 g + e, row j
    for (int i = tid; i < np * NT * 256; i += kFtThreads) {
      const int row = i & 15, t = (i >> 4) % (16 * NT), lp = i / (256 * NT);
      if (t >= M) continue;
      const int u = (pb + lp) >> 1, h16 = ((pb + lp) & 1) * 16;
      const int at = ((t >> 4) * 64 + ((t >> 2) & 3) * 16 + row) * 4 + (t & 3);
      const float* s0 = reinterpret_cast<const float*>(slots + (2 * lp) * NT * 64);
      const float* s1 = reinterpret_cast<const float*>(slots + (2 * lp + 1) * NT * 64);
      const bool mine = (p.umask[u] >> t) & 1u;
      p.act[(long long)t * (d.NB * 32) + u * 32 + h16 + row] = mine ? f2h(silu_mul(s0[at], s1[at])) : (uint16_t)0;
    }
    lds_barrier();
  }
}

// -------------------------------------------------------------------- down --
// K is the union's blocks in union order, 4 blocks (128 columns) a chunk:
// lane (j, g) loads the 16 packed bytes of row j of block 4 c + g (256
// contiguous bytes of each of 4 blocks per load).  A 4 x 4 transposition of the
// dwords over the lane groups makes dword i the B fragment of block 4 c + i
// (K slots 8 g .. 8 g + 7: its columns 8 g .. + 7), and the block's absmax
// multiplies its MFMA result.  A wave takes RT row tiles of 16 rows at a time.
template <int NT>
struct FdGeo {
  static constexpr int NCH = 6 / NT;                         // chunks a wave holds (96 VGPRs of activations)
  static constexpr int RT = 4 / NT;                          // row tiles of 16 rows per unit
  static constexpr int PD = NT == 1 ? 2 : 3;                 // units in flight (8 or 6 loads)
  static constexpr int kC2Word = kFtLutWords, kRefWord = kC2Word + 256, kCombWord = kRefWord + kFtWaves * NCH * 4 * 2;
  static constexpr size_t kLds = (size_t)(kCombWord + 2 * kFtWaves * RT * NT * 256) * 4;
  static_assert(kLds <= 160 * 1024 && NCH % PD == 0, "geometry");
};

template <bool DQ, bool HOST, int NT>
__global__ void __launch_bounds__(kFtThreads, 2) k_ft_down(FewTokArgs p) {
  using G = FdGeo<NT>;
  constexpr int NCH = G::NCH, RT = G::RT, PD = G::PD;
  extern __shared__ __attribute__((aligned(16))) uint32_t lds[];  // no static LDS: the table is at LDS address 0
  const DecodeArgs& d = p.d;
  float* c2 = reinterpret_cast<float*>(lds + G::kC2Word);
  float4_t* comb = reinterpret_cast<float4_t*>(lds + G::kCombWord);
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 15, g = lane >> 4;
  const int H = d.H, M = p.M, nu = p.nu[0], lda = d.NB * 32;
  const unsigned CG = (unsigned)p.nu[1], WPC = gridDim.x / CG, NRG = (unsigned)(H / (16 * RT));
  const unsigned cg = blockIdx.x % CG, wi = blockIdx.x / CG;
  if (wi >= WPC) return;
  const int rg_lo = (int)(wi * NRG / WPC), rg_hi = (int)((wi + 1) * NRG / WPC);
  if (rg_lo >= rg_hi) return;
  const unsigned nch_all = (unsigned)(nu + 3) / 4, gw = cg * kFtWaves + (unsigned)wave;
  const int c_lo = (int)(gw * nch_all / (CG * kFtWaves));
  const int kc = (int)((gw + 1) * nch_all / (CG * kFtWaves)) - c_lo;  // <= NCH
  {
    LutCodes codes;
    lut_codes_load(d.code_down, d.code_down, tid, codes);
    lut_store(lds, codes, tid);
    if constexpr (DQ) {
      if (tid < 256) c2[tid] = d.down.code2[tid];
    }
  }
  // (slot, or block id with bit 30 for a host copy; -1: none) and block id of
  // the wave's blocks
  int2* refs = reinterpret_cast<int2*>(lds + G::kRefWord) + wave * (NCH * 4);
  if (lane < NCH * 4) {
    const int u = 4 * c_lo + lane;
    int2 e = make_int2(-1, 0);
    if (lane < 4 * kc && u < nu) {
      const BlockRef br = resolve_id(d, p.ublk[u]);
      e.y = br.b;
      if (br.ok) e.x = br.dev ? (int)br.q : (0x40000000 | (int)br.q);
    }
    refs[lane] = e;
  }
  half8_t x[NCH][4][NT];
  {
    const rsrc_t rx = make_rsrc(p.act, M * lda * 2);
#pragma unroll
    for (int c = 0; c < NCH; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int n = 0; n < NT; ++n) {
          const int t = 16 * n + j, u = 4 * (c_lo + c) + i;
          const bool in = t < M && c < kc && u < nu;
          x[c][i][n] = as_h8(buf_ld16c(rx, in ? ((uint32_t)t * (uint32_t)lda + 32u * (uint32_t)u + 8u * (uint32_t)g) * 2u : kOffNone, 0));
        }
  }
  lds_barrier();
  const uint32_t bs = (uint32_t)d.down.blk_stride, as = (uint32_t)d.down.abs_blk_stride;
  const uint32_t Ad = (uint32_t)lda >> d.qbs_shift;
  const rsrc_t rw = make_rsrc(d.down.packed, d.n_slots > 0 ? d.n_slots * (int)bs : 0);
  const rsrc_t rwh = HOST ? make_rsrc(d.host_down.packed, d.NB * (int)bs) : rw;
  const rsrc_t ra = DQ ? make_rsrc(d.down.qabsmax, d.n_slots * (int)as) : make_rsrc(d.down.absmax, d.n_slots * (int)as * 4);
  const rsrc_t rah = !HOST ? ra
                     : DQ  ? make_rsrc(d.host_down.qabsmax, d.NB * (int)as)
                           : make_rsrc(d.host_down.absmax, d.NB * (int)as * 4);
  const rsrc_t r2 = DQ ? make_rsrc(d.down.absmax2, p.dn_a2bytes) : ra;

  struct Stage {
    uint4 w[RT];
    uint32_t qa[RT];
    float am[RT];
    bool ok;
  };
  auto issue = [&](Stage& st, int rg, int c) {
    const int2 e = refs[c * 4 + g];
    // opaque here: products with them are not kept in registers over the loop
    uint32_t Ao = Ad, bso = bs, aso = as;
    asm volatile("" : "+s"(Ao), "+s"(bso), "+s"(aso));
    const bool ok = rg < rg_hi && c < kc && e.x >= 0;
    const bool host = HOST && (e.x & 0x40000000) != 0;
    const bool dv = ok && !host, hv = ok && host;
    const uint32_t q = (uint32_t)(e.x & 0x3FFFFFFF);
    const uint32_t o = (uint32_t)(rg * 16 * RT + j);
    const uint32_t wo = q * bso + o * 16u, ao = (q * aso + o) * (DQ ? 1u : 4u);
    const uint32_t wd = dv ? wo : kOffNone, wh = hv ? wo : kOffNone, adv = dv ? ao : kOffNone, ahv = hv ? ao : kOffNone;
    const uint32_t f0 = o * Ao + ((32u * (uint32_t)e.y) >> d.qbs_shift);
    st.ok = ok;
#pragma unroll
    for (int m = 0; m < RT; ++m) {
      st.w[m] = buf_ld16(rw, wd, 256u * m);
      if constexpr (HOST) {
        const uint4 h = buf_ld16(rwh, wh, 256u * m);
        st.w[m] = make_uint4(st.w[m].x | h.x, st.w[m].y | h.y, st.w[m].z | h.z, st.w[m].w | h.w);
      }
      if constexpr (DQ) {
        st.qa[m] = buf_ldu8(ra, adv, 16u * m);
        if constexpr (HOST) st.qa[m] |= buf_ldu8(rah, ahv, 16u * m);
        st.am[m] = buf_ldfc(r2, ok ? ((f0 + 16u * m * Ao) >> d.dq_shift) * 4u : kOffNone, 0);
      } else {
        st.am[m] = buf_ldf(ra, adv, 64u * m);
        if constexpr (HOST) st.am[m] = __uint_as_float(__float_as_uint(st.am[m]) | __float_as_uint(buf_ldf(rah, ahv, 64u * m)));
      }
    }
  };
  float* part = p.part + (size_t)cg * M * H;
  Stage st[PD];
#pragma unroll
  for (int i = 0; i < PD; ++i) issue(st[i], rg_lo + i / NCH, i % NCH);
  sched_fence();
  uint32_t ad[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) ad[m] = (uint32_t)lane * 4u;
  float top = 0.0f;  // largest product seen where one may leave the range; inf or nan sums
  for (int rg = rg_lo; rg < rg_hi; ++rg) {
    float4_t acc[RT][NT];
#pragma unroll
    for (int m = 0; m < RT; ++m)
#pragma unroll
      for (int n = 0; n < NT; ++n) acc[m][n] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      Stage& su = st[c % PD];
      if (c < kc) {  // uniform over the wave
#pragma unroll
        for (int m = 0; m < RT; ++m) {
          uint4 w = su.w[m];
          swap16(w.x, w.y);
          swap16(w.z, w.w);
          swap32(w.x, w.z);
          swap32(w.y, w.w);
          const uint32_t dw[4] = {w.x, w.y, w.z, w.w};
          float4_t cc[4][NT];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const half8_t bf = ft_codes8(dw[i], ad);
#pragma unroll
            for (int n = 0; n < NT; ++n) cc[i][n] = mfma16(x[c][i][n], bf, float4_t{0.0f, 0.0f, 0.0f, 0.0f});
          }
          // the lane's absmax, finite (a token that did not select the block
          // has a zero product with it), then every block's in all lane groups
          float a = su.am[m];
          if constexpr (DQ) a = dq_absmax(c2[su.qa[m]], a, d.down.offset);
          a = su.ok ? fminf(fmaxf(a, -3.0e38f), 3.0e38f) : 0.0f;
          float am[4];
          group_values(a, am);
          mfma_drain();
          // |code sums| < 2^21 (32 products of |code| <= 1 and |act| < 2^16),
          // so a product outside the range needs an absmax of 4 or more
          if (__any(fabsf(a) >= 4.0f)) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
              for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int e = 0; e < 4; ++e) top = fmaxf(top, fabsf(cc[i][n][e] * am[i]));
          }
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
              for (int e = 0; e < 4; ++e) acc[m][n][e] = __builtin_fmaf(cc[i][n][e], am[i], acc[m][n][e]);
          // summed here: left to itself the compiler moves the sums down to
          // their use and keeps (or spills) every product until then
#pragma unroll
          for (int n = 0; n < NT; ++n) asm volatile("" : "+v"(acc[m][n]));
        }
      }
      issue(su, rg + (c + PD) / NCH, (c + PD) % NCH);
      sched_fence();
    }
    const int par = (rg - rg_lo) & 1;
#pragma unroll
    for (int m = 0; m < RT; ++m)
#pragma unroll
      for (int n = 0; n < NT; ++n) {
#pragma unroll
        for (int e = 0; e < 4; ++e) top = fabsf(acc[m][n][e]) < 3.4e38f ? top : kFtRange;
        comb[((par * kFtWaves + wave) * 4 + m * NT + n) * 64 + lane] = acc[m][n];
      }
    lds_barrier();
    // four (row tile, token tile) sums of the 8 waves, by four waves
    const int job = (wave - 4 * par) & 7;
    if (job < 4) {
      const int n = job % NT, m = job / NT;
      float4_t y = comb[((par * kFtWaves) * 4 + job) * 64 + lane];
#pragma unroll
      for (int w = 1; w < kFtWaves; ++w) y += comb[((par * kFtWaves + w) * 4 + job) * 64 + lane];
      const int o = (rg * RT + m) * 16 + j;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int t = 16 * n + 4 * g + e;
        if (t < M) part[(uint32_t)t * (uint32_t)H + (uint32_t)o] = y[e];
      }
    }
  }
  if (p.report_range && top >= kFtRange) atomicOr(d.status, NSMLP_STATUS_FIXED_RANGE);
}

__global__ void __launch_bounds__(256) k_ft_fin(FewTokArgs p) {
  const long long n = (long long)p.M * p.d.H;
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int CG = p.nu[1];
  float y = 0.0f;
  for (int s = 0; s < CG; ++s) y += p.part[(long long)s * n + i];
  if (p.d.down_bias != nullptr) y += h2f(p.d.down_bias[(int)(i % p.d.H)]);
  p.out[i] = f2h(y);
}

int ft_token_tiles(int M) { return M <= 16 ? 1 : 2; }

using FtFn = void (*)(FewTokArgs);
struct FtKernel {
  FtFn fn;
  size_t lds;
};
template <bool DQ, int NT, int NCH>
constexpr FtKernel ft_gu() {
  return FtKernel{k_ft_gu<DQ, NT, NCH>, FtGeo<NT, NCH>::kLds};
}
template <bool DQ, bool HOST, int NT>
constexpr FtKernel ft_down() {
  return FtKernel{k_ft_down<DQ, HOST, NT>, FdGeo<NT>::kLds};
}
// [dq][chunks - 5 of one token tile; 4 + chunks - 3 of two]
const FtKernel kFtGu[2][6] = {
    {ft_gu<false, 1, 5>(), ft_gu<false, 1, 6>(), ft_gu<false, 1, 7>(), ft_gu<false, 1, 8>(), ft_gu<false, 2, 3>(),
     ft_gu<false, 2, 4>()},
    {ft_gu<true, 1, 5>(), ft_gu<true, 1, 6>(), ft_gu<true, 1, 7>(), ft_gu<true, 1, 8>(), ft_gu<true, 2, 3>(),
     ft_gu<true, 2, 4>()}};
// [dq][host copies][token tiles - 1]
const FtKernel kFtDown[2][2][2] = {{{ft_down<false, false, 1>(), ft_down<false, false, 2>()},
                                    {ft_down<false, true, 1>(), ft_down<false, true, 2>()}},
                                   {{ft_down<true, false, 1>(), ft_down<true, false, 2>()},
                                    {ft_down<true, true, 1>(), ft_down<true, true, 2>()}}};

void ft_set_lds() {
  static std::once_flag once;
  std::call_once(once, [] {
    auto set = [](const FtKernel& k) {
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k.fn), hipFuncAttributeMaxDynamicSharedMemorySize, (int)k.lds);
    };
    for (int q = 0; q < 2; ++q) {
      for (const FtKernel& k : kFtGu[q]) set(k);
      for (int h = 0; h < 2; ++h)
        for (const FtKernel& k : kFtDown[q][h]) set(k);
    }
  });
}
void ft_launch(const FtKernel& k, int wgs, const FewTokArgs& p, hipStream_t s) {
  k.fn<<<dim3((unsigned)wgs), dim3(kFtThreads), k.lds, s>>>(p);
}

// Chunks a wave holds and the column waves of a workgroup for H columns: the
// fewest column groups (each a pass over the workgroup's tiles with its own
// tokens in registers), then the fewest chunks a wave, then the fewest
// column waves.
void ft_columns(int H, int NT, int* nch, int* cw, int* cgs) {
  const int chunks = H / 128, top = 8 / NT, low = NT == 1 ? 5 : 3;
  const int waves = (chunks + top - 1) / top;
  *cgs = (waves + kFtWaves - 1) / kFtWaves;
  const int per = (chunks + *cgs - 1) / *cgs;
  int w = 1;
  while (w < kFtWaves && w * top < per) w *= 2;
  *cw = w;
  int n = (per + w - 1) / w;
  *nch = n < low ? low : n;
}

}  // namespace

size_t few_tokens_workspace(int H, int NB, int M, int k) {
  auto up = [](size_t v) { return (v + 255) / 256 * 256; };
  const long long nu = (long long)M * k < NB ? (long long)M * k : NB;
  const int cg = ft_groups_min((int)nu, ft_token_tiles(M)) + kFtGroupsTried - 1;
  return 256 + 2 * up((size_t)NB * 4) + up((size_t)M * NB * 64) + up((size_t)cg * M * H * 4);
}

// Up to 32 tokens (two 16-token tiles of 128 VGPRs between them).  The grouped
// kernels these replace there read the weights once per block as well, but
// work tile by tile on token lists (hidden 16384, 1664 blocks, top-k 208,
// double-quantised, whole prefill call with its route): 2 tokens 376 -> 132
// us, 8 tokens 579 -> 290, 16 tokens 520 -> 367, 32 tokens 539 -> 473; hidden
// 4096, 448 blocks, top-k 64: 8 tokens 144 -> 74, 24 tokens 103 -> 94.  Four
// tiles (33 to 64 tokens, 2 chunks a wave) were slower than the grouped
// kernels: 1138 against 544 and 167 against 106 us.
bool few_tokens_shape(int H, int NB, int M) { return M <= kFtMaxTok && NB <= kFtMaxNB && H % 256 == 0; }

bool few_tokens_fit(const DecodeArgs& d, int M) {
  if (!few_tokens_shape(d.H, d.NB, M) || d.qbs < 64 || device_cus() < 64) return false;
  const long long lim = 1LL << 31, n_abs = (long long)d.H * d.NB * 32 / d.qbs;
  const long long slots = d.n_slots > d.NB ? d.n_slots : d.NB;
  return slots * d.H * 16 < lim && n_abs < lim && 16LL * d.H < lim && (d.n_slots < (1 << 30));
}

void launch_few_tokens(const FewTokArgs& args, void* ws, hipStream_t s) {
  FewTokArgs p = args;
  const DecodeArgs& d = p.d;
  auto up = [](size_t v) { return (v + 255) / 256 * 256; };
  const int NT = ft_token_tiles(p.M), cus = device_cus();
  p.NT = NT;
  p.wgs = cus;
  char* w = (char*)ws;
  p.nu = (int32_t*)w;
  w += 256;
  p.ublk = (int32_t*)w;
  w += up((size_t)d.NB * 4);
  p.umask = (uint32_t*)w;
  w += up((size_t)d.NB * 4);
  p.act = (uint16_t*)w;
  w += up((size_t)p.M * d.NB * 64);
  p.part = (float*)w;
  int nch;
  ft_columns(d.H, NT, &nch, &p.gu_cw, &p.gu_cgs);
  const long long n2 = (((long long)d.H * d.NB * 32 / d.qbs) + (1LL << d.dq_shift) - 1) >> d.dq_shift;
  p.gu_a2bytes = p.dn_a2bytes = (int)(n2 * 4);
  k_ft_list<<<dim3(1), dim3(1024), 0, s>>>(p);
  ft_set_lds();
  ft_launch(kFtGu[d.dq ? 1 : 0][NT == 1 ? nch - 5 : 4 + nch - 3], cus, p, s);
  ft_launch(kFtDown[d.dq ? 1 : 0][d.host_down.packed != nullptr ? 1 : 0][NT - 1], cus, p, s);
  const long long n = (long long)p.M * d.H;
  k_ft_fin<<<dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s>>>(p);
}

}  // namespace nsmlp
