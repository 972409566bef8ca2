// Few-token products over NF4 rows on v_mfma_f32_16x16x32_f16: the sparse MLP
// of up to 32 tokens over the union of their blocks (a short prefill chunk, a
// batch of sequences decoded together), and an LM head of three rows or more.
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
//              them; partial sums per group of waves;
//   k_ft_fin   the groups' partial sums + bias, rounded once.
//
// Weights go into the MFMAs as their fp16 code values (exact products, fp32
// sums); the absmax multiplies the fp32 result of its own 64 columns
// (gate/up) or of its block (down), as in the decode kernels.  For that an
// MFMA's 32 K slots have to lie in one absmax block, while a lane loads 16
// packed bytes (32 columns) at once: the lane groups' dwords are exchanged
// with v_permlane32_swap / v_permlane16_swap, 2 (4) VALU operations per 16
// bytes, instead of narrower loads.
//
// Gate/up sums are taken in a fixed order, which depends on the hidden size
// and the number of token tiles only.  The down sums are exact: a block's place
// in the union (its wave and group) depends on what the other tokens select,
// and a token's output does not (see kFdGrid).
//
// At hidden 16384 and 8 tokens (1092 of 1664 blocks, 894 MB) gate/up takes 146
// us (4.0 TB/s) and down 107 (2.8 TB/s; 89 with fp32 sums, at 32 tokens 214
// against 162): two waves a SIMD (the tokens'
// registers) leave the lookups' and MFMAs' latency partly open (without the
// weight loads gate/up still takes 133 us); the loads are temporal, as a row's
// 128-byte line serves two chunks (172 -> 158 us against nontemporal ones).
#include <cstring>
#include <mutex>
#include <utility>

#include "nsmlp_replut.h"

namespace nsmlp {

namespace {

constexpr int kFtThreads = 512;
constexpr int kFtWaves = 8;
constexpr int kFtLutWords = kRepLutBytes / 4;
// 2^23, the range of the grouped down's partial products: a product outside it
// is right here, and reported where the grouped down would report it, so that a
// checked call does not depend on the number of tokens
constexpr float kFtRange = 8388608.0f;

typedef unsigned u32x2v_t __attribute__((ext_vector_type(2)));
typedef double double2_t __attribute__((ext_vector_type(2)));

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
__device__ __forceinline__ uint64_t ft_lane64(uint64_t v, int lane) {
  return ((uint64_t)ft_lane((uint32_t)(v >> 32), lane) << 32) | ft_lane((uint32_t)v, lane);
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

// Down sums: fp64, over multiples of 2^-31 (the unit of the grouped kernels'
// fixed-point sums).  A wave's sum starts at kFdGrid = 1.5 2^21, whose ulp is
// 2^-31, so every fma rounds the exact product of a block's fp32 code sum and
// its absmax to that grid and adds it without another error, as long as the sum
// stays below 2^20; sums on the grid add exactly in any order.  A product that
// is a tie would round by the sum's parity: the absmax's lowest fp64 bit is set
// (a relative 2^-52), so that a tie takes a product of 2^20.  Sums of 2^20 and
// more lose the order independence, not the result.
constexpr double kFdGrid = 3145728.0;
__device__ __forceinline__ double fd_absmax(float a) {
  return __longlong_as_double(__double_as_longlong((double)a) | 1ll);
}

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
  static constexpr bool kPipe = NT == 1 && NCH <= 6;  // the chunks' own pipeline (see below)
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

//
// HEAD: the rows of one dense matrix instead (the LM head: d.gate and d.up are
// both the matrix, p.rows its rows, a pair 32 of them), their sums rounded to
// fp16 and, with p.out_f32, also written before that.
template <bool DQ, int NT, int NCH, bool HEAD>
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
  // pairs: (union block, 16-row half), each a gate and an up tile
  const unsigned pairs = HEAD ? (unsigned)(p.rows + 31) / 32 : 2u * (unsigned)p.nu[0];
  const int p_lo = (int)(blockIdx.x * pairs / gridDim.x);
  const int p_hi = (int)((blockIdx.x + 1) * pairs / gridDim.x);
  {
    LutCodes codes;
    lut_codes_load(d.code, d.code_up, tid, codes);
    lut_store(lds, codes, tid);
    if constexpr (DQ) c2[tid] = tid < 256 ? d.gate.code2[tid] : d.up.code2[tid - 256];
  }
  lds_barrier();
  const rsrc_t rx = make_rsrc(p.x, M * H * 2);
  // opaque to the compiler, which otherwise loads the fields again for every
  // tile (a scalar load's round trip, waited for together with the LDS reads)
  uint32_t rs = (uint32_t)d.gate.row_stride, A = (uint32_t)d.gate.abs_row_stride;
  uint32_t qsh = (uint32_t)d.qbs_shift, dsh = (uint32_t)d.dq_shift;
  uint64_t s_g = reinterpret_cast<uint64_t>(d.gate.absmax2), s_u = reinterpret_cast<uint64_t>(d.up.absmax2);
  float off_g = d.gate.offset, off_u = d.up.offset;
  asm volatile("" : "+s"(rs), "+s"(A), "+s"(qsh), "+s"(dsh), "+s"(s_g), "+s"(s_u), "+s"(off_g), "+s"(off_u));
  // by value: a conditional over the variables themselves selects an address
  auto pick = [](bool c, auto a, auto b) { return c ? a : b; };

  struct Stage {
    uint4 w[SU];
    uint32_t qa[NH];
    float am[NH];
  };
  // equal batches of at most kSlots tiles
  const int batches = (p_hi - p_lo + G::kSlots / 2 - 1) / (G::kSlots / 2);
  const int step = HEAD ? (p_hi - p_lo + batches - 1) / max(batches, 1) : G::kSlots / 2;
  for (int pb = p_lo; pb < p_hi; pb += step) {
    const int np = min(p_hi - pb, step), ntl = 2 * np;
    const int R = (ntl + RW - 1) / RW, VT = R * CGS;
    // lane t: tile t's packed rows and its block's absmax (addresses), the
    // flat index of its first absmax; bit 31 of that: the block is unavailable
    uint64_t tw = 0, ta = 0;
    uint32_t tf = 0x80000000u;
    if (HEAD && lane < ntl) {
      const int r0 = 32 * pb + 16 * lane;
      if (r0 < p.rows) {
        tw = reinterpret_cast<uint64_t>(d.gate.packed + (long long)r0 * rs);
        ta = DQ ? reinterpret_cast<uint64_t>(d.gate.qabsmax + (long long)r0 * A)
                : reinterpret_cast<uint64_t>(d.gate.absmax + (long long)r0 * A);
        tf = (uint32_t)r0 * A;
      }
    }
    if (!HEAD && lane < ntl) {
      const int pi = pb + (lane >> 1), h16 = (pi & 1) * 16;
      const bool up = (lane & 1) != 0;
      const BlockRef br = resolve_id(d, p.ublk[pi >> 1]);
      if (br.ok) {
        const ProjView& pv = up ? (br.dev ? d.up : d.host_up) : (br.dev ? d.gate : d.host_gate);
        tw = reinterpret_cast<uint64_t>(pv.packed + br.q * pv.blk_stride + (long long)h16 * rs);
        ta = DQ ? reinterpret_cast<uint64_t>(pv.qabsmax + br.q * pv.abs_blk_stride + (long long)h16 * A)
                : reinterpret_cast<uint64_t>(pv.absmax + br.q * pv.abs_blk_stride + (long long)h16 * A);
        tf = (32u * (uint32_t)br.b + (uint32_t)h16) * A;
      } else if (wave == 0) {
        atomicOr(d.status, NSMLP_STATUS_BLOCK_UNAVAILABLE);
      }
    }
    int icg = 0, ir = 0;  // column group and round of the next tile to issue
    auto issue = [&](Stage& st, auto unit) {
      constexpr int U = decltype(unit)::value;
      const int t = ir * RW + rw;
      const bool live = icg < CGS && t < ntl;
      const int l = live ? t : 0;
      const uint32_t f = ft_lane(tf, l);
      const bool ok = live && (int)f >= 0;
      const int chb = (icg * CW + cw) * NCH;
      constexpr int c0 = U == 0 ? 0 : SU, c1 = U == 0 ? SU : NCH;
      // the tile's rows; none for a unit past the last chunk where blocks may be
      // host copies (hidden 5120, 32 tokens, half of them: 753 -> 729 us)
      const int nr = !ok || (!HEAD && chb + c0 >= chunks) ? 0 : HEAD ? min(p.rows - 32 * pb - 16 * l, 16) : 16;
      const rsrc_t rp = make_rsrc(reinterpret_cast<const void*>(ft_lane64(tw, l)), nr * (int)rs);
      // temporal: a row's 128-byte line serves two chunks.  A unit's chunk past
      // the last reads the next row (or zeros past the tile): its tokens are zero
      const uint32_t voff = (uint32_t)j * rs + (uint32_t)(chb * 64) + 16u * (uint32_t)g;
#pragma unroll
      for (int c = c0; c < c1; ++c) st.w[c - c0] = buf_ld16c(rp, voff + 64u * (uint32_t)c, 0);
      const rsrc_t ra = make_rsrc(reinterpret_cast<const void*>(ft_lane64(ta, l)), nr * (int)(A * (DQ ? 1u : 4u)));
      const rsrc_t r2 = make_rsrc(reinterpret_cast<const void*>(pick((t & 1) != 0, s_u, s_g)), ok ? p_a2 : 0);
#pragma unroll
      for (int i = 0; i < (2 * (c1 - c0) + 3) / 4; ++i) {
        const uint32_t e = (uint32_t)(128 * chb + 64 * (2 * c0 + 4 * i + g)) >> qsh;
        if constexpr (DQ) {
          // a slot's codes of rows 2 i and 2 i + 1 are interleaved
          st.qa[i] = buf_ldu8c(ra, HEAD ? (uint32_t)j * A + e : (uint32_t)(j & 14) * A + 2u * e + (uint32_t)(j & 1), 0);
          st.am[i] = buf_ldfc(r2, ((f + (uint32_t)j * A + e) >> dsh) * 4u, 0);
        } else {
          st.qa[i] = 0;
          st.am[i] = buf_ldfc(ra, ((uint32_t)j * A + e) * 4u, 0);
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

    // With up to 6 chunks a wave the registers allow a pipeline of the chunks
    // (kPipe): chunk c + 1's lookups go out before chunk c's MFMAs, and the
    // absmax multiplies chunk c - 1's results after them (16 lookups and their
    // address moves and the MFMAs of a chunk lie between an MFMA and the first
    // read of its result; the last chunk of a tile has the drain instead).
    // With more, a chunk's lookups, MFMAs, drain and scaling follow each other.
    uint32_t ad[4];
    auto set_ad = [&](int t) {
#pragma unroll
      for (int m = 0; m < 4; ++m) ad[m] = ((t & 1) ? 128u : 0u) + (uint32_t)(lane & 31) * 4u;
    };
    auto lookup = [&](half8_t (&b)[4], uint4 w) {
      swap32(w.x, w.z);
      swap32(w.y, w.w);
      b[0] = ft_codes8(w.x, ad);
      b[1] = ft_codes8(w.y, ad);
      b[2] = ft_codes8(w.z, ad);
      b[3] = ft_codes8(w.w, ad);
    };
    half8_t bq[2][4];
    set_ad(rw);
    if constexpr (G::kPipe) lookup(bq[0], st[0].w[0]);
    int cg = 0, r = 0;
    for (int v0 = 0; v0 < VT; v0 += RB) {
#pragma unroll
      for (int i = 0; i < RB; ++i) {
        if (v0 + i < VT) {  // uniform over the workgroup
          if (r == 0 && v0 + i > 0) load_x(cg);
          const int t = r * RW + rw, tn = (r + 1 < R ? r + 1 : 0) * RW + rw;
          const int mych = min(chunks - (cg * CW + cw) * NCH, NCH);
          const bool ok = t < ntl && (int)ft_lane(tf, t < ntl ? t : 0) >= 0;
          float4_t acc[NT], cc[2][2][NT];
#pragma unroll
          for (int n = 0; n < NT; ++n) acc[n] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
          // absmax of the lane's halves (lane group g: halves 4 q + g of a unit)
          auto resolve = [&](float (&o)[NH], const Stage& su, int first, int count) {
#pragma unroll
            for (int q = 0; q < (2 * count + 3) / 4; ++q) {
              float a = su.am[q];
              if constexpr (DQ) a = dq_absmax(c2[((t & 1) ? 256 : 0) + su.qa[q]], a, pick((t & 1) != 0, off_u, off_g));
              o[q] = ok && 2 * first + 4 * q + g < 2 * mych ? a : 0.0f;
            }
          };
          float ar[NH], am[4];
          resolve(ar, st[2 * i], 0, SU);
          auto scale = [&](auto cc_) {
            constexpr int c = decltype(cc_)::value;
            constexpr int h = 2 * (c < SU ? c : c - SU);  // the chunk's first half in its unit
            if constexpr (h % 4 == 0) group_values(ar[h / 4], am);
#pragma unroll
            for (int hb = 0; hb < 2; ++hb)
#pragma unroll
              for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[n][e] = __builtin_fmaf(cc[G::kPipe ? c & 1 : 0][hb][n][e], am[(h + hb) % 4], acc[n][e]);
#pragma unroll
            for (int n = 0; n < NT; ++n) asm volatile("" : "+v"(acc[n]));  // summed here, not at its use
          };
          auto products = [&](auto cc_, const half8_t (&b)[4]) {
            constexpr int c = decltype(cc_)::value, o = G::kPipe ? c & 1 : 0;
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
              for (int n = 0; n < NT; ++n)
                cc[o][s >> 1][n] = mfma16(x[c][s][n], b[s], (s & 1) ? cc[o][s >> 1][n] : float4_t{0.0f, 0.0f, 0.0f, 0.0f});
          };
          auto weights = [&](auto cc_) {
            constexpr int c = decltype(cc_)::value;
            if constexpr (c < SU)
              return st[2 * i].w[c];
            else
              return st[2 * i + 1].w[c - SU];
          };
          auto chunk = [&](auto cc_) {
            constexpr int c = decltype(cc_)::value;
            if constexpr (G::kPipe) {
              if constexpr (c + 1 < NCH) {
                lookup(bq[(c + 1) & 1], weights(std::integral_constant<int, c + 1>{}));
              } else {
                set_ad(tn);
                lookup(bq[(c + 1) & 1], st[(2 * i + 2) % PD].w[0]);
              }
              sched_fence();
              products(cc_, bq[c & 1]);
              sched_fence();
              if constexpr (c > 0) {
                scale(std::integral_constant<int, (c > 0 ? c - 1 : 0)>{});
                if constexpr (c == SU) resolve(ar, st[2 * i + 1], SU, NCH - SU);
              }
              if constexpr (c == SU - 1) issue(st[2 * i], U0{});
              if constexpr (c == (NCH - 2 > SU ? NCH - 2 : SU)) issue(st[2 * i + 1], U1{});
              if constexpr (c == NCH - 1) {
                mfma_drain();
                scale(cc_);
              }
            } else {
              if constexpr (c == 0) set_ad(t);
              if constexpr (c == SU) resolve(ar, st[2 * i + 1], SU, NCH - SU);
              lookup(bq[0], weights(cc_));
              products(cc_, bq[0]);
              mfma_drain();
              scale(cc_);
              if constexpr (c == SU - 1) issue(st[2 * i], U0{});
              if constexpr (c == NCH - 1) issue(st[2 * i + 1], U1{});
            }
            sched_fence();
          };
          [&]<int... C>(std::integer_sequence<int, C...>) {
            (chunk(std::integral_constant<int, C>{}), ...);
          }(std::make_integer_sequence<int, NCH>{});
          if constexpr (G::kPipe && NCH % 2 != 0) {
#pragma unroll
            for (int s = 0; s < 4; ++s) bq[0][s] = bq[1][s];
          }
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
    if constexpr (HEAD) {
      const int nr = min(16 * ntl, p.rows - 32 * pb);
      for (int t = wave; t < M; t += kFtWaves)
        for (int r = lane; r < nr; r += kWave) {
          const float y = reinterpret_cast<const float*>(
              slots + (r >> 4) * NT * 64)[((t >> 4) * 64 + ((t >> 2) & 3) * 16 + (r & 15)) * 4 + (t & 3)];
          const long long o = (long long)t * p.rows + 32 * pb + r;
          p.out[o] = f2h(y);
          if (p.out_f32 != nullptr) p.out_f32[o] = y;
        }
      lds_barrier();
      continue;
    }
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
  static constexpr int kC2Word = kFtLutWords, kRefWord = kC2Word + 256, kMaskWord = kRefWord + kFtWaves * NCH * 4 * 2,
                       kNanWord = kMaskWord + kFtWaves * NCH * 4, kCombWord = kNanWord + 2 * RT * 16;
  static constexpr size_t kLds = (size_t)(kCombWord + kFtWaves * RT * NT * 512) * 4;
  static_assert(kLds <= 160 * 1024 && NCH % PD == 0 && kCombWord % 4 == 0 && RT * NT == 4, "geometry");
};

template <bool DQ, bool HOST, int NT>
__global__ void __launch_bounds__(kFtThreads, 2) k_ft_down(FewTokArgs p) {
  using G = FdGeo<NT>;
  constexpr int NCH = G::NCH, RT = G::RT, PD = G::PD;
  extern __shared__ __attribute__((aligned(16))) uint32_t lds[];  // no static LDS: the table is at LDS address 0
  const DecodeArgs& d = p.d;
  float* c2 = reinterpret_cast<float*>(lds + G::kC2Word);
  double2_t* comb = reinterpret_cast<double2_t*>(lds + G::kCombWord);
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
  // rows of a unit: the tokens whose sum is NaN (two units' buffers)
  uint32_t* nans = lds + G::kNanWord;
  if (tid < 2 * RT * 16) nans[tid] = 0;
  // (slot, or block id with bit 30 for a host copy; -1: none) and block id of
  // the wave's blocks, and the tokens that selected them
  int2* refs = reinterpret_cast<int2*>(lds + G::kRefWord) + wave * (NCH * 4);
  uint32_t* masks = lds + G::kMaskWord + wave * (NCH * 4);
  if (lane < NCH * 4) {
    const int u = 4 * c_lo + lane;
    int2 e = make_int2(-1, 0);
    uint32_t mask = 0;
    if (lane < 4 * kc && u < nu) {
      mask = p.umask[u];
      const BlockRef br = resolve_id(d, p.ublk[u]);
      e.y = br.b;
      if (br.ok) e.x = br.dev ? (int)br.q : (0x40000000 | (int)br.q);
    }
    refs[lane] = e;
    masks[lane] = mask;
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
  double* part = p.part + (size_t)cg * M * H;
  Stage st[PD];
#pragma unroll
  for (int i = 0; i < PD; ++i) issue(st[i], rg_lo + i / NCH, i % NCH);
  sched_fence();
  uint32_t ad[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) ad[m] = (uint32_t)lane * 4u;
  float top = 0.0f;  // largest product seen where one may leave the range; inf or nan sums
  for (int rg = rg_lo; rg < rg_hi; ++rg) {
    double acc[RT][NT][4];
#pragma unroll
    for (int m = 0; m < RT; ++m)
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[m][n][e] = kFdGrid;
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      Stage& su = st[c % PD];
      if (c < kc) {  // uniform over the wave
        // row tile m's lookups and MFMAs go out before the absmax multiplies
        // m - 1's results: those lookups and MFMAs lie between an MFMA and the
        // first read of its result (the last tile has the drain instead; a drain
        // a tile cost 4 of 91 us at hidden 16384, 8 tokens)
        // (with host copies and two token tiles the registers do not hold two
        // tiles' products: a drain a tile there)
        constexpr bool kAhead = !(HOST && NT == 2);
        float4_t cc[kAhead ? 2 : 1][4][NT];  // tile m's: cc[m & kPar]
        constexpr int kPar = kAhead ? 1 : 0;
        auto scale = [&](int m) {
          // the lane's absmax, then every block's in all lane groups.  One
          // that is not finite makes its row's sum NaN for the tokens that
          // selected the block (weights 0 and infinite, or NaN), and only
          // for those (the others' products with the block are zero).
          float a = su.am[m];
          if constexpr (DQ) a = dq_absmax(c2[su.qa[m]], a, d.down.offset);
          a = su.ok ? a : 0.0f;
          const bool wide = __any(!(fabsf(a) < 4.0f));
          if (wide && !(fabsf(a) <= 3.402823466e38f)) {
            atomicOr(&nans[((rg - rg_lo) & 1) * (RT * 16) + m * 16 + j], masks[c * 4 + g]);
            top = kFtRange;
            a = 0.0f;
          }
          float am[4];
          group_values(a, am);
          // |code sums| < 2^21 (32 products of |code| <= 1 and |act| < 2^16),
          // so a product outside the range needs an absmax of 4 or more
          if (wide) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
              for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int e = 0; e < 4; ++e) top = fmaxf(top, fabsf(cc[m & kPar][i][n][e] * am[i]));
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const double a64 = fd_absmax(am[i]);
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
              for (int e = 0; e < 4; ++e) acc[m][n][e] = __builtin_fma((double)cc[m & kPar][i][n][e], a64, acc[m][n][e]);
          }
          // summed here: left to itself the compiler moves the sums down to
          // their use and keeps (or spills) every product until then
#pragma unroll
          for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int e = 0; e < 4; ++e) asm volatile("" : "+v"(acc[m][n][e]));
        };
#pragma unroll
        for (int m = 0; m < RT; ++m) {
          uint4 w = su.w[m];
          swap16(w.x, w.y);
          swap16(w.z, w.w);
          swap32(w.x, w.z);
          swap32(w.y, w.w);
          const uint32_t dw[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const half8_t bf = ft_codes8(dw[i], ad);
#pragma unroll
            for (int n = 0; n < NT; ++n) cc[m & kPar][i][n] = mfma16(x[c][i][n], bf, float4_t{0.0f, 0.0f, 0.0f, 0.0f});
          }
          if constexpr (kAhead) {
            sched_fence();
            if (m > 0) scale(m - 1);
            sched_fence();
          } else {
            mfma_drain();
            scale(m);
          }
        }
        if constexpr (kAhead) {
          mfma_drain();
          scale(RT - 1);
        }
      }
      issue(su, rg + (c + PD) / NCH, (c + PD) % NCH);
      sched_fence();
    }
    if (rg > rg_lo) lds_barrier();  // the sums and marks of the unit before have been read
    if (tid < RT * 16) nans[(~(rg - rg_lo) & 1) * (RT * 16) + tid] = 0;
#pragma unroll
    for (int m = 0; m < RT; ++m)
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const double2_t v = {acc[m][n][2 * h] - kFdGrid, acc[m][n][2 * h + 1] - kFdGrid};
          top = fabs(v[0]) < 1.0e300 && fabs(v[1]) < 1.0e300 ? top : kFtRange;
          comb[((wave * 4 + m * NT + n) * 2 + h) * 64 + lane] = v;
        }
    lds_barrier();
    // four (row tile, token tile) sums of the 8 waves: two waves a tile, each
    // two of a lane's four tokens
    const int job = wave >> 1, h = wave & 1, n = job % NT, m = job / NT;
    double2_t y = comb[(job * 2 + h) * 64 + lane];
#pragma unroll
    for (int w = 1; w < kFtWaves; ++w) y += comb[((w * 4 + job) * 2 + h) * 64 + lane];
    const int o = (rg * RT + m) * 16 + j;
    const uint32_t nan = nans[((rg - rg_lo) & 1) * (RT * 16) + m * 16 + j];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int t = 16 * n + 4 * g + 2 * h + e;
      if (t < M) part[(uint32_t)t * (uint32_t)H + (uint32_t)o] = (nan >> t) & 1u ? __builtin_nan("") : y[e];
    }
  }
  if (p.report_range && top >= kFtRange) atomicOr(d.status, NSMLP_STATUS_FIXED_RANGE);
}

__global__ void __launch_bounds__(256) k_ft_fin(FewTokArgs p) {
  const long long n = (long long)p.M * p.d.H;
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int CG = p.nu[1];
  double sum = 0.0;
#pragma unroll 4
  for (int s = 0; s < CG; ++s) sum += p.part[(long long)s * n + i];
  float y = (float)sum;
  if (p.d.down_bias != nullptr) y += h2f(p.d.down_bias[(int)(i % p.d.H)]);
  p.out[i] = f2h(y);
}

int ft_token_tiles(int M) { return M <= 16 ? 1 : 2; }

using FtFn = void (*)(FewTokArgs);
struct FtKernel {
  FtFn fn;
  size_t lds;
};
template <bool DQ, int NT, int NCH, bool HEAD>
constexpr FtKernel ft_gu() {
  return FtKernel{k_ft_gu<DQ, NT, NCH, HEAD>, FtGeo<NT, NCH>::kLds};
}
template <bool DQ, bool HOST, int NT>
constexpr FtKernel ft_down() {
  return FtKernel{k_ft_down<DQ, HOST, NT>, FdGeo<NT>::kLds};
}
// [dq][one token tile of 4, 5, 6, 8 chunks, two of 3, 4]
#define NSMLP_FT_GU(DQ) \
  {ft_gu<DQ, 1, 4, false>(), ft_gu<DQ, 1, 5, false>(), ft_gu<DQ, 1, 6, false>(), \
   ft_gu<DQ, 1, 8, false>(), ft_gu<DQ, 2, 3, false>(), ft_gu<DQ, 2, 4, false>()}
const FtKernel kFtGu[2][6] = {NSMLP_FT_GU(false), NSMLP_FT_GU(true)};
#undef NSMLP_FT_GU
// [dq][3 or 4 chunks][token tiles - 1]: the LM head has one order of its sums
// for one and two token tiles, so a row's bits do not depend on the rows with it
#define NSMLP_FT_HEAD(DQ) \
  {{ft_gu<DQ, 1, 3, true>(), ft_gu<DQ, 2, 3, true>()}, {ft_gu<DQ, 1, 4, true>(), ft_gu<DQ, 2, 4, true>()}}
const FtKernel kFtHead[2][2][2] = {NSMLP_FT_HEAD(false), NSMLP_FT_HEAD(true)};
#undef NSMLP_FT_HEAD
constexpr int kFtGuChunks[6] = {4, 5, 6, 8, 3, 4};
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
      for (int c = 0; c < 2; ++c)
        for (const FtKernel& k : kFtHead[q][c]) set(k);
      for (int h = 0; h < 2; ++h)
        for (const FtKernel& k : kFtDown[q][h]) set(k);
    }
  });
}
void ft_launch(const FtKernel& k, int wgs, const FewTokArgs& p, hipStream_t s) {
  k.fn<<<dim3((unsigned)wgs), dim3(kFtThreads), k.lds, s>>>(p);
}

// The kernel (by the chunks a wave holds), column waves of a workgroup and
// column groups (each a pass over the workgroup's tiles with its own tokens in
// registers) for H columns: the fewest column groups, then the fewest chunk
// slots, then the fewest chunks a wave.  Whole prefill call, top-k an eighth of
// the blocks, chunks x waves (groups where more than one), the rule's choice
// first, in us.  8 tokens: hidden 3072 6x4 58, 4x8 58; 4096 4x8 63, 8x4 64; 5120
// 5x8 72, 4x4(3) 76; 6144 6x8 79, 4x4(3) 82; 8192 8x8 98, 4x8(2) 100; 10240
// 5x8(2) 132, 4x4(5) 131; 11264 6x8(2) 157, 4x8(3) 159; 12288 6x8(2) 167, 4x8(3)
// 164; 14336 8x8(2) 216, 4x4(7) 217; 16384 8x8(2) 251, 4x8(4) 259.  24 tokens:
// 3072 3x8 66, 4x8 69; 5120 3x8(2) 106, 4x4(3) 112; 6144 3x8(2) 111, 4x4(3) 118;
// 7168 4x8(2) 138, 3x8(3) 147; 16384 4x8(4) 435, 3x8(6) 484.
int ft_columns(int H, int NT, int* cw, int* cgs) {
  const int chunks = H / 128;
  int best = 0, cost = 0x7FFFFFFF;
  for (int i = NT == 1 ? 0 : 4; i < (NT == 1 ? 4 : 6); ++i)
    for (int w = 1; w <= kFtWaves; w *= 2) {
      const int n = kFtGuChunks[i], c = (chunks + w * n - 1) / (w * n);
      const int v = c * 100000 + c * n * w * 16 + n;
      if (v < cost) {
        cost = v;
        best = i;
        *cw = w;
        *cgs = c;
      }
    }
  return best;
}

}  // namespace

size_t few_tokens_workspace(int H, int NB, int M, int k) {
  auto up = [](size_t v) { return (v + 255) / 256 * 256; };
  const long long nu = (long long)M * k < NB ? (long long)M * k : NB;
  const int cg = ft_groups_min((int)nu, ft_token_tiles(M)) + kFtGroupsTried - 1;
  return 256 + 2 * up((size_t)NB * 4) + up((size_t)M * NB * 64) + up((size_t)cg * M * H * 8);
}

// Up to 32 tokens (two 16-token tiles of 128 VGPRs between them).  The grouped
// kernels these replace there read the weights once per block as well, but
// work tile by tile on token lists (hidden 16384, 1664 blocks, top-k 208,
// double-quantised, whole prefill call with its route, which is 6 us shorter
// in the second figures): 2 tokens 366 -> 113 us, 8 tokens 578 -> 276, 16 tokens
// 521 -> 345, 32 tokens 541 -> 513; hidden 4096, 448 blocks, top-k 64: 8 tokens
// 144 -> 70, 32 tokens 103 -> 93; hidden 5120, 432 blocks, top-k 61, 32 tokens,
// the closest: 109 -> 108 (its 40 chunks leave column waves idle; the grouped
// kernels behind the present route would take about 103).  Four
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
  p.part = (double*)w;
  const int gu = ft_columns(d.H, NT, &p.gu_cw, &p.gu_cgs);
  const long long n2 = (((long long)d.H * d.NB * 32 / d.qbs) + (1LL << d.dq_shift) - 1) >> d.dq_shift;
  p.gu_a2bytes = p.dn_a2bytes = (int)(n2 * 4);
  k_ft_list<<<dim3(1), dim3(1024), 0, s>>>(p);
  ft_set_lds();
  ft_launch(kFtGu[d.dq ? 1 : 0][gu], cus, p, s);
  ft_launch(kFtDown[d.dq ? 1 : 0][d.host_down.packed != nullptr ? 1 : 0][NT - 1], cus, p, s);
  const long long n = (long long)p.M * d.H;
  k_ft_fin<<<dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s>>>(p);
}

// The few-row LM head against passes of one or two rows (k_rows_rep), fp32
// absmax, 128256 rows, one call: hidden 4096, 3 rows 145 -> 62 us, 5 rows 227 ->
// 62 (4.8 TB/s), 16 rows 701 -> 67, 32 rows 1397 -> 90; hidden 16384, 5 rows 831
// -> 227.  Calls of one and two rows stay there: they give bit-equal logits with
// each other, and one row is faster (190 us at hidden 16384, 51 at 4096).  A call
// of three rows or more takes every row here, and the column split is the
// two-tile one for every number of rows, so that all the rows of all such calls
// have one order of sums; 4 rows against the one-tile split: hidden 9216 189 ->
// 151 us, 12288 205 -> 178, 5120 99 -> 98, 16384 230 -> 226, 2304 44 -> 47, the
// worst.
// MFMA chunks want whole 128 columns, and an absmax of whole 64-column halves.
bool few_tokens_rows_fit(const RowsArgs& a, int rows) {
  return rows > 2 && a.in % 128 == 0 && a.qbs_shift >= 6 && device_cus() >= 64;
}

int launch_few_tokens_rows(const RowsArgs& a, int rows, hipStream_t s) {
  FewTokArgs p;
  memset(&p, 0, sizeof(p));
  DecodeArgs& d = p.d;
  d.H = a.in;
  d.qbs_shift = a.qbs_shift;
  d.dq = a.dq;
  d.dq_shift = a.dq_shift;
  d.gate.packed = a.packed;
  d.gate.row_stride = a.rs;
  d.gate.absmax = a.absmax;
  d.gate.qabsmax = a.qabsmax;
  d.gate.abs_row_stride = a.ars;
  d.gate.absmax2 = a.absmax2;
  d.gate.code2 = a.code2;
  d.gate.offset = a.offset;
  d.up = d.gate;
  d.code = d.code_up = a.code;
  p.x = a.x;
  p.M = rows < kFtMaxTok ? rows : kFtMaxTok;
  p.rows = a.out;
  p.out = a.y;
  p.out_f32 = a.out_f32;
  p.gu_a2bytes = a.a2_bytes;
  p.NT = ft_token_tiles(p.M);
  const int gu = ft_columns(a.in, 2, &p.gu_cw, &p.gu_cgs);  // the two-tile choice, whatever the rows
  ft_set_lds();
  ft_launch(kFtHead[a.dq ? 1 : 0][kFtGuChunks[gu] - 3][p.NT - 1], device_cus(), p, s);
  return p.M;
}

}  // namespace nsmlp
