// Matrix products with few output tiles, for gfx950: the same products and epilogues as gemm.hip (formats, formulas
// and the order of their float steps there), for shapes whose 256 x 256 tiles would leave most compute units idle.
//
// What bounds such a product is the L2 -> LDS stream of its operands and the latency of its start and end, not the
// matrix units. So the tiles are small (32 x 32 to 96 x 128) and the waves of a workgroup split K: wave g multiplies
// the whole tile over the 128-byte K slices g, g + NWK, g + 2 NWK, ... from LDS slots of its own, filled by LDS-direct
// loads NST steps ahead. No wave waits for another before the end: its own vmcnt orders its loads and there is no
// barrier in the loop. Slices are whole 128-byte cache lines (64-byte slices: 300 x 4096 x 4096 bf16 23.6 us against
// 19.1). At the end the partial tiles meet in LDS (float32, added in the order of the waves; int32 sums are exact)
// and all threads run the epilogue on 4 consecutive columns each; what it needs from memory (scales, bias, row types)
// is loaded before the first slice (loaded in the epilogue: +1.5 to 2 us).
// h8 weights stay int8 in LDS and are widened in registers (exact), so no widened copy of the weights is made.
// Tiles are ordered down the rows first and each XCD takes a contiguous range, so that it reads its own columns of
// W once and the (small) A from its L2.
// Measured (us a call, 256 x 256 tiles -> here): 300 x 4096 x 4096 h8 99 -> 18.8, bf16 82 -> 18.8, q8 48 -> 14.2;
// 16 x 4096 x 4096 q8 44 -> 8.7; 128 x 2048 x 8192 q8 into the residual 89 -> 10.2.
#include "gemm_common.h"

namespace h3 {
namespace {

// 8 int8 values to half, exact: u = code + 128 as the low byte of the half 1024 + u, minus 1152.
__device__ __forceinline__ i32x4 widen8(unsigned lo, unsigned hi) {
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  const unsigned s[2] = {lo ^ 0x80808080u, hi ^ 0x80808080u};
  const h2 off = {(_Float16)1152.0f, (_Float16)1152.0f};
  i32x4 r;
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const h2 a = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, s[i], 0x04010400u)) - off;
    const h2 b = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, s[i], 0x04030402u)) - off;
    r[2 * i] = __builtin_bit_cast(int, a);
    r[2 * i + 1] = __builtin_bit_cast(int, b);
  }
  return r;
}

template <int WFMT, int TM_, int TN_, int NWK_, int NST_>
struct KCfg {
  static constexpr int KS = 128;                          // K bytes of A per step of a wave (whole cache lines)
  static constexpr int NC = KS / 32;                      // MFMAs along K per step
  static constexpr bool H8 = WFMT == 6;
  static constexpr int AT = WFMT == 1 ? A_I8 : WFMT == 5 ? A_BF16 : A_F16;
  static constexpr int SM = WFMT == 1 ? S_ROW_COL : H8 ? S_COL : S_NONE;
  static constexpr int TM = TM_, TN = TN_, NWK = NWK_, NST = NST_;
  static constexpr int MI = TM / 32, NJ = TN / 32;
  static constexpr int WB = H8 ? KS / 2 : KS;             // bytes of a W row in a K slice
  static constexpr int SLOT = TM * KS + TN * WB;          // LDS bytes of one wave's K slice
  static constexpr int NQA = TM * KS / 1024, NQW = TN * WB / 1024;  // 1 KB loads per slice: A, W
  static constexpr int LPS = NQA + NQW;
  static constexpr int RS = TN * 4 + 16;                  // bytes of a row of a partial tile
  static constexpr int PI = MI == 1 || NWK * TM * RS <= 160 * 1024 ? MI : MI / 2;  // MFMA row tiles per pass of the end
  static constexpr int PR = 32 * PI;                      // rows of a pass
  static constexpr int LDS = NWK * (NST * SLOT > PR * RS ? NST * SLOT : PR * RS);
  static_assert(TN * WB % 1024 == 0 && MI % PI == 0 && LDS <= 160 * 1024 && (NST - 1) * LPS <= 63, "tile configuration");
};

// 16-byte piece p of an LDS row of RBY bytes sits at slot p ^ ((row / rows per 256 bytes) % pieces): the 16 rows of a
// pass of a 16-byte read then cover all banks.
template <int RBY>
__device__ __forceinline__ int kslot(int row, int piece) {
  return piece ^ ((row / (256 / RBY)) % (RBY / 16));
}
// the piece of a row's slice (its byte in the slice) that lane `lane` of load q fetches, and its byte among rows of
// `str` bytes
template <int RBY>
__device__ __forceinline__ int kpiece(int q, int lane) {
  constexpr int NP = RBY / 16;
  return kslot<RBY>(q * (64 / NP) + lane / NP, lane % NP) * 16;
}
template <int RBY>
__device__ __forceinline__ int kfetch(int q, int lane, int str) {
  constexpr int NP = RBY / 16;
  return (q * (64 / NP) + lane / NP) * str + kpiece<RBY>(q, lane);
}

template <class C>
__global__ __launch_bounds__(C::NWK * 64) void gemm_ksplit_kernel(GemmArgs g, GemmParams p, int ntm, int ot, int epi) {
  constexpr int TM = C::TM, TN = C::TN, MI = C::MI, NJ = C::NJ, NST = C::NST, NWK = C::NWK, LPS = C::LPS, KS = C::KS, NC = C::NC;
  constexpr int AT = C::AT, ES = AT == A_I8 ? 1 : 2, WES = AT == A_I8 || C::H8 ? 1 : 2;
  using Acc = AccOf<AT>;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, hl = lane >> 5, l32 = lane & 31;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int astr = p.a_stride * ES, wstr = p.w_stride * WES;

  // XCD-contiguous tile ranges (workgroup b runs on XCD b % 8), row tiles first
  const int nb = gridDim.x, b = blockIdx.x;
  const int per = nb >> 3, rem = nb & 7, xcd = b & 7, loc = b >> 3;
  const int lid = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + loc;
  const int nt = lid / ntm, mt = lid - nt * ntm;
  const int m0 = mt * TM, n0 = nt * TN;

  const int reca = __builtin_amdgcn_readfirstlane(max(0, min(TM, p.M - m0)) * astr);
  const int recw = __builtin_amdgcn_readfirstlane(max(0, min(TN, p.N - n0)) * wstr);
  const __amdgpu_buffer_rsrc_t ra =
      __builtin_amdgcn_make_buffer_rsrc((void *)(g.a + (size_t)m0 * astr), (short)0, reca, 0x00020000);
  const __amdgpu_buffer_rsrc_t rw =
      __builtin_amdgcn_make_buffer_rsrc((void *)(g.w + (size_t)n0 * wstr), (short)0, recw, 0x00020000);
  const int nk = (p.K * ES + KS - 1) / KS;          // K slices (the last may be half of one)
  const int steps = (nk + NWK - 1) / NWK;           // of each wave (slices past the last read as zero)
  const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) char *)smem + w * (NST * C::SLOT);
  const char *own = smem + w * (NST * C::SLOT);

  // a load fills 1 KB of LDS; each lane fetches the piece that its slot holds
  int offa[C::NQA], offw[C::NQW];
#pragma unroll
  for (int q = 0; q < C::NQA; q++) offa[q] = kfetch<KS>(q, lane, astr);
#pragma unroll
  for (int q = 0; q < C::NQW; q++) offw[q] = kfetch<C::WB>(q, lane, wstr);
  const int krow = p.K * ES;  // bytes of a row's K; the last slice may hold half of it (K is a multiple of 64 bytes)
  auto dma = [&](int s) __attribute__((always_inline)) {
    const unsigned st = lds0 + ((unsigned)s % NST) * C::SLOT;
    const int kt = s * NWK + w;
    if ((kt + 1) * KS <= krow) {
#pragma unroll
      for (int q = 0; q < C::NQA; q++) dma16(st + q * 1024, (unsigned)(offa[q] + kt * KS), ra);
#pragma unroll
      for (int q = 0; q < C::NQW; q++) dma16(st + TM * KS + q * 1024, (unsigned)(offw[q] + kt * C::WB), rw);
    } else {
      // pieces past the end of K read as zero
      const int left = max(0, krow - kt * KS);  // bytes of A's slice, WB / KS of them of W's
#pragma unroll
      for (int q = 0; q < C::NQA; q++)
        dma16(st + q * 1024, kpiece<KS>(q, lane) < left ? (unsigned)(offa[q] + kt * KS) : 0x80000000u, ra);
#pragma unroll
      for (int q = 0; q < C::NQW; q++)
        dma16(st + TM * KS + q * 1024,
              kpiece<C::WB>(q, lane) < left * C::WB / KS ? (unsigned)(offw[q] + kt * C::WB) : 0x80000000u, rw);
    }
  };

  Acc acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; i++)
#pragma unroll
    for (int j = 0; j < NJ; j++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[i][j][e] = 0;

  // Operands of a step. h8: lane half hl takes the 16 codes of W piece 2 d + hl, the first 8 for MFMA 2 d, the others
  // for MFMA 2 d + 1, so its A pieces are 2 (2 d + hl) and the one after it instead of 2 c + hl (any order of K that
  // both sides share).
  struct Ops {
    i32x4 a[NC][MI], w[C::H8 ? NC / 2 : NC][NJ];
  };
  auto read_ops = [&](Ops &o, int s) __attribute__((always_inline)) {
    const char *sA = own + ((unsigned)s % NST) * C::SLOT, *sW = sA + TM * KS;
#pragma unroll
    for (int c = 0; c < NC; c++) {
      const int pa = C::H8 ? 2 * ((c & ~1) + hl) + (c & 1) : 2 * c + hl;
#pragma unroll
      for (int i = 0; i < MI; i++) {
        const int r = 32 * i + l32;
        o.a[c][i] = *(const i32x4 *)(sA + r * KS + kslot<KS>(r, pa) * 16);
      }
      if (!C::H8 || (c & 1) == 0) {
#pragma unroll
        for (int j = 0; j < NJ; j++) {
          const int r = 32 * j + l32;
          o.w[C::H8 ? c / 2 : c][j] = *(const i32x4 *)(sW + r * C::WB + kslot<C::WB>(r, (C::H8 ? c : 2 * c) + hl) * 16);
        }
      }
    }
  };
  // Step s: its operands are in registers (cur), so its slot is free and takes step s + NST; then the reads of step
  // s + 1 (once landed) run beside the MFMAs of step s.
  auto mfmas = [&](const Ops &o, int c0, int c1) __attribute__((always_inline)) {
#pragma unroll
    for (int c = c0; c < c1; c++) {
      i32x4 wv[NJ];
#pragma unroll
      for (int j = 0; j < NJ; j++) {
        if constexpr (C::H8) wv[j] = widen8((unsigned)o.w[c / 2][j][2 * (c & 1)], (unsigned)o.w[c / 2][j][2 * (c & 1) + 1]);
        else wv[j] = o.w[c][j];
      }
#pragma unroll
      for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++) acc[i][j] = mma<AT>(wv[j], o.a[c][i], acc[i][j]);
    }
  };
  auto step = [&](int s, const Ops &cur, Ops &nxt) __attribute__((always_inline)) {
    // with one slot the wait below is for the load just issued: half of the MFMAs go before it
    constexpr int CB = NST == 1 ? NC / 2 : 0;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    dma(s + NST);
    mfmas(cur, 0, CB);
    if constexpr (CB > 0) __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NST - 1) * LPS) : "memory");
    read_ops(nxt, s + 1);
    mfmas(cur, CB, NC);
  };

  // What the end needs from memory is loaded first: each thread writes the 4 columns n of rows m0 + row0 + RPI it
  constexpr int PPR = TN / 4, NT = NWK * 64, RPI = NT / PPR, PI = C::PI, PR = C::PR, RS = C::RS;
  constexpr int IT = PR > RPI ? PR / RPI : 1, NP = MI / PI;  // rows per thread and pass, passes
  static_assert(NT % PPR == 0 && (PR % RPI == 0 || (RPI % PR == 0 && NP == 1)), "rows per thread");
  const int row0 = tid / PPR, nl = 4 * (tid % PPR), n = n0 + nl;
  const bool all = g.vec;  // N is then a multiple of the output's 16-byte vector, so of 4
  int nc[4];
  float sw[4], bn[4], sam[NP * IT];
  int gro[NP * IT];
#pragma unroll
  for (int r = 0; r < 4; r++) {
    nc[r] = min(n + r, p.N - 1);
    sw[r] = C::SM != S_NONE ? g.sw[nc[r]] : 1.0f;
    bn[r] = g.bias ? g.bias[nc[r]] : 0.0f;
  }
#pragma unroll
  for (int k = 0; k < NP * IT; k++) {
    const int m = min(m0 + row0 + RPI * k, p.M - 1);
    sam[k] = C::SM == S_ROW_COL ? g.sa[m] : 1.0f;
    gro[k] = epi ? min((int)g.rtype[m], g.ntypes - 1) * p.g_stride : 0;
  }

#pragma unroll
  for (int s = 0; s < NST; s++) dma(s);
  Ops o0, o1;
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NST - 1) * LPS) : "memory");
  read_ops(o0, 0);
  for (int s = 0; s < steps; s += 2) {
    step(s, o0, o1);
    if (s + 1 < steps) step(s + 1, o1, o0);
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");

  // partial tiles, PR rows at a time: wave w's at w * PR rows; element e of MFMA tile (i, j) is
  // C[32 i + l32][32 j + 8 (e / 4) + 4 hl + e % 4]
#pragma unroll
  for (int ps = 0; ps < NP; ps++) {
    float xv[IT][4], gv[IT][4];
    if (epi) {
#pragma unroll
      for (int k = 0; k < IT; k++) {
        const int m = min(m0 + row0 + RPI * (ps * IT + k), p.M - 1);
        const float *xr = (const float *)g.out + (size_t)m * p.c_stride, *gr = g.gate + gro[ps * IT + k];
#pragma unroll
        for (int r = 0; r < 4; r++) {
          xv[k][r] = xr[nc[r]];
          gv[k][r] = gr[nc[r]];
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PI; i++)
#pragma unroll
      for (int j = 0; j < NJ; j++) {
        const Acc v = acc[ps * PI + i][j];
        const i32x16 vi = __builtin_bit_cast(i32x16, v);
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const i32x4 f = q == 0   ? __builtin_shufflevector(vi, vi, 0, 1, 2, 3)
                          : q == 1 ? __builtin_shufflevector(vi, vi, 4, 5, 6, 7)
                          : q == 2 ? __builtin_shufflevector(vi, vi, 8, 9, 10, 11)
                                   : __builtin_shufflevector(vi, vi, 12, 13, 14, 15);
          *(i32x4 *)(smem + (w * PR + 32 * i + l32) * RS + (32 * j + 8 * q + 4 * hl) * 4) = f;
        }
      }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < IT; k++) {
      const int ml = row0 + RPI * k, m = m0 + ps * PR + ml;
      if (ml >= PR || m >= p.M || n >= p.N) continue;
      float v[4];
      if constexpr (AT == A_I8) {
        i32x4 t = *(const i32x4 *)(smem + ml * RS + nl * 4);
#pragma unroll
        for (int u = 1; u < NWK; u++) t += *(const i32x4 *)(smem + (u * PR + ml) * RS + nl * 4);
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int ti = t[r];
          v[r] = (float)ti;
        }
      } else {
        float4 t = *(const float4 *)(smem + ml * RS + nl * 4);
#pragma unroll
        for (int u = 1; u < NWK; u++) {
          const float4 d = *(const float4 *)(smem + (u * PR + ml) * RS + nl * 4);
          t.x += d.x, t.y += d.y, t.z += d.z, t.w += d.w;
        }
        v[0] = t.x, v[1] = t.y, v[2] = t.z, v[3] = t.w;
      }
#pragma unroll
      for (int r = 0; r < 4; r++) {
        if constexpr (C::SM == S_ROW_COL) v[r] = v[r] * sam[ps * IT + k] * sw[r];
        else if constexpr (C::SM == S_COL) v[r] = v[r] * sw[r];
        if (g.bias) v[r] += bn[r];
        if (epi) v[r] = xv[k][r] + gv[k][r] * v[r];
      }
      const size_t at = (size_t)m * p.c_stride + n;
      if (ot == T_F32) {
        float *dst = (float *)g.out + at;
        if (all) {
          *(float4 *)dst = make_float4(v[0], v[1], v[2], v[3]);
        } else {
#pragma unroll
          for (int r = 0; r < 4; r++)
            if (n + r < p.N) dst[r] = v[r];
        }
      } else {
        unsigned short h[4];
#pragma unroll
        for (int r = 0; r < 4; r++)
          h[r] = ot == T_BF16 ? __builtin_bit_cast(unsigned short, (__bf16)v[r])
                              : __builtin_bit_cast(unsigned short, (_Float16)v[r]);
        unsigned short *dst = (unsigned short *)g.out + at;
        if (all) {
          *(uint2 *)dst = make_uint2(h[0] | (unsigned)h[1] << 16, h[2] | (unsigned)h[3] << 16);
        } else {
#pragma unroll
          for (int r = 0; r < 4; r++)
            if (n + r < p.N) dst[r] = h[r];
        }
      }
    }
  }
}

template <class C>
int launch(int ot, int epi, const GemmArgs &g, const GemmParams &p, hipStream_t stream, std::string *err) {
  auto kern = gemm_ksplit_kernel<C>;
  static bool attr_set = false;
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS);
    if (e != hipSuccess) {
      *err = std::string("hipFuncSetAttribute: ") + hipGetErrorString(e);
      return -1;
    }
    attr_set = true;
  }
  const int ntm = (p.M + C::TM - 1) / C::TM, ntn = (p.N + C::TN - 1) / C::TN;
  hipLaunchKernelGGL(kern, dim3((unsigned)(ntm * ntn)), dim3(C::NWK * 64), C::LDS, stream, g, p, ntm, ot, epi);
  return 0;
}

template <int WFMT>
int launch_fmt(int kcfg, int ot, int epi, const GemmArgs &g, const GemmParams &p, hipStream_t stream, std::string *err) {
  switch (kcfg) {
    case KSPLIT_32x32: return launch<KCfg<WFMT, 32, 32, 8, 2>>(ot, epi, g, p, stream, err);
    case KSPLIT_64x64: return launch<KCfg<WFMT, 64, 64, 4, 2>>(ot, epi, g, p, stream, err);
    case KSPLIT_96x64: return launch<KCfg<WFMT, 96, 64, 4, 2>>(ot, epi, g, p, stream, err);
    case KSPLIT_96x128:
      if constexpr (WFMT != 1) return launch<KCfg<WFMT, 96, 128, 4, WFMT == 6 ? 2 : 1>>(ot, epi, g, p, stream, err);
      [[fallthrough]];
    default: *err = "no such tile configuration"; return -1;
  }
}

}  // namespace

int launch_gemm_ksplit(int wfmt, int kcfg, int ot, int epi, const GemmArgs &g, const GemmParams &p, hipStream_t stream,
                       std::string *err) {
  switch (wfmt) {
    case 1: return launch_fmt<1>(kcfg, ot, epi, g, p, stream, err);
    case 4: return launch_fmt<4>(kcfg, ot, epi, g, p, stream, err);
    case 5: return launch_fmt<5>(kcfg, ot, epi, g, p, stream, err);
    default: return launch_fmt<6>(kcfg, ot, epi, g, p, stream, err);
  }
}

}  // namespace h3
