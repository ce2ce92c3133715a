// Flash attention for gfx950 at sizes that leave most compute units idle with 256-row tiles: few heads, short
// sequences, causal masks. Semantics as attention.hip's kernels (scores in log2 units, key masking at L and by the
// causal offset, int8 scores scaled by qs_i * ks_j, P rounded to the value type, O divided by the row sum).
//
// What bounds such a call is the length of one workgroup's chain of key blocks and the number of workgroups (and, as the
// sizes grow, the L2 -> LDS stream of K and V, which a tile of 32 rows reads 8 times as often as one of 256), so here a
// workgroup owns only 32 NU query rows of one head (NU 1; 2 for longer calls at head dim 96, where two tiles still leave
// two waves per SIMD) and its 4 waves split the keys: wave g takes the 32-key blocks g, g + 4, ... of all the rows, with
// a running maximum, row sum and O of its own, and the four partial states meet in LDS at the end (the online-softmax
// merge), so there is no second launch and no partial state in memory. The waves share nothing in the loop: each stages
// its K and V blocks in LDS of its own by LDS-direct loads ordered by its own vmcnt, with no barrier. The K slot is
// refilled while the softmax and P V of a block run, the V slot while the next block's scores do. Two waves per SIMD
// (registers held to that; V operands read 16 keys at a time) cover each other's waits: 8 to 10% over one.
// Measured against 256-row tiles: small_tiles in attention.hip.
// Layouts (S^T = K Q^T with K rows in pi order, O^T = V^T P^T, transposing V reads, swizzles) as in attention.hip.
// Head dim 96 keeps 256-byte LDS rows (the missing pieces are never fetched and never read).
#include "attention_common.h"

#include <algorithm>

namespace h3 {
namespace {

constexpr int NWS = 4;             // waves per workgroup (key groups)
constexpr int KB = 32;             // keys per block
constexpr float SLACK_S = 8.0f;    // log2 units the running maximum may lag behind a score

template <int DG, int QKT, int NU_>
struct CfgS {
  static constexpr bool QK8 = QKT == T_I8;
  static constexpr int NU = NU_;
  static constexpr int D = DG == 96 ? 128 : DG;          // channels of an LDS row
  static constexpr int ESZ = QK8 ? 1 : 2;
  static constexpr int RB = D * ESZ, RBG = DG * ESZ;     // bytes of a K row: in LDS, in memory
  static constexpr int NP = RB / 16;                     // 16-byte pieces of a K row in LDS
  static constexpr int NCH = DG * ESZ / 32;              // score MFMAs per 32 x 32 tile
  static constexpr int NDB = DG / 32;                    // 32-channel blocks of O
  static constexpr int KBYTES = KB * RB, VBYTES = KB * D * 2;
  static constexpr int KDMA = KBYTES / 1024, VDMA = VBYTES / 1024;  // 1 KB loads per block
  static constexpr int SBYTES = QK8 ? 256 : 0;           // key scales of a block (one 256-byte load)
  static constexpr int SLOT = KBYTES + VBYTES + SBYTES;  // LDS of a wave
  static constexpr int NKL = KDMA + (QK8 ? 1 : 0);       // loads of a K block
  static constexpr int ORS = (DG + 4) * 4;               // bytes of a row of a partial state
  static constexpr int MERGE = NWS * (32 * ORS + 32 * 8);  // 32 rows of each wave: O, then (m, l)
  static constexpr int LDS = NWS * SLOT > MERGE ? NWS * SLOT : MERGE;
};

template <int DG, int QKT, int VT, int NU, bool DUMP>
__global__ __launch_bounds__(NWS * 64) __attribute__((amdgpu_waves_per_eu(2)))
void attention_small_kernel(const char *__restrict__ Q, const char *__restrict__ K, const char *__restrict__ V,
                            char *__restrict__ O, const float *__restrict__ qs, const float *__restrict__ ks,
                            int *__restrict__ dump, AttnParams p, int nqb, int causal, int ot) {
  using C = CfgS<DG, QKT, NU>;
  constexpr int D = C::D, NDB = C::NDB, NCH = C::NCH;
  constexpr bool QK8 = C::QK8;
  using VT8 = typename Vec8<VT>::type;
  using VE = typename Vec8<VT>::elem;
  using VP2 = typename Vec8<VT>::pair;
  using SAcc = typename std::conditional<QK8, i32x16, f32x16>::type;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, hl = lane >> 5, l32 = lane & 31;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);

  // XCD-contiguous tile ranges (workgroup b runs on XCD b % 8), so that an XCD's tiles share their heads' K and V in
  // its L2; with a causal mask a head's longest tiles go first
  const int nb = gridDim.x, b = blockIdx.x;
  const int per = nb >> 3, rem = nb & 7, xcd = b & 7, loc = b >> 3;
  const int lid = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + loc;
  const int h = lid / nqb, qt = lid - h * nqb, qb = causal ? nqb - 1 - qt : qt;
  const int kvh = h / (p.H / p.KVH);
  const int qt0 = qb * 32 * NU;  // first query row of the tile

  const char *Kh = K + (size_t)kvh * p.k_rows * C::RBG;
  const char *Vh = V + (size_t)kvh * p.k_rows * DG * 2;
  const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc((void *)Kh, (short)0, p.L * C::RBG, 0x00020000);
  const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc((void *)Vh, (short)0, p.L * DG * 2, 0x00020000);
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      (void *)(QK8 ? ks + (size_t)kvh * p.k_rows : nullptr), (short)0, QK8 ? p.L * 4 : 0, 0x00020000);
  const int kend = causal ? min(p.L, qt0 + 32 * NU + p.causal_off) : p.L;
  const int nblk = kend > 0 ? (kend + KB - 1) / KB : 0;

  // LDS-direct loads of a block: load r of a wave fills 1 KB; each lane fetches the 16-byte piece whose swizzled
  // place that is. Rows at or past L, and pieces past a row in memory (head dim 96), read as zero.
  const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) char *)smem + w * C::SLOT;
  const char *own = smem + w * C::SLOT;
  unsigned kgo[C::KDMA], vgo[C::VDMA];
#pragma unroll
  for (int r = 0; r < C::KDMA; r++) {
    const int o = r * 1024 + 16 * lane, row = o / C::RB, pc = ((o / 16) % C::NP) ^ kswz<C::RB, C::NP>(row);
    kgo[r] = pc * 16 < C::RBG ? row * C::RBG + pc * 16 : 0x80000000u;
  }
#pragma unroll
  for (int r = 0; r < C::VDMA; r++) {
    constexpr int R = 256 / (D * 2) > 0 ? 256 / (D * 2) : 1;
    const int o = r * 1024 + 16 * lane, row = o / (D * 2), in = o % (D * 2);
    const int pc = 2 * ((in >> 5) ^ (2 * ((row & 3) / R))) + ((in >> 4) & 1);
    vgo[r] = pc * 16 < DG * 2 ? row * (DG * 2) + pc * 16 : 0x80000000u;
  }
  auto load_k = [&](int blk) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < C::KDMA; r++) dma16(lds0 + r * 1024, kgo[r] + (unsigned)blk * (KB * C::RBG), rk);
    if constexpr (QK8) dma4(lds0 + C::KBYTES + C::VBYTES, (unsigned)(blk * KB + lane) * 4, rs);
  };
  auto load_v = [&](int blk) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < C::VDMA; r++)
      dma16(lds0 + C::KBYTES + r * 1024, vgo[r] + (unsigned)blk * (KB * DG * 2), rv);
  };

  // Q operands (B of S^T = K Q^T) of the NU query tiles
  i32x4 qreg[NU][NCH];
  float qsc[NU];
#pragma unroll
  for (int u = 0; u < NU; u++) {
    const int q = qt0 + 32 * u + l32;
    const bool ok = q < p.Lq;
    const char *qrow = Q + ((size_t)h * p.q_rows + (ok ? q : 0)) * C::RBG;
#pragma unroll
    for (int c = 0; c < NCH; c++) {
      const i32x4 v = *(const i32x4 *)(qrow + (2 * c + hl) * 16);
      qreg[u][c] = ok ? v : i32x4{0, 0, 0, 0};
    }
    qsc[u] = p.scale;
    if constexpr (QK8) qsc[u] = ok ? fmaxf(qs[(size_t)h * p.q_rows + q] * p.scale, FLT_MIN) : 1.0f;
  }

  f32x16 o[NU][NDB];
  float m[NU], l[NU];
#pragma unroll
  for (int u = 0; u < NU; u++) {
    m[u] = -INFINITY;
    l[u] = 0.0f;
#pragma unroll
    for (int db = 0; db < NDB; db++)
#pragma unroll
      for (int i = 0; i < 16; i++) o[u][db][i] = 0.0f;
  }

  const int krow = 16 * (l32 >> 4) + 8 * ((l32 >> 2) & 1) + 4 * ((l32 >> 3) & 1) + (l32 & 3);
  const int l16 = lane & 15, tr_row = l16 >> 2, tr_col = (l16 & 3) * 8;
  const char *Ks = own, *Vs = own + C::KBYTES;
  const float *Ss = (const float *)(own + C::KBYTES + C::VBYTES);

  // one block: the scores of the NU tiles, then softmax and P V of each; `next` (a block number, or -1) is what the
  // slots take after their last reads
  auto block = [&](int blk, bool next) __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(C::VDMA) : "memory");  // K(blk) has landed (V(blk) may be in flight)
    i32x4 ka[NCH];
#pragma unroll
    for (int c = 0; c < NCH; c++)
      ka[c] = *(const i32x4 *)(Ks + krow * C::RB + (((2 * c + hl) ^ kswz<C::RB, C::NP>(krow)) * 16));
    f32x4 k4[4];
    if constexpr (QK8) {
#pragma unroll
      for (int g = 0; g < 4; g++) k4[g] = *(const f32x4 *)(Ss + 16 * (g >> 1) + 8 * hl + 4 * (g & 1));
    }
    SAcc s[NU];
#pragma unroll
    for (int u = 0; u < NU; u++) {
#pragma unroll
      for (int i = 0; i < 16; i++) s[u][i] = 0;
#pragma unroll
      for (int c = 0; c < NCH; c++) s[u] = mma_qk<QKT>(ka[c], qreg[u][c], s[u]);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the K slot's reads are done
    if constexpr (DUMP) {  // the scores hook: the raw accumulators, [H][Lq][L]
#pragma unroll
      for (int u = 0; u < NU; u++) {
        const i32x16 a = __builtin_bit_cast(i32x16, s[u]);
        const i32x4 g[4] = {__builtin_shufflevector(a, a, 0, 1, 2, 3), __builtin_shufflevector(a, a, 4, 5, 6, 7),
                            __builtin_shufflevector(a, a, 8, 9, 10, 11), __builtin_shufflevector(a, a, 12, 13, 14, 15)};
        const int q = qt0 + 32 * u + l32;
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const int key = blk * KB + 16 * (r >> 1) + 8 * hl + 4 * (r & 1) + e;
            if (q < p.Lq && key < p.L) dump[((size_t)h * p.Lq + q) * p.L + key] = g[r][e];
          }
      }
    }
    if (next) load_k(blk + NWS);
    i32x4 pb[NU][2];
#pragma unroll
    for (int u = 0; u < NU; u++) {
      f32x16 x;
      if constexpr (QK8) {
#pragma unroll
        for (int i = 0; i < 16; i++) {
          const int si = s[u][i];
          x[i] = (float)si * k4[i >> 2][i & 3];
        }
      } else {
        x = s[u];
      }
      const int q0 = qt0 + 32 * u;
      if (blk * KB + KB > p.L || (causal && blk * KB + KB - 1 > q0 + p.causal_off)) {
        // element i of lane half hl holds key KB blk + 16 (i / 8) + 8 hl + i % 8
        const int last = causal ? min(p.L - 1, q0 + l32 + p.causal_off) : p.L - 1;
#pragma unroll
        for (int i = 0; i < 16; i++)
          if (blk * KB + 16 * (i >> 3) + 8 * hl + (i & 7) > last) x[i] = -INFINITY;
      }
      float am[2] = {x[0], x[1]};
#pragma unroll
      for (int i = 2; i < 16; i++) am[i & 1] = fmaxf(am[i & 1], x[i]);
      const float amax = fmaxf(am[0], am[1]);
      // lazy running maximum (wave-uniform branch); partner lanes (the same query) always update together
      if (__any(amax * qsc[u] > m[u] + SLACK_S)) {
        const float ap = fmaxf(amax, __shfl_xor(amax, 32));
        const float mn = fmaxf(m[u], ap * qsc[u]);
        const float f = mn == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m[u] - mn);
        m[u] = mn;
        l[u] *= f;
#pragma unroll
        for (int db = 0; db < NDB; db++)
#pragma unroll
          for (int i = 0; i < 16; i++) o[u][db][i] *= f;
      }
      const float nm = m[u] == -INFINITY ? 0.0f : -m[u];
      float ls[2] = {0.0f, 0.0f};
#pragma unroll
      for (int i = 0; i < 16; i += 2) {
        const float p0 = __builtin_amdgcn_exp2f(fmaf(x[i], qsc[u], nm));
        const float p1 = __builtin_amdgcn_exp2f(fmaf(x[i + 1], qsc[u], nm));
        const VP2 pr = {(VE)p0, (VE)p1};
        pb[u][i >> 3][(i & 7) >> 1] = __builtin_bit_cast(int, pr);
        ls[(i >> 1) & 1] = sum2<VT>(pr, ls[(i >> 1) & 1]);
      }
      l[u] += ls[0] + ls[1];
    }
    if (next) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(C::NKL) : "memory");  // V(blk) has landed
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int s2 = 0; s2 < 2; s2++) {
      const int k0 = 16 * s2 + 8 * hl + tr_row;
      i16x8 va[NDB];
#pragma unroll
      for (int db = 0; db < NDB; db++) {
        const int pc = (db * 32 + (l32 & 16)) / 8;
        const i16x4 lo = lds_tr16(Vs + voff<D>(k0, pc) + tr_col);
        const i16x4 hi = lds_tr16(Vs + voff<D>(k0 + 4, pc) + tr_col);
        va[db] = i16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
#pragma unroll
      for (int u = 0; u < NU; u++)
#pragma unroll
        for (int db = 0; db < NDB; db++)
          o[u][db] = mma_pv<VT>(va[db], __builtin_bit_cast(VT8, pb[u][s2]), o[u][db]);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the V slot's reads are done
    if (next) load_v(blk + NWS);
  };

  int blk = w;
  if (blk < nblk) {
    load_k(blk);
    load_v(blk);
    for (; blk + NWS < nblk; blk += NWS) block(blk, true);
    block(blk, false);
  }

  // merge, 32 rows (one query tile) at a time: each wave leaves its O, m and l; then 8 channels of a row per thread
#pragma unroll
  for (int u = 0; u < NU; u++) {
    const float lt = l[u] + __shfl_xor(l[u], 32);
    __syncthreads();
    char *orow = smem + (w * 32 + l32) * C::ORS;
#pragma unroll
    for (int db = 0; db < NDB; db++)
#pragma unroll
      for (int g = 0; g < 4; g++)
        store4<T_F32>(orow + (db * 32 + 8 * g + 4 * hl) * 4, o[u][db][4 * g], o[u][db][4 * g + 1], o[u][db][4 * g + 2],
                      o[u][db][4 * g + 3]);
    float *ml = (float *)(smem + NWS * 32 * C::ORS);
    if (hl == 0) *(float2 *)(ml + (w * 32 + l32) * 2) = make_float2(m[u], lt);
    __syncthreads();
    constexpr int PPR = DG / 8;
#pragma unroll
    for (int c = tid; c < 32 * PPR; c += NWS * 64) {
      const int r = c / PPR, d0 = 8 * (c - r * PPR), q = qt0 + 32 * u + r;
      if (q >= p.Lq) continue;
      float2 s[NWS];
      float mx = -INFINITY, lsum = 0.0f;
#pragma unroll
      for (int k = 0; k < NWS; k++) {
        s[k] = *(const float2 *)(ml + (k * 32 + r) * 2);
        mx = fmaxf(mx, s[k].x);
      }
      float v[8] = {};
#pragma unroll
      for (int k = 0; k < NWS; k++) {
        const float wt = s[k].x == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(s[k].x - mx);
        lsum += wt * s[k].y;
        const char *pr = smem + (k * 32 + r) * C::ORS + d0 * 4;
        const f32x4 a = *(const f32x4 *)pr, bq = *(const f32x4 *)(pr + 16);
#pragma unroll
        for (int e = 0; e < 4; e++) {
          v[e] += wt * a[e];
          v[4 + e] += wt * bq[e];
        }
      }
      const float inv = lsum > 0.0f ? 1.0f / lsum : 0.0f;
#pragma unroll
      for (int e = 0; e < 8; e++) v[e] *= inv;
      const int seq = h / p.seq_heads;
      const size_t at = ((size_t)seq * p.seq_rows + q) * p.o_stride + (size_t)(h - seq * p.seq_heads) * DG + d0;
      // 4 elements at a time: the caller's rows are aligned to that
      if (ot == T_F32) {
        store4<T_F32>(O + at * 4, v[0], v[1], v[2], v[3]);
        store4<T_F32>(O + at * 4 + 16, v[4], v[5], v[6], v[7]);
      } else if (ot == T_BF16) {
        store4<T_BF16>(O + at * 2, v[0], v[1], v[2], v[3]);
        store4<T_BF16>(O + at * 2 + 8, v[4], v[5], v[6], v[7]);
      } else {
        store4<T_F16>(O + at * 2, v[0], v[1], v[2], v[3]);
        store4<T_F16>(O + at * 2 + 8, v[4], v[5], v[6], v[7]);
      }
    }
  }
}

template <int DG, int QKT, int VT, int NU, bool DUMP>
int run(int ot, bool causal, const Exec &ex, const Arg *args, const AttnParams &p, std::string *err) {
  using C = CfgS<DG, QKT, NU>;
  auto kern = attention_small_kernel<DG, QKT, VT, NU, DUMP>;
  static bool attr_set = false;
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS);
    if (e != hipSuccess) {
      *err = std::string("hipFuncSetAttribute: ") + hipGetErrorString(e);
      return -1;
    }
    attr_set = true;
  }
  const int nqb = (p.Lq + 32 * NU - 1) / (32 * NU);
  hipLaunchKernelGGL(kern, dim3((unsigned)(nqb * p.H)), dim3(NWS * 64), C::LDS, ex.stream, args[0].ptr, args[1].ptr,
                     args[2].ptr, args[3].ptr, (const float *)args[5].ptr, (const float *)args[6].ptr,
                     DUMP ? (int *)args[7].ptr : nullptr, p, nqb, (int)causal, ot);
  return 0;
}

template <int DG, int QKT, int VT>
int run_nu(int nu, int ot, bool causal, bool dump, const Exec &ex, const Arg *args, const AttnParams &p,
           std::string *err) {
  if constexpr (DG == 96) {
    if (nu == 2) return run<DG, QKT, VT, 2, false>(ot, causal, ex, args, p, err);
  }
  if constexpr (DG == 128) {
    if (dump) return run<DG, QKT, VT, 1, true>(ot, causal, ex, args, p, err);
  }
  return run<DG, QKT, VT, 1, false>(ot, causal, ex, args, p, err);
}

template <int DG>
int run_types(int qkt, int vt, int nu, int ot, bool causal, bool dump, const Exec &ex, const Arg *args,
              const AttnParams &p, std::string *err) {
  if (qkt == T_I8)
    return vt == T_BF16 ? run_nu<DG, T_I8, T_BF16>(nu, ot, causal, dump, ex, args, p, err)
                        : run_nu<DG, T_I8, T_F16>(nu, ot, causal, dump, ex, args, p, err);
  return qkt == T_BF16 ? run_nu<DG, T_BF16, T_BF16>(nu, ot, causal, dump, ex, args, p, err)
                       : run_nu<DG, T_F16, T_F16>(nu, ot, causal, dump, ex, args, p, err);
}

}  // namespace

int launch_attention_small(int d, int qkt, int vt, int ot, int nu, bool causal, bool dump, const Exec &ex,
                           const Arg *args, const AttnParams &p, std::string *err) {
  switch (d) {
    case 64: return run_types<64>(qkt, vt, nu, ot, causal, dump, ex, args, p, err);
    case 96: return run_types<96>(qkt, vt, nu, ot, causal, dump, ex, args, p, err);
    default: return run_types<128>(qkt, vt, nu, ot, causal, dump, ex, args, p, err);
  }
}

}  // namespace h3
