// Queries/keys pre-pass for attention, fused in one kernel for gfx950:
// per-head RMS norm, rotary embedding, Walsh-Hadamard rotation with fixed
// signs, and per-row int8 quantisation; values are copied through.
//
// Semantics of the reference kernel qk_norm_rope (kernels/ops.metal:365-468,
// parameters :344-349, launcher h3metal/ops.py:225-239):
//  * Input rows hold Hq query heads, then Hk key heads, then Hv value heads of
//    HDIM channels each (a "slot" is one of them); row m is row r = m % seq_len
//    of sequence m / seq_len, whose heads are output heads sq*H .. sq*H + H-1,
//    row r of each (:381, :448).
//  * norm: v = (v * 1/sqrt(sum(v^2)/HDIM + eps)) * w (:394-402).
//  * rot: the first `rot` channels are rotated in pairs (i, i + rot/2) by the
//    row's angle table: v_i c - v_{i+rot/2} s and v_{i+rot/2} c + v_i s (:403-419).
//  * QKROT (int8 outputs only): v_c = -v_c where popcount(c * 0x2545F491) is odd,
//    then a 128-point fast Walsh-Hadamard transform with its butterfly stages in
//    increasing channel-bit order, each (a + b, a - b) with a the lower channel,
//    then a multiply by 1/sqrt(HDIM) (:420-446).
//  * QK8: scale = amax > 0 ? amax / 127 : 1, code = rint(v / scale) (:450-458).
// Every floating-point step is a single IEEE-rounded operation in that order
// (this file is compiled without FMA contraction; division and square root are
// correctly rounded), so a float32 restatement reproduces codes and scales bit
// for bit. The sum of squares is summed per lane, then over the lanes of a
// head with an xor butterfly (halving strides): a fixed order.
//
// gfx950 layout: a head's channels are spread over a group of lanes, PER
// consecutive channels per lane: PER = 8 (16-byte loads of 16-bit rows; 16
// lanes per head at HDIM 128) whenever the rotary pairs (c, c + rot/2) stay
// lane-aligned (rot/2 a multiple of 8), else the reference's HDIM / 32. Every
// cross-lane step of the transform and the reductions stays inside the group
// and runs on DPP lane patterns at 16 lanes per slot (ds_swizzle at other
// shapes; no LDS memory traffic). A workgroup of 256 threads covers 4 waves'
// groups of slots of 8 consecutive rows; each wave issues all 8 rows' loads
// before processing them, and a slot's 8 scales are stored together.
// With the norm, the rotary embedding, the transform and the int8 rounding the
// kernel was bound by its vector instructions (about 300 per row and wave,
// 172-178 us at 16896 rows of 32 + 32 + 32 heads where the bytes take 135), so
// the work of a row is cut to about 190: what is one value per row (1 / sqrt,
// the scale and its reciprocal) is computed once for 8 rows, a row per lane;
// the angle tables of the 8 rows are made once per workgroup in LDS, in
// channel order, with the rotary signs and the transform's fixed signs folded
// in; and codes are rounded by one fma each. 140 us (5.0 TB/s) there, 49 -> 44
// us at 4608 rows; 16-bit outputs 176 -> 152 us. int8 outputs without norm and
// rotary embedding (PLAIN) take one row at a time: there is little to share.
#include "h3hip_internal.h"

#include <cmath>
#include <cstring>
#include <type_traits>

namespace h3 {
namespace {

enum { T_I8 = 0, T_BF16 = 1, T_F16 = 2, T_F32 = 3 };

template <int T> struct Elem;
template <> struct Elem<T_BF16> { using type = __bf16; };
template <> struct Elem<T_F16> { using type = _Float16; };
template <> struct Elem<T_F32> { using type = float; };

template <int N, typename E> struct VecOf { typedef E type __attribute__((ext_vector_type(N))); };

constexpr int RPW = 8;  // rows per workgroup; each wave walks them with all their loads in flight

template <int HDIM>
constexpr double inv_sqrt_hdim() {
  return HDIM == 128 ? 0.0883883476483184405501055452631 : HDIM == 64 ? 0.125 : 0.1767766952966368811;
}

// PER channels per lane, LPS = HDIM / PER lanes per (row, head) slot, 64 / LPS slots per wave. Workgroup
// (bx, by): rows bx*RPW .. bx*RPW + RPW-1, slots by*SPG .. by*SPG + SPG-1 (SPG = 4 waves' slots). A lane group
// owns one slot and walks the rows; its lane r keeps the scale of row r so that a slot's RPW scales (consecutive
// in memory within a sequence) are stored together after the rows.
template <int HDIM, int PER>
struct PrepassShape {
  static constexpr int LPS = HDIM / PER;     // lanes per slot
  static constexpr int SPG = 4 * 64 / LPS;   // slots per workgroup
  static_assert(LPS >= RPW && LPS <= 32 && (LPS & (LPS - 1)) == 0, "lane group");
};

// Channel groups and lanes. With 16 lanes per slot the group g (channels 8 g .. 8 g + 7) sits in lane
// L(g) = g0 ^ 2 g1 ^ 7 g2 ^ 8 g3 (g_b the bits of g): the partner along group bit 0, 1, 2, 3 is then lane L ^ 1,
// ^ 2, ^ 7, ^ 8 -- all four DPP lane patterns within a 16-lane row (quad_perm, row_half_mirror, row_ror:8), so
// every cross-lane step of the transform and of the reductions is one VALU instruction with no LDS traffic.
// Other lane counts keep g = lane.
template <int LPS>
__device__ __forceinline__ int group_of_lane(int l) {
  if constexpr (LPS != 16) return l;
  const int g2 = (l >> 2) & 1, r = l ^ (7 * g2);
  return (r & 1) | (r & 2) | (g2 << 2) | (r & 8);
}
template <int LPS>
__device__ __forceinline__ int lane_of_group(int g) {
  if constexpr (LPS != 16) return g;
  return (g & 1) ^ (g & 2) ^ (7 * ((g >> 2) & 1)) ^ (g & 8);
}
// the value of the lane whose group differs in group bit B
template <int LPS, int B>
__device__ __forceinline__ float gshfl(float v) {
  if constexpr (LPS == 16 && B == 4)
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xF, 0xF, true));
  else return xshfl<B>(v);
}
// one cross-lane Hadamard stage along group bit B (see hadamard_lane_stage for the sign convention)
template <int LPS, int B, int N>
__device__ __forceinline__ void group_stage(float (&v)[N], float c) {
  if constexpr (LPS == 16 && B == 4) {
    H3_DPP_FMAC_STAGE("row_half_mirror row_mask:0xf bank_mask:0xf bound_ctrl:1");
  } else {
    hadamard_lane_stage<B>(v, c);
  }
}

// the value of lane R of the slot's lane group, on every lane of it
template <int LPS, int R>
__device__ __forceinline__ float group_bcast(float v, int gbase) {
  if constexpr (LPS == 16)  // row_newbcast:R
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x150 + R, 0xF, 0xF, true));
  else return __shfl(v, gbase + R);
}

template <int R> using RowConst = std::integral_constant<int, R>;
// f(RowConst<0>) ... f(RowConst<nr - 1>): the rows as compile-time constants (a DPP control has to be one). It ends at the
// last row, so that a row's store is known to be behind the loads of the later rows and no wait for them waits for it
template <class F>
__device__ __forceinline__ void each_row(int nr, F &&f) {
  auto go = [&](auto rc) { return decltype(rc)::value < nr && (f(rc), true); };
  (void)(go(RowConst<0>{}) && go(RowConst<1>{}) && go(RowConst<2>{}) && go(RowConst<3>{}) && go(RowConst<4>{}) &&
         go(RowConst<5>{}) && go(RowConst<6>{}) && go(RowConst<7>{}));
  static_assert(RPW == 8, "rows");
}

// QKROT's fixed sign of channel c, as a sign bit
__device__ __forceinline__ unsigned sign_bit(int c) {
  return (__builtin_popcount((unsigned)c * 0x2545F491u) & 1u) ? 0x80000000u : 0u;
}
__device__ __forceinline__ float flip(float v, unsigned bit) {
  return __builtin_bit_cast(float, __builtin_bit_cast(unsigned, v) ^ bit);
}

template <int HDIM, int PER, int IN_T, int QK_T, int V_T, bool QKROT, bool PLAIN>
__global__ __launch_bounds__(256) void qk_norm_rope_kernel(const char *__restrict__ in, const float *__restrict__ wq,
                                                            const float *__restrict__ wk,
                                                            const float *__restrict__ cs,
                                                            const float *__restrict__ sn, char *__restrict__ Qo,
                                                            char *__restrict__ Ko, char *__restrict__ Vo,
                                                            float *__restrict__ qsc, float *__restrict__ ksc,
                                                            QkRopeParams p, int nd) {
  const bool norm = !PLAIN && p.norm;  // PLAIN: int8 outputs without norm and rotary embedding (launch_qk)
  const int rot = PLAIN ? 0 : p.rot;
  using SH = PrepassShape<HDIM, PER>;
  constexpr int LPS = SH::LPS;
  using IE = typename Elem<IN_T>::type;
  typedef typename VecOf<PER, IE>::type IV;
  // the rows' angle tables, per channel: cos, and sin with the sign of the channel's half, both times QKROT's sign of
  // the channel. Channel c at tab_at(c): lanes read 16 consecutive bytes each (PER 8: two runs of 4 channels)
  __shared__ __attribute__((aligned(16))) float tab[RPW][2][HDIM];
  auto tab_at = [](int c) { return PER == 8 ? (((c >> 2) & 1) * LPS + (c >> 3)) * 4 + (c & 3) : c; };
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int l32 = lane & (LPS - 1);  // lane within the slot's group
  const int gbase = lane & ~(LPS - 1);  // first lane of the group
  const int g = group_of_lane<LPS>(l32);  // this lane's channel group: channels g * PER .. g * PER + PER - 1
  // order of the workgroups: the row groups of a slot group first, or the nd > 0 slot groups of a row group (launch_qk)
  const int bx = nd ? blockIdx.x / nd : blockIdx.x, by = nd ? blockIdx.x - bx * nd : blockIdx.y;
  const int slot = by * SH::SPG + w * (64 / LPS) + lane / LPS;
  const int m0 = bx * RPW;
  const int nslots = p.Hq + p.Hk + p.Hv;
  const int nr = min(RPW, p.M - m0);
  // outputs are streamed out with nontemporal stores (nothing in this kernel reads them again; measured +6%)
  auto st = [](auto *dst, auto val) { __builtin_nontemporal_store(val, dst); };

  // rows past the last one repeat it and are not stored
  IV xin[RPW];
  {
    const IE *src = (const IE *)in + (size_t)m0 * p.in_stride + (size_t)min(slot, nslots - 1) * HDIM + g * PER;
#pragma unroll
    for (int r = 0; r < RPW; r++) xin[r] = *(const IV *)(src + (size_t)min(r, nr - 1) * p.in_stride);
  }
  const int half_rot = rot / 2;
  if (rot && by * SH::SPG < p.Hq + p.Hk) {  // (uniform over the workgroup)
    for (int i = threadIdx.x; i < nr * rot; i += 256) {
      const int r = i / rot, c = i - r * rot;
      const bool first = c < half_rot;
      const size_t at = (size_t)((m0 + r) % p.seq_len) * half_rot + (first ? c : c - half_rot);
      const unsigned sb = QKROT ? sign_bit(c) : 0u;
      tab[r][0][tab_at(c)] = flip(cs[at], sb);
      tab[r][1][tab_at(c)] = flip(sn[at], sb ^ (first ? 0x80000000u : 0u));
    }
    __syncthreads();
  }
  if (slot >= nslots) return;  // whole lane groups only; no cross-lane step leaves a group
  const bool isqk = slot < p.Hq + p.Hk, isq = slot < p.Hq;
  const int h = isq ? slot : isqk ? slot - p.Hq : slot - p.Hq - p.Hk;
  const int heads = isq ? p.Hq : isqk ? p.Hk : p.Hv;
  auto hrow_of = [&](int m) {
    const int sq = m / p.seq_len, r = m - sq * p.seq_len;
    return ((size_t)sq * heads + h) * p.out_rows + r;
  };
  if (!isqk) {
    using OE = typename Elem<V_T>::type;
    typedef typename VecOf<PER, OE>::type OV;
#pragma unroll
    for (int rr = 0; rr < RPW; rr++) {
      if (rr >= nr) break;
      OE *dst = (OE *)Vo + hrow_of(m0 + rr) * HDIM + g * PER;
      if constexpr (V_T == IN_T) {
        st((OV *)dst, xin[rr]);  // same type: a plain copy
      } else {
        OV out;
#pragma unroll
        for (int i = 0; i < PER; i++) out[i] = (OE)(float)xin[rr][i];
        st((OV *)dst, out);
      }
    }
    return;
  }

  // What is one value per row (the norm's 1 / sqrt, the int8 scale) is computed once for the 8 rows of a slot: lane r
  // of the group takes row r's sum (or maximum), and the result is broadcast back row by row.
  const bool rotated = g * PER < rot;  // this lane's channels are in rotary pairs (they then get their signs there)
  auto sign_of = [&](int i) { return QKROT && !rotated ? sign_bit(g * PER + i) : 0u; };
  float wv[PER], inv_l = 1.0f;  // a channel's weight, with its sign
#pragma unroll
  for (int i = 0; i < PER; i++) wv[i] = flip(1.0f, sign_of(i));
  if (norm) {
    const float *ws = (isq ? wq : wk) + g * PER;
#pragma unroll
    for (int i = 0; i < PER; i++) wv[i] = flip(ws[i], sign_of(i));
    float mine = 1.0f;
    each_row(RPW, [&](auto rc) {
      constexpr int r = decltype(rc)::value;
      float ss = (float)xin[r][0] * (float)xin[r][0];
#pragma unroll
      for (int i = 1; i < PER; i++) ss = ss + (float)xin[r][i] * (float)xin[r][i];
      // over the groups in halving strides (the partner of group g is g ^ stride)
      if constexpr (LPS > 16) ss = ss + gshfl<LPS, 16>(ss);
      if constexpr (LPS > 8) ss = ss + gshfl<LPS, 8>(ss);
      ss = ss + gshfl<LPS, 4>(ss);
      ss = ss + gshfl<LPS, 2>(ss);
      ss = ss + gshfl<LPS, 1>(ss);
      if (l32 == r) mine = ss;
    });
    inv_l = 1.0f / sqrtf(mine / (float)HDIM + p.eps);
  }
  const int lanes = half_rot / PER;  // lanes holding the first half of the rotated channels
  const int src_group = g < lanes ? g + lanes : (g < 2 * lanes ? g - lanes : g);
  const int from = (gbase + lane_of_group<LPS>(src_group)) * 4;
  // row r normalised and rotated (and, on QKROT, with its signs)
  auto row = [&](auto rc, float (&v)[PER]) __attribute__((always_inline)) {
    constexpr int r = decltype(rc)::value;
    if (norm) {
      const float inv = group_bcast<LPS, r>(inv_l, gbase);
#pragma unroll
      for (int i = 0; i < PER; i++) v[i] = ((float)xin[r][i] * inv) * wv[i];
    } else {
#pragma unroll
      for (int i = 0; i < PER; i++) v[i] = (float)xin[r][i] * wv[i];
    }
    if (rot) {
      float pv[PER];
#pragma unroll
      for (int i = 0; i < PER; i++)
        pv[i] = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(from, __builtin_bit_cast(int, v[i])));
      if (rotated) {
        // v_i c - v_p s on the first half of the channels, v_i c + v_p s on the second (the sign is in the table)
#pragma unroll
        for (int i = 0; i < PER; i++) {
          const int at = tab_at(g * PER + i);
          v[i] = v[i] * tab[r][0][at] + pv[i] * tab[r][1][at];
        }
      }
    }
  };
  if constexpr (QK_T != T_I8) {
    using OE = typename Elem<QK_T>::type;
    typedef typename VecOf<PER, OE>::type OV;
    each_row(nr, [&](auto rc) {
      constexpr int r = decltype(rc)::value;
      float v[PER];
      row(rc, v);
      OV out;
#pragma unroll
      for (int i = 0; i < PER; i++) out[i] = (OE)v[i];
      st((OV *)((isq ? Qo : Ko) + (hrow_of(m0 + r) * HDIM + g * PER) * sizeof(OE)), out);
    });
  } else {
    // the transform's final factor 1 / sqrt(HDIM), with the sign that the lane carries (an exact sign change)
    constexpr float rn = QKROT ? (float)inv_sqrt_hdim<HDIM>() : 1.0f;
    const float rns = QKROT && (__builtin_popcount(g) & 1) ? -rn : rn;
    // a row normalised, rotated and transformed, but for that factor, and the largest magnitude of its values
    auto transform = [&](auto rc, float (&v)[PER]) __attribute__((always_inline)) {
      row(rc, v);
      if constexpr (QKROT) {
#pragma unroll
        for (int s = 1; s < PER; s <<= 1) {
#pragma unroll
          for (int i = 0; i < PER; i++) {
            if (!(i & s)) {
              const float a = v[i], b = v[i + s];
              v[i] = a + b;
              v[i + s] = a - b;
            }
          }
        }
        // across lanes: channel c pairs with c ^ (ls * PER), stages in increasing bit order; the lower channel
        // becomes a + b, the upper one a - b (a the lower channel's value); each lane ends with its values
        // times (-1)^popcount(g) (hadamard_lane_stage)
        auto stage = [&](auto ls_const) {
          constexpr int LS = decltype(ls_const)::value;
          group_stage<LPS, LS>(v, (g & LS) ? -1.0f : 1.0f);
        };
        stage(std::integral_constant<int, 1>{});
        stage(std::integral_constant<int, 2>{});
        stage(std::integral_constant<int, 4>{});
        if constexpr (LPS > 8) stage(std::integral_constant<int, 8>{});
        if constexpr (LPS > 16) stage(std::integral_constant<int, 16>{});
      }
      float amax = 0.0f;
#pragma unroll
      for (int i = 0; i < PER; i++) amax = fmaxf(amax, fabsf(v[i]));
      if constexpr (LPS > 16) amax = fmaxf(amax, gshfl<LPS, 16>(amax));
      if constexpr (LPS > 8) amax = fmaxf(amax, gshfl<LPS, 8>(amax));
      amax = fmaxf(amax, gshfl<LPS, 4>(amax));
      amax = fmaxf(amax, gshfl<LPS, 2>(amax));
      return fmaxf(amax, gshfl<LPS, 1>(amax));
    };
    // rounding is monotonic, so the largest |v * rn| is the rounded product of the largest |v|
    auto scale_of = [&](float amax) {
      const float am = QKROT ? amax * rn : amax;
      return am > 0.0f ? am / 127.0f : 1.0f;
    };
    // Codes are the nearest integers of fl(v * rns) / scale. y = v * (rns * rs) is within 2^-14 of that quotient
    // (|y| <= 128; four roundings of at most 1 ulp), so their nearest integers agree unless y lies within 2^-14 of
    // a half-integer, and then the wave divides (one row of four slots in sixteen, and exact). t = fma(v, f, 1.5 * 2^23)
    // rounds y to the nearest integer (half to even), whose two's complement is in t's low bits. A scale whose
    // reciprocal (rs, 1 ulp) is not a normal float (amax below ~2^-119) divides too, and so does a NaN (`far` keeps it).
    auto code = [&](auto rc, const float (&v)[PER], float rs, auto scale) __attribute__((always_inline)) {
      constexpr int r = decltype(rc)::value;
      const float f = rs * rns;
      constexpr float MG = 12582912.0f;
      unsigned t[PER];
      float far = 0.0f;
#pragma unroll
      for (int i = 0; i < PER; i++) {
        const float ti = __builtin_fmaf(v[i], f, MG);
        far = __builtin_elementwise_maximum(far, fabsf(__builtin_fmaf(v[i], f, -(ti - MG))));
        t[i] = __builtin_bit_cast(unsigned, ti);
      }
      bool divide = !(far <= 0.5f - 0x1p-14f) || !(rs < 0x1p126f);
      if constexpr (!PLAIN) divide = __builtin_amdgcn_ballot_w64(divide);  // so that a broadcast's source lanes are active
      if (divide) {
        const float s = scale(rc);
#pragma unroll
        for (int i = 0; i < PER; i++) t[i] = (unsigned)(int)rintf((QKROT ? v[i] * rns : v[i]) / s);
      }
      typedef typename VecOf<PER, signed char>::type CV;
      CV codes;
#pragma unroll
      for (int i = 0; i < PER; i++) codes[i] = (signed char)t[i];
      st((CV *)((isq ? Qo : Ko) + hrow_of(m0 + r) * HDIM + g * PER), codes);
    };
    float scale_l = 1.0f;  // of row l32
    if constexpr (PLAIN) {
      // one row at a time
      each_row(nr, [&](auto rc) {
        constexpr int r = decltype(rc)::value;
        float v[PER];
        const float scale = scale_of(transform(rc, v));
        code(rc, v, __builtin_amdgcn_rcpf(scale), [&](auto) { return scale; });
        if (l32 == r) scale_l = scale;
      });
    } else {
      float v[RPW][PER], mine = 0.0f;
      each_row(RPW, [&](auto rc) {
        constexpr int r = decltype(rc)::value;
        const float amax = transform(rc, v[r]);
        if (l32 == r) mine = amax;
      });
      scale_l = scale_of(mine);
      const float rs_l = __builtin_amdgcn_rcpf(scale_l);
      each_row(nr, [&](auto rc) {
        constexpr int r = decltype(rc)::value;
        code(rc, v[r], group_bcast<LPS, r>(rs_l, gbase),
             [&](auto q) { return group_bcast<LPS, decltype(q)::value>(scale_l, gbase); });
      });
    }
    if (l32 < nr) (isq ? qsc : ksc)[hrow_of(m0 + l32)] = scale_l;
  }
}

int esize(int t) { return t == T_I8 ? 1 : t == T_F32 ? 4 : 2; }

template <int HDIM, int IN_T, int QK_T, int V_T, bool QKROT>
int launch_qk(const Pipeline &pl, const Exec &ex, const Arg *a, int nargs, const void *params,
              uint32_t params_len, std::string *err) {
  (void)pl;
  if (params_len != sizeof(QkRopeParams)) {
    *err = "parameter block of " + std::to_string(params_len) + " bytes, expected " +
           std::to_string(sizeof(QkRopeParams));
    return -1;
  }
  QkRopeParams p;
  memcpy(&p, params, sizeof p);
  const int PER = HDIM / 32;
  const int nslots = p.Hq + p.Hk + p.Hv;
  if (p.M < 0 || p.Hq < 0 || p.Hk < 0 || p.Hv < 0 || nslots < 1 || p.seq_len < 1 || p.out_rows < 1 ||
      p.in_stride < nslots * HDIM) {
    *err = "bad shape: M " + std::to_string(p.M) + " heads " + std::to_string(p.Hq) + "/" + std::to_string(p.Hk) +
           "/" + std::to_string(p.Hv) + " in_stride " + std::to_string(p.in_stride) + " seq_len " +
           std::to_string(p.seq_len);
    return -1;
  }
  const int rows = p.M < p.seq_len ? p.M : p.seq_len;  // rows per sequence actually present
  if (rows > p.out_rows) {
    *err = "out_rows " + std::to_string(p.out_rows) + " smaller than the rows of a sequence";
    return -1;
  }
  if (p.rot < 0 || p.rot > HDIM || p.rot % 2 || (p.rot / 2) % PER) {
    *err = "rot " + std::to_string(p.rot) + " must be even, at most HD, and rot/2 a multiple of " +
           std::to_string(PER);
    return -1;
  }
  if (p.norm && !(p.eps >= 0.0f)) {
    *err = "eps must be non-negative";
    return -1;
  }
  if (nargs < 11 && QK_T == T_I8) {
    *err = "int8 outputs need buffers q_scale and k_scale (indices 9, 10)";
    return -1;
  }
  if (nargs < 8) {
    *err = "expected buffers qkv, wq, wk, cos, sin, Q, K, V";
    return -1;
  }
  auto need = [&](int i, uint64_t bytes, const char *what, bool required) {
    if (!required || bytes == 0) return true;
    if (!a[i].ptr) {
      *err = std::string(what) + " is not bound";
      return false;
    }
    if (bytes > a[i].avail) {
      *err = std::string(what) + " needs " + std::to_string(bytes) + " bytes, its buffer holds " +
             std::to_string(a[i].avail);
      return false;
    }
    return true;
  };
  const uint64_t nseq = p.M ? (uint64_t)(p.M - 1) / p.seq_len + 1 : 0;
  const uint64_t in_bytes = p.M ? ((uint64_t)(p.M - 1) * p.in_stride + (uint64_t)nslots * HDIM) * esize(IN_T) : 0;
  // Rows written per output: head-major rows up to (last head) * out_rows + (rows of a sequence). Callers pass
  // views that start inside a head's row block (h3metal/flux2.py:417-426 writes text rows, then image rows at
  // offset r0), so the check is on the extent actually touched, not on heads * out_rows.
  auto extent = [&](int heads) -> uint64_t {
    return heads && nseq ? (nseq * heads - 1) * (uint64_t)p.out_rows + (uint64_t)rows : 0;
  };
  const uint64_t hq = extent(p.Hq), hk = extent(p.Hk), hv = extent(p.Hv);
  const uint64_t tab = (uint64_t)rows * (p.rot / 2) * 4;
  if (!need(0, in_bytes, "qkv", true) || !need(1, HDIM * 4, "wq", p.norm && p.Hq) ||
      !need(2, HDIM * 4, "wk", p.norm && p.Hk) || !need(3, tab, "cos", p.rot > 0 && (p.Hq + p.Hk)) ||
      !need(4, tab, "sin", p.rot > 0 && (p.Hq + p.Hk)) || !need(5, hq * HDIM * esize(QK_T), "Q", p.Hq > 0) ||
      !need(6, hk * HDIM * esize(QK_T), "K", p.Hk > 0) || !need(7, hv * HDIM * esize(V_T), "V", p.Hv > 0))
    return -1;
  if (QK_T == T_I8 && (!need(9, hq * 4, "q_scale", p.Hq > 0) || !need(10, hk * 4, "k_scale", p.Hk > 0))) return -1;
  if (p.M == 0) return 0;
  // 8 channels per lane (16-byte loads for 16-bit inputs) unless the rotary pairs would straddle lanes, then
  // the reference's HDIM / 32
  auto go = [&](auto per_const, auto plain) {
    constexpr int P = decltype(per_const)::value;
    constexpr int SPG = PrepassShape<HDIM, P>::SPG;
    const int nx = (p.M + RPW - 1) / RPW, ny = (nslots + SPG - 1) / SPG;
    // The order of the workgroups. int8 calls with a rotary embedding whose 16-bit rows outgrow the 256 MB last-level
    // cache together with the outputs run a row group's slot groups first, so that the value copies overlap the queries'
    // and keys' arithmetic (415 MB of rows: 153 -> 139 us, 221 MB: 72 -> 69). Otherwise the row groups of a slot group's
    // columns go first (113 MB of rows just written by a projection: 50 -> 45 us; 415 MB without norm and embedding: 138
    // -> 130; float32 rows, 207 MB: 56 -> 45).
    const bool rows_first = QK_T == T_I8 && IN_T != T_F32 && p.rot &&
                            (uint64_t)p.M * nslots * HDIM * esize(IN_T) > 160000000ull;
    // PLAIN is bound by HBM, and its 54 to 96 registers would let 5 to 8 waves run on a SIMD: an unused LDS request holds it
    // to 5 (4 with float32 rows), whose accesses lie closer together (415 MB of rows without the transform: 130 -> 125 us)
    const unsigned lds = !decltype(plain)::value ? 0 : IN_T == T_F32 ? 40000 : 32000;
    const dim3 grid = rows_first ? dim3((unsigned)nx * ny) : dim3((unsigned)nx, (unsigned)ny);
    hipLaunchKernelGGL((qk_norm_rope_kernel<HDIM, P, IN_T, QK_T, V_T, QKROT, decltype(plain)::value>), grid, dim3(256), lds, ex.stream, a[0].ptr,
                       (const float *)a[1].ptr, (const float *)a[2].ptr, (const float *)a[3].ptr,
                       (const float *)a[4].ptr, a[5].ptr, a[6].ptr, a[7].ptr,
                       nargs > 9 ? (float *)a[9].ptr : nullptr, nargs > 10 ? (float *)a[10].ptr : nullptr, p,
                       rows_first ? ny : 0);
  };
  if constexpr (QK_T == T_I8) {
    // PLAIN: what is one value per row is little here, and holding 8 rows' values for it took 126 registers (with the order
    // and the occupancy above 10.1 -> 9.1 us at 1000 rows of 32 + 32 + 32 heads, 35.0 -> 31.1 at 4608; without the transform
    // 133 -> 125 at 16896)
    if (!p.norm && !p.rot) {
      go(std::integral_constant<int, 8>{}, std::true_type{});
      return 0;
    }
  }
  if ((p.rot / 2) % 8 == 0) go(std::integral_constant<int, 8>{}, std::false_type{});
  else go(std::integral_constant<int, HDIM / 32>{}, std::false_type{});
  return 0;
}

template <int HDIM, int IN_T>
LaunchFn pick_out(int qk_t, int v_t, bool rot, std::string *err) {
  if (qk_t == T_I8) {
    if (v_t == T_BF16) return rot ? launch_qk<HDIM, IN_T, T_I8, T_BF16, true> : launch_qk<HDIM, IN_T, T_I8, T_BF16, false>;
    return rot ? launch_qk<HDIM, IN_T, T_I8, T_F16, true> : launch_qk<HDIM, IN_T, T_I8, T_F16, false>;
  }
  if (rot) {
    *err = "QKROT needs QK8 (int8 outputs)";
    return nullptr;
  }
  if (qk_t == T_BF16)
    return v_t == T_BF16 ? launch_qk<HDIM, IN_T, T_BF16, T_BF16, false> : launch_qk<HDIM, IN_T, T_BF16, T_F16, false>;
  return v_t == T_BF16 ? launch_qk<HDIM, IN_T, T_F16, T_BF16, false> : launch_qk<HDIM, IN_T, T_F16, T_F16, false>;
}

template <int HDIM>
LaunchFn pick_in(int in_t, int qk_t, int v_t, bool rot, std::string *err) {
  switch (in_t) {
    case T_BF16: return pick_out<HDIM, T_BF16>(qk_t, v_t, rot, err);
    case T_F16: return pick_out<HDIM, T_F16>(qk_t, v_t, rot, err);
    default: return pick_out<HDIM, T_F32>(qk_t, v_t, rot, err);
  }
}

int type_of(const std::string &s) {
  if (s == "bfloat" || s == "bf16") return T_BF16;
  if (s == "half" || s == "f16") return T_F16;
  if (s == "float" || s == "f32") return T_F32;
  return -1;
}

}  // namespace

// Specialisation macros: HDIM (64 or 128), IN_T (input: half | bfloat | float),
// QK8 (int8 Q/K + scales), QKROT (rotation; needs QK8), QK_T (Q/K without QK8:
// half | bfloat, default half as in the reference), V_T (half | bfloat, default
// half). NSG (the reference's SIMD-groups per threadgroup) is accepted and unused.
bool make_ops(const std::string &fn, const Macros &m, Pipeline *pl, std::string *err) {
  if (fn == "rot_q8") return make_rot_q8(m, pl, err);
  if (fn != "qk_norm_rope") {
    *err = "unknown function (have: qk_norm_rope, rot_q8)";
    return false;
  }
  int hd, q8, rot, nsg;
  if (!macro_int(m, "HDIM", 128, &hd, err) || !macro_int(m, "QK8", 0, &q8, err) ||
      !macro_int(m, "QKROT", 0, &rot, err) || !macro_int(m, "NSG", 8, &nsg, err))
    return false;
  for (auto &kv : m) {
    static const char *known[] = {"HDIM", "IN_T", "QK8", "QKROT", "QK_T", "V_T", "NSG"};
    bool ok = false;
    for (const char *k : known) ok = ok || kv.first == k;
    if (!ok) {
      *err = "unknown macro " + kv.first;
      return false;
    }
  }
  const int in_t = type_of(macro_str(m, "IN_T", "half"));
  const int qk_t = q8 ? T_I8 : type_of(macro_str(m, "QK_T", "half"));
  const int v_t = type_of(macro_str(m, "V_T", "half"));
  if (in_t < 0 || qk_t < 0 || qk_t == T_F32 || v_t < 0 || v_t == T_F32) {
    *err = "IN_T must be half|bfloat|float, QK_T and V_T half|bfloat";
    return false;
  }
  LaunchFn f = nullptr;
  if (hd == 128) f = pick_in<128>(in_t, qk_t, v_t, rot != 0, err);
  else if (hd == 64) f = pick_in<64>(in_t, qk_t, v_t, rot != 0, err);
  else *err = "HDIM " + std::to_string(hd) + " not supported (64 or 128)";
  if (!f) return false;
  pl->launch = f;
  pl->threads = 256;
  return true;
}

}  // namespace h3
