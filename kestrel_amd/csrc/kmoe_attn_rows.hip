// kmoe_attn_rows.hip — causal GQA attention over the f16 cache for prompt
// chunks (transformer.rs:591-631) on the f16 matrix cores, with 32-bit
// arithmetic kept: q and the softmax weights enter as two f16 pieces each.
#include "kmoe_device.h"
#include "kmoe_launch.h"

namespace kmoe {

namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4a4 __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kQT = 32;  // query rows per work-group
constexpr int kKB = 32;  // key positions per block
// Calls that end at most here run four waves per work-group, whichever form was
// launched: a row's bits do not depend on the cache's capacity or on where its
// position is kept.
constexpr int kNarrow = 8 * kKB;

// A pair of f32 as two dwords of f16 pairs: hi, the nearest f16, and lo, the
// nearest f16 of 2^12 times what hi leaves. x = hi + lo * 2^-12 to 2^-23 of x
// for |x| in 2^-14..2^15 and to 2^-37 below that. (Without the 2^12, lo's
// exponent ends at 2^-25: elements some 2^20 below their row's largest, or
// softmax weights so far below a first position's, would lose their bits.)
constexpr float kLo = 0x1p-12f;
__device__ __forceinline__ void split2(float a, float b, uint32_t &hi, uint32_t &lo) {
  const h2 h = {(_Float16)a, (_Float16)b};
  const h2 l = {(_Float16)fmaf((float)h.x, -1.0f / kLo, a * (1.0f / kLo)),
                (_Float16)fmaf((float)h.y, -1.0f / kLo, b * (1.0f / kLo))};
  hi = __builtin_bit_cast(uint32_t, h);
  lo = __builtin_bit_cast(uint32_t, l);
}

// exp(x) * 2^14 for x <= 0 (or NaN). x = n ln 2 + r with n the nearest integer,
// ln 2 taken off in two parts (the argument reduction of Cody and Waite,
// Software Manual for the Elementary Functions, 1980; the first part leaves no
// rounding), so r is good to 2^-26 and exp(x) = 2^n * 2^(r / ln 2).
__device__ __forceinline__ float exp14(float x) {
  constexpr double ln2 = 0.69314718055994530942;
  constexpr float ln2hi = (float)ln2, ln2lo = (float)(ln2 - (double)ln2hi), inv = (float)(1.0 / ln2);
  x = x < -150.0f ? -150.0f : x;
  const float n = rintf(x * inv);
  const float r = fmaf(n, -ln2lo, fmaf(n, -ln2hi, x));
  return ldexpf(__builtin_amdgcn_exp2f(r * inv), (int)n + 14);
}

__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Work-group: NW waves, one query head, 32 query rows; wave w takes the key
// blocks w, w + nw, ... (32 positions each) with its own running softmax, and
// the waves are merged through LDS in wave order. NW = 4, two work-groups per
// CU, or 8 (see launch_attn_rows).
//
// Per block and wave, v_mfma_f32_32x32x16_f16 throughout:
//   scores S^T[key, query] = K . q^T: A = K rows (through the wave's LDS tile),
//     B = q, scaled by a power of two per row to [2^14, 2^15) and split into
//     two f16 pieces (LDS, for the whole kernel). Lane l ends with query
//     l % 32 and 16 of the 32 keys, so the row maximum is in-lane plus one
//     exchange with lane l ^ 32.
//   O^T[dim, query] = f * O^T + V^T . P: B = the weights of the lane's own 16
//     keys, times 2^14, as two f16 pieces, straight from the score registers
//     (the key order inside an MFMA only has to agree with A's); A = V^T: lane
//     m loads dims DL*m .. +DL-1 of its half's 16 keys (whole rows per load
//     instruction) and turns them with byte permutes, tile t holding dim
//     DL*m + t.
// K and V are exact in f16 and all sums are fp32; the small pieces' products
// are summed first, and a block's sum before it joins O, so the roundings stay
// as small as in a sum by chunks. The next block's K and V load while a block
// is worked on.
// An infinity or NaN among a tile's q, K or V would spread here (0 * inf in
// the small pieces, and to rows before its position), so a result that is not
// finite is formed again from its row's own positions, in plain f32.
// Measured on MI355X (16 heads of 128 over 4, 777 rows after 611 positions):
// the work-group per (row, 64 positions) of attn_batch takes 2400 us, bound by
// its per-row loads, hand-offs and VALU products; this kernel 31.6 us, bound by
// the softmax's VALU work between the two products. Error against 64 bits 2.2e-7
// there, 1.9e-7 here; where all but e^-20 of the weight lies on a position with a
// zero value, 6.1e-7 in both.
template <int HD, int NW>
__global__ void __launch_bounds__(64 * NW, NW == 4 ? 2 : 1) k_attn_rows(const float *__restrict__ q, const uint16_t *__restrict__ kc,
                                                      const uint16_t *__restrict__ vc, int64_t s_rows, int nh,
                                                      int nkv, int64_t pos0, const int32_t *__restrict__ pos_dev,
                                                      int64_t n_ctx, float *__restrict__ out) {
  constexpr int NS = HD / 16;       // K steps of the score product
  constexpr int DL = HD / 32;       // head dims per lane of V, and O tiles
  constexpr int KPL = HD / 16;      // 16-byte K pieces per lane and block
  constexpr int CPR = HD / 8;       // 16-byte pieces per K row
  constexpr int KROW = CPR + 1;     // the same in LDS (one pad: rows start 4 banks apart)
  constexpr int OROW = HD + 4;      // f32 per query row in the merge
  union Lds {
    struct {
      u32x4 k[NW][kKB][KROW];
      u32x4 q[2][kQT][KROW];  // hi and lo pieces
    } a;
    float o[NW][kQT][OROW];
  };
  __shared__ __attribute__((aligned(16))) Lds L;
  __shared__ float ml[NW][kQT], ll[NW][kQT];
  const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = blockIdx.x;
  const int g = h / (nh / nkv);
  const int64_t s0 = (int64_t)(gridDim.y - 1 - blockIdx.y) * kQT;  // long rows first
  const int64_t pos = pos0 + (pos_dev ? (int64_t)*pos_dev : 0);
  auto visible = [&](int64_t r) {
    r = r < s_rows ? r : s_rows - 1;
    return (int)(pos + r + 1 < n_ctx ? pos + r + 1 : n_ctx);
  };
  const int n_me = visible(s0 + l32), n_first = visible(s0), n_max = visible(s0 + kQT - 1);
  const int nblk = (n_max + kKB - 1) / kKB;
  const int nw = NW == 4 || pos + s_rows > kNarrow ? NW : 4;
  const int64_t rowb = (int64_t)nkv * HD * 2;  // bytes per position
  const char *kg = (const char *)(kc + (int64_t)g * HD), *vg = (const char *)(vc + (int64_t)g * HD);

  u32x4 kp[KPL];
  uint32_t vp[16][DL / 2];
  // key i of the lane's 16: the positions its score registers hold
  auto key = [&](int i) { return 8 * (i >> 2) + 4 * half + (i & 3); };
  // Rows past n_max read as zeros: a block's buffer ends with its last row, and
  // the row is in the lane's offset, which the bounds check covers (a scalar
  // offset is not promised to be checked).
  const int ko = (int)((lane / CPR) * rowb) + 16 * (lane % CPR);
  const int vo = (int)(4 * half * rowb) + 2 * DL * l32;
  auto block = [&](const char *base, int b) {
    const int nr = n_max - b * kKB < kKB ? n_max - b * kKB : kKB;
    return __builtin_amdgcn_make_buffer_rsrc((void *)(base + (int64_t)b * kKB * rowb), (short)0,
                                             (int)((nr - 1) * rowb) + 2 * HD, 0x00020000);
  };
  auto load_k = [&](int b) {
    const auto rs = block(kg, b);
    int o = ko;
    asm volatile("" : "+v"(o));  // formed here, not held in registers over the loop
#pragma unroll
    for (int i = 0; i < KPL; ++i, o += (int)((64 / CPR) * rowb)) kp[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, o, 0, 0);
  };
  auto load_v = [&](int b) {
    const auto rs = block(vg, b);
    int o = vo;
    asm volatile("" : "+v"(o));
#pragma unroll
    for (int i = 0; i < 16; ++i, o += (int)((i & 3) ? rowb : 5 * rowb)) {  // row 8 * (i / 4) + i % 4
      if constexpr (DL == 4) {
        const auto u = __builtin_amdgcn_raw_buffer_load_b64(rs, o, 0, 0);
        vp[i][0] = u[0];
        vp[i][1] = u[1];
      } else {
        vp[i][0] = __builtin_amdgcn_raw_buffer_load_b32(rs, o, 0, 0);
      }
    }
  };
  const int b0 = wave < nw ? wave : nblk;
  if (b0 < nblk) {
    load_k(wave);
    load_v(wave);
  }
  // q pieces: thread (row tid / 8, dims HD/8 * (tid % 8) ..); the row's shift by its 8 threads
  if (NW == 4 || tid < 256) {
    constexpr int DQ = HD / 8;
    const int r = tid >> 3, c = tid & 7;
    const int64_t sr = s0 + r < s_rows ? s0 + r : s_rows - 1;
    const float *qp = q + (sr * nh + h) * HD + DQ * c;
    f32x4a4 v[DQ / 4];
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < DQ / 4; ++i) v[i] = *(const f32x4a4 *)(qp + 4 * i);
#pragma unroll
    for (int i = 0; i < DQ; ++i) amax = fmaxf(amax, fabsf(v[i >> 2][i & 3]));
    amax = group_max<8>(amax);
    int sh = 15 - ((int)(__float_as_uint(amax) >> 23) - 126);
    sh = sh < 100 ? sh : 100;
#pragma unroll
    for (int i = 0; i < DQ / 8; ++i) {
      u32x4 hi, lo;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        uint32_t x, y;
        split2(ldexpf(v[2 * i + (j >> 1)][2 * (j & 1)], sh), ldexpf(v[2 * i + (j >> 1)][2 * (j & 1) + 1], sh), x, y);
        hi[j] = x;
        lo[j] = y;
      }
      L.a.q[0][r][DQ / 8 * c + i] = hi;
      L.a.q[1][r][DQ / 8 * c + i] = lo;
    }
    if (c == 0) ml[0][r] = ldexpf(1.0f / sqrtf((float)HD), -sh);
  }
  lds_barrier();
  const float fs = ml[0][l32], fsl = fs * kLo;
  lds_barrier();
  f32x16 O[DL];
#pragma unroll
  for (int t = 0; t < DL; ++t) O[t] = f32x16{0};
  float m = -INFINITY, l = 0.0f;  // l and O times 2^14
  for (int b = b0; b < nblk; b += nw) {
#pragma unroll
    for (int i = 0; i < KPL; ++i) L.a.k[wave][(64 / CPR) * i + lane / CPR][lane % CPR] = kp[i];
    const bool more = b + nw < nblk;
    if (more) load_k(b + nw);
    wave_lds_order();
    f32x16 S = f32x16{0}, Sh[2] = {f32x16{0}, f32x16{0}};
#pragma unroll
    for (int t = 0; t < NS; ++t) {
      const h8 a = __builtin_bit_cast(h8, L.a.k[wave][l32][2 * t + half]);
      S = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, __builtin_bit_cast(h8, L.a.q[1][l32][2 * t + half]), S, 0, 0, 0);
      Sh[t & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
          a, __builtin_bit_cast(h8, L.a.q[0][l32][2 * t + half]), Sh[t & 1], 0, 0, 0);
    }
    wave_lds_order();  // the tile is read before the next block writes it
    const bool edge = b * kKB + kKB > n_first;  // some row does not see the whole block
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float t = fmaf(Sh[0][i] + Sh[1][i], fs, S[i] * fsl);
      if (edge) t = b * kKB + key(i) < n_me ? t : -INFINITY;
      S[i] = t;
      mx = fmaxf(mx, t);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const float mn = fmaxf(m, mx);
    const float mb = mn == -INFINITY ? 0.0f : mn;  // no visible position yet: every weight is 0
    const float f = exp14(m - mb) * 0x1p-14f;
    m = mn;
    u32x4 ph[2], pl[2];
    float ls[2] = {0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < 16; i += 2) {
      const float e0 = exp14(S[i] - mb), e1 = exp14(S[i + 1] - mb);
      ls[i >> 3] += e0 + e1;
      uint32_t x, y;
      split2(e0, e1, x, y);
      ph[i >> 3][(i >> 1) & 3] = x;
      pl[i >> 3][(i >> 1) & 3] = y;
    }
    l = fmaf(l, f, ls[0] + ls[1]);
    u32x4 a[2][DL];
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int c = 0; c < DL / 2; ++c) {
          const uint32_t x = vp[8 * st + 2 * i][c], y = vp[8 * st + 2 * i + 1][c];
          a[st][2 * c][i] = __builtin_amdgcn_perm(y, x, 0x05040100u);
          a[st][2 * c + 1][i] = __builtin_amdgcn_perm(y, x, 0x07060302u);
        }
#pragma unroll
    for (int t = 0; t < DL; ++t) {
      f32x16 T = f32x16{0};
#pragma unroll
      for (int st = 0; st < 2; ++st)
        T = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8, a[st][t]), __builtin_bit_cast(h8, pl[st]), T, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 16; ++i) T[i] *= kLo;
#pragma unroll
      for (int st = 0; st < 2; ++st)
        T = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8, a[st][t]), __builtin_bit_cast(h8, ph[st]), T, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 16; ++i) O[t][i] = fmaf(O[t][i], f, T[i]);
    }
    if (more) load_v(b + nw);
  }
  // merge the waves: element i of tile t is dim DL * key(i) + t of query l32
  lds_barrier();  // every wave is done with its K tile and q
  l += __shfl_xor(l, 32);
  if (half == 0) {
    ml[wave][l32] = m;
    ll[wave][l32] = l;
  }
#pragma unroll
  for (int i = 0; i < 16; ++i)
#pragma unroll
    for (int t = 0; t < DL; ++t) L.o[wave][l32][DL * key(i) + t] = O[t][i];
  lds_barrier();
  constexpr int TPR = 2 * NW, DPT = HD / TPR;  // threads per query row, dims per thread
  const int qi = tid / TPR, d0 = (tid % TPR) * DPT;
  if (s0 + qi >= s_rows) return;
  float M = -INFINITY, f[NW], Ls = 0.0f;
#pragma unroll
  for (int w = 0; w < NW; ++w) M = fmaxf(M, ml[w][qi]);
  const float Mb = M == -INFINITY ? 0.0f : M;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    f[w] = exp14(ml[w][qi] - Mb) * 0x1p-14f;
    Ls += ll[w][qi] * f[w];
  }
  const float inv = 1.0f / Ls;
  const int64_t row = (s0 + qi) * nh + h;
  float *o = out + row * HD + d0;
  bool finite = true;
#pragma unroll
  for (int d = 0; d < DPT; d += 4) {
    f32x4a4 r;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      float v = 0.0f;
#pragma unroll
      for (int w = 0; w < NW; ++w) v += L.o[w][qi][d0 + d + c] * f[w];
      r[c] = v * inv;
      finite = finite && fabsf(r[c]) < INFINITY;
    }
    *(f32x4a4 *)(o + d) = r;
  }
  if (!finite) {  // one row's dims from its own positions, in plain f32
    const float *qp = q + row * HD;
    const int n = visible(s0 + qi);
    const float scale = 1.0f / sqrtf((float)HD);
    auto score = [&](int p) {
      const _Float16 *kr = (const _Float16 *)(kg + p * rowb);
      float sc = 0.0f;
      for (int d = 0; d < HD; ++d) sc += qp[d] * (float)kr[d];
      return sc * scale;
    };
    float mr = -INFINITY, lr = 0.0f, acc[DPT];
    for (int p = 0; p < n; ++p) mr = fmaxf(mr, score(p));
#pragma unroll
    for (int d = 0; d < DPT; ++d) acc[d] = 0.0f;
    for (int p = 0; p < n; ++p) {
      const float e = exp14(score(p) - mr);
      lr += e;
#pragma unroll
      for (int d = 0; d < DPT; ++d) acc[d] += e * (float)((const _Float16 *)(vg + p * rowb))[d0 + d];
    }
#pragma unroll
    for (int d = 0; d < DPT; ++d) o[d] = acc[d] * (1.0f / lr);
  }
}

}  // namespace

hipError_t launch_attn_rows(hipStream_t st, const float *q, const uint16_t *kc, const uint16_t *vc, int64_t s_rows,
                            int nh, int nkv, int hd, int64_t pos0, const int32_t *pos_dev, int64_t n_ctx,
                            float *out) {
  const int64_t tiles = (s_rows + kQT - 1) / kQT;
  if (s_rows < kAttnRowsMin || tiles > 65535 || (((uintptr_t)kc | (uintptr_t)vc) & 15)) return hipErrorNotSupported;
  const dim3 grid((unsigned)nh, (unsigned)tiles);
  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
#define KMOE_ATTN(H, W)                                                                                          \
  KMOE_LAUNCH((k_attn_rows<H, W>), grid, dim3(64 * W), 0, st, q, kc, vc, s_rows, nh, nkv, pos0, pos_dev, n_ctx, \
              out)
  // 8 waves per work-group where the grid has at most one per CU and the rows
  // see more than 8 blocks: 64 rows after 1000 positions, 32 heads 22.0 -> 17.7
  // us, 24 after 900, 16 heads 19.6 -> 16.4; but 16 rows after none 8.5 -> 10.2,
  // where the larger merge is all that is added. (With a position on the device
  // the kernel finds out itself.)
  const bool wide = nh * tiles <= cus && (pos_dev ? n_ctx : pos0 + s_rows) > kNarrow;
  if (hd == 64) {
    if (wide) KMOE_ATTN(64, 8);
    else KMOE_ATTN(64, 4);
  } else if (hd == 128) {
    if (wide) KMOE_ATTN(128, 8);
    else KMOE_ATTN(128, 4);
  } else {
    return hipErrorNotSupported;
  }
#undef KMOE_ATTN
  return hipGetLastError();
}

}  // namespace kmoe
