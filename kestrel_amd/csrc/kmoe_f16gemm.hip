// kmoe_f16gemm.hip — the reference's f32 regime (quant.rs:242-260) for many
// activation rows on the f16 matrix cores: Q4_K, Q6_K and Q8_0 rows of the
// expert tier (gate/up + SwiGLU, transformer.rs:551-558, and down) and plain
// GGUF rows (quant::matmul itself, a shared expert's front).
#include "kmoe_device.h"
#include "kmoe_launch.h"

namespace kmoe {

namespace {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2a2 __attribute__((ext_vector_type(2), aligned(2)));

// ------------------------------------------------ activation rows as f16 pieces
//
// A row is scaled by a power of two so that its largest finite magnitude lies
// in [2^14, 2^15), and each element becomes two f16 pieces: hi, the nearest
// f16, and lo, the nearest f16 of 2^12 times what hi leaves (a factor of its
// own: lo's exponent would end 2^-39 below the row's largest otherwise, and
// elements some 2^20 below it lose their bits). x = hi + lo * 2^-12 to 2^-23 of
// x, and to 2^-51 of the row's largest element for elements too small for that.
// (An infinity keeps hi = inf, lo = 0.) Row r of the result is cols hi pieces,
// then cols lo pieces (cols rounded up to 128, the rest zeros): the row's own
// size in f32, so rows whose length is a multiple of 128 convert in place.
// Inside every 8 elements the order is 0,2,1,3,4,6,5,7, the order in which
// the weights' 4-bit pairs come out of a dword. For Q4_K's minimum term the
// sums of 32 scaled elements, times 2^-5, go to `sums` as two such pieces: per
// 256 elements 8 hi pieces, then 8 lo.
struct SplitArgs {
  const float *x;
  int64_t rows, cols;
  F16Rows o;
  // grouped rows (slots in dispatch order): only rows of experts with at least
  // min_rows rows; idx null: every row
  const uint32_t *idx, *perm, *offsets;
  int min_rows;
};

constexpr float kLo = 0x1p-12f;  // the lo pieces' unit

__device__ __forceinline__ uint32_t pack_h2(float a, float b) {
  h2 v;
  v.x = (_Float16)a;
  v.y = (_Float16)b;
  return __builtin_bit_cast(uint32_t, v);
}

// WV waves per row, lane: 8 columns of every 512 * WV, at most NIT times.
// Every load of the row is consumed before its first store (in-place rows).
template <int WV, int NIT>
__global__ void __launch_bounds__(64 * WV) k_split_f16(SplitArgs a) {
  const int64_t r = blockIdx.x;
  if (a.idx) {
    const uint32_t e = a.idx[a.perm[r]];
    if ((int)(a.offsets[e + 1] - a.offsets[e]) < a.min_rows) return;
  }
  const int tid = threadIdx.x;
  const float *x = a.x + r * a.cols;
  float4 v[NIT][2];
  float m = 0.0f;
#pragma unroll
  for (int i = 0; i < NIT; ++i) {
    const int64_t c = 8 * (tid + (int64_t)(64 * WV) * i);
    const bool in = c < a.cols;
    v[i][0] = in ? *(const float4 *)(x + c) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    v[i][1] = in ? *(const float4 *)(x + c + 4) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  }
#pragma unroll
  for (int i = 0; i < NIT; ++i)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const float t[4] = {v[i][u].x, v[i][u].y, v[i][u].z, v[i][u].w};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float f = fabsf(t[k]);
        m = f < __builtin_inff() ? fmaxf(m, f) : m;
      }
    }
  m = group_max<64>(m);
  if constexpr (WV > 1) {
    __shared__ float wm[WV];
    if ((tid & 63) == 0) wm[tid >> 6] = m;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < WV; ++i) m = fmaxf(m, wm[i]);
  }
  const int sh = m > 0.0f ? 14 - ilogbf(m) : 0;
  if (tid == 0) a.o.ex[r * a.o.ex_stride] = sh;
  const int64_t kp = (a.cols + 127) / 128 * 128;
  uint16_t *hi = a.o.planes + r * 2 * kp, *lo = hi + kp;
  uint8_t *sums = (uint8_t *)a.o.sums + r * a.o.sums_stride;
#pragma unroll
  for (int i = 0; i < NIT; ++i) {
    const int64_t c = 8 * (tid + (int64_t)(64 * WV) * i);
    if (c >= kp) continue;
    const float t[8] = {v[i][0].x, v[i][0].y, v[i][0].z, v[i][0].w, v[i][1].x, v[i][1].y, v[i][1].z, v[i][1].w};
    float hf[8], lf[8], s = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float y = ldexpf(t[k], sh);
      hf[k] = (float)(_Float16)y;
      lf[k] = fabsf(y) < __builtin_inff() ? (y - hf[k]) * (1.0f / kLo) : 0.0f;
      s += y;
    }
    *(u32x4 *)(hi + c) = u32x4{pack_h2(hf[0], hf[2]), pack_h2(hf[1], hf[3]), pack_h2(hf[4], hf[6]), pack_h2(hf[5], hf[7])};
    *(u32x4 *)(lo + c) = u32x4{pack_h2(lf[0], lf[2]), pack_h2(lf[1], lf[3]), pack_h2(lf[4], lf[6]), pack_h2(lf[5], lf[7])};
    if (a.o.sums) {  // 4 lanes hold a 32-element sub-block
      s = ldexpf(group_sum<4>(s), -5);
      if ((tid & 3) == 0) {
        const _Float16 sh16 = (_Float16)s;
        const _Float16 sl16 = (_Float16)(fabsf(s) < __builtin_inff() ? (s - (float)sh16) * (1.0f / kLo) : 0.0f);
        _Float16 *p = (_Float16 *)(sums + c / 256 * 32) + (c / 32 % 8);
        p[0] = sh16;
        p[8] = sl16;
      }
    }
  }
}

// ------------------------------------------- int8 activation rows as f16 pieces
//
// Rows of int8 values (Q8_K or Q8) as one f16 piece each, exact, in the same
// order within 8; row r is cols pieces. sums (Q8_K, for Q4_K's minimum term):
// the sums of 32 from the row's 16-sums, times 2^-5, as above (both pieces
// together exact: at most 12 bits). One lane per 16 columns.
__global__ void __launch_bounds__(256) k_i8_f16(const int8_t *__restrict__ q, const int32_t *__restrict__ s16,
                                                int64_t n16, int64_t cols, uint16_t *__restrict__ planes,
                                                uint16_t *__restrict__ sums, int64_t sums_stride) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n16) return;
  const u32x4 v = *(const u32x4 *)(q + 16 * i);
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
  u32x4 o[2];
#pragma unroll
  for (int k = 0; k < 4; ++k) {  // 4 values: (0, 2), (1, 3) of the dword
    const uint32_t u = w[k] ^ 0x80808080u;
    const h2 off = {(_Float16)-1152.0f, (_Float16)-1152.0f};
    const h2 a = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, u, 0x04020400u)) + off;
    const h2 b = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, u, 0x04030401u)) + off;
    o[k >> 1][2 * (k & 1)] = __builtin_bit_cast(uint32_t, a);
    o[k >> 1][2 * (k & 1) + 1] = __builtin_bit_cast(uint32_t, b);
  }
  *(u32x4 *)(planes + 16 * i) = o[0];
  *(u32x4 *)(planes + 16 * i + 8) = o[1];
  if (sums && (i & 1) == 0) {
    const float s = (float)(s16[i] + s16[i + 1]) * 0.03125f;
    const int64_t r = 16 * i / cols, c = 16 * i - r * cols;
    _Float16 *p = (_Float16 *)((uint8_t *)sums + r * sums_stride + c / 256 * 32) + (c / 32 % 8);
    const _Float16 hi = (_Float16)s;
    p[0] = hi;
    p[8] = (_Float16)((s - (float)hi) * (1.0f / kLo));
  }
}

// ------------------------------------------------------------------ the product

struct F16Args {
  ExpertTier tier;
  Routing rt;
  int64_t rows, cols;      // weight rows and columns of one part
  F16Rows x;               // gate/up: the layer input's rows; down: the slots' h rows
  float *out;              // gate/up: h [slots, rows]; down: y [slots, rows]; plain: out [s_rows, rows]
  int min_rows, max_rows;  // grouped: experts with min_rows..max_rows rows
  int n_expert;
  const uint8_t *pw, *pw2;  // plain: GGUF rows; with SwiGLU the gate and the up rows
  int64_t s_rows;           // plain: activation rows
  int split_stages;         // columns split over blockIdx.y: stages per split (even), each split's
  int64_t split_stride;     // sums at out + split * split_stride
  const float *ad;          // int8 rows: their block scales [.., cols / 256 or / 32]
  BlockDbg dbg;             // int8 rows with DBG: per-block integers (gate/down 0, up 1),
  const int32_t *s16;       // the rows' 16-sums (Q6_K)
};

__device__ __forceinline__ void lds_dma16(const void *g, uint8_t *lds_wave_base) {
  __builtin_amdgcn_global_load_lds(g, (__attribute__((address_space(3))) void *)lds_wave_base, 16, 0, 0);
}

// One stage (128 columns) of one 32-row weight tile as loaded: lane l holds its
// 8 of every 16 elements of row l % 32 (elements 16s + 8*(l/32) ..+7).
template <int T>
struct Raw;
template <>
struct Raw<T_Q4_K> {
  u32x2 n[2][2];  // nibble bytes of (quarter, 16-byte half)
  u32x4 hd;
};
template <>
struct Raw<T_Q8_0> {
  u32x2 n[4][2];  // block, 16-element half
  uint16_t d[4];
};
template <>
struct Raw<T_Q6_K> {
  u32x2 n[2][2];  // tiled: nibbles of (row pair, half); GGUF: ql of (row & 1, half)
  u32x2 q[2];     // tiled: high bits of the row pair; GGUF: qh of the half
  u32x2 sc;       // the 8 scales
  uint16_t d;
};

template <int T, bool TILED>
__device__ __forceinline__ void load_raw(Raw<T> &w, const uint8_t *m, uint32_t ro, int64_t nb, int64_t st) {
  // ro: byte offset of the lane's row in the matrix plus 8 * (lane / 32) (the quants); the rest is uniform
  // opaque in each stage, so that the loads keep a scalar base and a 32-bit
  // lane offset instead of 64-bit lane addresses held over the loop
  asm volatile("" : "+v"(ro));
  const uint32_t r0 = ro - 8 * ((threadIdx.x & 63) >> 5);
  if constexpr (T == T_Q4_K) {
    const int64_t b = st >> 1;
    const int k0 = 2 * (int)(st & 1);
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        w.n[q][j] = *(const u32x2 *)(m + (TILED ? tq4_qs_off(nb, b, k0 + q, j) : 144 * b + 16 + 32 * (k0 + q) + 16 * j) + ro);
    w.hd = *(const u32x4 *)(m + (TILED ? 16 : 144) * b + r0);
  } else if constexpr (T == T_Q8_0) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int64_t b = 4 * st + q < nb ? 4 * st + q : nb - 1;
      w.d[q] = *(const uint16_t *)(m + 34 * b + r0);
#pragma unroll
      for (int j = 0; j < 2; ++j) w.n[q][j] = *(const u32x2a2 *)(m + 34 * b + 2 + 16 * j + ro);
    }
  } else {
    const int64_t b = st >> 1;
    const int h = (int)(st & 1);
#pragma unroll
    for (int p = 0; p < 2; ++p) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
        w.n[p][j] = *(const u32x2a2 *)(m + (TILED ? tq6_piece_off(nb, b, 2 * h + p, j) : 210 * b + 64 * h + 32 * p + 16 * j) + ro);
      w.q[p] = *(const u32x2a2 *)(m + (TILED ? tq6_piece_off(nb, b, 2 * h + p, 2) : 210 * b + 128 + 32 * h + 16 * p) + ro);
    }
    w.sc = *(const u32x2a2 *)(m + (TILED ? 192 * nb + 16 * b : 210 * b + 192) + 8 * h + r0);
    w.d = *(const uint16_t *)(m + (TILED ? 208 * nb + 2 * b : 210 * b + 208) + r0);
  }
}

// Groups of columns with one scale per stage, and their f32 scale.
template <int T>
constexpr int kGroups = T == T_Q4_K ? 1 : T == T_Q8_0 ? 4 : 8;

// One v_and_or_b32 (at most one of its constants may come from a scalar
// register, so the other is kept in a vector register: `k1024`).
__device__ __forceinline__ uint32_t and_or(uint32_t a, uint32_t m, uint32_t o) { return (a & m) | o; }

// Weights of the stage as MFMA operands (f16, exact): Q4_K sc*q (<= 945),
// Q8_0 q, Q6_K q - 32; g: the f32 factor of each group (Q4_K d, Q8_0 d, Q6_K
// d*sc as dequant_row forms it; INT: the bits of the integer sc).
template <int T, bool TILED, bool INT>
__device__ __forceinline__ void unpack(const Raw<T> &w, int64_t st, int64_t nb, h8 (&o)[8], float (&g)[kGroups<T>]) {
  uint32_t r[8][4];
  if constexpr (T == T_Q4_K) {
    uint32_t k1024 = 0x64006400u, mlo = 0x000f000fu, mhi = 0x00f000f0u;
    asm("" : "+v"(k1024));
    asm("" : "+s"(mlo), "+s"(mhi));
    g[0] = f16_bits_to_f32(w.hd.x);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      int sA, mA, sB, mB;
      q4k_scale_min_pair(w.hd.y, w.hd.z, w.hd.w, 2 * (int)(st & 1) + q, sA, mA, sB, mB);
      // 0x6400 | v is the f16 value 1024 + v: low nibbles (1024 + q)*s - 1024*s,
      // high nibbles (1024 + 16q)*(s/16) - 64*s, both exact
      const _Float16 s0 = (_Float16)(float)sA, s1 = (_Float16)((float)sB * 0.0625f);
      const h2 sl = {s0, s0}, sh = {s1, s1};
      const h2 nl = sl * (_Float16)-1024.0f, nh = sh * (_Float16)-1024.0f;
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const uint32_t v = u ? w.n[q][j].y : w.n[q][j].x, v8 = v >> 8;
          const uint32_t t[4] = {and_or(v, mlo, k1024), and_or(v8, mlo, k1024), and_or(v, mhi, k1024),
                                 and_or(v8, mhi, k1024)};
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const h2 f = __builtin_elementwise_fma(__builtin_bit_cast(h2, t[i]), i < 2 ? sl : sh, i < 2 ? nl : nh);
            r[4 * q + 2 * (i >> 1) + j][2 * u + (i & 1)] = __builtin_bit_cast(uint32_t, f);
          }
        }
    }
  } else if constexpr (T == T_Q8_0) {
    const h2 off = {(_Float16)-1152.0f, (_Float16)-1152.0f};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      g[q] = 4 * st + q < nb ? f16_bits_to_f32(w.d[q]) : 0.0f;  // past the row's end the activations are zeros
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const uint32_t v = (u ? w.n[q][j].y : w.n[q][j].x) ^ 0x80808080u;  // q + 128
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const uint32_t t = __builtin_amdgcn_perm(0x64646464u, v, i ? 0x04030401u : 0x04020400u);
            r[2 * q + j][2 * u + i] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2, t) + off);
          }
        }
    }
  } else {
    const h2 off = {(_Float16)-1056.0f, (_Float16)-1056.0f};
    const float d = f16_bits_to_f32(w.d);
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int row = s >> 1, j = s & 1;
      const uint32_t sw = s < 4 ? w.sc.x : w.sc.y;
      const int sc = (int8_t)(sw >> (8 * (s & 3)));
      g[s] = INT ? __builtin_bit_cast(float, sc) : d * (float)sc;
      // the nibbles of 32-row `row` and its 2 high bits
      const u32x2 nv = TILED ? w.n[row >> 1][j] : w.n[row & 1][j], qv = TILED ? w.q[row >> 1] : w.q[j];
      const int ns = TILED ? 4 * (row & 1) : 4 * (row >> 1), qs = TILED ? 4 * j + 2 * (row & 1) : 2 * row;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const uint32_t n = (u ? nv.y : nv.x) >> ns, q = u ? qv.y : qv.x;
        const uint32_t b = (qs <= 4 ? q << (4 - qs) : q >> (qs - 4)) & 0x30303030u;
        const uint32_t v = (n & 0x0f0f0f0fu) | b;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const uint32_t t = __builtin_amdgcn_perm(0x64646464u, v, i ? 0x04030401u : 0x04020400u);
          r[s][2 * u + i] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2, t) + off);
        }
      }
    }
  }
#pragma unroll
  for (int s = 0; s < 8; ++s) o[s] = __builtin_bit_cast(h8, u32x4{r[s][0], r[s][1], r[s][2], r[s][3]});
}

// The lane's number, read where it is used: a register held for it over the K
// loop would spill others (the down product's two by two tiles: 2 registers, 181
// us at 1777 Qwen3-shaped tokens, 165 without).
__device__ __forceinline__ uint32_t lane_here() {
  uint32_t all = 0xffffffffu;
  asm volatile("" : "+s"(all));
  return __builtin_amdgcn_mbcnt_hi(all, __builtin_amdgcn_mbcnt_lo(all, 0));
}

// The 8 minimums of a Q4_K superblock, times 32, as the MFMA's B operand (the K
// halves: against the sums' hi and lo pieces).
__device__ __forceinline__ h8 mins_operand(const u32x4 &hd) {
  h8 o;
  // 32 in the lower lanes, 32 * kLo in the upper ones
  const float f = __builtin_bit_cast(float, 0x42000000u - (lane_here() >> 5) * (12u << 23));
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    int sA, mA, sB, mB;
    q4k_scale_min_pair(hd.y, hd.z, hd.w, k, sA, mA, sB, mB);
    o[2 * k] = (_Float16)((float)mA * f);
    o[2 * k + 1] = (_Float16)((float)mB * f);
  }
  return o;
}

// Row blocks of `rpb` weight rows times token blocks of BN rows, as one list:
// expert by expert, and inside one row block by row block, its token blocks
// side by side (they share the weights). Work-groups are dealt to the XCDs
// round-robin, so XCD x takes the x-th eighth of the list and neighbours share
// its L2. Every wave finds its work-group's entry itself.
template <int BN, bool PLAIN>
__device__ __forceinline__ bool find_block(const F16Args &a, int rblocks, int lane, int &e, int &rb, int &tb, int &n) {
  const int b = (int)blockIdx.x;
  auto eighth = [&](int total, int &want) {
    const int per = (total + 7) / 8;
    want = (b & 7) * per + (b >> 3);
    return (b >> 3) < per && want < total;
  };
  if constexpr (PLAIN) {
    e = 0;
    n = (int)a.s_rows;
    const int nt = (n + BN - 1) / BN;
    int want;
    if (!eighth(nt * rblocks, want)) return false;
    rb = want / nt;
    tb = want - rb * nt;
    return true;
  } else {
    auto rows_of = [&](int i) {
      int r = 0;
      if (i < a.n_expert) r = (int)(a.rt.offsets[i + 1] - a.rt.offsets[i]);
      return r >= a.min_rows && r <= a.max_rows ? r : 0;
    };
    int total = 0;
    for (int base = 0; base < a.n_expert; base += 64) total += group_sum_i<64>((rows_of(base + lane) + BN - 1) / BN);
    int want;
    if (!eighth(total * rblocks, want)) return false;
    int before = 0;  // entries of the experts below this chunk
    for (int base = 0; base < a.n_expert; base += 64) {
      const int r = rows_of(base + lane);
      const int own = (r + BN - 1) / BN * rblocks;
      int incl = own;
#pragma unroll
      for (int s = 1; s < 64; s <<= 1) {
        const int o = __shfl_up(incl, s);
        if (lane >= s) incl += o;
      }
      const int all = __builtin_amdgcn_readlane(incl, 63);
      if (want < before + all) {
        const int lo = before + incl - own;
        const uint64_t m = __ballot(want >= lo && want < lo + own);
        const int l = (int)__builtin_ctzll(m);
        e = base + l;
        n = __builtin_amdgcn_readlane(r, l);
        const int rem = want - __builtin_amdgcn_readlane(lo, l);
        const int nt = (n + BN - 1) / BN;
        rb = rem / nt;
        tb = rem - rb * nt;
        return true;
      }
      before += all;
    }
    return false;
  }
}

// MODE 0: grouped gate/up + SwiGLU, 1: grouped down (tier rows); 2: plain GGUF
// rows; 3: two plain matrices (gate, up) and SwiGLU.
//
// For a group of columns with one scale, sum_k w_k x_k = scale * sum_k q_k x_k
// with q exact in f16 (Q4_K: sc*q over the whole superblock, the minimum term
// -dmin * sum_j m_j S_j apart), and x is two f16 pieces, so
// v_mfma_f32_32x32x16_f16 forms the exact products and sums them in fp32: two
// MFMAs per product, the small pieces' first.
//
// Work-group: 4 waves, each RT tiles of 32 weight rows (MODE 0, 3: the gate
// and the up rows of the same 32) by up to NT tiles of 32 tokens. A = the
// tokens' pieces (LDS), B = the weights, unpacked by the wave that multiplies
// them straight into operand registers, once for all its token tiles. Lane l
// ends with weight row l % 32 and 16 tokens of each tile, so a scale is one
// register and the stores of a half wave are one run of 128 bytes.
// Stages of 128 columns: the next stage's pieces go to the other LDS buffer by
// direct loads and its weights to registers while this one multiplies; one
// barrier per stage. A piece row is 256 bytes in LDS, its 16-byte chunks at
// chunk ^ (token % 16): 8 consecutive tokens read 8 different bank groups.
// Two work-groups per CU (256 registers per lane): one unpacks while the
// other's MFMAs run.
// Measured on MI355X against the bf16-split and fp32 kernels (us, with the
// split and reduction kernels): Qwen3 shape, 1777 tokens, gate/up 1195 -> 308,
// down 680 -> 187; Q4_K 4096x4096 by 512 rows 184 -> 66; DeepSeek-V2-Lite
// shape, 203 tokens, gate/up 293 -> 143, Q8_0 down 180 -> 79, shared Q6_K down
// 278 -> 32. Its MFMAs run 29% of the time (counted); the rest is the weights'
// load requests (a row per lane: 32 lines per instruction), the unpacking and
// the short K loops' ends. Error against 64 bits: 3.1e-7 -> 1.7e-7 (Q4_K
// matrix). No form spills but Q8_0 gate/up by two token tiles (24 registers; 64
// experts of 1408 by 2048, 1777 tokens 1118 us per layer, one tile 1371).
//
// INT: int8 activation rows (the int8 path, quant.rs:262-281) as one exact f16
// piece. The MFMAs' sums are integers below 2^24 (Q4_K: 128 * 15*63 * 127 per
// stage), so exact, and join y once per superblock with the block scales, as
// the int8 kernels do: Q4_K d * (both stages) - dmin * mins; Q6_K the int32
// sum of sc * sum (mad_i24); Q8_0 the stage's four blocks first, the weight's
// f16 scale times the integer before the activation's. Long rows' sums move to
// LDS every kIntChain stages, so that no chain of roundings is longer than the
// int8 kernels' (which run parts of a row in parallel): error of the down
// product against 64 bits 7.3e-8 (Q4_K, 768 columns), 8.8e-8 (Q6_K, 14336),
// 8.9e-8 (Q8_0, 1408), there 7.3e-8, 8.9e-8 and 8.9e-8. A superblock's sums take
// the registers of two tiles: gate and up by one token tile, or down by two
// token tiles with one weight tile per wave, which unpacks a weight once per 64
// tokens (Mixtral shape, Q6_K down, 512 tokens 1666 -> 1401 us per layer).
// DBG adds the exact integers to the capture (its kernels spill; they are not
// timed).
// SPLIT: the columns over blockIdx.y (a form of its own: the bounds' registers).
// Stages per chain of roundings: 8 superblocks, or 4 sums of 4 blocks.
template <int T>
constexpr int kIntChain = T == T_Q8_0 ? 4 : 16;

template <int T, int MODE, int RT, int NT, bool INT = false, bool DBG = false, bool SPLIT = false>
__global__ void __launch_bounds__(256, 2) k_f16_gemm(F16Args a) {
  constexpr bool PLAIN = MODE >= 2, TILED = !PLAIN, SWIGLU = MODE == 0 || MODE == 3;
  static_assert(!SWIGLU || RT == 2, "gate and up tiles");
  constexpr int BN = 32 * NT, RPB = SWIGLU ? 128 : 128 * RT;
  constexpr int G = kGroups<T>, SPG = 8 / G;  // scale groups of a stage, MFMA steps per group
  constexpr int PLANE = BN * 256;             // bytes of one piece plane of a stage
  constexpr int SUMS = T == T_Q4_K ? BN * 32 : 0;  // the superblock's sums, with its second stage
  constexpr int NP = INT ? 1 : 2;                  // pieces per activation
  constexpr int ADW = T == T_Q8_0 ? 16 : 4, ADS = INT ? BN * ADW : 0;  // block scales of the stage's tokens
  __shared__ __attribute__((aligned(16))) uint8_t st0[NP * PLANE + ADS], st1[NP * PLANE + ADS + SUMS];
  __shared__ int exs[BN];
  __shared__ float4 yl[INT ? 4 * RT * NT : 1][INT ? 256 : 1];  // each thread's own sums
  static_assert(!INT || RT * NT == 2, "the registers of two tiles");
  const int tid = threadIdx.x, lane = tid & 63, hh = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int e, rb, tb, n;
  if (!find_block<BN, PLAIN>(a, (int)((a.rows + RPB - 1) / RPB), lane, e, rb, tb, n)) return;
  e = __builtin_amdgcn_readfirstlane(e);
  rb = __builtin_amdgcn_readfirstlane(rb);
  tb = __builtin_amdgcn_readfirstlane(tb);
  n = __builtin_amdgcn_readfirstlane(n);
  const int64_t p0 = PLAIN ? 0 : (int64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)a.rt.offsets[e]);
  const int tok0 = tb * BN;
  const int nbt = n - tok0 < BN ? n - tok0 : BN;
  const int ntt = (nbt + 31) / 32;
  const int64_t rows = a.rows, cols = a.cols;
  const int64_t nb = cols / (T == T_Q8_0 ? 32 : 256);
  const int64_t row_bytes = nb * (T == T_Q4_K ? 144 : T == T_Q6_K ? 210 : 34);
  const int64_t kp = (cols + 127) / 128 * 128;
  const int nst_all = (int)(kp / 128);
  const int st_lo = SPLIT ? (int)blockIdx.y * a.split_stages : 0;
  const int nst = SPLIT && st_lo + a.split_stages < nst_all ? st_lo + a.split_stages : nst_all;
  const int64_t rbase = (int64_t)rb * RPB + wave * (SWIGLU ? 32 : 32 * RT);
  const uint8_t *wm[RT];  // matrix (uniform) and row offset of each tile (launch: a matrix is below 4 GiB)
  uint32_t wr[RT];
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    int64_t r = rbase + (SWIGLU ? 0 : 32 * i) + l32;
    r = r < rows ? r : rows - 1;
    wm[i] = PLAIN ? (SWIGLU && i == 1 ? a.pw2 : a.pw)
                  : a.tier.base + (int64_t)e * a.tier.stride + a.tier.off[SWIGLU ? i : 2];
    wr[i] = (uint32_t)(r * row_bytes) + 8 * hh;
  }
  auto src_row = [&](int t) -> int64_t {  // the activation row of token t of this block
    const int64_t p = p0 + tok0 + (t < nbt ? t : nbt - 1);
    return MODE == 0 ? (int64_t)(a.rt.perm[p] / (uint32_t)a.rt.topk) : p;
  };
  if constexpr (!INT) {
    if (tid < BN) exs[tid] = a.x.ex[src_row(tid) * a.x.ex_stride];
  }
  // direct loads: instruction i of a wave takes tokens 4q .. 4q+3, q = wave * 2 NT + i, of both planes
  uint32_t xsrc[2 * NT];  // (launch: the pieces are below 4 GiB)
#pragma unroll
  for (int i = 0; i < 2 * NT; ++i) {
    const int t = 4 * (wave * 2 * NT + i) + (lane >> 4);
    xsrc[i] = (uint32_t)(src_row(t) * 2 * NP * kp) + 16 * ((lane & 15) ^ (t & 15));
  }
  const int64_t asrc = INT ? src_row(lane) * (cols / (T == T_Q8_0 ? 32 : 256)) : 0;
  auto load_x = [&](uint8_t *dst, int st) {
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
      for (int i = 0; i < 2 * NT; ++i) {
        uint32_t o = xsrc[i];
        asm volatile("" : "+v"(o));  // as in load_raw
        lds_dma16((const uint8_t *)a.x.planes + 2 * kp * p + 256 * (int64_t)st + o, dst + p * PLANE + (wave * 2 * NT + i) * 1024);
      }
    if constexpr (INT) {  // wave 0: token l's scale of the superblock, or scales of the stage's four blocks
      if (wave == 0 && lane < BN) {
        const float *p = a.ad + asrc + (T == T_Q8_0 ? 4 * st : st >> 1);
        auto *l = (__attribute__((address_space(3))) void *)(dst + NP * PLANE);
        if constexpr (T == T_Q8_0) __builtin_amdgcn_global_load_lds(p, l, 16, 0, 0);
        else __builtin_amdgcn_global_load_lds(p, l, 4, 0, 0);
      }
    }
  };
  // Q4_K: the superblock's sums of tokens 32w .. 32w+31 by wave w < NT
  uint32_t ssrc = 0;
  if constexpr (T == T_Q4_K && MODE == 0)
    ssrc = (uint32_t)(src_row(32 * (wave % NT) + (lane >> 1)) * a.x.sums_stride) + 16 * (lane & 1);
  // LDS offset of this lane's A piece of K step s: aoff ^ 32s
  const int aoff = 256 * l32 + 16 * (hh ^ (l32 & 15));

  float y[RT][NT][16];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) y[i][t][v] = 0.0f;
  Raw<T> raw[RT];
  load_x(st0, st_lo);
#pragma unroll
  for (int i = 0; i < RT; ++i) load_raw<T, TILED>(raw[i], wm[i], wr[i], nb, st_lo);

  // INT: sums on their way to y. Q4_K: the superblock's first half; Q8_0: the
  // stage's blocks; Q6_K (as int): the superblock's sum of sc * (bits of P).
  float z[INT ? RT : 1][NT][16];
  int zi[INT && T == T_Q6_K ? RT : 1][NT][16];
  // A group's sums P into y. Lane l's tokens of tile t are 8k + 4(l/32) + 0..3.
  auto int_epilogue = [&](int t, int gi, f32x16 (&P)[RT], const uint8_t *cur, bool odd, int st, const float (&g)[RT][G],
                          const h8 (&mo)[RT], const float (&dm)[RT]) {
    const uint8_t *ads = cur + NP * PLANE;
    auto capture = [&](int i, int v, int32_t *const (&arr)[2], int val) {
      const int tk = 32 * t + 8 * (v >> 2) + 4 * hh + (v & 3);
      const int64_t r = rbase + (SWIGLU ? 0 : 32 * i) + l32;
      if (tk < nbt && r < rows)
        dbg_add(arr[SWIGLU ? i : 0], ((p0 + tok0 + tk) * rows + r) * nb + (T == T_Q8_0 ? 4 * st + gi : st >> 1), val);
    };
    if constexpr (T == T_Q6_K) {
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        const int sc = __builtin_bit_cast(int, g[i][gi]);
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int p = sc * ((int)P[i][v] << 8 >> 8);
          zi[i][t][v] = gi == 0 && !odd ? p : zi[i][t][v] + p;
          asm volatile("" : "+v"(zi[i][t][v]));
        }
        if constexpr (DBG) {
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            const int tk = 32 * t + 8 * (v >> 2) + 4 * hh + (v & 3);
            const int o = sc * a.s16[src_row(tk) * (cols / 16) + 8 * st + gi];
            capture(i, v, a.dbg.m, o);
            capture(i, v, a.dbg.s, sc * (int)P[i][v] + 32 * o);
          }
        }
      }
      if (gi < G - 1 || !odd) return;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        float sc[4];
        *(float4 *)sc = *(const float4 *)(ads + 4 * (32 * t + 8 * k + 4 * hh));
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const int v = 4 * k + c;
            y[i][t][v] = fmaf(dm[i] * sc[c], (float)zi[i][t][v], y[i][t][v]);
          }
      }
    } else if constexpr (T == T_Q8_0) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        float sc[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) sc[c] = *(const float *)(ads + 16 * (32 * t + 8 * k + 4 * hh + c) + 4 * gi);
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const int v = 4 * k + c;
            if constexpr (DBG) capture(i, v, a.dbg.s, (int)P[i][v]);
            const float f = g[i][gi] * P[i][v];  // an f16 times a small integer: hardly rounded
            z[i][t][v] = gi == 0 ? sc[c] * f : fmaf(sc[c], f, z[i][t][v]);
            if (gi == G - 1) y[i][t][v] += z[i][t][v];
            asm volatile("" : "+v"(z[i][t][v]));
          }
      }
    } else {
      if constexpr (DBG) {
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
          for (int v = 0; v < 16; ++v) capture(i, v, a.dbg.s, (int)P[i][v]);
      }
      if (!odd) {
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            z[i][t][v] = P[i][v];
            asm volatile("" : "+v"(z[i][t][v]));
          }
        return;
      }
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        const h8 sm = *(const h8 *)(cur + NP * PLANE + ADS + 1024 * t + 32 * l32 + 16 * hh);
        f32x16 M;
#pragma unroll
        for (int v = 0; v < 16; ++v) M[v] = 0.0f;
        M = __builtin_amdgcn_mfma_f32_32x32x16_f16(sm, mo[i], M, 0, 0, 0);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          float sc[4];
          *(float4 *)sc = *(const float4 *)(ads + 4 * (32 * t + 8 * k + 4 * hh));
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const int v = 4 * k + c;
            if constexpr (DBG) capture(i, v, a.dbg.m, (int)M[v]);
            const float x = fmaf(g[i][gi], z[i][t][v] + P[i][v], -(dm[i] * M[v]));
            y[i][t][v] = fmaf(sc[c], x, y[i][t][v]);
            asm volatile("" : "+v"(y[i][t][v]));
          }
        }
      }
    }
  };
  auto stage = [&](int st, const uint8_t *cur, uint8_t *next, bool odd) {
    __builtin_amdgcn_s_waitcnt(7 << 4);  // this wave's loads of the stage are in, its LDS reads of the last one done
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    if (st + 1 < nst) {
      load_x(next, st + 1);
      if constexpr (T == T_Q4_K) {
        uint32_t o = ssrc;
        const uint8_t *sb = (const uint8_t *)a.x.sums;
        if constexpr (MODE == 0) {
          asm volatile("" : "+v"(o));
        } else {  // contiguous rows: formed here
          const uint32_t l = lane_here(), t = 32 * (wave % NT) + (l >> 1), last = (uint32_t)(nbt - 1);
          o = (t < last ? t : last) * (uint32_t)a.x.sums_stride + 16 * (l & 1);
          sb += (p0 + tok0) * a.x.sums_stride;
        }
        if (!odd && wave < NT)
          lds_dma16(sb + 32 * (int64_t)(st >> 1) + o, next + NP * PLANE + ADS + wave * 1024);
      }
    }
    if constexpr (T == T_Q4_K && !INT) {  // y -= dmin * sum_j m_j S_j, once per superblock
      if (odd) {
#pragma unroll
        for (int i = 0; i < RT; ++i) {
          const h8 mo = mins_operand(raw[i].hd);
          const float dm = f16_bits_to_f32(raw[i].hd.x >> 16);
#pragma unroll
          for (int t = 0; t < NT; ++t) {
            const h8 sm = *(const h8 *)(cur + NP * PLANE + ADS + 1024 * t + 32 * l32 + 16 * hh);
            f32x16 M;
#pragma unroll
            for (int v = 0; v < 16; ++v) M[v] = 0.0f;
            M = __builtin_amdgcn_mfma_f32_32x32x16_f16(sm, mo, M, 0, 0, 0);
#pragma unroll
            for (int v = 0; v < 16; ++v) y[i][t][v] = fmaf(-dm, M[v], y[i][t][v]);
          }
        }
      }
    }
    h8 w[RT][8], mo[RT];
    float g[RT][G], dm[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      if constexpr (T == T_Q4_K && INT) {
        if (odd) {
          mo[i] = mins_operand(raw[i].hd);
          dm[i] = f16_bits_to_f32(raw[i].hd.x >> 16);
        }
      }
      if constexpr (T == T_Q6_K && INT) dm[i] = f16_bits_to_f32(raw[i].d);
      unpack<T, TILED, INT>(raw[i], st, nb, w[i], g[i]);
#pragma unroll
      for (int s = 0; s < 8; ++s) asm volatile("" : "+v"(w[i][s]));  // unpacked here, before raw is loaded again
    }
    auto next_weights = [&]() {
      if (st + 1 < nst) {
#pragma unroll
        for (int i = 0; i < RT; ++i) load_raw<T, TILED>(raw[i], wm[i], wr[i], nb, st + 1);
      }
    };
    if (T == T_Q4_K || NT == 1) next_weights();
    // The A pieces of a tile (16, INT 8) in reads of 4, each issued one read
    // ahead of its MFMAs. Q4_K: the small pieces of steps 0-3, 4-7, then the
    // large ones; Q8_0: a block's two steps, small then large; Q6_K: two groups
    // of one step, small then large; INT: steps 0-3, 4-7.
    constexpr int NR = INT ? 2 : 4;
    auto pl_of = [](int j, int u) {
      return INT ? 0 : T == T_Q4_K ? (j < 2 ? 1 : 0) : T == T_Q8_0 ? (u < 2 ? 1 : 0) : 1 - (u & 1);
    };
    auto st_of = [](int j, int u) {
      return INT ? 4 * j + u : T == T_Q4_K ? 4 * (j & 1) + u : T == T_Q8_0 ? 2 * j + (u & 1) : 2 * j + (u >> 1);
    };
    auto first_of = [&](int j, int u) { return INT ? (4 * j + u) % SPG == 0 : (T == T_Q4_K ? j + u : T == T_Q8_0 ? u : u & 1) == 0; };
    auto last_of = [&](int j, int u) {
      return INT ? (4 * j + u) % SPG == SPG - 1 : T == T_Q4_K ? j == 3 && u == 3 : T == T_Q8_0 ? u == 3 : (u & 1) == 1;
    };
    h8 x[2][4];
    auto read = [&](int t, int j) {
#pragma unroll
      for (int u = 0; u < 4; ++u)
        x[j & 1][u] = *(const h8 *)(cur + (aoff ^ (32 * st_of(j, u))) + pl_of(j, u) * PLANE + t * 8192);
    };
    read(0, 0);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      if (T != T_Q4_K && t == 1) next_weights();  // two tiles and these types' larger stage: registers
      if (t >= ntt) break;
      f32x16 P[RT];
      uint32_t lo2 = 0x0c000c00u;  // two f16 kLo, opaque per tile (products of both tiles' would be kept in registers)
      asm volatile("" : "+s"(lo2));
#pragma unroll
      for (int j = 0; j < NR; ++j) {
        if (j < NR - 1) read(t, j + 1);
        else if (t + 1 < NT) read(t + 1, 0);  // also past the last tile: any LDS bytes
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int s = st_of(j, u), gi = s / SPG;
          if (first_of(j, u)) {  // a group's first
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
              for (int v = 0; v < 16; ++v) P[i][v] = 0.0f;
          }
#pragma unroll
          for (int i = 0; i < RT; ++i) {
            h8 wv = w[i][s];
            // the lo pieces' unit: in the weights (still exact in f16), or Q4_K, whose
            // small products are all summed first, in their sum
            if constexpr (T != T_Q4_K) {
              if (!INT && pl_of(j, u) == 1) wv *= __builtin_bit_cast(h8, u32x4{lo2, lo2, lo2, lo2});
            }
            P[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[j & 1][u], wv, P[i], 0, 0, 0);
            if (!INT && T == T_Q4_K && j == 1 && u == 3) {
#pragma unroll
              for (int v = 0; v < 16; ++v) P[i][v] *= kLo;
            }
          }
          if (INT && last_of(j, u)) {
            int_epilogue(t, gi, P, cur, odd, st, g, mo, dm);
          } else if (last_of(j, u)) {  // its last
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
              for (int v = 0; v < 16; ++v) {
                y[i][t][v] = fmaf(g[i][gi], P[i][v], y[i][t][v]);
                asm volatile("" : "+v"(y[i][t][v]));  // here, not sunk past the next groups' products (their registers)
              }
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  for (int st = st_lo; st < nst; st += 2) {
    stage(st, st0, st1, false);
    if (st + 1 < nst) stage(st + 1, st1, st0, true);
    if constexpr (INT) {  // (see kIntChain)
      if ((st & (kIntChain<T> - 1)) == kIntChain<T> - 2 && st + 2 < nst) {
#pragma unroll
        for (int j = 0; j < 4 * RT * NT; ++j) {
          float *yv = &y[j / (4 * NT)][j / 4 % NT][4 * (j % 4)];
          float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
          if (st >= kIntChain<T>) v = yl[j][tid];
          yl[j][tid] = make_float4(v.x + yv[0], v.y + yv[1], v.z + yv[2], v.w + yv[3]);
          yv[0] = yv[1] = yv[2] = yv[3] = 0.0f;
        }
      }
    }
  }
  if constexpr (INT) {
    if (nst > kIntChain<T>) {
#pragma unroll
      for (int j = 0; j < 4 * RT * NT; ++j) {
        float *yv = &y[j / (4 * NT)][j / 4 % NT][4 * (j % 4)];
        const float4 v = yl[j][tid];
        yv[0] += v.x;
        yv[1] += v.y;
        yv[2] += v.z;
        yv[3] += v.w;
      }
    }
  }
#pragma unroll
  for (int t = 0; t < NT; ++t) {
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int tk = 32 * t + 8 * (v >> 2) + 4 * hh + (v & 3);
      if (tk >= nbt) continue;
      const int sh = INT ? 0 : -exs[tk];
      float *o = a.out + (p0 + tok0 + tk) * rows + (SPLIT ? (int64_t)blockIdx.y * a.split_stride : 0);
      if constexpr (SWIGLU) {  // g / (1 + exp(-g)) * u
        const int64_t r = rbase + l32;
        const float gv = INT ? y[0][t][v] : ldexpf(y[0][t][v], sh), uv = INT ? y[1][t][v] : ldexpf(y[1][t][v], sh);
        const float den = 1.0f + expf_cr(-gv);
        const float qv = gv / den;
        if (r < rows) o[r] = qv * uv;
      } else {
#pragma unroll
        for (int i = 0; i < RT; ++i) {
          const int64_t r = rbase + 32 * i + l32;
          if (r < rows) o[r] = INT ? y[i][t][v] : ldexpf(y[i][t][v], sh);
        }
      }
    }
  }
}

// out[p] = the column splits' sums of row p, in split order. idx (grouped rows):
// only rows of experts with at least min_rows rows.
__global__ void __launch_bounds__(256) k_split_sum(const float *__restrict__ part, int ks, int64_t stride, int64_t rows,
                                                   int64_t n4, float *__restrict__ out,
                                                   const uint32_t *__restrict__ idx, const uint32_t *__restrict__ perm,
                                                   const uint32_t *__restrict__ offsets, int min_rows) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n4) return;
  if (idx) {
    const uint32_t e = idx[perm[4 * i / rows]];
    if ((int)(offsets[e + 1] - offsets[e]) < min_rows) return;
  }
  float4 s = *(const float4 *)(part + 4 * i);
  for (int k = 1; k < ks; ++k) {
    const float4 v = *(const float4 *)(part + k * stride + 4 * i);
    s.x += v.x;
    s.y += v.y;
    s.z += v.z;
    s.w += v.w;
  }
  *(float4 *)(out + 4 * i) = s;
}

constexpr int64_t kSplitCols = 16384;  // the widest row k_split_f16 takes

}  // namespace

bool f16_gemm_supported(int type, int64_t rows, int64_t cols, int64_t n) {
  if (rows <= 0 || n <= 0 || cols <= 0 || cols > kSplitCols) return false;
  if (!(type == T_Q8_0 ? cols % 32 == 0 : (type == T_Q4_K || type == T_Q6_K) && cols % 256 == 0)) return false;
  // 32-bit offsets into the pieces and into one matrix, a 31-bit grid
  const int64_t lim = (int64_t)UINT32_MAX - 1024, kp = (cols + 127) / 128 * 128;
  const int64_t row_bytes = type == T_Q8_0 ? cols / 32 * 34 : cols / 256 * (type == T_Q4_K ? 144 : 210);
  return n <= lim / (4 * kp) && rows <= lim / row_bytes && 2 * n <= (INT32_MAX / 2) / ((rows + 127) / 128);
}

hipError_t launch_split_f16(hipStream_t st, const float *x, int64_t rows, int64_t cols, const F16Rows &o,
                            const Routing *rt, const uint32_t *idx, int min_rows) {
  if (cols <= 0 || cols > kSplitCols || cols % 32 || ((uintptr_t)x & 15u) || ((uintptr_t)o.planes & 15u))
    return hipErrorNotSupported;
  if (rows <= 0) return hipSuccess;
  if (rows > INT32_MAX) return hipErrorNotSupported;
  SplitArgs a{x, rows, cols, o, rt ? idx : nullptr, rt ? rt->perm : nullptr, rt ? rt->offsets : nullptr, min_rows};
  const dim3 g((unsigned)rows);
  // one wave holds rows of up to 2048 columns in registers, four waves wider ones
  if (cols <= 1024) KMOE_LAUNCH((k_split_f16<1, 2>), g, dim3(64), 0, st, a);
  else if (cols <= 2048) KMOE_LAUNCH((k_split_f16<1, 4>), g, dim3(64), 0, st, a);
  else if (cols <= 4096) KMOE_LAUNCH((k_split_f16<4, 2>), g, dim3(256), 0, st, a);
  else if (cols <= 8192) KMOE_LAUNCH((k_split_f16<4, 4>), g, dim3(256), 0, st, a);
  else KMOE_LAUNCH((k_split_f16<4, 8>), g, dim3(256), 0, st, a);
  return hipGetLastError();
}

namespace {

int num_cus() {
  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  return cus;
}

int64_t splits_for(int64_t total, int nst, int rt) {
  const int64_t ks = (rt == 1 ? 4 : 2) * (int64_t)num_cus() / (total > 0 ? total : 1);
  return ks < nst / 6 ? ks : nst / 6;
}

// Where the partial sums of a column split may go; grouped: all slots and their flat expert choice.
struct Split {
  float *part = nullptr;
  int64_t part_floats = 0, n_slots = 0;
  const uint32_t *idx = nullptr;
};

// blocks: an upper bound of the token blocks over all experts.
template <int T, int MODE, int RT, int NT, bool INT = false, bool DBG = false>
hipError_t launch_t(hipStream_t st, const F16Args &a, int64_t blocks, const Split &sp = {}) {
  constexpr int RPB = MODE == 0 || MODE == 3 ? 128 : 128 * RT;
  const int64_t total = blocks * ((a.rows + RPB - 1) / RPB);
  const unsigned grid = (unsigned)((total + 7) / 8 * 8);
  if constexpr (!INT && (MODE == 1 || MODE == 2)) {
    // A grid that leaves the chip idle splits the columns, at least six stages
    // (768 columns) to a work-group, over as many as fill it twice (one row
    // tile per wave: four times) and the partial sums' buffer holds. 4096x4096
    // by 16 rows: Q4_K 37 -> 17.5 us, Q6_K 66 -> 24, Q8_0 75 -> 26.
    const int nst = (int)((a.cols + 127) / 128);
    const int64_t stride = (MODE == 1 ? sp.n_slots : a.s_rows) * a.rows;
    int64_t ks = splits_for(total, nst, RT);
    if (ks * stride > sp.part_floats) ks = sp.part_floats / stride;
    if (ks >= 2 && a.rows % 4 == 0 && stride / 4 < (int64_t)INT32_MAX * 128) {
      F16Args b = a;
      b.split_stages = (int)((nst + ks - 1) / ks + 1) / 2 * 2;
      b.split_stride = stride;
      b.out = sp.part;
      ks = (nst + b.split_stages - 1) / b.split_stages;
      KMOE_LAUNCH((k_f16_gemm<T, MODE, RT, NT, false, false, true>), dim3(grid, (unsigned)ks), dim3(256), 0, st, b);
      hipLaunchKernelGGL(k_split_sum, dim3((unsigned)((stride / 4 + 255) / 256)), dim3(256), 0, st, sp.part, (int)ks,
                         stride, a.rows, stride / 4, a.out, MODE == 1 ? sp.idx : nullptr, a.rt.perm, a.rt.offsets,
                         a.min_rows);
      return hipGetLastError();
    }
  }
  KMOE_LAUNCH((k_f16_gemm<T, MODE, RT, NT, INT, DBG>), dim3(grid), dim3(256), 0, st, a);
  return hipGetLastError();
}

template <int T, bool INT = false, bool DBG = false>
hipError_t launch_grouped_t(hipStream_t st, int mode, const F16Args &a, int64_t n_slots, int max_active,
                            const Split &sp = {}) {
  const int64_t ne = n_slots / a.min_rows < max_active ? n_slots / a.min_rows : max_active;
  if (ne == 0) return hipSuccess;
  if constexpr (!INT) {  // few token blocks: one row tile per wave, columns split
    if (mode == 1 && (n_slots / 32 + ne) * ((a.rows + 255) / 256) < 2 * num_cus())
      return launch_t<T, 1, 1, 1>(st, a, n_slots / 32 + ne, sp);
  }
  const bool wide = n_slots > 32 * (int64_t)max_active;
  const int64_t blocks = n_slots / (wide ? 64 : 32) + ne;
  if constexpr (INT) {  // (two tiles)
    if (mode == 1 && wide) return launch_t<T, 1, 1, 2, INT, DBG>(st, a, blocks);
  }
  // one token tile: Q6_K's scale per 16 columns and the int8 rows' sums take the registers of two
  if constexpr (T == T_Q6_K || INT) {
    return mode == 0 ? launch_t<T, 0, 2, 1, INT, DBG>(st, a, n_slots / 32 + ne)
                     : launch_t<T, 1, 2, 1, INT, DBG>(st, a, n_slots / 32 + ne, sp);
  } else {
    // (Q8_0: two by two tiles spill 31 registers; DeepSeek-V2-Lite shape, 1777
    // tokens 1077 us per layer so, 1001 with one weight tile per wave)
    constexpr int RT = T == T_Q8_0 ? 1 : 2;
    if (wide) return mode == 0 ? launch_t<T, 0, 2, 2>(st, a, blocks) : launch_t<T, 1, RT, 2>(st, a, blocks, sp);
    return mode == 0 ? launch_t<T, 0, 2, 1>(st, a, blocks) : launch_t<T, 1, 2, 1>(st, a, blocks, sp);
  }
}

// Row tiles per wave, token tiles and token blocks of a plain product: the
// largest tile that still fills the chip (twice, where two tiles of tokens do).
struct PlainShape {
  int rt, nt;
  int64_t blocks;
};
PlainShape plain_shape(int type, int64_t rows, int64_t s_rows) {
  const int64_t cus = num_cus(), r2 = (rows + 255) / 256, n64 = (s_rows + 63) / 64, n32 = (s_rows + 31) / 32;
  if (type != T_Q6_K && r2 * n64 >= 2 * cus) return {type == T_Q8_0 ? 1 : 2, 2, n64};  // (Q8_0: as in an expert's down)
  return {r2 * n32 >= cus ? 2 : 1, 1, n32};
}

template <int T>
hipError_t launch_plain_t(hipStream_t st, const F16Args &a, const Split &sp) {
  const int64_t cus = num_cus();
  const int64_t n64 = (a.s_rows + 63) / 64, n32 = (a.s_rows + 31) / 32;
  if (a.pw2) {
    if constexpr (T == T_Q4_K) {
      const int64_t r = (a.rows + 127) / 128;
      if (r * n64 >= 2 * cus) return launch_t<T, 3, 2, 2>(st, a, n64);
      return launch_t<T, 3, 2, 1>(st, a, n32);
    } else {
      return hipErrorNotSupported;
    }
  }
  const PlainShape p = plain_shape(T, a.rows, a.s_rows);
  if constexpr (T != T_Q6_K) {
    if (p.nt == 2) return launch_t<T, 2, T == T_Q8_0 ? 1 : 2, 2>(st, a, p.blocks, sp);
  }
  if (p.rt == 2) return launch_t<T, 2, 2, 1>(st, a, p.blocks, sp);
  return launch_t<T, 2, 1, 1>(st, a, p.blocks, sp);
}

}  // namespace

int64_t f16_gemm_part_floats(int type, int64_t rows, int64_t cols, int64_t s_rows) {
  const PlainShape p = plain_shape(type, rows, s_rows);
  const int64_t ks = splits_for(p.blocks * ((rows + 128 * p.rt - 1) / (128 * p.rt)), (int)((cols + 127) / 128), p.rt);
  return ks > 1 && rows % 4 == 0 ? ks * s_rows * rows : 0;
}

hipError_t launch_f16_gemm(hipStream_t st, int mode, int type, const ExpertTier &tier, int64_t rows, int64_t cols,
                           const Routing &rt, int n_expert, int max_active, int64_t n_slots, int min_rows,
                           int max_rows, const F16Rows &x, float *out, float *part, int64_t part_floats,
                           const uint32_t *idx) {
  const Split sp{part, idx ? part_floats : 0, n_slots, idx};
  if (!f16_gemm_supported(type, rows, cols, n_slots) || min_rows < 1) return hipErrorNotSupported;
  if (max_active <= 0 || max_rows < min_rows) return hipSuccess;
  F16Args a{};
  a.tier = tier;
  a.rt = rt;
  a.rows = rows;
  a.cols = cols;
  a.x = x;
  a.out = out;
  a.min_rows = min_rows;
  a.max_rows = max_rows;
  a.n_expert = n_expert;
  switch (type) {
    case T_Q4_K: return launch_grouped_t<T_Q4_K>(st, mode, a, n_slots, max_active, sp);
    case T_Q6_K: return launch_grouped_t<T_Q6_K>(st, mode, a, n_slots, max_active, sp);
    default: return launch_grouped_t<T_Q8_0>(st, mode, a, n_slots, max_active, sp);
  }
}

hipError_t launch_f16_gemm_i8(hipStream_t st, int mode, int type, const ExpertTier &tier, int64_t rows, int64_t cols,
                              const Routing &rt, int n_expert, int max_active, int64_t n_rows, int64_t n_slots,
                              int min_rows, int max_rows, const int8_t *q, const float *ad, const int32_t *s16,
                              uint8_t *scratch, float *out, const BlockDbg *dbg) {
  if (!f16_gemm_supported(type, rows, cols, n_slots) || cols % 128 || min_rows < 1 || ((uintptr_t)q & 15u) ||
      ((uintptr_t)ad & 15u) || ((uintptr_t)scratch & 15u))
    return hipErrorNotSupported;
  if (max_active <= 0 || max_rows < min_rows) return hipSuccess;
  const int64_t n16 = n_rows * (cols / 16);
  F16Args a{};
  a.x.planes = (uint16_t *)scratch;
  a.x.sums = type == T_Q4_K ? (uint16_t *)(scratch + 2 * n_rows * cols) : nullptr;
  a.x.sums_stride = cols / 8;
  hipLaunchKernelGGL(k_i8_f16, dim3((unsigned)((n16 + 255) / 256)), dim3(256), 0, st, q, s16, n16, cols, a.x.planes,
                     a.x.sums, a.x.sums_stride);
  a.tier = tier;
  a.rt = rt;
  a.rows = rows;
  a.cols = cols;
  a.out = out;
  a.min_rows = min_rows;
  a.max_rows = max_rows;
  a.n_expert = n_expert;
  a.ad = ad;
  a.s16 = s16;
  if (dbg) {
    a.dbg = *dbg;
    switch (type) {
      case T_Q4_K: return launch_grouped_t<T_Q4_K, true, true>(st, mode, a, n_slots, max_active);
      case T_Q6_K: return launch_grouped_t<T_Q6_K, true, true>(st, mode, a, n_slots, max_active);
      default: return launch_grouped_t<T_Q8_0, true, true>(st, mode, a, n_slots, max_active);
    }
  }
  switch (type) {
    case T_Q4_K: return launch_grouped_t<T_Q4_K, true>(st, mode, a, n_slots, max_active);
    case T_Q6_K: return launch_grouped_t<T_Q6_K, true>(st, mode, a, n_slots, max_active);
    default: return launch_grouped_t<T_Q8_0, true>(st, mode, a, n_slots, max_active);
  }
}

hipError_t launch_f16_gemm_plain(hipStream_t st, int type, const uint8_t *w, int64_t rows, int64_t cols,
                                 const F16Rows &x, int64_t s_rows, float *out, const uint8_t *w_up, float *part,
                                 int64_t part_floats) {
  const Split sp{part, part_floats, s_rows, nullptr};
  const uintptr_t al = type == T_Q4_K ? 15u : 1u;
  if (!f16_gemm_supported(type, rows, cols, s_rows) || ((uintptr_t)w & al) || ((uintptr_t)w_up & al))
    return hipErrorNotSupported;
  F16Args a{};
  a.rows = rows;
  a.cols = cols;
  a.x = x;
  a.out = out;
  a.pw = w;
  a.pw2 = w_up;
  a.s_rows = s_rows;
  switch (type) {
    case T_Q4_K: return launch_plain_t<T_Q4_K>(st, a, sp);
    case T_Q6_K: return launch_plain_t<T_Q6_K>(st, a, sp);
    default: return launch_plain_t<T_Q8_0>(st, a, sp);
  }
}

}  // namespace kmoe
