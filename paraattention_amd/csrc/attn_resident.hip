// Attention of many query rows to keys that fit the LDS of one compute unit: cross-attention to a text prompt or to an
// image's tokens, short self-attention.  It takes up to 288 keys at head_dim 128, 256 with a bias; 576 and 512 at head_dim 64, where it is
// chosen up to 512.
//
// A workgroup copies all keys and values of one (batch, head) into LDS once and keeps them; its 8 wavefronts then take
// blocks of 32 query rows on their own: no barrier, no tile copies, and while one of a SIMD's two wavefronts changes
// blocks (output stores, the next block's Q) the other is somewhere else in its sweep.  The kernels that stream K and V
// through LDS pay a workgroup's ends (Q, first tiles, last stores, all wavefronts at once) around every 256 rows.
// Against them (attn_fwd_d128_pipe / _stream_kernel, attn_fwd_d64_pipe_kernel; device time per call, bf16):
//   2 x 24 heads x 7800 rows x 256 keys   96 -> 69 us                     40 x 32760 x 257       299 -> 226 us
//   the same, padding as a bias          101 -> 57 (with the far key      2 x 24 x 5598 x 77     69 -> 36
//     tiles computed too                 107 -> 69)                       24 x 257 x 257       13.3 -> 10.1
//   24 x 4000 x 256                       42 -> 22
//   head_dim 64: 2 x 40 x 31316 x 457    464 -> 379                       24 x 17776 x 226       60 -> 43
// What bounds it is the traffic of Q and the output together with the clock that leaves: without stores the first of these takes
// 60, without reading new Q 62, without both 53 us; touching the next block's Q a block ahead gains nothing.
#include "attn_resident.h"

#include "resident_plan.h"

#include <type_traits>

namespace pa {

namespace {

constexpr float LN2 = 0.6931471805599453f;
constexpr float LOG2E = 1.4426950408889634f;
constexpr float RESCALE_SLACK = 8.0f;            // as in the kernels that stream their keys
constexpr float NO_MAX = -3.402823466e38f;       // running maximum of a row before its first key that is not at -inf
constexpr int LDS_BYTES = 160 * 1024;

typedef __attribute__((address_space(3))) char lds_char;

// HALF: the last tile of 64 keys holds only 32 (not with a bias, whose last tiles come and go)
template <typename T, int D, bool BIAS, bool HALF>
__global__ __launch_bounds__(512, 1) void attn_fwd_resident_kernel(const ResidentCall p) {
  typedef typename T::vec8 vec8;
  constexpr int DC = D / 16, DB = D / 32, ROW = 2 * D;
  constexpr int CHUNKS = ROW / 16;       // 16-byte chunks of a row
  constexpr int RPC = 64 / CHUNKS;       // rows one copy instruction moves
  const float c = p.scale_log2;
  extern __shared__ __attribute__((aligned(1024))) char smem[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31;
  const int hh = lane >> 5;

  int wg = blockIdx.x;
  if (p.xcd_chunk > 0) wg = (wg & 7) * p.xcd_chunk + (wg >> 3);  // the workgroups of a head share an L2
  if (wg >= p.B * p.H * p.parts) return;
  const int bh = wg / p.parts, part = wg - bh * p.parts;
  const int batch = bh / p.H, head = bh - batch * p.H;
  const int u_end = (int)((int64_t)(part + 1) * p.n_units / p.parts), u_begin = (int)((int64_t)part * p.n_units / p.parts);
  int unit = u_begin + wave;

  const int n_full = p.n_full;                        // tiles of 64 keys
  const int nsub = 2 * n_full + (HALF ? 1 : 0);       // blocks of 32 keys
  char* const sK = smem;
  char* const sV = smem + nsub * (32 * ROW);
  char* const sO = smem + 2 * nsub * (32 * ROW);
  float* const sB = (float*)(smem + 2 * nsub * (32 * ROW) + 16384);  // BIAS: one value per key, divided by the scale

  uint32_t* const sM = (uint32_t*)(sB + 64 * n_full);          // BIAS: largest squared norm of a key

  // ---- all keys and values of this head, once; rows past the last key arrive as zeros ----------------------------
  {
    auto rsrc = [&](const void* base, uint32_t row_bytes) {
      const uint64_t a = (uint64_t)base;
      u32x4 r;
      r[0] = __builtin_amdgcn_readfirstlane((uint32_t)a);
      r[1] = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32) & 0xffffu);
      r[2] = __builtin_amdgcn_readfirstlane((uint32_t)(p.Skv - 1) * row_bytes + ROW);
      r[3] = 0x00020000u;
      return r;
    };
    const uint32_t ks_bytes = (uint32_t)(p.ks_s * 2), vs_bytes = (uint32_t)(p.vs_s * 2);
    const u32x4 krs = rsrc((const uint16_t*)p.k + batch * p.ks_b + head * p.ks_h, ks_bytes);
    const u32x4 vrs = rsrc((const uint16_t*)p.v + batch * p.vs_b + head * p.vs_h, vs_bytes);
    const int r0 = lane / CHUNKS, pc = lane % CHUNKS;
    const int row = RPC * wave + r0;  // + 8 RPC i: the swizzles below repeat every 16 rows
    const int k_chunk = pc ^ (D == 128 ? row & 15 : (row >> 1) & 7);
    const int v_chunk = pc ^ (4 * (D == 128 ? row & 3 : (row >> 1) & 1));
    const uint32_t k_off = row * ks_bytes + 16 * k_chunk, v_off = row * vs_bytes + 16 * v_chunk;
    const uint32_t lk = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_char*)sK + wave * 1024);
    const uint32_t lv = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_char*)sV + wave * 1024);
    for (int i = 0; 8 * RPC * i + RPC * wave < 32 * nsub; ++i) {
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                   :: "s"(__builtin_amdgcn_readfirstlane(lk + i * 8192)), "v"(k_off), "s"(krs),
                      "s"(__builtin_amdgcn_readfirstlane(8 * RPC * i * ks_bytes)) : "memory");
    }
    for (int i = 0; 8 * RPC * i + RPC * wave < 32 * nsub; ++i) {
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                   :: "s"(__builtin_amdgcn_readfirstlane(lv + i * 8192)), "v"(v_off), "s"(vrs),
                      "s"(__builtin_amdgcn_readfirstlane(8 * RPC * i * vs_bytes)) : "memory");
    }
  }

  // ---- Q of a block of rows (B operand of the first product) ------------------------------------------------------
  const uint16_t* const qbase = (const uint16_t*)p.q + batch * p.qs_b + head * p.qs_h + 8 * hh;
  vec8 qf[DC];
  auto load_q = [&](int u) __attribute__((always_inline)) {
    int r = 32 * u + l32;
    r = r < p.Sq ? r : p.Sq - 1;
    const uint16_t* qp = qbase + (int64_t)r * p.qs_s;
#pragma unroll
    for (int dc = 0; dc < DC; ++dc) qf[dc] = *(const vec8*)(qp + 16 * dc);
  };
  if (unit < u_end) load_q(unit);

  // BIAS: bit j of `biased`: some key of tile j has a bias other than 0.  n_near tiles remain when the last ones are left out
  // whose keys lie so far below the others (padding at -10000) that their probabilities are 0 to the last bit; a row
  // may leave them out if its squared norm is below q2_limit, see below.
  uint32_t biased = 0, q2_limit = 0;
  int n_near = n_full;
  if constexpr (BIAS) {
    if (tid == 0) *sM = 0;
    const float per_scale = 1.0f / (p.scale_log2 * LN2);  // bias / scale, so that (s + that) * c = s * c + bias * log2(e)
    const int64_t at = batch * p.ms_b + head * p.ms_h;
    for (int n = tid; n < 64 * (n_full); n += 512) {
      float b = 0.f;
      if (n < p.Skv) b = (p.bias_act ? T::lo(((const uint16_t*)p.bias)[at + n * p.ms_k]) : ((const float*)p.bias)[at + n * p.ms_k]) * per_scale;
      sB[n] = b;
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wavefront's copies have landed
  __syncthreads();
  if constexpr (BIAS) {
    float top = -INFINITY, far = -INFINITY;  // largest bias of all keys, and of those in the tiles left out
    auto tile_top = [&](int j) {
      float b = sB[64 * j + lane];
      if ((__float_as_uint(b) & 0x7fffffffu) > 0x7f800000u) b = INFINITY;  // a NaN is not far below anything
      if (64 * j + lane >= p.Skv) b = -INFINITY;
#pragma unroll
      for (int d = 32; d > 0; d >>= 1) b = fmaxf(b, __shfl_xor(b, d));
      return b;
    };
    for (int j = 0; j < n_full; ++j) {
      if (__any((__float_as_uint(sB[64 * j + lane]) << 1) != 0)) biased |= 1u << j;
    }
    // Finding the far tiles takes 2 us, which one pass of the 8 wavefronts does not earn back (24 heads x 257 rows, a third of the keys
    // padding: 512 keys, head_dim 64, 12.2 -> 9.8 us without (11.3 where they are streamed), 256 keys, head_dim 128, 11.0 -> 8.9).  Two
    // passes do: 120 heads x 1000 rows x 512 keys, head_dim 64, gain 1.27 with that padding on what streams them, 1.14 without padding.
    if (u_end - u_begin > 8) {
      for (int j = 0; j < n_full; ++j) top = fmaxf(top, tile_top(j));
      for (; n_near > 1; --n_near) {
        const float b = tile_top(n_near - 1);
        if (!(b * c + 256.f < top * c)) break;
        far = fmaxf(far, b);
      }
      n_near = __builtin_amdgcn_readfirstlane(n_near);
    }
    // A score lies within |q| |k| c of its bias.  With every |k|^2 <= k2 and |q| |k| c below half of what the far tiles lie
    // deeper (less 176: 2^-150 and below rounds to 0, the running maximum may trail the true one by RESCALE_SLACK, the rest covers
    // roundings), every probability of a far key is 0.  Squares are compared by their bits, where NaN and infinity are large.
    if (n_near < n_full) {
      uint32_t k2 = 0;
      for (int n = tid >> 1; n < 64 * n_full; n += 256) {
        float x = 0.f;
#pragma unroll
        for (int i = 0; i < CHUNKS / 2; ++i) {
          const u32x4 w = *(const u32x4*)(sK + n * ROW + 16 * (((i + (n & 7)) % (CHUNKS / 2)) + (CHUNKS / 2) * (tid & 1)));
#pragma unroll
          for (int e = 0; e < 4; ++e) x = T::dot2(w[e], w[e], x);
        }
        x += __shfl_xor(x, 1);
        k2 = max(k2, __float_as_uint(x));
        if (n >= 64 * n_near) {  // a far key's value that is no number makes one of 0 times it
          x = 0.f;
#pragma unroll
          for (int i = 0; i < CHUNKS / 2; ++i) {
            const u32x4 w = *(const u32x4*)(sV + n * ROW + 16 * (((i + (n & 7)) % (CHUNKS / 2)) + (CHUNKS / 2) * (tid & 1)));
#pragma unroll
            for (int e = 0; e < 4; ++e) x = T::dot2(w[e], w[e], x);
          }
          if (__float_as_uint(x) >= 0x7f800000u) k2 = 0x7f800000u;
        }
      }
#pragma unroll
      for (int d = 32; d > 0; d >>= 1) k2 = max(k2, (uint32_t)__shfl_xor((int)k2, d));
      if (lane == 0) atomicMax(sM, k2);
      __syncthreads();
      k2 = __builtin_amdgcn_readfirstlane(*sM);
      const float room = ((top - far) * c - 176.f) * 0.49f;
      // (k2 = 0: any finite q; the cap keeps q2_limit below infinity)
      const float lim = fminf(room * room, 1e30f) / fmaxf(__uint_as_float(k2 < 0x7f800000u ? k2 : 0x7f7fffffu) * c * c, 1e-6f);
      q2_limit = k2 < 0x7f800000u ? __float_as_uint(lim) : 0;
      q2_limit = __builtin_amdgcn_readfirstlane(q2_limit);
    }
  }
  if (unit >= u_end) return;  // (no barrier from here on)

  // ---- fragment reads: the layout of the kernels that stream their keys.  A lane's address is that of its first chunk
  // with the chunk's number flipped in (rows are aligned to their size): one register per tile instead of one per chunk
  const uint32_t kb0 = (uint32_t)(uintptr_t)(lds_char*)sK + l32 * ROW + 16 * (hh ^ (D == 128 ? l32 & 15 : (l32 >> 1) & 7));
  uint32_t vb0;
  {
    const int g16 = lane >> 4, lg = lane & 15, r = lg >> 2, cq = lg & 3, dhalf = g16 & 1;
    vb0 = (uint32_t)(uintptr_t)(lds_char*)sV + (4 * hh + r) * ROW + 16 * ((2 * dhalf + (cq >> 1)) ^ (4 * (D == 128 ? r : (r >> 1) & 1))) + 8 * (cq & 1);
  }
  typedef __attribute__((__vector_size__(4 * sizeof(short)))) short s16x4;
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
  typedef __attribute__((address_space(3))) vec8 lds_vec8;
  auto read_k = [&](uint32_t at, int t, int dc) __attribute__((always_inline)) -> vec8 {
    return *(const lds_vec8*)((lds_char*)(uintptr_t)(at ^ (32 * dc)) + t * 32 * ROW);
  };
  auto read_vt = [&](uint32_t at, int t, int c, int db) __attribute__((always_inline)) -> vec8 {
    lds_char* a = (lds_char*)(uintptr_t)(at ^ (64 * db)) + (32 * t + 16 * c) * ROW;
    s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(a));
    s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(a + 8 * ROW));
    typedef __attribute__((__vector_size__(8 * sizeof(short)))) short s16x8;
    s16x8 v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_bit_cast(vec8, v);
  };

  constexpr std::integral_constant<int, 0> none{};
  constexpr std::integral_constant<int, 1> one{};
  constexpr std::integral_constant<int, 2> two{};
  constexpr std::true_type yes{};
  constexpr std::false_type no{};
  floatx16 o[DB];
  floatx16 sn0, sn1;  // scores of the coming tile (keys 0..31, 32..63)
  float mx, m_run = 0.f, l_run = 0.f;
  vec8 f[8];
  floatx16 zero;
#pragma unroll
  for (int r = 0; r < 16; ++r) zero[r] = 0.f;

  auto across = [&](float x) {  // the other half of a query row lives in lane ^ 32
    auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
  };
  // biases, and -inf on the keys past the last one; SUB: blocks of 32 keys the tile has
  auto finish_scores = [&](auto SUB, int j) __attribute__((always_inline)) {
    constexpr int sub = decltype(SUB)::value;
    if constexpr (BIAS) {
      if ((biased >> j) & 1u) {
        const float* b = sB + 64 * j + 4 * hh;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          const floatx4 x = *(const floatx4*)(b + 8 * a);
#pragma unroll
          for (int i = 0; i < 4; ++i) sn0[4 * a + i] += x[i];
          if constexpr (sub == 2) {
            const floatx4 y = *(const floatx4*)(b + 32 + 8 * a);
#pragma unroll
            for (int i = 0; i < 4; ++i) sn1[4 * a + i] += y[i];
          }
        }
      }
    }
    const int valid = p.Skv - 64 * j;
    if (valid < 32 * sub) {
      int lim = valid - 4 * hh;
      asm volatile("" : "+v"(lim));  // (nor these masks)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        if (8 * (r >> 2) + (r & 3) >= lim) sn0[r] = -INFINITY;
        if (sub == 2 && 8 * (r >> 2) + (r & 3) + 32 >= lim) sn1[r] = -INFINITY;
      }
    }
  };

  // The softmax and second product of tile j (CUR blocks of 32 keys) and, in front of them, the scores of tile j + 1 (NXT
  // blocks; 0: the sweep ends here).  FIRST: nothing has been accumulated yet.
  auto step = [&](auto CUR, auto NXT, auto FIRST, int j) __attribute__((always_inline)) {
    constexpr int cur = decltype(CUR)::value, nxt = decltype(NXT)::value;
    constexpr bool first = decltype(FIRST)::value;
    constexpr int NA = nxt * DC, NB = cur * 2 * DB;
    // (the compiler must not work out the tiles' addresses and masks in front of the loop over blocks: it spills them there)
    asm volatile("" : "+s"(j));
    const uint32_t tKn = kb0 + (j + 1) * (64 * ROW), tV = vb0 + j * (64 * ROW);
    auto fetch = [&](int i) __attribute__((always_inline)) {
      if (i < NA) f[i & 7] = nxt == 2 ? read_k(tKn, i & 1, i >> 1) : read_k(tKn, 0, i);
      else if (i < NA + NB) f[i & 7] = read_vt(tV, (i - NA) / (2 * DB), (i - NA) / DB % 2, (i - NA) % DB);
    };
    floatx16 c0 = sn0, c1 = sn1;
#pragma unroll
    for (int i = 0; i < 8; ++i) fetch(i);
    if constexpr (first) {
      m_run = BIAS ? fmaxf(mx * c, NO_MAX) : mx * c;
      l_run = 0.f;
    } else {
      const float mx_s = mx * c;
      if (__any(mx_s > m_run + RESCALE_SLACK)) {
        const float m_new = fmaxf(m_run, mx_s);
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
        l_run *= alpha;
#pragma unroll
        for (int i = 0; i < DB; ++i)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[i][r] *= alpha;
        m_run = m_new;
      }
    }
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);

    uint32_t pk[16];
    float lsum = 0.f;
    float tf[2][2], te[2][2];
    constexpr int PAIRS = 8 * cur;
    auto expo_slot = [&](int n) __attribute__((always_inline)) {  // a score pair takes three consecutive slots
      if (n >= 2 && n < PAIRS + 2) {
        const int i = n - 2;
        lsum += te[i & 1][0] + te[i & 1][1];
        asm volatile("" : "+v"(lsum));  // holds the slot's arithmetic where the source puts it
        pk[i] = T::pack2(te[i & 1][0], te[i & 1][1]);
      }
      if (n >= 1 && n < PAIRS + 1) {
        const int i = n - 1;
        te[i & 1][0] = __builtin_amdgcn_exp2f(tf[i & 1][0]);
        te[i & 1][1] = __builtin_amdgcn_exp2f(tf[i & 1][1]);
      }
      if (n < PAIRS) {
        const floatx16& cs = n < 8 ? c0 : c1;
        tf[n & 1][0] = __builtin_fmaf(cs[2 * (n & 7)], c, -m_run);
        tf[n & 1][1] = __builtin_fmaf(cs[2 * (n & 7) + 1], c, -m_run);
      }
    };
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      if (nxt == 2 && (i & 1)) sn1 = T::mfma32(f[i & 7], qf[i >> 1], i < nxt ? zero : sn1);
      else sn0 = T::mfma32(f[i & 7], qf[nxt == 2 ? i >> 1 : i], i < nxt ? zero : sn0);
      fetch(i + 8);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (nxt > 0) finish_scores(std::integral_constant<int, nxt>{}, j + 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < 6; ++n) expo_slot(n);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
    __builtin_amdgcn_sched_barrier(0);
    float mxa = 0.f, mxb = 0.f;
    if constexpr (nxt > 0) mxa = sn0[0];
    if constexpr (nxt > 1) mxb = sn1[0];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int t = i / (2 * DB), cc = i / DB % 2, db = i % DB;
      const uint32_t* w = pk + 8 * t + 4 * cc;
      const u32x4 bw = {w[0], w[1], w[2], w[3]};
      const int at = NA + i;
      o[db] = T::mfma32(f[at & 7], __builtin_bit_cast(vec8, bw), first && i < DB ? zero : o[db]);
      fetch(at + 8);
      // four softmax slots under the MFMAs of every 16 keys: those of the next 16 are packed when they are reached
#pragma unroll
      for (int n = 6 + i * 4 / DB; n < 6 + (i + 1) * 4 / DB; ++n) expo_slot(n);
#pragma unroll
      for (int n = 1 + 15 * i / NB; n < 1 + 15 * (i + 1) / NB; ++n) {
        if constexpr (nxt > 0) mxa = fmaxf(mxa, sn0[n]);
        if constexpr (nxt > 1) mxb = fmaxf(mxb, sn1[n]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    l_run += lsum;
    if constexpr (nxt == 1) mx = across(mxa);
    if constexpr (nxt == 2) mx = across(fmaxf(mxa, mxb));
  };
  // the scores of the first tile, which is whole (past the last key: -inf)
  auto open = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 8; ++i) f[i] = read_k(kb0, i & 1, i >> 1);
    __builtin_amdgcn_s_setprio(0);
#pragma unroll
    for (int i = 0; i < 2 * DC; ++i) {
      if (i & 1) sn1 = T::mfma32(f[i & 7], qf[i >> 1], i < 2 ? zero : sn1);
      else sn0 = T::mfma32(f[i & 7], qf[i >> 1], i < 2 ? zero : sn0);
      if (i + 8 < 2 * DC) f[i & 7] = read_k(kb0, i & 1, (i + 8) >> 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    finish_scores(two, 0);
    float a = sn0[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) a = fmaxf(a, sn0[r]);
#pragma unroll
    for (int r = 0; r < 16; ++r) a = fmaxf(a, sn1[r]);
    mx = across(a);
  };

  char* const obase = (char*)((uint16_t*)p.out + batch * p.os_b + head * p.os_h);
  float* const lbase = p.lse ? p.lse + ((int64_t)batch * p.H + head) * p.Sq : nullptr;

  for (; unit < u_end; unit += 8) {
    int n = n_full;
    if constexpr (BIAS) {
      if (n_near < n_full) {
        float x = 0.f;
#pragma unroll
        for (int dc = 0; dc < DC; ++dc) {
          const u32x4 w = __builtin_bit_cast(u32x4, qf[dc]);
#pragma unroll
          for (int e = 0; e < 4; ++e) x = T::dot2(w[e], w[e], x);
        }
        auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
        x = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
        if (!__any(__float_as_uint(x) >= q2_limit)) n = n_near;
      }
    }
    open();
    if (n > 1) {
      step(two, two, yes, 0);
      for (int j = 1; j < n - 1; ++j) step(two, two, no, j);
      if constexpr (HALF) step(two, one, no, n - 1);
    } else if constexpr (HALF) {
      step(two, one, yes, 0);
    }
    // behind the last scores of this block its Q is done with: the next block's is sent for
    if (unit + 8 < u_end) load_q(unit + 8);
    if constexpr (HALF) {
      step(one, none, no, n);
    } else {
      if (n > 1) step(two, none, no, n - 1);
      else step(two, none, yes, 0);
    }
    // ---- output: through 2 KB of LDS, 16 rows x 128 bytes at a time, so that stores write whole lines.  (Stored from the accumulators,
    // 32 bytes of a row per instruction: 77 keys 36 -> 40 us, 257 keys 226 -> 239.  Past the caches: head_dim 64 46 -> 43, 4000
    // rows 24 -> 22, 77 keys 35 -> 36.)
    float l_tot;
    {
      auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(l_run), __float_as_uint(l_run), false, false);
      l_tot = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
    }
    const float inv = l_tot > 0.f ? 1.0f / l_tot : 0.f;
    int ln = lane;
    asm volatile("" : "+v"(ln));  // (addresses worked out here, not in front of the loop)
    const int m16 = ln & 15, rr = ln >> 3, cc8 = ln & 7, h2 = ln >> 5, hm = (ln >> 4) & 1;
    char* const stage = sO + wave * 2048;
#pragma unroll
    for (int ch = 0; ch < DB / 2; ++ch) {
      u32x4 w[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const floatx16& x = o[2 * ch + (k >> 1)];
        const int a = 2 * (k & 1);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const uint32_t x0 = T::pack2(x[4 * a + 2 * i] * inv, x[4 * a + 2 * i + 1] * inv);
          const uint32_t x1 = T::pack2(x[4 * a + 4 + 2 * i] * inv, x[4 * a + 5 + 2 * i] * inv);
          auto sw = __builtin_amdgcn_permlane32_swap(x0, x1, false, false);
          w[k][i] = sw[0];
          w[k][2 + i] = sw[1];
        }
      }
#pragma unroll
      for (int rh = 0; rh < 2; ++rh) {
        if (hm == rh) {
#pragma unroll
          for (int k = 0; k < 4; ++k) *(u32x4*)(stage + m16 * 128 + 16 * ((2 * k + h2) ^ ((m16 >> 1) & 7))) = w[k];
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int r = 8 * i + rr;
          const u32x4 w = *(const u32x4*)(stage + r * 128 + 16 * (cc8 ^ ((r >> 1) & 7)));
          const int orow = 32 * unit + 16 * rh + r;
          char* const op = obase + (int64_t)orow * p.os_s * 2 + 16 * cc8;
          if (orow < p.Sq) __builtin_nontemporal_store(w, (u32x4*)(op + 128 * ch));
        }
        __builtin_amdgcn_wave_barrier();
      }
    }
    const int row = 32 * unit + l32;
    if (lbase != nullptr && hh == 0 && row < p.Sq) lbase[row] = l_tot > 0.f ? (m_run + __builtin_amdgcn_logf(l_tot)) * LN2 : -INFINITY;
  }
}

// blocks of 32 keys held: the first tile of 64 is always whole, with a bias all are
int key_blocks(int Skv, bool bias) { return Skv <= 32 || bias ? 2 * ((Skv + 63) / 64) : (Skv + 31) / 32; }
size_t lds_bytes(int D, int Skv, bool bias) {
  const size_t nsub = (size_t)key_blocks(Skv, bias);
  return nsub * 32 * 2 * D * 2 + 16384 + (bias ? nsub * 32 * sizeof(float) + 16 : 0);
}

template <typename T, int D, bool BIAS, bool HALF>
int launch(const ResidentCall& c, hipStream_t stream) {
  const size_t smem = lds_bytes(D, c.Skv, BIAS);
  static bool attr_done[PA_MAX_DEVICES] = {};  // benign race: the call is idempotent
  const int dev = current_device();
  if (dev < 0 || !attr_done[dev]) {
    hipError_t e = hipFuncSetAttribute((const void*)attn_fwd_resident_kernel<T, D, BIAS, HALF>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES);
    if (e != hipSuccess) PA_FAIL(PA_ERR_LAUNCH, "hipFuncSetAttribute: %s", hipGetErrorString(e));
    if (dev >= 0) attr_done[dev] = true;
  }
  const int64_t n = c.xcd_chunk > 0 ? 8 * (int64_t)c.xcd_chunk : (int64_t)c.B * c.H * c.parts;
  hipLaunchKernelGGL((attn_fwd_resident_kernel<T, D, BIAS, HALF>), dim3((unsigned)n), dim3(512), smem, stream, c);
  PA_CHECK_LAUNCH("attention kernel (resident keys)");
  return PA_OK;
}

template <typename T, int D>
int launch_form(const ResidentCall& c, hipStream_t stream) {
  if (c.bias != nullptr) return launch<T, D, true, false>(c, stream);
  return key_blocks(c.Skv, false) & 1 ? launch<T, D, false, true>(c, stream) : launch<T, D, false, false>(c, stream);
}

}  // namespace

bool resident_takes(ResidentCall& c, int D, int want) {
  if (want == 0 || (D != 128 && D != 64) || c.Skv <= 0 || c.Sq <= 0 || c.B <= 0 || c.H <= 0) return false;
  if (c.Skv > 1024 || lds_bytes(D, c.Skv, c.bias != nullptr) > (size_t)LDS_BYTES) return false;
  // 32-bit offsets of the copies (rows past the last key included)
  if ((uint64_t)(c.Skv + 64) * (uint64_t)c.ks_s * 2 + 256 > 0xfffff000u || (uint64_t)(c.Skv + 64) * (uint64_t)c.vs_s * 2 + 256 > 0xfffff000u) return false;
  const int cus = device_cus();
  if (cus <= 0) return false;
  const int64_t heads = (int64_t)c.B * c.H;
  c.n_units = (c.Sq + 31) / 32;
  c.n_full = key_blocks(c.Skv, c.bias != nullptr) / 2;
  if (heads * c.n_units > 0x7fffffff || heads * ((c.n_units + 3) / 4) > 0x3fffffff) return false;
  if (want < 0) {
    // Copying all keys in before the first product must pay.  Each line lies between the points measured on its sides (before -> with
    // this kernel, inputs that change from call to call); with everything in the caches this kernel still gains 1.05 .. 1.4 beyond some
    // of them (300 x 128 x 64, head_dim 64, 7.4 -> 6.7; 224 x 4000 x 400 146 -> 126; 520 x 300 x 288, head_dim 128, 84 -> 57).
    // Where the other kernel is one with a workgroup per query tile that streams the keys:
    // - one tile of 128 rows, and the LDS of all heads together (keys, values and 16 KB of staging each) above 8 MB: head_dim 64, 512 keys,
    //   80 heads 11.7 -> 12.5 us, 24 heads (3.5 MB) 10.5 -> 9.8
    // - up to 512 rows and more heads than compute units: 300 x 128 x 512 16.2 -> 23.0, 300 x 256 x 226 17.5 -> 19.6
    // - head_dim 64 and more than 384 keys, from five eighths as many heads as compute units on: 257 x 2000 x 512 112 -> 119, 40 x 32760 x 512
    //   248 -> 219, 2 x 40 x 31316 x 457 464 -> 379
    // Where it is the one with resident workgroups (head_dim 128, no bias):
    // - its pieces of 256 rows make whole rounds (it cuts the last round otherwise, which costs it 20 us: 510 x 256 x 128 63 -> 31) and are more
    //   than half full, up to two of them per head and more heads than compute units: 512 x 256 x 128 25.2 -> 30.6, 768 x 150 x 230 41.8 -> 49.8,
    //   384 x 440 x 230 42.6 -> 46.7, 640 x 500 x 128 50.0 -> 55.8.  Not with up to 96 keys (384 x 440 x 77 31.4 -> 29.8), nor half-full ones
    //   (512 x 300 rows), nor two each of whole rounds of heads beyond 192 keys (768 x 440 x 230 83.8 -> 79.8)
    const bool tiled = D == 64 || c.bias != nullptr;
    if (tiled && c.n_units <= 4 && heads * (double)lds_bytes(D, c.Skv, false) > 8.0e6) return false;
    if (heads > cus && c.n_units <= 16) {
      if (tiled) return false;
      const bool whole = heads * ((c.n_units + 7) / 8) % cus == 0, filled = (c.n_units - 1) % 8 >= 4;
      if (whole && filled && c.Skv > 96 && (c.n_units <= 8 || heads % cus != 0 || c.Skv <= 192)) return false;
    }
    if (D == 64 && (c.Skv > 512 || (c.Skv > 384 && 8 * heads > 5 * cus))) return false;
  }
  return true;
}

bool plan_resident(ResidentCall& c, int D, int want) {
  if (!resident_takes(c, D, want)) return false;
  const int cus = device_cus();
  const int64_t heads = (int64_t)c.B * c.H;
  c.parts = resident_parts(heads, c.n_units, cus);
  c.xcd_chunk = cus == 256 ? (int)((heads * c.parts + 7) / 8) : 0;
  return true;
}

int launch_resident(const ResidentCall& c, int dtype, int D, hipStream_t stream) {
  if (c.out == nullptr) PA_FAIL(PA_ERR_INVALID, "null output pointer");
  if (dtype == PA_DTYPE_BF16) return D == 128 ? launch_form<BF16, 128>(c, stream) : launch_form<BF16, 64>(c, stream);
  return D == 128 ? launch_form<F16, 128>(c, stream) : launch_form<F16, 64>(c, stream);
}

}  // namespace pa
