// Role-masked prefill of a short prompt from an empty cache (bf16, head dims 32, 64 and 128) in one launch.
//
// A short prompt is bound by the chain of launches and of trips to memory behind each other, not by any rate: the key-limit
// kernel, then a workgroup that reads tile summaries, builds its list, fetches Q and its first tiles and walks them, one
// workgroup for four q heads and 64 queries.  Here a workgroup owns 32 query rows of ONE q head, so that even 173 tokens
// give the device 192 workgroups, and its four wavefronts deal the 32-key tiles among themselves, each with its own O, row
// maxima and row sums, which meet in LDS at the end.  Every wavefront requests Q and one of the four newest tiles before it
// knows the roles (the newest tile is always visible, the others mostly); the row limits come from the roles themselves
// while those requests travel.
//
//   S^T = K Q^T   on v_mfma_f32_32x32x16_bf16, K straight from global memory in A-operand form, Q in B-operand form
//   O^T = V^T P^T V through LDS (global_load_lds, wave-private double buffer, no barrier), transposed by
//                 ds_read_b64_tr_b16; the probabilities leave the softmax in B-operand form
//
// Mask semantics and limits are those of key_lim_kernel for a prefill from empty (components/masks/utils.py:85-94,
// components/cache/nats_chunk_layer_cache.py:603-616).
// Measured (32 / 8 heads of 128, chunk 64, attention call with its key limits): 40 / 173 / 512 tokens 11.3 -> 5.8, 14.6 -> 8.0, 28.4 -> 15.4
// us; what is left is the launch, one trip to memory for Q, K and V, a tile or four per wavefront, and the merge.
#include <stdlib.h>

#include "nats_prefill.h"

namespace nats {

constexpr int kShortRows = 32;   // query rows of a workgroup, keys of a tile
constexpr int kShortWaves = 4;
constexpr int kShortMaxLen = 2048;  // (64 tiles: one bit each)

struct ShortArgs {
  const void *q, *k, *v;
  const uint8_t* roles;  // [B * Hkv, S]
  void* o;
  int64_t qs_b, qs_h, qs_l, ks_b, ks_h, ks_l, vs_b, vs_h, vs_l, os_b, os_h, os_l;
  int B, Hq, Hkv, n_rep, L, S, C, wc;  // wc = W / C
  float scale;
};

template <int D>
struct ShortSmem {
  static constexpr int kOPitch = D + 4;  // floats per query row of a wavefront's partial result
  int lim[kShortMaxLen];                 // last query token that sees the row
  uint64_t globals[kShortMaxLen / kWave];
  float m[kShortWaves][kShortRows], l[kShortWaves][kShortRows];
  union {
    uint16_t v[kShortWaves][2][kShortRows * D];
    float o[kShortWaves][kShortRows * kOPitch];
  };
};

template <int D>
__global__ __launch_bounds__(kShortWaves * kWave, 2) void prefill_short_kernel(ShortArgs a) {
  constexpr int OCT = D / 8;       // 16-byte chunks per row
  constexpr int DSTEPS = D / 16;
  constexpr int DT = D / 32;
  constexpr int NDMA = kShortRows * OCT / kWave;  // 1 KiB transfers per V tile
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  ShortSmem<D>& sm = *reinterpret_cast<ShortSmem<D>*>(smem_raw);

  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hl = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // kv streams change fastest (with eight of them a stream's workgroups share an XCD), late blocks come first
  const int n_streams = a.B * a.Hkv;
  const int stream = blockIdx.x % n_streams;
  const int rest = blockIdx.x / n_streams;
  const int rep = rest % a.n_rep;
  const int t_last = (a.L - 1) / kShortRows - rest / a.n_rep;  // block of query rows = its newest key tile
  const int b = stream / a.Hkv, hkv = stream % a.Hkv, hq = hkv * a.n_rep + rep;
  const uint16_t* qp = static_cast<const uint16_t*>(a.q) + b * a.qs_b + hq * a.qs_h;
  const uint16_t* kp = static_cast<const uint16_t*>(a.k) + b * a.ks_b + hkv * a.ks_h;
  const uint16_t* vp = static_cast<const uint16_t*>(a.v) + b * a.vs_b + hkv * a.vs_h;
  const uint8_t* roles = a.roles + (int64_t)stream * a.S;
  const int q0 = t_last * kShortRows, rlast = min(q0 + kShortRows, a.L) - 1;
  const int qtok = q0 + l32;
  const float c = a.scale * 1.4426950408889634f;

  auto v_swizzle = [](int row) { return OCT >= 16 ? (row & 3) << 2 : OCT >= 8 ? ((row >> 1) & 1) << 2 : 0; };
  bf16x8 kreg[DSTEPS];
  // (rows past the end repeat the last one: they are later than every query, which masks them)
  auto load_k = [&](int t) {
    const uint16_t* rp = kp + (int64_t)min(t * kShortRows + l32, a.L - 1) * a.ks_l + hl * 8;
#pragma unroll
    for (int s = 0; s < DSTEPS; ++s) kreg[s] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(rp + s * 16));
  };
  // (From assembly, with one buffer per tile: the builtin's transfers were waited for, next tile's and all, before this tile's first V
  // fragment.  32 / 8 heads of 128, 1000 / 1700 tokens 27.4 / 30.1 -> 25.7 / 28.5 us, even roles 39.7 -> 36.8; 8 heads of 64 13.2 / 17.4 ->
  // 12.1 / 16.0.)
  const uint32_t v_lds = lds_address(&sm.v[wave][0][0]);
  auto load_v = [&](int t, int buf) {
    const int row0 = t * kShortRows;
    const RowBuffer rows(vp + (int64_t)row0 * a.vs_l, (uint32_t)((min(kShortRows, a.L - row0) - 1) * (int)a.vs_l + D) * 2);  // (rows past the end are zeros)
    int ln = lane;
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+v"(ln));
#endif
    const int row = ln / OCT, chunk = (ln % OCT) ^ v_swizzle(ln / OCT);
#pragma unroll
    for (int j = 0; j < NDMA; ++j) {
      constexpr int kRows = kWave / OCT;  // of one transfer
      // (the permutation of the rows repeats within a transfer, or the lane's own row says)
      const int c = kRows % 4 == 0 ? chunk : (ln % OCT) ^ v_swizzle(j * kRows + row);
      rows.template to_lds<16>(v_lds + (buf * kShortRows * D + j * kWave * 8) * 2, (row * (int)a.vs_l + c * 8) * 2, (uint32_t)(j * kRows * (int)a.vs_l * 2));
    }
  };

  // ---- requests: roles, Q, this wavefront's guess of a tile ----
  uint8_t role[kShortMaxLen / (kShortWaves * kWave)];
#pragma unroll
  for (int j = 0; j < kShortMaxLen / (kShortWaves * kWave); ++j) {
    const int s = j * kShortWaves * kWave + tid;
    role[j] = s < a.S ? roles[s] : uint8_t(NATS_ROLE_SW);
  }
  bf16x8 qreg[DSTEPS];
  {
    const uint16_t* rp = qp + (int64_t)min(qtok, a.L - 1) * a.qs_l + hl * 8;
#pragma unroll
    for (int s = 0; s < DSTEPS; ++s) qreg[s] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(rp + s * 16));
  }
  int t = t_last - wave;
  if (t >= 0) {
    load_k(t);
    load_v(t, 0);
  }

  // ---- row limits ----
  // (a local slot is visible up to the first global slot at or after it, which may lie behind this workgroup's keys)
#pragma unroll
  for (int j = 0; j < kShortMaxLen / (kShortWaves * kWave); ++j) {
    const int s = j * kShortWaves * kWave + tid;
    const uint64_t bits = __ballot(s < a.S && (role[j] == NATS_ROLE_GLOBAL || s == a.S - 1));
    if (lane == 0) sm.globals[s / kWave] = bits;
  }
  __syncthreads();
  for (int row = tid; row < (t_last + 1) * kShortRows; row += kShortWaves * kWave) {
    const int s = min(row, a.L - 1) / a.C;
    const uint8_t r = roles[s];
    int lim = kLimGlobal;
    if (r != NATS_ROLE_GLOBAL) {
      int last = s + a.wc;  // last query slot
      if (r != NATS_ROLE_SW) {
        int blk = s / kWave;
        uint64_t bits = sm.globals[blk] >> (s % kWave) << (s % kWave);
        while (bits == 0) bits = sm.globals[++blk];  // (slot S - 1 counts as global: there is one)
        last = blk * kWave + __builtin_ctzll(bits);
      }
      lim = (int)min((int64_t)kLimGlobal, ((int64_t)last + 1) * a.C - 1);
    }
    sm.lim[row] = row < a.L ? lim : -1;
  }
  __syncthreads();

  // ---- which tiles: the four newest are dealt already, the visible ones before them go round the wavefronts ----
  uint64_t mine = 0, mixed = 0;  // bit = tile
  int turn = 0;
  for (int p = 0; p <= t_last; p += 2) {
    const int row = p * kShortRows + lane;  // (row < kShortMaxLen: pairs of the at most 64 tiles)
    const int lim = p + hl <= t_last ? sm.lim[row] : -1;
    const uint64_t vis = __ballot(lim >= q0), part = __ballot(lim < rlast);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int tt = p + h;
      const bool seen = (uint32_t)(vis >> (32 * h)) != 0;
      if ((uint32_t)(part >> (32 * h)) != 0 || tt == t_last) mixed |= uint64_t(1) << tt;
      if (!seen || tt > t_last) continue;
      const int owner = tt > t_last - kShortWaves ? t_last - tt : turn++ & (kShortWaves - 1);
      if (owner == wave) mine |= uint64_t(1) << tt;
    }
  }

  f32x16 oacc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) oacc[dt][i] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;
  const int r16 = lane & 15, dsel = (lane >> 4) & 1;
  auto v_frag = [&](const uint16_t* Vt, int kt, int dt) {
    const int chunk0 = dt * 4 + dsel * 2 + ((r16 & 3) >> 1);
    const int half4 = (r16 & 1) * 4;
    const int row_lo = kt * 16 + hl * 4 + (r16 >> 2), row_hi = row_lo + 8;
    const uint16_t* pl = Vt + row_lo * D + ((chunk0 ^ v_swizzle(row_lo)) * 8) + half4;
    const uint16_t* ph = Vt + row_hi * D + ((chunk0 ^ v_swizzle(row_hi)) * 8) + half4;
    bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((bf16x4 __attribute__((address_space(3)))*)pl);
    bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((bf16x4 __attribute__((address_space(3)))*)ph);
    return bf16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  };

  int cur = 0;
  if (t < 0 || !((mine >> t) & 1)) {  // the guess is not visible (or there is no such tile): on to the next one
    t = mine ? 63 - __builtin_clzll(mine) : -1;
    if (t >= 0) {
      load_k(t);
      load_v(t, 1);  // (the guess may still be on its way to the other buffer)
      cur = 1;
    }
  }
  while (t >= 0) {
    mine &= ~(uint64_t(1) << t);
    const int t_next = mine ? 63 - __builtin_clzll(mine) : -1;
    wait_transfers();  // K in registers, V in LDS
    f32x16 s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.f;
#pragma unroll
    for (int i = 0; i < DSTEPS; ++i) s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kreg[i], qreg[i], s, 0, 0, 0);
    if (t_next >= 0) {
      load_k(t_next);
      load_v(t_next, cur ^ 1);
    }
    // (the scale first: it may be 0 or negative)
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] *= c;
    if ((mixed >> t) & 1) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int key0 = t * kShortRows + 8 * g + 4 * hl;
        const int4 l4 = *reinterpret_cast<const int4*>(&sm.lim[key0]);
        const int lv[4] = {l4.x, l4.y, l4.z, l4.w};
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (!(key0 + e <= qtok && qtok <= lv[e])) s[g * 4 + e] = -INFINITY;
      }
    }
    float mx = s[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) mx = fmaxf(mx, s[i]);
    {
      auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
      mx = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    }
    if (__ballot(mx > m_run)) {
      const float m_new = fmaxf(m_run, mx);
      const float alpha = m_run == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run - m_new);
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) oacc[dt][i] *= alpha;
    }
    const float m_use = m_run == -INFINITY ? 0.f : m_run;
    bf16x8 pb[2];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float p = __builtin_amdgcn_exp2f(s[i] - m_use);
      l_run += p;
      pb[i >> 3][i & 7] = (__bf16)p;
    }
    const uint16_t* Vt = sm.v[wave][cur];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
        oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v_frag(Vt, kt, dt), pb[kt], oacc[dt], 0, 0, 0);
    t = t_next;
    cur ^= 1;
  }

  // ---- combine the wavefronts ----
  {
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(l_run), __float_as_uint(l_run), false, false);
    l_run = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
  wait_transfers();  // (a guess that was dropped has arrived: its buffer is about to be reused)
  if (hl == 0) sm.m[wave][l32] = m_run;
  __syncthreads();
  float m_all = sm.m[0][l32];
#pragma unroll
  for (int w = 1; w < kShortWaves; ++w) m_all = fmaxf(m_all, sm.m[w][l32]);
  const float f = m_run == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run - m_all);
  if (hl == 0) sm.l[wave][l32] = l_run * f;
  // accumulator i of block dt: head dimension dt * 32 + 8 * (i / 4) + 4 * hl + i % 4 of query l32
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<f32x4*>(&sm.o[wave][l32 * ShortSmem<D>::kOPitch + dt * 32 + 8 * g + 4 * hl]) =
          f32x4{oacc[dt][g * 4] * f, oacc[dt][g * 4 + 1] * f, oacc[dt][g * 4 + 2] * f, oacc[dt][g * 4 + 3] * f};
  __syncthreads();
  uint16_t* op = static_cast<uint16_t*>(a.o) + b * a.os_b + hq * a.os_h;
#pragma unroll
  for (int i = tid; i < kShortRows * OCT; i += kShortWaves * kWave) {
    const int row = i / OCT, piece = i % OCT;
    if (q0 + row >= a.L) continue;
    float l = 0.f;
    f32x4 lo = {0.f, 0.f, 0.f, 0.f}, hi = lo;
#pragma unroll
    for (int w = 0; w < kShortWaves; ++w) {
      const float* src = &sm.o[w][row * ShortSmem<D>::kOPitch + piece * 8];
      lo += *reinterpret_cast<const f32x4*>(src);
      hi += *reinterpret_cast<const f32x4*>(src + 4);
      l += sm.l[w][row];
    }
    const float inv = 1.f / l;
    const bf16x8 ob = {(__bf16)(lo[0] * inv), (__bf16)(lo[1] * inv), (__bf16)(lo[2] * inv), (__bf16)(lo[3] * inv),
                       (__bf16)(hi[0] * inv), (__bf16)(hi[1] * inv), (__bf16)(hi[2] * inv), (__bf16)(hi[3] * inv)};
    *reinterpret_cast<uint4*>(op + (int64_t)(q0 + row) * a.os_l + piece * 8) = __builtin_bit_cast(uint4, ob);
  }
}

// Where this kernel is the faster one (GPU time of the attention call with its key-limit launch, us, the other kernels / here):
//   * while its workgroups are about one round of the device: two per compute unit at head dim 128 (77 KB of LDS each), four
//     below.  32 / 8 heads of 128: 40 / 173 / 512 tokens 11.2 / 5.8, 14.7 / 8.0, 22.4 / 15.4, beyond that (700, 1024) 22.4 / 23.6,
//     24.4 / 31.2; batch 4, 128 / 173 tokens 13.3 / 9.3, 15.2 / 16.1.  8 heads of 64: 2048 tokens 29.4 / 16.8, batch 2 of them 31.8 /
//     29.3; 32 heads of 64, 1024 tokens 28.0 / 22.0, 1280 28.5 / 27.6.
//   * at head dim 64 (44 KB: three fit) and with groups of four q heads, which share a workgroup of the other kernel, fewer the longer
//     the prompt: four up to 768 tokens (300 tokens, 832 / 1024 workgroups 1.2 to 2.0 / 0.97 to 1.5 times its speed), three and a half up
//     to 1024 (850 tokens, 864 workgroups 1.06 to 1.44; 940, 960 0.86 to 1.09, chunk 1 1.22 and 1.09 to 1024 tokens: four there), three
//     beyond: 16 / 4 heads, 1536 / 1792 / 2048 tokens 19.5 / 17.3, 21.8 / 22.7, 22.6 / 29.6 (chunk 16: 21.3 / 18.0, 19.4 / 21.6,
//     19.7 / 27.8; chunk 1: 29.0 / 29.2, 33.5 / 29.7, 38.3 / 30.2).
//   * chunks of one to three tokens, whose old rows the other kernel gathers one by one: up to 1792 tokens.  Chunk 1, 1024 / 1536 /
//     1792 / 2048 tokens: 8 heads of 128 38.2 / 24.0, 38.0 / 35.6, 39.9 / 38.5, 40.3 / 44.9; 8 heads of 64 33.3 / 19.6, 33.6 / 26.1,
//     31.1 / 29.4, 31.7 / 33.4.  (Chunk 4, 2048 tokens: 41.2 / 30.8, 31.9 / 23.2; chunk 8 41.6 / 28.2, 32.1 / 21.3.)
// (NATS_PREFILL_SHORT=0 in the environment: nowhere, for comparison.)
bool prefill_short_takes(int64_t B, int64_t H_q, int64_t H_kv, int64_t D, int64_t L, int64_t C, int dtype) {
  if (dtype != NATS_DTYPE_BF16 || (D != 32 && D != 64 && D != 128) || L > kShortMaxLen) return false;
  if (const char* e = getenv("NATS_PREFILL_SHORT"); e && e[0] == '0') return false;
  if (C < 4 && D >= 64 && L > 1792) return false;
  const int64_t n_wg = B * H_q * ((L + kShortRows - 1) / kShortRows);
  const int64_t n_cu = device_cu_count();
  int64_t halves = D == 128 ? 4 : 8;  // of n_cu workgroups
  if (D == 64 && H_q / H_kv % 4 == 0 && L > (C < 4 ? 1024 : 768)) halves = L <= 1024 ? 7 : 6;
  return 2 * n_wg <= halves * n_cu;
}

template <int D>
static int launch_d(const ShortArgs& a, hipStream_t st) {
  constexpr int kMaxDev = 64;
  static bool configured[kMaxDev] = {};  // the LDS attribute is set once per device
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDev) return fail(NATS_ERR_LAUNCH, "prefill: no current device");
  if (!configured[dev]) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&prefill_short_kernel<D>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)sizeof(ShortSmem<D>));
    if (e != hipSuccess) return fail(NATS_ERR_LAUNCH, "prefill_short_kernel: LDS: %s", hipGetErrorString(e));
    configured[dev] = true;
  }
  const int64_t n_wg = (int64_t)a.B * a.Hq * ((a.L + kShortRows - 1) / kShortRows);
  hipLaunchKernelGGL((prefill_short_kernel<D>), dim3((unsigned)n_wg), dim3(kShortWaves * kWave), sizeof(ShortSmem<D>), st, a);
  NATS_CHECK_LAUNCH("prefill_short_kernel");
  return NATS_OK;
}

int launch_prefill_short(const void* q, const void* k, const void* v, const uint8_t* roles, void* o, int64_t B, int64_t H_q, int64_t H_kv,
                         int64_t L, int64_t D, int64_t C, int64_t W, const int64_t* q_strides, const int64_t* k_strides,
                         const int64_t* v_strides, const int64_t* o_strides, float sm_scale, hipStream_t st) {
  ShortArgs a;
  a.q = q; a.k = k; a.v = v; a.o = o; a.roles = roles;
  a.qs_b = q_strides[0]; a.qs_h = q_strides[1]; a.qs_l = q_strides[2];
  a.ks_b = k_strides[0]; a.ks_h = k_strides[1]; a.ks_l = k_strides[2];
  a.vs_b = v_strides[0]; a.vs_h = v_strides[1]; a.vs_l = v_strides[2];
  a.os_b = o_strides[0]; a.os_h = o_strides[1]; a.os_l = o_strides[2];
  a.B = (int)B; a.Hq = (int)H_q; a.Hkv = (int)H_kv; a.n_rep = (int)(H_q / H_kv);
  a.L = (int)L; a.S = (int)((L + C - 1) / C); a.C = (int)C;
  a.wc = (int)(W / C < (int64_t(1) << 29) ? W / C : (int64_t(1) << 29));
  a.scale = sm_scale;
  return D == 32 ? launch_d<32>(a, st) : D == 64 ? launch_d<64>(a, st) : launch_d<128>(a, st);
}

}  // namespace nats
