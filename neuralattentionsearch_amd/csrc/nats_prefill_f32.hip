// Role-masked prefill attention in fp32 on the fp32 matrix instruction (v_mfma_f32_32x32x2_f32: exact fp32 products,
// fp32 accumulation).
//
// A workgroup owns 32 query rows of one q head; its wavefronts share the visible 32-key tiles among themselves (every
// n_waves-th one each), keep their own O, row maxima and row sums, and are combined through LDS at the end.  A wavefront brings
// its K tile to LDS in whole rows and takes V from global memory (L2) in the form the instruction takes.
//
//   S^T = K Q^T   A = K, B = Q, both from LDS.  The contraction runs over head dimensions in any order, so a lane of half `hl`
//                 takes every second 16-byte piece of its row of K (of Q).
//   O^T = V^T P^T A = V, B = P.  Accumulator i of S^T holds, in half hl, key 8 * (i / 4) + 4 * hl + i % 4 of query
//                 lane % 32, which is what the i-th step of this product takes as B when its two keys are those two; its A
//                 operand is head dimension (lane % 32) * DT + dt of the same key, so the DT tiles of a step are one load
//                 of DT floats per lane and a row of V arrives as one contiguous read of a half wavefront.
//
// Bound: the fp32 matrix rate (64 FLOP per cycle and SIMD, 157 TFLOP/s): a 32 x 32 tile at D = 64 is 64 instructions of 64
// cycles.  One wavefront's tile is a chain of trips and products, so up to head dim 64 four of them share a SIMD: 128 registers
// each, which is why K goes through LDS (one buffer per wavefront: the next tile is requested when the scores of this one are
// done and travels under the softmax and the PV product, V of this one under the scores).  K straight from global memory in
// operand form, 16 bytes of each of 32 rows per instruction, kept L1 busy for 64 accesses per load, two thirds of all, and left
// registers for two wavefronts per SIMD.  Measured, the op with its two kernels in front (10 us), before / now, 8 heads, chunk 64,
// even roles: D = 64, L = 2048 44.5 / 35.5 us (batch 2 79.1 / 63.0, batch 8 203 now), L = 800 23.2 / 21.7; D = 32 27.4 / 23.1;
// D = 128 (one workgroup of eight wavefronts per compute unit) 75.6 / 66.9, L = 3000 133 / 116.  The plain kernel (a query row per lane)
// takes 0.88 ms at D = 64, L = 2048.
#include "nats_prefill.h"

namespace nats {

constexpr int kF32Rows = 32;      // query rows of a workgroup, keys of a tile
typedef float f32x2 __attribute__((ext_vector_type(2)));

// In LDS: Q (one copy per workgroup), and per wavefront one K tile and its row limits.  Four wavefronts at head dim 128 have 80 KiB to
// the byte, half of a compute unit's: their Q rows are permuted like K's instead of padded, and the row limits stay in registers.
template <int D, int kWaves>
struct F32Layout {
  static constexpr bool kTight = D == 128 && kWaves == 4;
  static constexpr int kQPitch = kTight ? D : D + 4;  // floats; rows of the 16-byte reads fall into different banks
  static constexpr int kOPitch = D + 1;               // floats per query row of a wavefront's partial result
  static constexpr int kWaveFloats = kF32Rows * D + (kTight ? 0 : kWave);  // K tile, row limits
  static constexpr int kOperands = kF32Rows * kQPitch + kWaves * kWaveFloats, kMerge = kWaves * kF32Rows * (kOPitch + 2);
  static constexpr int kBytes = (int)sizeof(float) * (kOperands > kMerge ? kOperands : kMerge);  // (the partial results take their place)
};
static_assert(2 * F32Layout<128, 4>::kBytes <= 160 * 1024, "two workgroups of four wavefronts on a compute unit");

template <int DT>
struct F32Vec;
template <>
struct F32Vec<1> { typedef float type; };
template <>
struct F32Vec<2> { typedef f32x2 type; };
template <>
struct F32Vec<4> { typedef f32x4 type; };
template <int DT>
__device__ __forceinline__ float f32_part(const typename F32Vec<DT>::type& v, int i) { return v[i]; }
template <>
__device__ __forceinline__ float f32_part<1>(const float& v, int) { return v; }

template <int DT>
__device__ __forceinline__ typename F32Vec<DT>::type row_part(const RowBuffer& buf, int lane_off, int row_off) {
#if defined(__HIP_DEVICE_COMPILE__)
  const __amdgpu_buffer_rsrc_t desc = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(buf.base), 0, (int)buf.bytes, RowBuffer::kFlags);
  if constexpr (DT == 1) {
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(desc, lane_off, row_off, 0));
  } else if constexpr (DT == 2) {
    return __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(desc, lane_off, row_off, 0));
  } else {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(desc, lane_off, row_off, 0));
  }
#else
  return {};
#endif
}

template <int D, int kWaves>
__global__ __launch_bounds__(kWaves * kWave, D <= 64 ? 4 : 2) void prefill_f32_kernel(PrefillArgs a, int blk_first, int n_blk, int paired) {
  using Lay = F32Layout<D, kWaves>;
  constexpr int HD = D / 2;   // head dimensions per half wavefront
  constexpr int DT = D / 32;  // 32-row tiles of O^T
  typedef typename F32Vec<DT>::type VecV;
  extern __shared__ __attribute__((aligned(16))) float smem[];

  const int lane = threadIdx.x & 63, l32 = lane & 31, hl = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr int n_waves = kWaves;
  // (q heads change fastest, so that with 8 heads and more the blocks of a head run on one XCD; heavy blocks first, or,
  // where the first `paired` ranks take every compute unit and the others join them, see launch_d, the light blocks in
  // falling order beside the others in rising order)
  const int n_heads = a.B * a.Hq;
  const int rank = (int)(blockIdx.x / n_heads);
  const int bh = blockIdx.x % n_heads;
  const int blk = blk_first + (rank < paired ? n_blk - paired + rank : n_blk - 1 - rank);
  const int b = bh / a.Hq, hq = bh % a.Hq, hkv = hq / a.n_rep;
  const int stream = b * a.Hkv + hkv;
  const float* qp = static_cast<const float*>(a.q) + b * a.qs_b + hq * a.qs_h;
  const float* kp = static_cast<const float*>(a.k) + b * a.ks_b + hkv * a.ks_h;
  const float* vp = static_cast<const float*>(a.v) + b * a.vs_b + hkv * a.vs_h;
  float* op = static_cast<float*>(a.o) + b * a.os_b + hq * a.os_h;
  const int32_t* lim = a.tok_lim + (int64_t)stream * a.N;
  const int2* gl = a.gran_lim + (int64_t)stream * a.Tk * (kTile / kGranule);

  const int q0 = blk * kF32Rows;  // region token of row 0
  const int qtok = q0 + l32;
  const int r0 = max(q0, a.r_begin), rlast = min(q0 + kF32Rows - 1, a.r_end - 1);
  const int t_last = (a.base + rlast) / kF32Rows;  // last key tile somebody may see
  const float c = a.scale * 1.4426950408889634f;

  float* k_lds = smem + kF32Rows * Lay::kQPitch + wave * Lay::kWaveFloats;
  int* lim_lds = reinterpret_cast<int*>(k_lds + kF32Rows * D);
  const uint32_t k_addr = lds_address(k_lds);

  f32x16 oacc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) oacc[dt][i] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;

  // ---- iterator over this wavefront's tiles: 64 tile summaries per ballot; the bits stay in scalar registers ----
  int w0 = 0;          // first tile of the window
  uint64_t mine = 0;   // this wavefront's visible tiles of the window that are still to come
  uint64_t mixed = 0;  // tiles of the window with rows that some query does not see
  int turn = 0;        // visible tiles before the window
  auto summary = [&](int t, int2& g0, int2& g1) {
    g0 = g1 = make_int2(-1, -1);
    if (t <= t_last) g0 = gl[2 * t], g1 = gl[2 * t + 1];  // (the granule table is filled up to whole 64-row tiles)
  };
  auto open_window = [&](const int2& g0, const int2& g1) {
    const int t = w0 + lane;
    const bool v = max(g0.x, g1.x) >= r0;
    const bool mx = !(min(g0.y, g1.y) >= rlast && t * kF32Rows + kF32Rows - 1 - a.base <= r0 && (t + 1) * kF32Rows <= a.N);
    const uint64_t vis = __ballot(v);
    mixed = __ballot(mx);
    const int nth = turn + __builtin_popcountll(vis & ((uint64_t(1) << lane) - 1));
    mine = __ballot(v && (nth & (n_waves - 1)) == wave);  // (n_waves is a power of two)
    turn += __builtin_popcountll(vis);
  };
  auto next_tile = [&](bool& masked) -> int {
    while (mine == 0) {
      w0 += 64;
      if (w0 > t_last) return -1;
      int2 g0, g1;
      summary(w0 + lane, g0, g1);
      open_window(g0, g1);
    }
    const int i = __builtin_ctzll(mine);
    mine &= mine - 1;
    masked = (mixed >> i) & 1;
    return w0 + i;
  };

  // K tile: global -> LDS (16 bytes per lane, whole rows per instruction).  The 16-byte chunks of a row are permuted so that the
  // rows which a quarter wavefront reads at once fall into different banks.
  constexpr int OCT = D / 4;                // 16-byte chunks per row
  constexpr int kRowsPerInst = kWave / OCT;
  auto swz = [](int row) { return D == 32 ? (row >> 1) & 7 : row & 15; };
  // (the buffer of a tile ends with the last row; the lane id is taken afresh for every tile so that nothing derived from it lives
  // from one to the next)
  auto tile_buffer = [&](const float* base, int64_t row_stride, int k0) {
    return RowBuffer(base + (int64_t)k0 * row_stride, ((min(kF32Rows, a.N - k0) - 1) * (int)row_stride + D) * 4);
  };
  auto load_k = [&](int t) {
    const RowBuffer buf = tile_buffer(kp, a.ks_l, t * kF32Rows);
    int ln = lane;
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+v"(ln));
#endif
    const int row0 = ln / OCT;
#pragma unroll
    for (int j = 0; j < kF32Rows / kRowsPerInst; ++j) {
      const int off = (row0 * (int)a.ks_l + ((ln % OCT) ^ swz(j * kRowsPerInst + row0)) * 4) * 4;
      buf.to_lds<16>(k_addr + j * kWave * 16, off, j * kRowsPerInst * (int)a.ks_l * 4);
    }
  };
  auto k_frag = [&](int i) { return *reinterpret_cast<const f32x4*>(k_lds + l32 * D + ((2 * i + hl) ^ swz(l32)) * 4); };
  auto q_frag = [&](int i) {
    const int chunk = 2 * i + hl;
    return *reinterpret_cast<const f32x4*>(smem + l32 * Lay::kQPitch + (Lay::kTight ? chunk ^ swz(l32) : chunk) * 4);
  };
  const int voff = (hl * 4 * (int)a.vs_l + l32 * DT) * 4;  // bytes

  // ---- Q goes to LDS (the B operand of the scores); the first tile summaries are requested before it and the first K tile
  // while it is under way: three trips to memory, of which two run side by side ----
  int2 g0, g1;
  summary(lane, g0, g1);
  constexpr int kQPieces = kF32Rows * D / 4, kQSteps = (kQPieces + n_waves * kWave - 1) / (n_waves * kWave);
  f32x4 qp_reg[kQSteps];
#pragma unroll
  for (int j = 0; j < kQSteps; ++j) {
    const int i = min(j * n_waves * kWave + (int)threadIdx.x, kQPieces - 1);
    const int m = min(max(q0 + i / (D / 4), a.r_begin), a.r_end - 1) - a.r_begin;
    qp_reg[j] = *reinterpret_cast<const f32x4*>(qp + (int64_t)m * a.qs_l + i % (D / 4) * 4);
  }
  open_window(g0, g1);
  bool masked = false;
  int t = next_tile(masked);
  if (t >= 0) load_k(t);
#pragma unroll
  for (int j = 0; j < kQSteps; ++j) {
    const int i = min(j * n_waves * kWave + (int)threadIdx.x, kQPieces - 1);
    const int row = i / (D / 4), chunk = i % (D / 4);
    *reinterpret_cast<f32x4*>(smem + row * Lay::kQPitch + (Lay::kTight ? chunk ^ swz(row) : chunk) * 4) = qp_reg[j];
  }
  __syncthreads();
  while (t >= 0) {
    const int k0 = t * kF32Rows;
    wait_transfers();  // K of this tile has landed in LDS
    __builtin_amdgcn_sched_barrier(0);
    // V rows of this tile (rows past the end are zeros, and so are their probabilities) and the row limits
    VecV vreg[16];
    {
      const RowBuffer buf = tile_buffer(vp, a.vs_l, k0);
#pragma unroll
      for (int i = 0; i < 16; ++i) vreg[i] = row_part<DT>(buf, voff, (8 * (i / 4) + i % 4) * (int)a.vs_l * 4);
    }
    int lim_reg = 0;
    if (masked) {
      lim_reg = lim[min(k0 + l32, a.N - 1)];
      if (!Lay::kTight) lim_lds[lane] = lim_reg;
    }
    __builtin_amdgcn_sched_barrier(0);

    // ---- S^T = K Q^T ----
    f32x16 s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.f;
    f32x4 kn = k_frag(0), qn = q_frag(0);
#pragma unroll
    for (int i = 0; i < HD / 4; ++i) {
      const f32x4 kv = kn, qv = qn;
      if (i + 1 < HD / 4) {
        kn = k_frag(i + 1);
        qn = q_frag(i + 1);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[e], qv[e], s, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    const bool was_masked = masked;
    const int t_next = next_tile(masked);
    if (t_next >= 0) load_k(t_next);
    __builtin_amdgcn_sched_barrier(0);

    // ---- mask, running maximum, probabilities (the scale first: it may be 0 or negative) ----
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] *= c;
    if (was_masked) {
      const int key0 = k0 - a.base;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        int lv[4];
        if (Lay::kTight) {
#pragma unroll
          for (int e = 0; e < 4; ++e) lv[e] = __shfl(lim_reg, 8 * g + 4 * hl + e);
        } else {
          const int4 l4 = *reinterpret_cast<const int4*>(lim_lds + 8 * g + 4 * hl);
          lv[0] = l4.x, lv[1] = l4.y, lv[2] = l4.z, lv[3] = l4.w;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int key = key0 + 8 * g + 4 * hl + e;  // (rows past the end are later than every query)
          if (!(key <= qtok && qtok <= lv[e])) s[g * 4 + e] = -INFINITY;
        }
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
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      s[i] = __builtin_amdgcn_exp2f(s[i] - m_use);
      l_run += s[i];
    }

    // ---- O^T += V^T P^T ----
#pragma unroll
    for (int i = 0; i < 16; ++i)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
        oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(f32_part<DT>(vreg[i], dt), s[i], oacc[dt], 0, 0, 0);
    t = t_next;
  }

  // ---- combine the wavefronts' partial results ----
  {
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(l_run), __float_as_uint(l_run), false, false);
    l_run = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
  float* o_part = smem;                                             // [n_waves][32][kOPitch]
  float* m_part = smem + n_waves * kF32Rows * Lay::kOPitch;         // [n_waves][32]
  float* l_part = m_part + n_waves * kF32Rows;                      // [n_waves][32]
  __syncthreads();  // (Q in LDS has been read by everybody)
  if (hl == 0) m_part[wave * kF32Rows + l32] = m_run;
  __syncthreads();
  float m_all = -INFINITY;
  for (int w = 0; w < n_waves; ++w) m_all = fmaxf(m_all, m_part[w * kF32Rows + l32]);
  const float f = m_run == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run - m_all);
  if (hl == 0) l_part[wave * kF32Rows + l32] = l_run * f;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int d = (8 * (i / 4) + 4 * hl + i % 4) * DT + dt;
      o_part[(wave * kF32Rows + l32) * Lay::kOPitch + d] = oacc[dt][i] * f;
    }
  __syncthreads();
  for (int i = threadIdx.x; i < kF32Rows * D; i += blockDim.x) {
    const int row = i / D, d = i % D;
    const int m = q0 + row;
    if (m < a.r_begin || m >= a.r_end) continue;
    float o = 0.f, l = 0.f;
    for (int w = 0; w < n_waves; ++w) {
      o += o_part[(w * kF32Rows + row) * Lay::kOPitch + d];
      l += l_part[w * kF32Rows + row];
    }
    op[(int64_t)(m - a.r_begin) * a.os_l + d] = o / l;
  }
}

bool prefill_f32_takes(const PrefillArgs& a, int D) {
  if (D != 32 && D != 64 && D != 128) return false;
  const uintptr_t p = reinterpret_cast<uintptr_t>(a.q) | reinterpret_cast<uintptr_t>(a.k) | reinterpret_cast<uintptr_t>(a.v);
  return p % 16 == 0 && (a.qs_b | a.qs_h | a.qs_l | a.ks_b | a.ks_h | a.ks_l | a.vs_b | a.vs_h | a.vs_l) % 4 == 0;
}

template <int D>
static int launch_d(const PrefillArgs& a, hipStream_t st) {
  constexpr int kMaxDev = 64;
  static bool configured[kMaxDev] = {};  // the LDS attribute is set once per device
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDev) return fail(NATS_ERR_LAUNCH, "prefill: no current device");
  const int blk_first = a.r_begin / kF32Rows, n_blk = (a.r_end - 1) / kF32Rows - blk_first + 1;
  const int64_t n_wg = (int64_t)a.B * a.Hq * n_blk;
  NATS_REQUIRE(n_wg < (int64_t(1) << 31), NATS_ERR_BAD_SHAPE, "prefill: grid too large");
  // How many wavefronts share a block's tiles.  Eight make the heaviest block, which ends the launch, short; four waste less on the
  // ends of a workgroup, more of them the shorter the lists.  LDS holds two workgroups of eight or three of four on a compute unit at
  // head dim 64 (76 and 42 KB; registers would allow a fourth), so just above two per compute unit and between three and six four leave more
  // of a round empty than eight do, around three less.  At head dim 128 it holds one of eight or two of four.  Four / eight, by workgroups
  // per compute unit, for heads of up to 20 and of more blocks (even and sparse roles):
  //   D = 64   up to 2: 0.98 to 1.06 / 1.00 to 1.09.  2.2: - / 1.05 to 1.12.  2.5 to 2.75: 0.76 to 0.84 / 0.90 to 0.92.  3: - / 0.86 to 1.12.  4 to 4.4:
  //            0.97 / 0.99 to 1.09.  5 to 6: 0.88 to 0.91 / 0.98 to 1.08.  8 and more: 0.86 to 0.91 / 0.91 to 1.02.
  //   D = 32   four / eight in us: 1.4: 21 / 20, 18 / 18.  2: 24 / 23, 20 / 20.  2.66: 33 / 33, 25 / 28.  4: 34 / 36, 27 / 30.  13: 139 / 150, 83 / 97.
  //   D = 128  up to 2: 0.81 to 1.06 / 0.89 to 1.17.  2.1 to 2.6: 0.86 to 0.91 / 0.89 to 1.13.  3: - / 0.97 to 1.07.  4 to 6: 0.75 to 0.85 / 0.86 to
  //            0.98.  8 and more: 0.74 to 0.82 / 0.80 to 0.94 (64 heads, 1024 tokens 165 -> 141 us).
  const int n_cu = device_cu_count();
  auto up_to = [&](int half_rounds) { return 2 * n_wg <= half_rounds * (int64_t)n_cu; };  // (halves of a workgroup per compute unit)
  const bool few = up_to(4) || (n_blk > 20 && (D == 64 ? up_to(5) || (!up_to(7) && up_to(12)) : D == 128 && up_to(6)));
  // Between one and two workgroups per compute unit: workgroups i and i + n_cu share one, so the lightest blocks come last, in
  // falling order, beside the lightest of the others, and the heaviest have a compute unit to themselves (8 heads of 64, 2048
  // tokens 39.0 -> 35.8 us, 1400 31.6 -> 26.1, 4 heads, 3000 tokens 41.4 -> 34.0).
  const int per_round = (int)(n_cu / ((int64_t)a.B * a.Hq));  // blocks of a head that take every compute unit once
  const int paired = per_round > 0 && n_blk > per_round && n_blk <= 2 * per_round ? per_round : 0;
  constexpr int kBytes8 = F32Layout<D, 8>::kBytes, kBytes4 = F32Layout<D, 4>::kBytes;
  if (!configured[dev]) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&prefill_f32_kernel<D, 8>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                       kBytes8);
    if (e == hipSuccess)
      e = hipFuncSetAttribute(reinterpret_cast<const void*>(&prefill_f32_kernel<D, 4>), hipFuncAttributeMaxDynamicSharedMemorySize,
                              kBytes4);
    if (e != hipSuccess) return fail(NATS_ERR_LAUNCH, "prefill_f32_kernel: LDS: %s", hipGetErrorString(e));
    configured[dev] = true;
  }
  const dim3 grid((unsigned)n_wg);
  if (few) {
    hipLaunchKernelGGL((prefill_f32_kernel<D, 8>), grid, dim3(8 * kWave), kBytes8, st, a, blk_first, n_blk, paired);
  } else {
    hipLaunchKernelGGL((prefill_f32_kernel<D, 4>), grid, dim3(4 * kWave), kBytes4, st, a, blk_first, n_blk, paired);
  }
  NATS_CHECK_LAUNCH("prefill_f32_kernel");
  return NATS_OK;
}

int launch_prefill_f32(const PrefillArgs& a, int D, hipStream_t st) {
  return D == 32 ? launch_d<32>(a, st) : D == 64 ? launch_d<64>(a, st) : launch_d<128>(a, st);
}

}  // namespace nats
