// Role-masked prefill attention in fp32 on the fp32 matrix instruction (v_mfma_f32_32x32x2_f32: exact fp32 products,
// fp32 accumulation).
//
// A workgroup owns 32 query rows of one q head; its wavefronts share the visible 32-key tiles among themselves (every
// n_waves-th one each), keep their own O, row maxima and row sums, and are combined through LDS at the end.  Nothing is
// staged: every operand is laid out so that it comes from global memory (K, V: L2) in the form the instruction takes.
//
//   S^T = K Q^T   A = K, B = Q.  The contraction runs over head dimensions in any order, so a lane of half `hl` holds every
//                 second 16-byte piece of its row of K (of Q): the two halves of a load take 32 contiguous bytes of a row.
//   O^T = V^T P^T A = V, B = P.  Accumulator i of S^T holds, in half hl, key 8 * (i / 4) + 4 * hl + i % 4 of query
//                 lane % 32, which is what the i-th step of this product takes as B when its two keys are those two; its A
//                 operand is head dimension (lane % 32) * DT + dt of the same key, so the DT tiles of a step are one load
//                 of DT floats per lane and a row of V arrives as one contiguous read of a half wavefront.
//
// Bound: the fp32 matrix rate (64 FLOP per cycle and SIMD, 157 TFLOP/s): a 32 x 32 tile at D = 64 is 64 instructions of 64
// cycles.  K of the next tile is requested when the scores of this one are done, V of this one before they begin, so
// both travel under matrix instructions.  Measured (8 heads, D = 64, chunk 64): all keys visible, L = 2048, batch 8 0.357 ms =
// 96 TFLOP/s; even roles at batch 8 0.236 ms, at batch 1 (two workgroups per compute unit, of which the heaviest has 44
// tiles and the average one 17) 0.048 ms, where the plain kernel (a query row per lane, one wavefront per workgroup)
// takes 0.88 ms.  The ends of a workgroup (Q, the tile summaries, the first K tile, the combination) are a third of an
// average workgroup's life there.
#include "nats_prefill.h"

namespace nats {

constexpr int kF32Rows = 32;      // query rows of a workgroup, keys of a tile
typedef float f32x2 __attribute__((ext_vector_type(2)));

// The Q operand is in LDS (one copy per workgroup): at D = 64 a wavefront then fits 168 registers, three to a SIMD (5 to 8 %
// faster than two with Q in registers), at D = 128 it fits 256.
template <int D>
struct F32Layout {
  static constexpr bool kQInLds = D >= 64;
  static constexpr int kQPitch = D + 4;   // floats; rows of the 16-byte reads fall into different banks
  static constexpr int kOPitch = D + 1;   // floats per query row of a wavefront's partial result
  static size_t smem_bytes(int n_waves) {
    const size_t q = (kQInLds ? sizeof(float) * kF32Rows * kQPitch : 0) + sizeof(int) * n_waves * kWave;  // Q, row limits
    const size_t merge = sizeof(float) * n_waves * kF32Rows * (kOPitch + 2);
    return q > merge ? q : merge;  // (the partial results take their place)
  }
};

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

template <int D, int kMaxWaves>
__global__ __launch_bounds__(kMaxWaves * kWave, kMaxWaves == 4 && D <= 64 ? 3 : 2) void prefill_f32_kernel(PrefillArgs a, int blk_first, int n_blk) {
  using Lay = F32Layout<D>;
  constexpr int HD = D / 2;   // head dimensions per half wavefront
  constexpr int DT = D / 32;  // 32-row tiles of O^T
  typedef typename F32Vec<DT>::type VecV;
  extern __shared__ __attribute__((aligned(16))) float smem[];

  const int lane = threadIdx.x & 63, l32 = lane & 31, hl = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n_waves = __builtin_amdgcn_readfirstlane(blockDim.x >> 6);
  // (q heads change fastest, so that with 8 heads and more the blocks of a head run on one XCD; heavy blocks first)
  const int n_heads = a.B * a.Hq;
  const int bh = blockIdx.x % n_heads, blk = blk_first + n_blk - 1 - (int)(blockIdx.x / n_heads);
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

  // ---- Q: the B operand of the scores ----
  float qreg[Lay::kQInLds ? 1 : HD];
  if (Lay::kQInLds) {
    for (int i = threadIdx.x; i < kF32Rows * D / 4; i += blockDim.x) {
      const int row = i / (D / 4), piece = i % (D / 4);
      const int m = min(max(q0 + row, a.r_begin), a.r_end - 1) - a.r_begin;
      *reinterpret_cast<f32x4*>(smem + row * Lay::kQPitch + piece * 4) =
          *reinterpret_cast<const f32x4*>(qp + (int64_t)m * a.qs_l + piece * 4);
    }
    __syncthreads();
  } else {
    const int m = min(max(qtok, a.r_begin), a.r_end - 1) - a.r_begin;
    const f32x4* rp = reinterpret_cast<const f32x4*>(qp + (int64_t)m * a.qs_l + hl * 4);
#pragma unroll
    for (int i = 0; i < HD / 4; ++i) {
      const f32x4 x = rp[2 * i];
#pragma unroll
      for (int e = 0; e < 4; ++e) qreg[(i * 4 + e) % (Lay::kQInLds ? 1 : HD)] = x[e];
    }
  }
  int* lim_lds = reinterpret_cast<int*>(smem + (Lay::kQInLds ? kF32Rows * Lay::kQPitch : 0)) + wave * kWave;
  const float* q_lds = smem + l32 * Lay::kQPitch + hl * 4;

  f32x16 oacc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) oacc[dt][i] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;

  // ---- iterator over this wavefront's tiles: 64 tile summaries per ballot; the bits stay in scalar registers ----
  int w0 = -64;        // first tile of the window
  uint64_t mine = 0;   // this wavefront's visible tiles of the window that are still to come
  uint64_t mixed = 0;  // tiles of the window with rows that some query does not see
  int turn = 0;        // visible tiles before the window
  auto next_tile = [&](bool& masked) -> int {
    while (mine == 0) {
      w0 += 64;
      if (w0 > t_last) return -1;
      const int t = w0 + lane;
      bool v = false, mx = true;
      if (t <= t_last) {
        const int2 g0 = gl[2 * t], g1 = gl[2 * t + 1];  // (the granule table is filled up to whole 64-row tiles)
        v = max(g0.x, g1.x) >= r0;
        mx = !(min(g0.y, g1.y) >= rlast && t * kF32Rows + kF32Rows - 1 - a.base <= r0 && (t + 1) * kF32Rows <= a.N);
      }
      const uint64_t vis = __ballot(v);
      mixed = __ballot(mx);
      const int nth = turn + __builtin_popcountll(vis & ((uint64_t(1) << lane) - 1));
      mine = __ballot(v && (nth & (n_waves - 1)) == wave);  // (n_waves is a power of two)
      turn += __builtin_popcountll(vis);
    }
    const int i = __builtin_ctzll(mine);
    mine &= mine - 1;
    masked = (mixed >> i) & 1;
    return w0 + i;
  };

  f32x4 kreg[HD / 4];
  // (a tile's rows at a lane offset from a uniform base; the last tile's rows past the end repeat the last row)
  const uint32_t koff = uint32_t(l32 * a.ks_l + hl * 4), voff = uint32_t(hl * 4 * a.vs_l + l32 * DT);
  auto load_k = [&](int t) {
    const int k0 = t * kF32Rows;
    const float* tb = kp + (int64_t)k0 * a.ks_l;
    const uint32_t off = k0 + kF32Rows <= a.N ? koff : uint32_t(min(l32, a.N - 1 - k0) * a.ks_l + hl * 4);
#pragma unroll
    for (int i = 0; i < HD / 4; ++i) kreg[i] = *reinterpret_cast<const f32x4*>(tb + off + i * 8);
  };

  bool masked = false;
  int t = next_tile(masked);
  if (t >= 0) load_k(t);
  while (t >= 0) {
    const int k0 = t * kF32Rows;
    // V rows of this tile (rows past the end repeat the last one: their probabilities are 0) and the row limits
    VecV vreg[16];
    if (k0 + kF32Rows <= a.N) {
#pragma unroll
      for (int i = 0; i < 16; ++i) vreg[i] = *reinterpret_cast<const VecV*>(vp + (int64_t)(k0 + 8 * (i / 4) + i % 4) * a.vs_l + voff);
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int n = min(k0 + 8 * (i / 4) + 4 * hl + i % 4, a.N - 1);
        vreg[i] = *reinterpret_cast<const VecV*>(vp + (int64_t)n * a.vs_l + l32 * DT);
      }
    }
    if (masked) lim_lds[lane] = lim[min(k0 + l32, a.N - 1)];
    __builtin_amdgcn_sched_barrier(0);

    // ---- S^T = K Q^T ----
    f32x16 s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.f;
#pragma unroll
    for (int i = 0; i < HD / 4; ++i) {
      f32x4 qv;
      if (Lay::kQInLds) {
        qv = *reinterpret_cast<const f32x4*>(q_lds + i * 8);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) qv[e] = qreg[(i * 4 + e) % (Lay::kQInLds ? 1 : HD)];
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kreg[i][e], qv[e], s, 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
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
        const int4 l4 = *reinterpret_cast<const int4*>(lim_lds + 8 * g + 4 * hl);
        const int lv[4] = {l4.x, l4.y, l4.z, l4.w};
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
  // Eight wavefronts per workgroup while the launch is at most four workgroups per compute unit: the heaviest block is the
  // end of the launch there and has to be short; above, four (three workgroups per compute unit at D = 64) waste less on the
  // ends of a workgroup.  8 heads, L = 2048, D = 64: 0.048 against 0.057 ms at batch 1 (2 workgroups per compute unit), 0.085 /
  // 0.088 at batch 2, 0.165 / 0.146 at batch 4.
  const int n_cu = device_cu_count();
  const int waves = n_wg <= 4 * (int64_t)n_cu ? 8 : 4;
  if (!configured[dev]) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&prefill_f32_kernel<D, 4>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)F32Layout<D>::smem_bytes(4));
    if (e == hipSuccess)
      e = hipFuncSetAttribute(reinterpret_cast<const void*>(&prefill_f32_kernel<D, 8>), hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)F32Layout<D>::smem_bytes(8));
    if (e != hipSuccess) return fail(NATS_ERR_LAUNCH, "prefill_f32_kernel: LDS: %s", hipGetErrorString(e));
    configured[dev] = true;
  }
  const dim3 grid((unsigned)n_wg), block(waves * kWave);
  const size_t smem = F32Layout<D>::smem_bytes(waves);
  if (waves == 8) {
    hipLaunchKernelGGL((prefill_f32_kernel<D, 8>), grid, block, smem, st, a, blk_first, n_blk);
  } else {
    hipLaunchKernelGGL((prefill_f32_kernel<D, 4>), grid, block, smem, st, a, blk_first, n_blk);
  }
  NATS_CHECK_LAUNCH("prefill_f32_kernel");
  return NATS_OK;
}

int launch_prefill_f32(const PrefillArgs& a, int D, hipStream_t st) {
  return D == 32 ? launch_d<32>(a, st) : D == 64 ? launch_d<64>(a, st) : launch_d<128>(a, st);
}

}  // namespace nats
