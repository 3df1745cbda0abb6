// What the prefill kernels share: the arguments of one segment and the entry of the fp32 matrix kernel.
#pragma once

#include "nats_common.h"

namespace nats {

struct PrefillArgs {
  const void* q;
  const void* k;
  const void* v;
  void* o;
  const int32_t* tok_lim;  // [B*Hkv, N], then one entry holding -1
  const int2* tile_lim;    // [B*Hkv, Tk] {max, min}
  const int2* gran_lim;    // [B*Hkv, Tk * 4] {max, min} of every 16 key rows
  int64_t qs_b, qs_h, qs_l;
  int64_t ks_b, ks_h, ks_l;
  int64_t vs_b, vs_h, vs_l;
  int64_t os_b, os_h, os_l;
  int B, Hq, Hkv, n_rep;
  int N, Tk;             // key rows and 64-row key tiles
  int base;              // first key row of the region
  int r_begin, r_end;    // region tokens that are queries; query i of q / o is token r_begin + i
  int qt_first, qt_last; // 64-token region tiles that hold queries
  int hpw;       // q heads of one kv head handled by one workgroup (mfma kernel)
  int qpw;       // 64-row query tiles handled by one workgroup (mfma kernel)
  int n_hg;      // head groups per kv head = n_rep / hpw
  int n_qg;      // query tile groups = ceil(n query tiles / qpw)
  int xcd_mode;  // 1: workgroups of one kv stream share an XCD (needs B*Hkv % 8 == 0)
  // The query groups with the fewest visible keys (the last pool_ranks ranks of every stream) are not bound to a
  // workgroup: a few workgroups at the end of the grid draw them from counters, one queue per XCD (heaviest first),
  // for as long as there are any, so that an XCD that reaches its last workgroups earlier takes more of them.
  int pool_ranks;    // 0: every workgroup has its fixed query group
  int heavy_first;   // launches with the balanced map: how far above the mean the largest stream has to be, in hundredths
  int32_t* ticket;   // one counter per XCD, kTicketStride entries apart, zero at launch
  float scale;   // softmax scale
  // few query tiles over many key rows: n_split workgroups share the tile list of one (kv stream, head group,
  // query group) and leave partial results, which prefill_split_merge_kernel combines
  int n_split;      // 1: no split
  float* part_acc;  // [workgroup, split, wavefront, 32 rows, D]
  float* part_ml;   // [workgroup, split, wavefront, 32 rows, 2] running maximum (base-2 exponent) and row sum
  // packed tiles of chunks shorter than a granule: rows more than t_long tokens behind a query group come from the
  // lists of long-lived rows (long_rows_kernel), gathered row by row; NULL = every row is walked granule by granule
  const int32_t* long_rows;    // [streams, 2, long_cap]: list A (rows every later query sees), list B (rows with a last query)
  const int32_t* long_lim;     // [streams, 2, long_cap]
  const int32_t* long_before;  // [streams, 2, n_gran + 1] entries of A / of B before every granule
  const int32_t* long_alive;   // [streams, n_rtile] first entry of B that a query of the 64-token region tile may see
  int long_cap, n_gran, n_rtile, t_long;
};

// Workgroup `bid` of ns * n_hg * n_qg -> its item, where the streams in `heavy` (a set of the first ns <= 64) come first.
__host__ __device__ inline void balanced_item(uint64_t heavy, int ns, int n_hg, int n_qg, int bid, int& ks, int& hg, int& rank) {
  const uint64_t light = ~heavy & (ns < 64 ? (uint64_t(1) << ns) - 1 : ~uint64_t(0));
  const uint64_t every8 = 0x0101010101010101ull;
  const int total = ns * n_hg * n_qg;
  const int n_heavy = (int)__builtin_popcountll(heavy) * n_hg * n_qg;
  uint64_t set = heavy;
  int i = bid;  // the item's place among those of the streams in `set`, rank by rank
  if (bid >= n_heavy) {
    // Workgroup i runs on XCD i mod 8.  An XCD works through the light streams that are its own as far as its workgroups
    // reach; what is left of them (their lightest query groups) goes to the XCDs that have workgroups to spare.
    auto own = [&](int y) -> int { return (int)__builtin_popcountll(light & (every8 << y)) * n_hg * n_qg; };
    auto slots = [&](int y) -> int { return (total + 7 - y) / 8 - (n_heavy + 7 - y) / 8; };  // workgroups of [n_heavy, total) on XCD y
    auto kept = [&](int y) -> int { return own(y) < slots(y) ? own(y) : slots(y); };
    const int x = bid & 7;
    i = (bid - x) / 8 - (n_heavy + 7 - x) / 8;  // this workgroup's place among those of its XCD
    int home = x;
    if (i >= kept(x)) {
      int o = i - kept(x);  // ... among the workgroups to spare, then among the items left over
      for (int y = 0; y < x; ++y) o += slots(y) - kept(y);
      for (home = 0; home < 7 && o >= own(home) - kept(home); ++home) o -= own(home) - kept(home);
      i = kept(home) + o;
    }
    set = light & (every8 << home);
  }
  const int n_slot = (int)__builtin_popcountll(set) * n_hg;
  rank = i / n_slot;
  const int slot = i % n_slot;
  hg = slot % n_hg;
  for (int n = slot / n_hg; n > 0; --n) set &= set - 1;
  ks = __builtin_ctzll(set);
}

// fp32 kernel on the fp32 matrix instruction (nats_prefill_f32.hip)
bool prefill_f32_takes(const PrefillArgs& a, int D);
int launch_prefill_f32(const PrefillArgs& a, int D, hipStream_t st);
// short prompts from an empty cache in one launch (nats_prefill_short.hip)
bool prefill_short_takes(int64_t B, int64_t H_q, int64_t H_kv, int64_t D, int64_t L, int64_t C, int dtype);
int launch_prefill_short(const void* q, const void* k, const void* v, const uint8_t* roles, void* o, int64_t B, int64_t H_q, int64_t H_kv,
                         int64_t L, int64_t D, int64_t C, int64_t W, const int64_t* q_strides, const int64_t* k_strides,
                         const int64_t* v_strides, const int64_t* o_strides, float sm_scale, hipStream_t st);
// compute units of the current device (0: unknown)
int device_cu_count();

}  // namespace nats
