// What the prefill kernels share: the arguments of one segment and the entry of the fp32 matrix kernel.
#pragma once

#include "nats_balanced_map.h"
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

// Rows of K or V (or row limits) as a raw buffer of `bytes` bytes: reads beyond its end give zero, and a row is a scalar offset
// beside a lane's own, where addresses per row would take two registers and vector arithmetic each.
// A vector memory instruction may read a scalar register five wait states after a vector instruction wrote it at the earliest (the
// v_readlane that brings a spilled scalar back, for one).  The compiler keeps that distance for its own instructions only, so every
// assembly block has it inside, in front of its first transfer.
struct RowBuffer {
  typedef int Words __attribute__((ext_vector_type(4)));
  static constexpr int kFlags = 0x00027000;  // last word of a raw buffer's descriptor
  const void* base;
  uint32_t bytes;
  Words desc;
  __device__ __forceinline__ RowBuffer(const void* base, uint32_t bytes)
      : base(base), bytes(bytes), desc{(int)(uintptr_t)base, (int)((uintptr_t)base >> 32) & 0xffff, (int)bytes, kFlags} {}
  template <int kBytes>
  __device__ __forceinline__ void to_lds(uint32_t lds_addr, int lane_off, uint32_t row_off) const {
    static_assert(kBytes == 16 || kBytes == 4, "sizes a transfer can have here");
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (kBytes == 16) {
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 3\n\tbuffer_load_dwordx4 %0, %1, %3 offen lds" ::"v"(lane_off), "s"(desc), "s"(lds_addr), "s"(row_off)
                   : "memory", "m0");
    } else {
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 3\n\tbuffer_load_dword %0, %1, %3 offen lds" ::"v"(lane_off), "s"(desc), "s"(lds_addr), "s"(row_off)
                   : "memory", "m0");
    }
#endif
  }
  // two transfers of 16 bytes to consecutive KiB of LDS
  __device__ __forceinline__ void to_lds_pair(uint32_t lds_addr, int lane_off0, int lane_off1, uint32_t row_off) const {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile(
        "s_mov_b32 m0, %3\n\ts_nop 3\n\tbuffer_load_dwordx4 %0, %2, %4 offen lds\n\t"
        "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %4 offen lds" ::"v"(lane_off0), "v"(lane_off1), "s"(desc), "s"(lds_addr),
        "s"(row_off)
        : "memory", "m0", "scc");
#endif
  }
  // four transfers of 16 bytes to consecutive KiB of LDS, their rows `step` bytes apart
  __device__ __forceinline__ void to_lds_quad(uint32_t lds_addr, int off0, int off1, int off2, int off3, uint32_t row_off, uint32_t step) const {
#if defined(__HIP_DEVICE_COMPILE__)
    uint32_t row;
    asm volatile(
        "s_mov_b32 m0, %6\n\ts_mov_b32 %0, %7\n\ts_nop 2\n\tbuffer_load_dwordx4 %1, %5, %0 offen lds\n\t"
        "s_add_u32 m0, m0, 0x400\n\ts_add_u32 %0, %0, %8\n\tbuffer_load_dwordx4 %2, %5, %0 offen lds\n\t"
        "s_add_u32 m0, m0, 0x400\n\ts_add_u32 %0, %0, %8\n\tbuffer_load_dwordx4 %3, %5, %0 offen lds\n\t"
        "s_add_u32 m0, m0, 0x400\n\ts_add_u32 %0, %0, %8\n\tbuffer_load_dwordx4 %4, %5, %0 offen lds"
        : "=&s"(row)
        : "v"(off0), "v"(off1), "v"(off2), "v"(off3), "s"(desc), "s"(lds_addr), "s"(row_off), "s"(step)
        : "memory", "m0", "scc");
#endif
  }
};

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
