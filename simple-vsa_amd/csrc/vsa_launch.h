// Host-side helpers for the C ABI entry points: dtype dispatch and launch checks.
#pragma once

#include <hip/hip_runtime.h>

#include "../../include/vsa_capi.h"

// Instantiate BODY with T bound to the element type named by `dtype`;
// returns VSA_ERR_DTYPE from the enclosing function for anything else.
#define VSA_DISPATCH_ALL(dtype, T, BODY)      \
  do {                                        \
    if ((dtype) == VSA_BF16) {                \
      typedef __bf16 T;                       \
      BODY;                                   \
    } else if ((dtype) == VSA_F16) {          \
      typedef _Float16 T;                     \
      BODY;                                   \
    } else if ((dtype) == VSA_F32) {          \
      typedef float T;                        \
      BODY;                                   \
    } else {                                  \
      return VSA_ERR_DTYPE;                   \
    }                                         \
  } while (0)

// Same, for the MFMA kernels (bf16 / fp16 only).
#define VSA_DISPATCH_MFMA(dtype, T, BODY)     \
  do {                                        \
    if ((dtype) == VSA_BF16) {                \
      typedef __bf16 T;                       \
      BODY;                                   \
    } else if ((dtype) == VSA_F16) {          \
      typedef _Float16 T;                     \
      BODY;                                   \
    } else {                                  \
      return VSA_ERR_DTYPE;                   \
    }                                         \
  } while (0)

// Alignment the kernels' accesses need (NULL, an absent optional buffer,
// passes): 16 bytes for rows of the element type and the fp32 score /
// probability rows, 8 for int64 index arrays, 4 for int32 arrays and
// lse / delta.
template <unsigned A, typename... P>
static inline bool vsa_aligned(P... p) {
  return ((((uintptr_t)(const void*)p) % A == 0) && ...);
}

static inline int vsa_check_launch() {
  return hipGetLastError() == hipSuccess ? VSA_OK : VSA_ERR_LAUNCH;
}

// CUs of the current device (cached per device; a racy first fill writes the
// same value)
static inline int cu_count() {
  static int cached[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
  if (cached[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      n = 256;
    cached[dev] = n;
  }
  return cached[dev];
}

namespace vsa {
// out = T(out_c[block] * gate + fine) with an fp32 gate (common.hip); out may
// alias fine.  gate_mode is 1, 2 or 3 (without the VSA_GATE_F32 flag).
int combine_f32gate(const void* fine, const void* out_c, const void* gate, int gate_mode,
                    int gate_heads, void* out, int64_t bh, int64_t sq, int D, int be, int dtype,
                    hipStream_t s);
// The shape checks combine_f32gate makes, for callers that must reject a call
// before launching anything else.
bool combine_f32gate_shape_ok(int64_t bh, int64_t sq, int D, int be, int dtype);
// Up to four tensors whose blocks of be rows become blocks of kbe rows, or back
// (block_move, tiling.hip): rows of the result, bytes of a source and a result
// row.
struct BlockMove {
  const void* src[4];
  void* dst[4];
  int64_t rows[4];
  int src_bytes[4], dst_bytes[4], unit[4];
  int n, be, kbe;
};
int block_move(BlockMove& m, bool pad, hipStream_t s);
// vsa_sparse_fwd / _bwd_dq / _bwd_dkdv for query blocks of which only the first
// `rows` rows exist (the caller's volume, where the blocks are padded to a
// volume the kernels have); the others are zero in q and dout, and no one reads
// their results.  The bf16 / fp16 forward and dQ multiply nothing for 32 rows
// that do not exist (their results are those of rows of zeros), and dK / dV at
// block 64 takes no items of them.
int sparse_fwd_rows(int rows, const void* q, const void* k, const void* v, const int32_t* selected,
                    const int32_t* kv_vbs, void* out, void* fine_out, float* lse,
                    const void* out_c, const void* gate, int32_t gate_mode, int32_t gate_heads,
                    int64_t bh, int64_t sq, int64_t skv, int32_t D, int32_t be, int32_t topk,
                    float scale, int32_t dtype, void* stream);
int sparse_bwd_dq_rows(int rows, const void* q, const void* k, const void* v, const void* dout,
                       const float* lse, const float* delta, const int32_t* selected,
                       const int32_t* kv_vbs, void* dq, const void* d_q_c, const int32_t* q_vbs,
                       int64_t bh, int64_t sq, int64_t skv, int32_t D, int32_t be, int32_t topk,
                       float scale, int32_t dtype, void* stream);
int sparse_bwd_dkdv_rows(int rows, const void* q, const void* k, const void* v, const void* dout,
                         const float* lse, const float* delta, const int32_t* counts,
                         const int32_t* offsets, const int32_t* inverse, const int32_t* kv_vbs,
                         void* dk, void* dv, const void* d_k_c, const void* d_v_c, int64_t bh,
                         int64_t sq, int64_t skv, int32_t D, int32_t be, int32_t topk, float scale,
                         int32_t* tile_order, int32_t dtype, void* stream);
// Scheduling counters (take_entry) of the persistent forward and dQ kernels for
// launches on stream s, from a file-scope device array (common.hip): one slot
// of zeroed counters per (device, stream), which every launch leaves zeroed.
// nullptr when the slots are all taken or s is not on the current device: the
// kernels then use a fixed stride over their XCD's range.
int32_t* sched_counters(hipStream_t s);
}  // namespace vsa
