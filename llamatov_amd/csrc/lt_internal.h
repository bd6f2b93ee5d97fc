// lt_internal.h -- shared declarations of the libllamatov_hip.so translation units.
#pragma once

#include <hip/hip_runtime.h>
#include <cstddef>
#include <cstdint>

#include "../../include/llamatov_hip.h"
#include "lt_numerics.h"

struct lt_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  bool capturing = false;
  int num_cus = 0;
  // the device address of lt_attn.hip's scratch array on this context's device (bound at
  // lt_init by lt_attn_scratch_bind), or null with the lookup's error in attn_scratch_err
  void* attn_scratch = nullptr;
  size_t attn_scratch_bytes = 0;
  hipError_t attn_scratch_err = hipSuccess;
};

// Binds ctx->attn_scratch to the device copy of the attention scratch array (the device
// must be current).  Never fails the caller: a failed lookup is kept in attn_scratch_err and
// reported by the entry point that needs the scratch.
void lt_attn_scratch_bind(lt_ctx* ctx);
// Gives the scratch back when ctx owns it (lt_free_ctx).
void lt_attn_scratch_release(lt_ctx* ctx);

int lt_fail(int code, const char* fmt, ...);
int lt_fail_hip(hipError_t e, const char* what, const char* file, int line);
int lt_check_launch(const char* kernel);

#define LT_CHECK(call)                                              \
  do {                                                              \
    hipError_t e_ = (call);                                         \
    if (e_ != hipSuccess) return lt_fail_hip(e_, #call, __FILE__, __LINE__); \
  } while (0)

#define LT_REQUIRE(cond, ...)                                       \
  do {                                                              \
    if (!(cond)) return lt_fail(LT_EINVAL, __VA_ARGS__);            \
  } while (0)

static inline bool lt_aligned(const void* p, size_t a) { return ((uintptr_t)p % a) == 0; }

// Split-K attention workspace for `rows` = batch * nh query heads and nsplit splits:
// per-split maxima m[rows][nsplit], sums z[rows][nsplit], outputs o[rows][nsplit][hd]
// (16-byte aligned).
struct AttnWs {
  float* m;
  float* z;
  float* o;
};

static inline size_t lt_attn_ws_bytes(int rows, int hd, int nsplit) {
  const size_t nrow = (size_t)rows * nsplit;
  return nrow * (size_t)(2 + hd) * sizeof(float) + 256;
}

static inline AttnWs lt_attn_ws_layout(void* ws, int rows, int hd, int nsplit) {
  const size_t nrow = (size_t)rows * nsplit;
  AttnWs w;
  w.m = (float*)ws;
  w.z = w.m + nrow;
  w.o = (float*)(((uintptr_t)(w.z + nrow) + 15) & ~(uintptr_t)15);
  return w;
}

// Causal prefill attention on the matrix cores (lt_attn_mm.hip): T query rows (q_stride floats
// apart) of one sequence over its cache, query t attending *len + t + 1 positions.
struct LtAttnMm {
  const float* q;
  int q_stride;
  const void* kc;
  const void* vc;
  const int* len;
  float* out;
  int T, nh, nkv;
  float scale;
  int maxt, nsplit;
  int cap, ntiles;   // set by the launcher: positions held in LDS, 16-row tiles in the grid
};
// Head sizes 64 and 128; one split past the shortest contexts (end: the most positions a row attends, as
// far as the caller knows), or a multiple of 16 splits over a long prompt whose context fits in LDS.
bool lt_attn_mm_covers(int hd, bool f16, int T, int maxt, int end, int nsplit);
int lt_attn_mm_prefill(lt_ctx* ctx, LtAttnMm A, int hd, bool f16);

// Unsplit decode attention, one workgroup per (head, sequence) (lt_attn_head.hip): the decode
// step (qkv, freqs; one sequence) or batched decode (q rows q_stride floats apart).
struct LtAttnHead {
  const float* qkv;
  const float* freqs;
  const float* q;
  int q_stride;
  void* kc;
  void* vc;
  const int* len;
  float* out;
  int8_t* oq;
  uint16_t* od;
  int obm;
  int batch, nh, nkv;
  float scale;
  int maxt;
  int rep;         // set by the launcher: nh / nkv
  uint32_t rnkv;   // set by the launcher: for pair / nkv
};
bool lt_attn_head_covers(const lt_ctx* ctx, int batch, int nh, int nkv, int hd, int maxt, bool step);
int lt_attn_head(lt_ctx* ctx, LtAttnHead A, int hd, bool f16, bool step);

// Device helpers shared by the kernel translation units.
__device__ __forceinline__ float lt_h2f(uint16_t h) {
  return static_cast<float>(__builtin_bit_cast(_Float16, h));
}
