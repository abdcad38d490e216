// Library-internal context, error plumbing and launch helpers.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdio>
#include <stdexcept>
#include <string>

#include "../../../include/malkin_hip.h"

struct mk_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  int n_cu = 0;
  char name[64] = {0};
  void* scratch = nullptr;  // per-context device scratch (partial reductions), allocated once at init
  size_t scratch_bytes = 0;
  void* topk_cand = nullptr;  // topk_workspace() bytes for mk_topk, allocated at init and never moved: a captured graph keeps
                              // its address
  int32_t* meta = nullptr;  // 64 bytes of per-call metadata (words 0..3: mk_attend_gqa's token layout, 4: attention's
                            // route), allocated at init
};

namespace mk {

void set_error(const char* fmt, ...);
// Counts one host wait on the device (a stream or event synchronization), for mk_host_waits().
void count_host_wait();
// Records the HIP error and returns MK_ERR_HIP.
int hip_fail(hipError_t e, const char* what);

// Errors raised inside library code; the extern "C" wrappers turn them into status codes.
struct Error : std::runtime_error {
  int code;
  Error(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

inline void check(hipError_t e, const char* what) {
  if (e != hipSuccess) throw Error(MK_ERR_HIP, std::string(what) + ": " + hipGetErrorString(e));
}

// The launch's own error (bad configuration) and any asynchronous fault reported so far.
inline void check_launch(const char* what) { check(hipGetLastError(), what); }

// Compute units of the current device (queried once: the library runs one device per process).
inline int device_cus() {
  static int n = 0;
  if (n == 0) {
    int dev = 0;
    check(hipGetDevice(&dev), "hipGetDevice");
    check(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev), "hipDeviceGetAttribute");
  }
  return n;
}

// Allows launches of Kernel up to `bytes` of dynamic LDS (past the default 64 KB); once per kernel, from any thread.
template <auto Kernel>
void allow_lds(int bytes) {
  static const bool set = (check(hipFuncSetAttribute(reinterpret_cast<const void*>(Kernel),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, bytes),
                                 "hipFuncSetAttribute"),
                           true);
  (void)set;
}

// The walks over a sequence's keys that attention on the matrix cores makes for a plain batch, per KV head: for each
// block of 16 / G consecutive tokens one per sequence among them. All blocks' and the most of one block.
struct AttnWalks {
  int all = 0, most = 0;
};
AttnWalks attention_walks(const int32_t* host_seq, int n, int G);

// mk_attention (xq NULL) and mk_attention_q8 for a caller that knows the batch's walks on the host.
int attention_batch(mk_ctx* ctx, const float* q, int64_t q_stride, float* out, int64_t out_stride, int n, int n_head,
                    const mk_kv_cache* kv, int layer, const int32_t* seq, const int32_t* n_keys, const int32_t* anc_off,
                    const int32_t* anc, int max_keys, void* xq, const AttnWalks* walks);

template <typename F>
int guard(F&& f) {
  try {
    f();
    return MK_OK;
  } catch (const Error& e) {
    set_error("%s", e.what());
    return e.code;
  } catch (const std::exception& e) {
    set_error("%s", e.what());
    return MK_ERR_INVALID;
  }
}

inline void require(bool ok, const char* msg) {
  if (!ok) throw Error(MK_ERR_INVALID, msg);
}

}  // namespace mk
