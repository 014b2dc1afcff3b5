// apcost — sharding-cost evaluation kernels for MI355X (gfx950) and their C ABI.
//
// Built with -ffp-contract=off: every fp64 operation below is a single IEEE
// rounding in the order the reference's Python evaluates it, so results are
// bit-identical to CPython's floats rather than merely close.
//
// Reference functions restated here (batched over the whole graph):
//   autoparallel/collective_runtime_estimation.py:22-153
//   autoparallel/compute_estimation.py:211-229, 302-365
//   autoparallel/optimize_sharding.py:306-379
//   torch/distributed/tensor/_collective_utils.py:230-313
//   torch/_prims_common/__init__.py:252-292
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstddef>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <type_traits>

#include "apcost.h"
#include "apcost_error.h"

static thread_local char g_err[512] = "";

int apc_internal::fail(int code, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

using apc_internal::check_params;
using apc_internal::fail;

namespace {

int check_launch(const char *what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(-3, "%s: %s", what, hipGetErrorString(e));
  return 0;
}

constexpr int kBlock = 256;

// ------------------------------------------------------------------------------------------
// placement codes
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ int kind_of(uint32_t c) { return (int)(c >> 6); }  // 0 R, 1 P, 2 S
__device__ __forceinline__ int dim_of(uint32_t c) { return (int)(c & 0x0F); }

// A load from a wave-uniform address of a table that no kernel of this library writes while it
// reads it (the uploaded encoding): through the constant address space, i.e. the scalar cache,
// into scalar registers.  (Left as a plain load the compiler takes such an address through vector
// memory, where the load queues behind the wavefront's other vector loads.)
#define APC_CONSTANT __attribute__((address_space(4)))
template <typename T>
__device__ __forceinline__ T uniform_load(const T *p) {
  return *(const APC_CONSTANT T *)p;
}
// A place in LDS as its address: what a lane looks up lies at addresses it adds up, and an offset known when the code is
// compiled becomes part of the load.
#define APC_LDS __attribute__((address_space(3)))
typedef uint32_t lds_address;
__device__ __forceinline__ lds_address address_in_lds(const void *p) { return (lds_address)(uintptr_t)(const APC_LDS char *)p; }
template <typename T>
__device__ __forceinline__ T lds_read(lds_address at) {
  return *(const APC_LDS T *)(uintptr_t)at;
}
template <typename T>
__device__ __forceinline__ void lds_write(lds_address at, T value) {
  *(APC_LDS T *)(uintptr_t)at = value;
}
// A lane's element of an array that starts at a wave-uniform address: the address stays a pair of scalar registers and
// a 32-bit offset per lane.  (As one 64-bit index per lane a tile's eleven loads took 40 vector instructions for their addresses.)
template <typename T>
__device__ __forceinline__ T load_of_lane(const T *base, uint32_t lane) {
  return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + lane * (uint32_t)sizeof(T));
}
// A plain store that is written through to memory (system scope, no ordering).  What a launch of
// a few tens of MB leaves in the L2 is written back when the kernel ends, after its last
// wavefront, and the launch lasts until that is done; written through, the lines leave while the
// wavefronts still work.  For the tables of a small pass only: a large table streams through the
// L2 anyway, and its tile kernels lose what the L2 does for them when neighbouring wavefronts fill
// a line together (write-through there: Llama-3-70B 126 -> 221 us, the stress table 1.19 -> 1.24 ms).
template <typename T>
__device__ __forceinline__ void store_through(T *p, T value) {
  __hip_atomic_store(p, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
// Where a launch's arguments lie.  The table kernels take more than a kilobyte of them, and what a launch passes by value
// is read from a segment that the host has just written: every compute unit fetches it past the caches.  A launch that
// is repeated keeps its arguments in a block of device memory, which the L2 holds, and passes the block's address; `kept`
// is NULL where a launch is made once, and its arguments are then the by-value ones, which every kernel takes last, behind
// kLaunchHeadBytes of others.  (Kernels that read 1 KB of arguments and store 2.3 MB, back to back: 5.6 us a launch by
// value, 3.15 from a block, 2.45 without the arguments.  The planner's pass: 1.7 M entries on (32, 8) over packed tiles 8.9 ->
// 8.15 us, 20 M on (16, 8, 4) in two launches 70.2 -> 68.7, 2.6 M on (12, 6) over staged tiles, whose wavefronts have other
// loads to wait for at that time, 18.4 -> 18.7.)
// The host fills the by-value arguments in, and waits for room for them, for every launch, read or not.  The kernels of small passes,
// which last no longer than that, have a form without them (KEPT); the others, the two-launch passes' among them, choose where
// they run (every such form is one more kernel to compile: the library 4.7 -> 6.0 MB).  (Together with a call that
// does not go through boxed values: one block on (64,) 4.95 -> 3.3 us a pass, 399 k entries on (8, 8, 8) 7.0 -> 6.55, 420 k on (12, 6)
// 7.1 -> 6.6.)
constexpr size_t kLaunchHeadBytes = 40;
template <typename Block, bool KEPT>
struct BlockByValue {
  Block block;
};
template <typename Block>
struct BlockByValue<Block, true> {};
template <bool KEPT, typename Block>
__device__ __forceinline__ const Block &launch_block(const Block *kept) {
  static_assert(alignof(Block) == 8, "the block follows the other arguments without padding");
  // (chosen as a number: of two pointers, of which one comes from the global address space, the compiler makes a generic
  // one, and of every load through it a flat one)
  const uint64_t by_value = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr() + kLaunchHeadBytes;
  const uint64_t at = KEPT || kept ? (uint64_t)kept : by_value;
  return *(const Block *)(const APC_CONSTANT Block *)at;
}
// (the arguments of every such kernel; `kept` arrives in registers with the wavefront, as do those in front of it)
#define APC_LAUNCH_PARAMS(BLOCK_, KEPT_) \
  const void *work, int n_tiles, int xcd_shift, int64_t tile_blocks, double *cost_out, const BLOCK_ *kept, BlockByValue<BLOCK_, KEPT_> by_value

typedef int32_t i32x16 __attribute__((ext_vector_type(16)));
typedef int64_t i64x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// The value lane `lane` (wave-uniform) holds.
__device__ __forceinline__ int64_t value_of_lane(int64_t x, int lane) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, lane);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)((uint64_t)x >> 32), lane);
  return (int64_t)(((uint64_t)hi << 32) | lo);
}

// Kernel arguments a wavefront will need, fetched now: the compiler loads an argument where it
// is first used, each behind the wait of whatever came before it, and a chain of such loads in
// front of a tile's own loads cost more than the loads themselves.  Naming the values as scalar
// operands of an (empty) asm statement puts their loads here, together, under one wait.
// One statement for all of them: a load may be moved past an asm statement that does not name it.
template <typename T0>
__device__ __forceinline__ void fetch_arguments_now(T0 v0) {
  __asm__ volatile("" ::"s"(v0));
}
template <typename T0, typename T1>
__device__ __forceinline__ void fetch_arguments_now(T0 v0, T1 v1) {
  __asm__ volatile("" ::"s"(v0), "s"(v1));
}
template <typename T0, typename T1, typename T2>
__device__ __forceinline__ void fetch_arguments_now(T0 v0, T1 v1, T2 v2) {
  __asm__ volatile("" ::"s"(v0), "s"(v1), "s"(v2));
}
template <typename T0, typename T1, typename T2, typename T3>
__device__ __forceinline__ void fetch_arguments_now(T0 v0, T1 v1, T2 v2, T3 v3) {
  __asm__ volatile("" ::"s"(v0), "s"(v1), "s"(v2), "s"(v3));
}
template <typename T0, typename T1, typename T2, typename T3, typename T4>
__device__ __forceinline__ void fetch_arguments_now(T0 v0, T1 v1, T2 v2, T3 v3, T4 v4) {
  __asm__ volatile("" ::"s"(v0), "s"(v1), "s"(v2), "s"(v3), "s"(v4));
}
template <typename T0, typename T1, typename T2, typename T3, typename T4, typename T5>
__device__ __forceinline__ void fetch_arguments_now(T0 v0, T1 v1, T2 v2, T3 v3, T4 v4, T5 v5) {
  __asm__ volatile("" ::"s"(v0), "s"(v1), "s"(v2), "s"(v3), "s"(v4), "s"(v5));
}
template <typename T0, typename T1, typename T2, typename T3, typename T4, typename T5, typename T6>
__device__ __forceinline__ void fetch_arguments_now(T0 v0, T1 v1, T2 v2, T3 v3, T4 v4, T5 v5, T6 v6) {
  __asm__ volatile("" ::"s"(v0), "s"(v1), "s"(v2), "s"(v3), "s"(v4), "s"(v5), "s"(v6));
}
template <typename T0, typename T1, typename T2, typename T3, typename T4, typename T5, typename T6, typename T7>
__device__ __forceinline__ void fetch_arguments_now(T0 v0, T1 v1, T2 v2, T3 v3, T4 v4, T5 v5, T6 v6, T7 v7) {
  __asm__ volatile("" ::"s"(v0), "s"(v1), "s"(v2), "s"(v3), "s"(v4), "s"(v5), "s"(v6), "s"(v7));
}
template <typename T0, typename T1, typename T2, typename T3, typename T4, typename T5, typename T6, typename T7, typename T8>
__device__ __forceinline__ void fetch_arguments_now(T0 v0, T1 v1, T2 v2, T3 v3, T4 v4, T5 v5, T6 v6, T7 v7, T8 v8) {
  __asm__ volatile("" ::"s"(v0), "s"(v1), "s"(v2), "s"(v3), "s"(v4), "s"(v5), "s"(v6), "s"(v7), "s"(v8));
}
template <typename T0, typename T1, typename T2, typename T3, typename T4, typename T5, typename T6, typename T7, typename T8, typename T9>
__device__ __forceinline__ void fetch_arguments_now(T0 v0, T1 v1, T2 v2, T3 v3, T4 v4, T5 v5, T6 v6, T7 v7, T8 v8, T9 v9) {
  __asm__ volatile("" ::"s"(v0), "s"(v1), "s"(v2), "s"(v3), "s"(v4), "s"(v5), "s"(v6), "s"(v7), "s"(v8), "s"(v9));
}
template <typename T0, typename T1, typename T2, typename T3, typename T4, typename T5, typename T6, typename T7, typename T8, typename T9, typename T10>
__device__ __forceinline__ void fetch_arguments_now(T0 v0, T1 v1, T2 v2, T3 v3, T4 v4, T5 v5, T6 v6, T7 v7, T8 v8, T9 v9, T10 v10) {
  __asm__ volatile("" ::"s"(v0), "s"(v1), "s"(v2), "s"(v3), "s"(v4), "s"(v5), "s"(v6), "s"(v7), "s"(v8), "s"(v9), "s"(v10));
}
template <typename T0, typename T1, typename T2, typename T3, typename T4, typename T5, typename T6, typename T7, typename T8, typename T9, typename T10, typename T11>
__device__ __forceinline__ void fetch_arguments_now(T0 v0, T1 v1, T2 v2, T3 v3, T4 v4, T5 v5, T6 v6, T7 v7, T8 v8, T9 v9, T10 v10, T11 v11) {
  __asm__ volatile("" ::"s"(v0), "s"(v1), "s"(v2), "s"(v3), "s"(v4), "s"(v5), "s"(v6), "s"(v7), "s"(v8), "s"(v9), "s"(v10), "s"(v11));
}
template <typename T0, typename T1, typename T2, typename T3, typename T4, typename T5, typename T6, typename T7, typename T8, typename T9, typename T10, typename T11, typename T12>
__device__ __forceinline__ void fetch_arguments_now(T0 v0, T1 v1, T2 v2, T3 v3, T4 v4, T5 v5, T6 v6, T7 v7, T8 v8, T9 v9, T10 v10, T11 v11, T12 v12) {
  __asm__ volatile("" ::"s"(v0), "s"(v1), "s"(v2), "s"(v3), "s"(v4), "s"(v5), "s"(v6), "s"(v7), "s"(v8), "s"(v9), "s"(v10), "s"(v11), "s"(v12));
}
template <typename T0, typename T1, typename T2, typename T3, typename T4, typename T5, typename T6, typename T7, typename T8, typename T9, typename T10, typename T11, typename T12, typename T13>
__device__ __forceinline__ void fetch_arguments_now(T0 v0, T1 v1, T2 v2, T3 v3, T4 v4, T5 v5, T6 v6, T7 v7, T8 v8, T9 v9, T10 v10, T11 v11, T12 v12, T13 v13) {
  __asm__ volatile("" ::"s"(v0), "s"(v1), "s"(v2), "s"(v3), "s"(v4), "s"(v5), "s"(v6), "s"(v7), "s"(v8), "s"(v9), "s"(v10), "s"(v11), "s"(v12), "s"(v13));
}
template <typename T0, typename T1, typename T2, typename T3, typename T4, typename T5, typename T6, typename T7, typename T8, typename T9, typename T10, typename T11, typename T12, typename T13, typename T14>
__device__ __forceinline__ void fetch_arguments_now(T0 v0, T1 v1, T2 v2, T3 v3, T4 v4, T5 v5, T6 v6, T7 v7, T8 v8, T9 v9, T10 v10, T11 v11, T12 v12, T13 v13, T14 v14) {
  __asm__ volatile("" ::"s"(v0), "s"(v1), "s"(v2), "s"(v3), "s"(v4), "s"(v5), "s"(v6), "s"(v7), "s"(v8), "s"(v9), "s"(v10), "s"(v11), "s"(v12), "s"(v13), "s"(v14));
}
template <typename T0, typename T1, typename T2, typename T3, typename T4, typename T5, typename T6, typename T7, typename T8, typename T9, typename T10, typename T11, typename T12, typename T13, typename T14, typename T15>
__device__ __forceinline__ void fetch_arguments_now(T0 v0, T1 v1, T2 v2, T3 v3, T4 v4, T5 v5, T6 v6, T7 v7, T8 v8, T9 v9, T10 v10, T11 v11, T12 v12, T13 v13, T14 v14, T15 v15) {
  __asm__ volatile("" ::"s"(v0), "s"(v1), "s"(v2), "s"(v3), "s"(v4), "s"(v5), "s"(v6), "s"(v7), "s"(v8), "s"(v9), "s"(v10), "s"(v11), "s"(v12), "s"(v13), "s"(v14), "s"(v15));
}
template <typename T0, typename T1, typename T2, typename T3, typename T4, typename T5, typename T6, typename T7, typename T8, typename T9, typename T10, typename T11, typename T12, typename T13, typename T14, typename T15, typename T16>
__device__ __forceinline__ void fetch_arguments_now(T0 v0, T1 v1, T2 v2, T3 v3, T4 v4, T5 v5, T6 v6, T7 v7, T8 v8, T9 v9, T10 v10, T11 v11, T12 v12, T13 v13, T14 v14, T15 v15, T16 v16) {
  __asm__ volatile("" ::"s"(v0), "s"(v1), "s"(v2), "s"(v3), "s"(v4), "s"(v5), "s"(v6), "s"(v7), "s"(v8), "s"(v9), "s"(v10), "s"(v11), "s"(v12), "s"(v13), "s"(v14), "s"(v15), "s"(v16));
}
template <typename T0, typename T1, typename T2, typename T3, typename T4, typename T5, typename T6, typename T7, typename T8, typename T9, typename T10, typename T11, typename T12, typename T13, typename T14, typename T15, typename T16, typename T17>
__device__ __forceinline__ void fetch_arguments_now(T0 v0, T1 v1, T2 v2, T3 v3, T4 v4, T5 v5, T6 v6, T7 v7, T8 v8, T9 v9, T10 v10, T11 v11, T12 v12, T13 v13, T14 v14, T15 v15, T16 v16, T17 v17) {
  __asm__ volatile("" ::"s"(v0), "s"(v1), "s"(v2), "s"(v3), "s"(v4), "s"(v5), "s"(v6), "s"(v7), "s"(v8), "s"(v9), "s"(v10), "s"(v11), "s"(v12), "s"(v13), "s"(v14), "s"(v15), "s"(v16), "s"(v17));
}
template <typename T0, typename T1, typename T2, typename T3, typename T4, typename T5, typename T6, typename T7, typename T8, typename T9, typename T10, typename T11, typename T12, typename T13, typename T14, typename T15, typename T16, typename T17, typename T18>
__device__ __forceinline__ void fetch_arguments_now(T0 v0, T1 v1, T2 v2, T3 v3, T4 v4, T5 v5, T6 v6, T7 v7, T8 v8, T9 v9, T10 v10, T11 v11, T12 v12, T13 v13, T14 v14, T15 v15, T16 v16, T17 v17, T18 v18) {
  __asm__ volatile("" ::"s"(v0), "s"(v1), "s"(v2), "s"(v3), "s"(v4), "s"(v5), "s"(v6), "s"(v7), "s"(v8), "s"(v9), "s"(v10), "s"(v11), "s"(v12), "s"(v13), "s"(v14), "s"(v15), "s"(v16), "s"(v17), "s"(v18));
}
template <typename T0, typename T1, typename T2, typename T3, typename T4, typename T5, typename T6, typename T7, typename T8, typename T9, typename T10, typename T11, typename T12, typename T13, typename T14, typename T15, typename T16, typename T17, typename T18, typename T19>
__device__ __forceinline__ void fetch_arguments_now(T0 v0, T1 v1, T2 v2, T3 v3, T4 v4, T5 v5, T6 v6, T7 v7, T8 v8, T9 v9, T10 v10, T11 v11, T12 v12, T13 v13, T14 v14, T15 v15, T16 v16, T17 v17, T18 v18, T19 v19) {
  __asm__ volatile("" ::"s"(v0), "s"(v1), "s"(v2), "s"(v3), "s"(v4), "s"(v5), "s"(v6), "s"(v7), "s"(v8), "s"(v9), "s"(v10), "s"(v11), "s"(v12), "s"(v13), "s"(v14), "s"(v15), "s"(v16), "s"(v17), "s"(v18), "s"(v19));
}
template <typename T0, typename T1, typename T2, typename T3, typename T4, typename T5, typename T6, typename T7, typename T8, typename T9, typename T10, typename T11, typename T12, typename T13, typename T14, typename T15, typename T16, typename T17, typename T18, typename T19, typename T20>
__device__ __forceinline__ void fetch_arguments_now(T0 v0, T1 v1, T2 v2, T3 v3, T4 v4, T5 v5, T6 v6, T7 v7, T8 v8, T9 v9, T10 v10, T11 v11, T12 v12, T13 v13, T14 v14, T15 v15, T16 v16, T17 v17, T18 v18, T19 v19, T20 v20) {
  __asm__ volatile("" ::"s"(v0), "s"(v1), "s"(v2), "s"(v3), "s"(v4), "s"(v5), "s"(v6), "s"(v7), "s"(v8), "s"(v9), "s"(v10), "s"(v11), "s"(v12), "s"(v13), "s"(v14), "s"(v15), "s"(v16), "s"(v17), "s"(v18), "s"(v19), "s"(v20));
}
template <typename T0, typename T1, typename T2, typename T3, typename T4, typename T5, typename T6, typename T7, typename T8, typename T9, typename T10, typename T11, typename T12, typename T13, typename T14, typename T15, typename T16, typename T17, typename T18, typename T19, typename T20, typename T21>
__device__ __forceinline__ void fetch_arguments_now(T0 v0, T1 v1, T2 v2, T3 v3, T4 v4, T5 v5, T6 v6, T7 v7, T8 v8, T9 v9, T10 v10, T11 v11, T12 v12, T13 v13, T14 v14, T15 v15, T16 v16, T17 v17, T18 v18, T19 v19, T20 v20, T21 v21) {
  __asm__ volatile("" ::"s"(v0), "s"(v1), "s"(v2), "s"(v3), "s"(v4), "s"(v5), "s"(v6), "s"(v7), "s"(v8), "s"(v9), "s"(v10), "s"(v11), "s"(v12), "s"(v13), "s"(v14), "s"(v15), "s"(v16), "s"(v17), "s"(v18), "s"(v19), "s"(v20), "s"(v21));
}
template <typename T0, typename T1, typename T2, typename T3, typename T4, typename T5, typename T6, typename T7, typename T8, typename T9, typename T10, typename T11, typename T12, typename T13, typename T14, typename T15, typename T16, typename T17, typename T18, typename T19, typename T20, typename T21, typename T22>
__device__ __forceinline__ void fetch_arguments_now(T0 v0, T1 v1, T2 v2, T3 v3, T4 v4, T5 v5, T6 v6, T7 v7, T8 v8, T9 v9, T10 v10, T11 v11, T12 v12, T13 v13, T14 v14, T15 v15, T16 v16, T17 v17, T18 v18, T19 v19, T20 v20, T21 v21, T22 v22) {
  __asm__ volatile("" ::"s"(v0), "s"(v1), "s"(v2), "s"(v3), "s"(v4), "s"(v5), "s"(v6), "s"(v7), "s"(v8), "s"(v9), "s"(v10), "s"(v11), "s"(v12), "s"(v13), "s"(v14), "s"(v15), "s"(v16), "s"(v17), "s"(v18), "s"(v19), "s"(v20), "s"(v21), "s"(v22));
}
template <typename T0, typename T1, typename T2, typename T3, typename T4, typename T5, typename T6, typename T7, typename T8, typename T9, typename T10, typename T11, typename T12, typename T13, typename T14, typename T15, typename T16, typename T17, typename T18, typename T19, typename T20, typename T21, typename T22, typename T23>
__device__ __forceinline__ void fetch_arguments_now(T0 v0, T1 v1, T2 v2, T3 v3, T4 v4, T5 v5, T6 v6, T7 v7, T8 v8, T9 v9, T10 v10, T11 v11, T12 v12, T13 v13, T14 v14, T15 v15, T16 v16, T17 v17, T18 v18, T19 v19, T20 v20, T21 v21, T22 v22, T23 v23) {
  __asm__ volatile("" ::"s"(v0), "s"(v1), "s"(v2), "s"(v3), "s"(v4), "s"(v5), "s"(v6), "s"(v7), "s"(v8), "s"(v9), "s"(v10), "s"(v11), "s"(v12), "s"(v13), "s"(v14), "s"(v15), "s"(v16), "s"(v17), "s"(v18), "s"(v19), "s"(v20), "s"(v21), "s"(v22), "s"(v23));
}

// Element `i` (a per-lane index below M) of one of the arrays of the kernel parameters, as a select chain over scalar registers.  (Indexing the array by a lane value
// makes the compiler read the kernel arguments through vector memory, and a vector load
// waits behind every store the compute unit has in flight.)
template <int M, typename T, int N>
__device__ __forceinline__ T pick(const T (&v)[N], int i) {
  static_assert(M <= N, "array shorter than the mesh");
  T e[M];  // every element is read (scalar loads) before the selects, so they stay selects
#pragma unroll
  for (int k = 0; k < M; ++k) e[k] = v[k];
  T r = e[0];
#pragma unroll
  for (int k = 1; k < M; ++k) r = i == k ? e[k] : r;
  return r;
}

// compute_estimation.py:302-314
__device__ __forceinline__ double rw_time(double bytes, const apc_params &p) {
  double t = bytes / p.hbm_bw * 1e6;
  t = t / p.rw_eff;
  return t > p.launch_floor ? t : p.launch_floor;
}

// torch _collective_utils.py:281-313: latency + bandwidth term of a ring collective over a dim of `size` devices
__device__ __forceinline__ double ring(double gb, const apc_params &p, int size, double lat, double bandwidth, int hops) {
  double latency = p.base_latency + (double)hops * lat;
  double bw = (gb * (double)hops / (double)size) / bandwidth;
  return latency + bw * 1e6;
}

// a / b for a divisor whose correctly rounded reciprocal y = RN(1 / b) is known: one
// multiply and two Newton corrections, each residual computed exactly by an FMA.  With y
// correctly rounded the second correction returns the correctly rounded quotient (Markstein),
// i.e. the same bits as the division instruction sequence, at a sixth of its cost.  The
// reciprocals travel in apc_params and are checked against 1.0 / b on the host.
__device__ __forceinline__ double div_by(double a, double b, double y) {
  double q = a * y;
  double r = __builtin_fma(-b, q, a);
  q = __builtin_fma(r, y, q);
  r = __builtin_fma(-b, q, a);
  return __builtin_fma(r, y, q);
}

__device__ __forceinline__ double rw_time_r(double bytes, const apc_params &p) {
  double t = div_by(bytes, p.hbm_bw, p.inv_hbm_bw) * 1e6;
  t = div_by(t, p.rw_eff, p.inv_rw_eff);
  return t > p.launch_floor ? t : p.launch_floor;
}

__device__ __forceinline__ double ring_r(double gb, const apc_params &p, int d, int hops) {
  const double latency = p.base_latency + (double)hops * p.lat[d];
  const double bw = div_by(div_by(gb * (double)hops, (double)p.mesh_size[d], p.inv_mesh[d]), p.bw[d], p.inv_bw[d]);
  return latency + bw * 1e6;
}

// collective_runtime_estimation.py:37-153 for one (producer spec, consumer spec) pair.
// gb = bytes / num_shards / 1024^3 of the producer spec, cont = global contiguity.
template <int M>
__device__ __forceinline__ double entry_cost(uint32_t srcp, uint32_t tgtp, double gb, bool cont,
                                             const apc_params &p) {
  if (srcp == 0u) {  // fully replicated producer (:56-62)
    bool tgt_partial = false;
#pragma unroll
    for (int i = 0; i < M; ++i) tgt_partial |= kind_of((tgtp >> (8 * i)) & 0xFF) == 1;
    return tgt_partial ? INFINITY : 0.0;
  }
  bool flip = false;
  if (M == 2) {  // :146-151
    flip = srcp == 0x4040u && kind_of(tgtp & 0xFF) == 2 && kind_of((tgtp >> 8) & 0xFF) == 2;
  }
  double cost = 0.0;
#pragma unroll
  for (int k = 0; k < M; ++k) {
    const int i = (M == 2 && flip) ? 1 - k : k;
    const uint32_t c = (srcp >> (8 * i)) & 0xFF, t = (tgtp >> (8 * i)) & 0xFF;
    if (c == t) continue;
    const int size = pick<M>(p.mesh_size, i);
    const double n = (double)size, lat = pick<M>(p.lat, i), bw = pick<M>(p.bw, i);
    if (!cont) cost += rw_time(gb * 2 * 1073741824.0, p);
    const int ck = kind_of(c), tk = kind_of(t);
    if (ck == 2 && tk == 0) {  // all-gather (:83-96)
      gb *= n;
      cost += ring(gb, p, size, lat, bw, size - 1);
      if (dim_of(c) != 0) cost += rw_time(gb * 2 * 1073741824.0, p);
    } else if (ck == 2 && tk == 2) {  // all-to-all (:97-113)
      double a2a = ring(gb, p, size, lat, bw, size - 1);
      a2a *= p.a2a_scale;
      cost += a2a;
      const int copies = (dim_of(c) != 0) + (dim_of(t) != 0);
      cost += (double)copies * rw_time(gb * 2 * 1073741824.0, p);
    } else if (ck == 1 && tk == 0) {  // all-reduce (:115-117)
      cost += ring(gb, p, size, lat, bw, 2 * (size - 1));
    } else if (ck == 1 && tk == 2) {  // reduce-scatter (:118-130)
      cost += ring(gb, p, size, lat, bw, size - 1);
      if (dim_of(t) != 0) cost += rw_time(gb * 2 * 1073741824.0, p);
      gb /= n;
    } else if (tk == 1 && ck != 1) {  // Shard->Partial, Replicate->Partial banned (:131-138)
      return INFINITY;
    }
    cont = true;  // :141
  }
  return cost;
}

// ------------------------------------------------------------------------------------------
// Running-bytes states.  The redistribution cost of an entry is a sum of per-mesh-dim terms,
// and every term is an expensive expression (fp64 divisions) of ONE quantity only: the
// running comm_bytes_gb at that dim.  For a given tensor that quantity takes few distinct
// values: it starts from bytes / num_shards (decided by WHICH mesh dims the producer
// shards: a mask of M bits) and every earlier dim either left it alone or applied its
// single possible update (x n after an all-gather when the producer shards that dim, / n
// after a reduce-scatter).  State (level L, mask, history) indexes every
// value that can occur; level L in [0, M) has 2^M masks x 2^L histories.  Behind the last dim
// (level M) only an all-gather there is charged, of a producer that shards it: mask and history
// hold the last dim, a quarter of the pairs, and are counted without it.  (4-D meshes: 304 states
// where all pairs are 496, in 22 KB of LDS instead of 36: four workgroups to a compute unit, not three.  5.1 M entries on
// (3, 2, 2, 2) 45.1 -> 33.7 us, 900 k 18.8 -> 13.7; 72 of 120 on 3-D meshes, 587 k on (6, 4, 2) 14.1 -> 12.0, 1.6 M 14.0 -> 12.2.)
// They are numbered mask by mask, and the states of a mask by level and history: a producer spec's first one and the
// place within its mask add up, so what an entry looks up by its two classes is the same for every producer spec.
// ------------------------------------------------------------------------------------------
template <int M>
struct States {
  static constexpr int kHalf = 1 << (M - 1);
  static constexpr int kPerMask = (1 << M) - 1;       // levels 0 .. M - 1
  static constexpr int kLast = kPerMask << M;         // of all masks; behind them, as they are counted below, level M
  static constexpr int kCount = kLast + kHalf * kHalf;
  // the first state of a mask
  __device__ static __forceinline__ int first(int mask) { return mask * kPerMask + (mask >= kHalf ? (mask & (kHalf - 1)) * kHalf : 0); }
  __device__ static __forceinline__ int index(int level, int mask, int hist) {
    return first(mask) + (level < M ? (1 << level) - 1 + hist : kPerMask + (hist & (kHalf - 1)));
  }
};
// ------------------------------------------------------------------------------------------
// XCD-aware work order.  The dispatcher deals workgroups to the chip's 8 XCDs round-robin by
// workgroup id, and every XCD has its own L2.  With the plain order, neighbouring tiles
// (which write neighbouring memory and share the cache lines at their boundaries) sit
// in eight different L2s and those lines are written back in parts.  Runs of kXcdRun consecutive tiles go to one XCD
// each, in turn; what is left behind the last full round of runs, in shares of one length.
// (An XCD used to take one contiguous share of all tiles: a table whose copies are tiled unevenly, 19 layers as an edge for 16
// and another for 3, then gave some XCDs five times the stores of others.  us a pass, contiguous shares / runs of 8 / 32 / 128
// tiles: 5.8 M entries in 19 layers on (64, 4) 22.6 / 18.1 / 17.7 / 20.4; 37 M in 40 layers on (8, 8, 8) 70 / 63 / 67 / 68,
// 73 M in 80 layers 131 / 137 / 126 / 127; the packed tables of 1.1 and 1.7 M as before.)
// ------------------------------------------------------------------------------------------
constexpr int kXcdRun = APC_TILE_RUN;
__device__ __forceinline__ int tile_of_block(int b, int n_tiles, int shift) {
  const int round = kXcdRun << shift, full = n_tiles & ~(round - 1);  // (a power of two)
  const int per = b < full ? kXcdRun : (n_tiles - full + (1 << shift) - 1) >> shift;
  const int within = b < full ? b & (round - 1) : b - full;
  return b - within + (within & ((1 << shift) - 1)) * per + (within >> shift);
}

// ------------------------------------------------------------------------------------------
// a7: bytes + contiguity per tensor
// ------------------------------------------------------------------------------------------
struct TensorTableArgs {
  int64_t n;
  const int32_t *rank, *itemsize;
  const int64_t *shape, *stride;
  int64_t *bytes;
  uint8_t *cont;
};

// Bytes and contiguity of one tensor (torch _collective_utils.py:230-232,
// _prims_common/__init__.py:252-292) from its zero-padded shape and stride rows, held in registers.
template <typename Row>
__device__ __forceinline__ void tensor_bytes_and_contiguity_of(int r, int64_t itemsize, const Row &x, const Row &y,
                                                               int64_t &nbytes, bool &contiguous) {
  nbytes = itemsize;
  int64_t expected = 1, expected_max = 1;
  bool ok = true;
#pragma unroll
  for (int i = APC_MAX_RANK - 1; i >= 0; --i) {
    if (i >= r) continue;
    nbytes *= x[i];
    if (x[i] == 1) continue;
    if (y[i] != expected && y[i] != expected_max) ok = false;
    expected_max *= (x[i] > 1 ? x[i] : 1);
    expected *= x[i];
  }
  contiguous = ok;
}

__device__ __forceinline__ void tensor_bytes_and_contiguity(int r, int64_t itemsize, const int64_t *sh, const int64_t *st,
                                                            int64_t &nbytes, bool &contiguous) {
  // the whole (zero-padded) rows are read at once, before the scan: one round of loads
  // instead of one per dim
  int64_t x[APC_MAX_RANK], y[APC_MAX_RANK];
#pragma unroll
  for (int i = 0; i < APC_MAX_RANK; ++i) {
    x[i] = sh[i];
    y[i] = st[i];
  }
  tensor_bytes_and_contiguity_of(r, itemsize, x, y, nbytes, contiguous);
}

// THROUGH: the rows are written through to memory (the packed pass: see store_through)
template <int BS, bool THROUGH = false>
__device__ __forceinline__ void tensor_tables_block(int64_t block, const TensorTableArgs &a) {
  const int64_t t = block * BS + threadIdx.x;
  if (t >= a.n) return;
  int64_t nbytes;
  bool ok;
  tensor_bytes_and_contiguity(a.rank[t], a.itemsize[t], a.shape + t * APC_MAX_RANK, a.stride + t * APC_MAX_RANK, nbytes, ok);
  if (THROUGH) {
    store_through(a.bytes + t, nbytes);
    store_through(a.cont + t, (uint8_t)(ok ? 1 : 0));
  } else {
    a.bytes[t] = nbytes;
    a.cont[t] = ok ? 1 : 0;
  }
}

__global__ __launch_bounds__(kBlock) void tensor_tables_kernel(TensorTableArgs a) {
  tensor_tables_block<kBlock>(blockIdx.x, a);
}

// ceil(x / m) for x >= 0 and a mesh size m whose correctly rounded reciprocal y is known.
// Below 2^52 the quotient is taken in fp64 (both operands exact, div_by rounds once, so the
// truncated value is off by at most one) and corrected by the exact integer remainder: a
// dozen instructions against the ~120 of a 64-bit integer division, which made this kernel
// VALU-bound.  Larger values take the integer division.
__device__ __forceinline__ int64_t ceil_div_by(int64_t x, int32_t m, double y) {
  const int64_t num = x + m - 1;
  if (num >> 52) return num / m;
  int64_t q = (int64_t)div_by((double)num, (double)m, y);
  int64_t rem = num - q * m;
  if (rem < 0) {
    q -= 1;
    rem += m;
  }
  if (rem >= m) q += 1;
  return q;
}

// ------------------------------------------------------------------------------------------
// a8: local shard shape / stride / counts per spec
// ------------------------------------------------------------------------------------------
struct SpecTableArgs {
  int64_t n;
  const uint32_t *codes;
  const int32_t *tensor, *rank, *itemsize;
  const int64_t *shape, *stride;
  int64_t *shards, *lshape, *lstride, *lnumel, *lbytes;
  int width;  // values per row of lshape / lstride: even, 2 .. APC_MAX_RANK, >= every tensor's rank
};

// s_rows: kBlock * (APC_MAX_RANK + 1) values of LDS
// Writes the staged rows of the workgroup (APC_MAX_RANK + 1 slots per row in LDS) to `out`, the
// first `width` values of each row, `live` values in all (rows x width), as one contiguous run,
// two values (one 16-byte store) per lane: width is even, so a pair never straddles rows.
template <int BS>
__device__ __forceinline__ void write_rows(int64_t *__restrict__ out, const int64_t *s_rows, int live, int width) {
  typedef int64_t pair_t __attribute__((ext_vector_type(2)));
  for (int k = 2 * threadIdx.x; k < live; k += 2 * BS) {
    const int r = k / width, c = k - r * width;
    const int64_t *src = s_rows + r * (APC_MAX_RANK + 1) + c;
    pair_t v = {src[0], src[1]};
    *reinterpret_cast<pair_t *>(out + k) = v;
  }
}

template <int BS>
__device__ __forceinline__ void spec_tables_block(int64_t block, const apc_params &p, const SpecTableArgs &a,
                                                  int64_t *s_rows) {
  const int64_t n = a.n;
  const uint32_t *__restrict__ codes = a.codes;
  const int32_t *__restrict__ tensor = a.tensor, *__restrict__ rank = a.rank, *__restrict__ itemsize = a.itemsize;
  const int64_t *__restrict__ shape = a.shape, *__restrict__ stride = a.stride;
  int64_t *__restrict__ shards = a.shards, *__restrict__ lshape = a.lshape, *__restrict__ lstride = a.lstride;
  int64_t *__restrict__ lnumel = a.lnumel, *__restrict__ lbytes = a.lbytes;
  // Each thread derives one spec in its own row of an LDS buffer (the Shard dim indexes the
  // row, so no register array is indexed by a lane value), first the shape and then, in the
  // same buffer, the stride; the workgroup (BS threads) writes each [BS][8] result block out
  // as one contiguous run.
  const int64_t base = block * BS;
  const int64_t s = base + threadIdx.x;
  int64_t *row = s_rows + threadIdx.x * (APC_MAX_RANK + 1);
  const int width = a.width;
  const int live = (int)(n - base < BS ? n - base : BS) * width;
  int t = -1, r = 0;
  uint32_t pc = 0;
  if (s < n) {
    t = tensor[s];
    if (t >= 0) {
      r = rank[t];
      pc = codes[s];
    }
  }
  // (every load is issued before the first store: a load behind stores waits for them)
  int64_t st[APC_MAX_RANK];
#pragma unroll
  for (int i = 0; i < APC_MAX_RANK; ++i) {
    row[i] = i < r ? shape[(int64_t)t * APC_MAX_RANK + i] : 0;
    st[i] = i < r ? stride[(int64_t)t * APC_MAX_RANK + i] : 0;
  }
  const int64_t item = t >= 0 ? itemsize[t] : 0;
  int64_t nsh = t >= 0 ? 1 : 0;
  for (int i = 0; i < p.mesh_ndim; ++i) {
    const uint32_t c = (pc >> (8 * i)) & 0xFF;
    if (kind_of(c) == 2) {
      const int d = dim_of(c);
      nsh *= p.mesh_size[i];
      if (d < APC_MAX_RANK) row[d] = ceil_div_by(row[d], p.mesh_size[i], p.inv_mesh[i]);
    }
  }
  if (s < n) {
    int64_t ne = 0, nb = 0;
    if (t >= 0) {
      ne = 1;
#pragma unroll
      for (int i = 0; i < APC_MAX_RANK; ++i)
        if (i < r) ne *= row[i];
      nb = ne * item;
    }
    shards[s] = nsh;
    lnumel[s] = ne;
    lbytes[s] = nb;
  }
  __syncthreads();
  write_rows<BS>(lshape + base * width, s_rows, live, width);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < APC_MAX_RANK; ++i) row[i] = st[i];
  for (int i = 0; i < p.mesh_ndim; ++i) {
    const uint32_t c = (pc >> (8 * i)) & 0xFF;
    if (kind_of(c) == 2) {
      const int d = dim_of(c);
      if (d - 1 > 0 && d - 1 < APC_MAX_RANK)  // compute_estimation.py:225-228
        row[d - 1] = ceil_div_by(row[d - 1], p.mesh_size[i], p.inv_mesh[i]);
    }
  }
  __syncthreads();
  write_rows<BS>(lstride + base * width, s_rows, live, width);
}

__global__ __launch_bounds__(kBlock) void spec_tables_kernel(apc_params p, SpecTableArgs a) {
  __shared__ int64_t s_rows[kBlock * (APC_MAX_RANK + 1)];
  spec_tables_block<kBlock>(blockIdx.x, p, a, s_rows);
}

// ------------------------------------------------------------------------------------------
// a9/a10: compute-cost tail per (node, strategy)
// ------------------------------------------------------------------------------------------
struct ComputeCostArgs {
  int64_t n;
  const int64_t *flops, *rw_bytes;
  const int8_t *dtype;
  const uint8_t *zero_cost;
  const int32_t *num_args;
  double *compute, *per_arg;
  int32_t *error_flag;
};

// Compute cost of one strategy (compute_estimation.py:334-365), the divisions taken through the checked reciprocals
// (div_by): gf / inv_gf = the device row's throughput for the strategy's dtype and its reciprocal, 0 when unsupported (then,
// with flops, the result is NaN).
__device__ __forceinline__ double compute_cost_through_reciprocals(const apc_params &p, bool zero_cost, int64_t rw_bytes,
                                                                   int64_t flops, double gf, double inv_gf) {
  if (zero_cost) return 0.0;
  const double rw = rw_time_r((double)rw_bytes, p);
  if (flops == 0) return rw;
  if (gf == 0.0) return NAN;  // compute_estimation.py:198-201 raises ValueError (flagged by compute_costs_block)
  double t = div_by((double)flops, gf, inv_gf) * 1e6;
  t = div_by(t, p.compute_eff, p.inv_compute_eff);
  return t > rw ? t : rw;
}

template <int BS, bool THROUGH = false>
__device__ __forceinline__ void compute_costs_block(int64_t block, const apc_params &p, const ComputeCostArgs &a) {
  const int64_t s = block * BS + threadIdx.x;
  if (s >= a.n) return;
  // (the divisions through the checked reciprocals: a third of the instructions; these workgroups share the chip with the
  // ones that write the matrices)
  const int dt = a.dtype[s];
  const bool zero = a.zero_cost[s] != 0;
  const int64_t flops = a.flops[s];
  const bool known = dt >= 0 && dt < APC_MAX_DTYPES;
  const double gf = known ? pick<APC_MAX_DTYPES>(p.gpu_flops, dt) : 0.0, inv_gf = known ? pick<APC_MAX_DTYPES>(p.inv_gpu_flops, dt) : 0.0;
  const double c = compute_cost_through_reciprocals(p, zero, a.rw_bytes[s], flops, gf, inv_gf);
  const bool unsupported = !zero && flops != 0 && gf == 0.0;
  if (unsupported && a.error_flag) *a.error_flag = 1;
  const double per_arg = c / (double)a.num_args[s];
  if (THROUGH) {
    if (a.compute) store_through(a.compute + s, c);
    if (a.per_arg) store_through(a.per_arg + s, per_arg);
  } else {
    if (a.compute) a.compute[s] = c;
    if (a.per_arg) a.per_arg[s] = per_arg;
  }
}

__global__ __launch_bounds__(kBlock) void compute_costs_kernel(apc_params p, ComputeCostArgs a) {
  compute_costs_block<kBlock>(blockIdx.x, p, a);
}

// ------------------------------------------------------------------------------------------
// a9, integer part: flop and byte counts per (node, strategy) from the local shard shapes.
// The reference runs every operator on fake tensors of the local shard shapes under torch's
// FlopCounterMode and adds the bytes of all tensor arguments and outputs
// (compute_estimation.py:232-299, 334-349).  For the operators torch's counter knows in the
// planned graphs the count is a closed form of the local shapes (torch/utils/flop_counter.py:
// mm_flop, bmm_flop, sdpa_flop_count, sdpa_backward_flop_count), and the bytes are the local
// bytes of the strategy's input and output specs (the rows of the spec table) plus a per-node
// constant (outputs of factories, tensor constants).  One recipe per node, written by the
// host; one thread per strategy.
// ------------------------------------------------------------------------------------------
struct StrategyInputArgs {
  int64_t n;
  const int32_t *strat_node;
  const int64_t *node_strat_begin;
  const int32_t *node_kind;        // APC_NODE_*
  const int8_t *node_dtype;
  const int64_t *node_const_bytes;
  const int64_t *node_row_begin;   // CSR over byte_rows
  const int32_t *byte_rows;        // first spec rows of the node's argument and output slots (strategy ss reads row + ss)
  const int32_t *node_flop_rows;   // [n_nodes, 4]: first spec rows of the tensors the flop formula reads
  const int64_t *local_shape;      // [n_specs, width]
  int32_t width;
  const int64_t *local_bytes;      // [n_specs]
  int64_t *flops, *rw_bytes;
  int8_t *dtype;
  uint8_t *zero_cost;
};

// b * m * n * 2 * k, in torch's order of multiplications (exact in int64 below 2^63)
__device__ __forceinline__ int64_t bmm_flops(int64_t b, int64_t m, int64_t k, int64_t n) { return b * m * n * 2 * k; }

__global__ __launch_bounds__(kBlock) void strategy_inputs_kernel(StrategyInputArgs a) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= a.n) return;
  const int node = a.strat_node[i];
  const int64_t ss = i - a.node_strat_begin[node];
  const int kind = a.node_kind[node];
  int64_t flops = 0, bytes = 0;
  if (kind != APC_NODE_ZERO_COST) {
    bytes = a.node_const_bytes[node];
    for (int64_t r = a.node_row_begin[node]; r < a.node_row_begin[node + 1]; ++r) bytes += a.local_bytes[a.byte_rows[r] + ss];
    const int32_t *rows = a.node_flop_rows + (int64_t)node * 4;
    const int w = a.width;
    // (a dim past the row's width reads as 1: the host checks ranks, this keeps the load inside the table)
    auto dim = [&](int t, int d) { return d < w ? a.local_shape[(rows[t] + ss) * w + d] : (int64_t)1; };
    if (kind == APC_NODE_MM) {  // [m, k] x [k, n]
      flops = dim(0, 0) * dim(1, 1) * 2 * dim(0, 1);
    } else if (kind == APC_NODE_BMM) {  // [b, m, k] x [b, k, n]
      flops = bmm_flops(dim(0, 0), dim(0, 1), dim(0, 2), dim(1, 2));
    } else if (kind == APC_NODE_SDPA || kind == APC_NODE_SDPA_BACKWARD) {
      // rows: query [b, h, s_q, d_q], key [b, h, s_k, d_q], value [b, h, s_k, d_v]
      const int64_t bh = dim(0, 0) * dim(0, 1), s_q = dim(0, 2), d_q = dim(0, 3), s_k = dim(1, 2), d_v = dim(2, 3);
      if (kind == APC_NODE_SDPA) {
        flops = bmm_flops(bh, s_q, d_q, s_k) + bmm_flops(bh, s_q, s_k, d_v);
      } else {  // recomputed scores, gradScores, gradV, gradQ, gradK
        flops = bmm_flops(bh, s_q, d_q, s_k) + bmm_flops(bh, s_q, d_v, s_k) + bmm_flops(bh, s_k, s_q, d_v) +
                bmm_flops(bh, s_q, s_k, d_q) + bmm_flops(bh, d_q, s_q, s_k);
      }
    }
  }
  a.flops[i] = flops;
  a.rw_bytes[i] = bytes;
  a.dtype[i] = a.node_dtype[node];
  a.zero_cost[i] = kind == APC_NODE_ZERO_COST ? 1 : 0;
}

// The three tables above in one launch: workgroups [0, spec_blocks) take the spec table (the
// largest), the next tensor_blocks the tensor table, the rest the compute costs.  None of the
// three reads another's output.
struct InputTablesBlock {
  apc_params p;
  TensorTableArgs t;
  SpecTableArgs sp;
  ComputeCostArgs c;
  int64_t spec_blocks, tensor_blocks;
};

template <bool KEPT>
__global__ __launch_bounds__(kBlock) void input_tables_kernel(APC_LAUNCH_PARAMS(InputTablesBlock, KEPT)) {
  __shared__ int64_t s_rows[kBlock * (APC_MAX_RANK + 1)];
  const InputTablesBlock &k = launch_block<KEPT>(kept);
  const int64_t b = blockIdx.x;
  if (b < k.spec_blocks) spec_tables_block<kBlock>(b, k.p, k.sp, s_rows);
  else if (b < k.spec_blocks + k.tensor_blocks) tensor_tables_block<kBlock>(b - k.spec_blocks, k.t);
  else compute_costs_block<kBlock>(b - k.spec_blocks - k.tensor_blocks, k.p, k.c);
}

// ------------------------------------------------------------------------------------------
// a1-a6: redistribution-cost matrices.  The unit of work is a tile: a rectangle of one edge's
// matrix.  A tile's producer and consumer specs and the per-state terms of the edge's tensor
// are staged in LDS (TileStage); the per-entry loop walks the mesh dims, looks the terms of
// the current state up and adds them in the reference's order, so results are bit-identical
// to evaluating every entry directly (entry_cost).  The direct evaluation remains the path
// for the rare case the states do not cover: producer specs of one edge that point at
// different tensors.
//
// One workgroup per tile.  (A variant in which a workgroup walked a run of tiles, one
// wavefront staging tile t+1 into a second LDS stage while the others computed and stored
// tile t, was measured 35 - 60 % slower on both large tables, also with the one-round
// staging below: fewer, longer-lived workgroups keep fewer stores in flight.)
// ------------------------------------------------------------------------------------------

// What is the same for every tile of a launch (see "Term arrays" and "Lookup words" below):
// the layout of the term arrays, the lookup words (by dim x 16 + producer class x 4 + consumer
// class), how a producer spec's running index starts and, for the power-of-two layout, the
// constants of every computed array.
constexpr int kMaxTermArrays = 16;
struct TermArrayConstants {  // value at exponent index j = max(lat + ldexp(B, j + shift), floor) x scale,
  double hops;               // B = RN(RN(RN(RN(bytes x hops) / div1) x 1e6) / div2)
  double div1, inv_div1;
  double div2, inv_div2;
  double lat;
  double floor;
  double scale;
  int32_t shift;
  int32_t pad_;
};
struct TermLayout {
  // What a tile's first wavefront copies into LDS, 16 bytes a lane (TileStage::image): the lookup words, then the constants
  // of arrays 2 .. of the power-of-two layout (TermArrayConstants)
  uint32_t image[APC_MAX_MESH * 16 + (kMaxTermArrays - 2) * (int)sizeof(TermArrayConstants) / 4];
  int32_t exponents;         // 0: general layout; else E, the number of exponents
  int32_t lg[APC_MAX_MESH];  // log2 of the mesh sizes (power-of-two layout)
  int32_t lg_total;          // L
  // the running index of a producer spec: index0 + the weights of the dims it shards + (general layout, where it shards
  // the last dim) last_weight x the mask of its other dims
  int32_t index0, index_weight[APC_MAX_MESH], last_weight;
  int32_t level_stride;      // bytes from one level's states to the next's (general layout; else 0), in units of 2^level - 1
  int32_t state_stride;      // bytes between the entries of two consecutive states / exponents
  uint32_t exponent_magic;   // ceil(65536 / E): t / E = (t * magic) >> 16 for t < 512
  double inv_rescale;        // 1.0 / params.rescale
};

struct TableArgs {
  const int64_t *tensor_bytes;
  const uint8_t *tensor_contiguous;
  const uint32_t *spec_codes;
  const int32_t *spec_tensor;
  const double *pt_values;
  const double *per_arg;
  const apc_tile *tiles;
  const int64_t *dup_entry_begin;
  double *comm_out;
  uint8_t *trans_out;
  double *cost_out;
  // When the tensor and compute-cost tables are produced by the same launch (build_tables_kernel)
  // a tile cannot read them: tensor_bytes / tensor_contiguous / per_arg are NULL and the tile
  // derives the few values it needs from the tables those are computed from.
  const int32_t *rank, *itemsize;
  const int64_t *shape, *stride;
  const int64_t *flops, *rw_bytes;
  const int8_t *dtype;
  const uint8_t *zero_cost;
  const int32_t *num_args;
  // Row minima written by the tiles themselves (NULL: not wanted).  Matrix rows are numbered
  // edge by edge (edge_row_begin[e] + consumer strategy); dup_row_begin[k] is the first row of
  // the identical edge whose first entry is dup_entry_begin[k].
  const int64_t *edge_row_begin;
  const int64_t *dup_row_begin;
  double *row_min_out;
  int32_t *row_arg_out;
  TermLayout lay;  // the launch's term-array layout and lookup-word bases
};

// Bytes and contiguity of tensor t: read from the tensor table, or (DERIVE) derived from its
// shape row.  A compile-time choice: as a run-time one it cost the tile kernel a third of
// its registers.
template <bool DERIVE>
__device__ __forceinline__ void tensor_info(const TableArgs &a, int t, int64_t &nbytes, bool &contiguous) {
  if (!DERIVE) {
    nbytes = a.tensor_bytes[t];
    contiguous = a.tensor_contiguous[t] != 0;
  } else {
    tensor_bytes_and_contiguity(a.rank[t], a.itemsize[t], a.shape + (int64_t)t * APC_MAX_RANK,
                                a.stride + (int64_t)t * APC_MAX_RANK, nbytes, contiguous);
  }
}


// What one mesh dim contributes, by (producer class, consumer class) with classes
// 0 Replicate, 1 Partial, 2 Shard(0), 3 Shard(d != 0); only consulted when the two placement
// codes differ.  One byte per pair:
//   bits 0-2  term array: 0 none, 1 all-gather, 2 reduce-scatter, 3 all-reduce, 4 all-to-all
//   bits 3-4  number of read+write reshuffles added after the collective
//   bit  5    banned transition (-> Partial from Replicate / Shard): cost is inf
//   bit  6    the running bytes change after this dim (x n after all-gather, / n after
//             reduce-scatter)
// collective_runtime_estimation.py:83-138.
__host__ __device__ constexpr uint32_t pair_action(int c, int t) {
  constexpr uint32_t AG = 1, RS = 2, AR = 3, A2A = 4, BAN = 1u << 5, UPD = 1u << 6;
  const uint32_t cn = c == 3, tn = t == 3;
  if (t == 1) return c == 1 ? 0u : BAN;            // -> Partial
  if (c == 0) return 0u;                           // Replicate -> Replicate / Shard: local
  if (c == 1) return t == 0 ? AR : (RS | (tn << 3) | UPD);
  return t == 0 ? (AG | (cn << 3) | UPD) : (A2A | ((cn + tn) << 3));
}
// (of the placement at mesh dim i of packed codes; a Shard's code is 0x80 | .. | its dim)
__device__ __forceinline__ uint32_t placement_class(uint32_t codes, int i) {
  const uint32_t kind = (codes >> (8 * i + 6)) & 3u;
  return kind + ((codes & (0x8Fu << (8 * i))) > (0x80u << (8 * i)) ? 1u : 0u);
}

// Term arrays staged per tile, interleaved: the entry of (state s, array a) sits at byte
// s x state_stride + 8 a, state_stride = 8 x (arrays + 1): an odd number of doubles, so that
// lanes reading one array at different states hit different LDS banks.  Two layouts, chosen per
// launch by the host (TermLayout):
//
// General (any mesh): one value per running-bytes state, 8 arrays: [0] zeros, [1] +inf (banned
// transitions), [2] one read+write, [3] two read+writes (2.0 x [2]: the same bits as
// (double)2 * rw), [4] all-gather, [5] reduce-scatter, [6] all-reduce, [7] all-to-all (=
// reduce-scatter shaped term x a2a_scale, :22-32).  An entry's running index is the history of
// the earlier dims.
//
// Power-of-two meshes (every mesh size a power of two, world size at most 2^31): the running
// bytes are the tensor's bytes times a power of two, bytes x 2^e with e in [-30 - L, -30],
// L = log2(world size): dividing by the shards, x n after an all-gather and / n after a
// reduce-scatter are exact.  Every term is then a rounding-free rescaling of ONE chain of
// operations on the tensor's bytes: RN(2^e x) = 2^e RN(x) for the multiplications and divisions
// of the ring and read+write formulas (no underflow: bytes < 2^53, e >= -61), so
//   ring term of dim d at exponent e = latency_d + ldexp(B_d, e - log2 n_d),
//       B_d = RN(RN(RN(bytes x hops_d) / bw_d) x 1e6)      (two hops per step: B doubles)
//   read+write at exponent e = max(ldexp(R, e + 31), launch floor),
//       R = RN(RN(RN(bytes / hbm_bw) x 1e6) / rw_eff)
// and one value per (array, exponent) replaces one per (array, state); 16 arrays: [0] zeros,
// [1] +inf, [2] one read+write, [3] two, then per mesh dim d [4 + 3d] one-hop ring (all-gather
// and reduce-scatter), [5 + 3d] two-hop ring (all-reduce), [6 + 3d] all-to-all; E = L + 1
// exponents.  An entry's running index is e + 30 + L.  Every computed array is one formula,
// max(lat + ldexp(B, j + shift), floor) x scale with B from one chain bytes x hops / div1 x 1e6
// / div2 (division by 1.0, x 1.0, 0.0 + x and max(x, -inf) return x), with constants the host
// works out per launch (TermArrayConstants): a lane per array takes B, then a lane per (array,
// exponent) the value.  (3-D mesh of 512 devices: 11 chains and 110 values of five operations,
// against 120 states x 6 terms of two divisions each.)
constexpr int kMaxExponents = 32;
constexpr int kGeneralStride = 8 * (8 + 1), kPow2Stride = 8 * (kMaxTermArrays + 1);  // bytes per state / exponent
template <int M>
struct TermTable {
  // (a 2-D mesh has one state more, behind the others: the bytes of an unsharded producer after dim 1, before dim 0, for
  // the order flip's words)
  static constexpr int kStates = States<M>::kCount + (M == 2 ? 1 : 0);
  static constexpr int kGeneral = kGeneralStride / 8 * kStates;
  static constexpr int kPow2 = kPow2Stride / 8 * kMaxExponents;
  static constexpr int kEntries = kGeneral > kPow2 ? kGeneral : kPow2;
};
static_assert(4 + 3 * APC_MAX_MESH <= kMaxTermArrays, "arrays of the power-of-two layout");

// Lookup words.  What a mesh dim adds to an entry depends on the producer's and the consumer's class at
// that dim and on the running index, which starts at the producer spec's own (general: the first state of its mask;
// power-of-two meshes: L - log2 of its shards) and goes on by the earlier dims.  One 32-bit word per (dim, producer
// class, consumer class), the same for every tile of a launch (TermLayout::image), in fields an instruction can take as a
// half or a byte of a register:
//   bits  0-15  byte offset of the collective's term from the running index' entry (general: array of
//               pair_action's term, state of the bytes the collective moves: after the update
//               for an all-gather, before it else; the +inf array for a banned transition)
//   bits 16-23  signed: bytes from there to the read+write term of the same state (zeros / one
//               / two reshuffles)
//   bits 24-31  signed step of the running index after this dim (general: the dim's history
//               bit; power-of-two meshes: + log2 n after an all-gather, - log2 n after a
//               reduce-scatter)
// Word 0 (dim 0, Replicate to Replicate) adds nothing and serves every dim of an entry whose placements are the same.
// A producer spec's record and a consumer spec's hold a byte per dim, (16 class) and (64 dim + 4 class): their sum is
// the offset of the dim's word, all dims in one addition.
// (The words used to be made for every producer spec of a tile, with its own index added: 85 vector instructions of a tile's
// first wavefront and 19 words of LDS a spec, 4.9 KB, read at a stride; now 20 instructions and two words, and lanes that
// share a word read it together.  us a pass: 704 k entries on (6, 4, 2) 13.0 -> 11.5, 5.9 M on (2, 4, 2, 2) 33.0 -> 29.8, on (64, 4)
// 28.5 -> 26.7, 584 k on (3, 2, 2, 2) 11.4 -> 10.8, 1.8 M on (16, 8, 4) 16.0 -> 15.6, 2.6 M on (12, 6) 11.8 -> 11.6; tables of which
// the stores are what takes the time, 20 M on (16, 8, 4) and 66 M in 80 layers, as before, 62.7 and 127.)
// A (Partial, Partial) producer on a 2-D mesh reaches an all-Shard consumer by two reduce-scatters, dim 1 first
// (collective_runtime_estimation.py:146-151): words kFlipWord.. hold that walk, of dim 1 to Shard(0) and to another Shard,
// then of dim 0, and byte 3 of the producer's codes holds the shift (kFlipShift, 0 for any other producer) that takes a
// consumer's flip slots in place of its plain ones (RowRecord).
constexpr uint32_t kFlipShift = 16;
constexpr int kFlipWord = 2 * 16;
template <int M>
constexpr int kPairWords = M * 16 + (M == 2 ? 4 : 0);
constexpr uint32_t kZerosArray = 0, kInfArray = 1, kRw1Array = 2;
static_assert(TermTable<APC_MAX_MESH>::kEntries * 8 <= 0xFFFF + 1, "term offsets fit their 16 bits");

static TermLayout term_layout(const apc_params &p) {
  TermLayout lay{};
  const int M = p.mesh_ndim;
  uint32_t pair[APC_MAX_MESH * 16] = {};
  TermArrayConstants arrays[kMaxTermArrays - 2] = {};
  bool pow2 = getenv("APC_GENERAL_TERMS") == nullptr;  // (testing override: the general layout on any mesh)
  int total = 0;
  for (int i = 0; i < M; ++i) {
    const int n = p.mesh_size[i];
    if (n < 1 || (n & (n - 1)) != 0) {
      pow2 = false;
      break;
    }
    int lg = 0;
    while ((1 << lg) < n) ++lg;
    lay.lg[i] = lg;
    total += lg;
  }
  if (total + 1 > kMaxExponents) pow2 = false;
  const int E = pow2 ? total + 1 : 0;
  lay.exponents = E;
  lay.lg_total = pow2 ? total : 0;
  lay.state_stride = pow2 ? kPow2Stride : kGeneralStride;
  lay.exponent_magic = pow2 ? (uint32_t)((65536 + E - 1) / E) : 0u;
  lay.inv_rescale = 1.0 / p.rescale;
  for (int i = 0; i < M; ++i)
    for (int c = 0; c < 4; ++c)
      for (int t = 0; t < 4; ++t) {
        const uint32_t e = pair_action(c, t);
        const uint32_t sel = e & 7u, copies = (e >> 3) & 3u;
        const bool ban = (e & 32u) != 0, upd = (e & 64u) != 0;
        const uint32_t rw_array = copies == 0u ? kZerosArray : kRw1Array + copies - 1u;
        uint32_t term_array, state = 0;
        int step;
        if (!pow2) {
          // the first state of the level within its mask; an all-gather (a sharding producer, a replicating consumer) is charged
          // on the gathered bytes, those of the next level, behind the last dim without its history bit (States)
          term_array = ban ? kInfArray : sel == 0u ? kZerosArray : 3u + sel;
          state = sel != 1u ? (1u << i) - 1u : (2u << i) - 1u + (i + 1 < M ? 1u << i : 0u);
          step = upd ? (1 << i) : 0;
        } else {
          if (sel == 1u) state = (uint32_t)lay.lg[i];  // an all-gather is charged on the gathered bytes
          term_array = ban ? kInfArray : sel == 0u ? kZerosArray : sel <= 2u ? 4u + 3u * i : sel == 3u ? 5u + 3u * i : 6u + 3u * i;
          step = !upd ? 0 : sel == 1u ? lay.lg[i] : -lay.lg[i];
        }
        const int to_rw = ((int)rw_array - (int)term_array) * 8;
        pair[i * 16 + c * 4 + t] = (state * (uint32_t)lay.state_stride + term_array * 8u) | ((uint32_t)(to_rw & 0xFF) << 16) |
                                       ((uint32_t)(step & 0xFF) << 24);
      }
  if (M == 2)
    for (int k = 0; k < 4; ++k) {  // the order flip: (Partial -> Shard at dim 1, then at dim 0), of an unsharded producer
      const int dim = k < 2 ? 1 : 0;
      const uint32_t word = pair[dim * 16 + 4 + 2 + (k & 1)];
      // (general layout: both states are named outright, no step between them)
      const uint32_t own = (1u << dim) - 1u, state = dim == 1 ? 1u : (uint32_t)States<2>::kCount;
      pair[kFlipWord + k] = pow2 ? word : (word & 0x00FFFFFFu) + (state - own) * (uint32_t)lay.state_stride;
    }
  lay.index0 = lay.lg_total;
  for (int i = 0; i < M; ++i) lay.index_weight[i] = pow2 ? -lay.lg[i] : ((1 << M) - 1) << i;
  lay.last_weight = pow2 ? 0 : 1 << (M - 1);
  lay.level_stride = pow2 ? 0 : kGeneralStride;
  if (pow2) {
    const double ninf = -INFINITY;
    // one read+write, two (compute_estimation.py:302-314 on bytes x 2^(e + 31))
    arrays[0] = {1.0, p.hbm_bw, p.inv_hbm_bw, p.rw_eff, p.inv_rw_eff, 0.0, p.launch_floor, 1.0, -total - 30 + 31, 0};
    arrays[1] = arrays[0];
    arrays[1].scale = 2.0;
    for (int d = 0; d < M; ++d) {  // torch _collective_utils.py:281-313 on bytes x 2^e
      const double h = (double)(p.mesh_size[d] - 1);
      const double lat1 = p.base_latency + h * p.lat[d];
      const double lat2 = p.base_latency + (2.0 * h) * p.lat[d];
      const int shift = -total - 30 - lay.lg[d];
      arrays[2 + 3 * d] = {h, p.bw[d], p.inv_bw[d], 1.0, 1.0, lat1, ninf, 1.0, shift, 0};
      arrays[3 + 3 * d] = {h, p.bw[d], p.inv_bw[d], 1.0, 1.0, lat2, ninf, 1.0, shift + 1, 0};
      arrays[4 + 3 * d] = {h, p.bw[d], p.inv_bw[d], 1.0, 1.0, lat1, ninf, p.a2a_scale, shift, 0};
    }
  }
  const size_t words = sizeof(uint32_t) * (size_t)(M * 16 + (M == 2 ? 4 : 0));  // (kPairWords)
  std::memcpy(lay.image, pair, words);
  std::memcpy(reinterpret_cast<char *>(lay.image) + words, arrays, sizeof(TermArrayConstants) * (size_t)(3 * M + 2));
  return lay;
}

// A consumer spec of a tile: its placement codes; per mesh dim i, in byte i of `slots`, its part of the byte offset of
// the dim's lookup word, 64 i + 4 class (byte 0 = 0xFF: not a DTensorSpec; on a 2-D mesh bytes 2 and 3 are what a (Partial,
// Partial) producer takes instead: the same, or, when every dim is a Shard, what leads to its two flip words); the compute
// cost / num_args of its strategy.  One 16-byte LDS read per entry.
struct alignas(16) RowRecord {
  uint32_t codes, slots;
  double cpa;
};
// A producer spec: its placement codes (2-D: the flip's shift in byte 3); its part of the words' offsets, 16 class (byte 0 =
// 0xFF as above); its running index, in the byte of `slots` behind the dims', on a 4-D mesh in a word of its own.
template <int M>
struct alignas(8) ColRecord {
  uint32_t codes, slots;
};
template <>
struct alignas(16) ColRecord<4> {
  uint32_t codes, slots, index, pad_;
};
static_assert(States<3>::kCount <= 256 && kMaxExponents <= 256 && APC_MAX_MESH == 4, "a running index fits its byte");
constexpr uint32_t kNotASpec = 0xFFu;

template <int M>
constexpr int kComputedArrays = 3 * M + 2;  // arrays 2 .. of the power-of-two layout
template <int M>
constexpr int kImagePieces = (kPairWords<M> * 4 + kComputedArrays<M> * (int)sizeof(TermArrayConstants) + 15) / 16;
static_assert(kPairWords<1> % 4 == 0 && kPairWords<2> % 4 == 0 && kPairWords<3> % 4 == 0 && kPairWords<4> % 4 == 0 && kImagePieces<APC_MAX_MESH> <= 128 &&
                  kImagePieces<APC_MAX_MESH> * 16 <= (int)sizeof(TermLayout::image), "an image in pieces of 16 bytes, two a lane at most");

// Everything the entry loops need about one tile, in LDS.
template <int M>
struct TileStage {
  RowRecord row[APC_TILE_MAX_ROWS];              // consumer specs
  ColRecord<M> col[APC_TILE_MAX_COLS];           // producer specs
  alignas(16) uint32_t image[kImagePieces<M> * 4];  // TermLayout::image: the lookup words, the constants of the term arrays
  double chain[kMaxTermArrays];                  // of the computed arrays, on the tensor's bytes
  int mixed[4];  // per wavefront: some spec is not a DTensorSpec on the tile's tensor (generic loop)
  int cont;      // the tile's tensor is contiguous
  // Last: the tile kernels size their LDS per launch for the entries the layout in use needs (stage_lds_bytes), so that the
  // small power-of-two layout leaves room for more workgroups.  Behind the entries, where the tile's row minima are taken,
  // the values of the rows each wavefront is walking (tile_entries_row_min).
  alignas(16) double terms[TermTable<M>::kEntries];
};

// Where its parts begin, in bytes.
template <int M>
__host__ __device__ constexpr uint32_t rows_at() {
  using Stage = TileStage<M>;
  return (uint32_t)offsetof(Stage, row);
}
template <int M>
__host__ __device__ constexpr uint32_t cols_at() {
  using Stage = TileStage<M>;
  return (uint32_t)offsetof(Stage, col);
}
template <int M>
__host__ __device__ constexpr uint32_t words_at() {
  using Stage = TileStage<M>;
  return (uint32_t)offsetof(Stage, image);
}
template <int M>
__host__ __device__ constexpr uint32_t terms_at() {
  using Stage = TileStage<M>;
  return (uint32_t)offsetof(Stage, terms);
}

// LDS a wavefront has to itself where the tile's row minima are taken: the values of the rows it is walking.
constexpr int kRowMinValues = 320;
template <bool RM>
constexpr size_t kWaveScratchBytes = RM ? kRowMinValues * sizeof(double) : 0;
// Bytes of the term arrays in the launch's layout.
template <int M>
__host__ __device__ __forceinline__ uint32_t term_bytes(const TermLayout &lay) {
  return lay.exponents ? (uint32_t)kPow2Stride * (uint32_t)lay.exponents : (uint32_t)TermTable<M>::kGeneral * 8u;
}

// LDS bytes of a tile stage whose term arrays hold what the launch's layout needs.
template <int M, bool RM>
static size_t stage_lds_bytes(const TermLayout &lay, int threads) {
  return terms_at<M>() + term_bytes<M>(lay) + kWaveScratchBytes<RM> * (size_t)(threads / 64);
}

// Where the copies of a tile's values go: lane k of EVERY wavefront holds the first entry and the
// first matrix row of the k-th identical edge (k < dup_count <= APC_TILE_MAX_DUPS <= 64), read
// back one by one as scalars (value_of_lane) when a value is stored to all copies: no LDS, no
// load in the store loop.  row_out (the same in every lane) is the first matrix row of the tile's own edge.
struct TileCopies {
  int64_t entry0, row0;
  int64_t row_out;
};
static_assert(APC_TILE_MAX_DUPS <= 64, "one lane per identical edge");

// Waits for the loads of `copies` now.  On this hardware loads and stores share one counter of
// outstanding vector-memory operations, and a wait for a load behind which stores were issued
// can only be a wait for all of them: offsets first touched inside the store loop would make
// every wavefront sit out the full round trip of its first store.  Called before the stores begin.
__device__ __forceinline__ void settle(TileCopies &copies) {
  __asm__ volatile("" : "+v"(copies.entry0), "+v"(copies.row0), "+v"(copies.row_out));
}

// The fields of a tile record the entry loops use.
struct TileView {
  int rows, cols, row_begin, col_begin, n_src, flags, dup_count, src_begin;
  int64_t entry_begin, pt_begin;
};

__device__ __forceinline__ int uniform_i32(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ int64_t uniform_i64(int64_t v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)v >> 32));
  return (int64_t)(((uint64_t)hi << 32) | lo);
}

__device__ __forceinline__ TileView view_of(const apc_tile &tile) {
  return TileView{tile.counts & 0xFFFF, tile.counts >> 16, tile.row_begin, tile.col_begin, tile.n_src,
                  tile.flags,           tile.dup_count,    tile.src_begin, tile.entry_begin, tile.pt_begin};
}

// ring_r on a per-lane mesh dim d, with mesh_size[d] - 1 hops and with twice as many: every step behind the first product
// of twice the hops doubles exactly.
template <int M>
__device__ __forceinline__ void rings_at(double gb, const apc_params &p, int d, double &one, double &two) {
  const int n = pick<M>(p.mesh_size, d);
  const double hops = (double)(n - 1), lat = pick<M>(p.lat, d);
  const double bw = div_by(div_by(gb * hops, (double)n, pick<M>(p.inv_mesh, d)), pick<M>(p.bw, d), pick<M>(p.inv_bw, d)) * 1e6;
  one = (p.base_latency + hops * lat) + bw;
  two = (p.base_latency + (2.0 * hops) * lat) + 2.0 * bw;
}

__device__ __forceinline__ int from_lane(int v, int lane) { return __builtin_amdgcn_ds_bpermute(lane << 2, v); }
__device__ __forceinline__ double from_lane(double v, int lane) {
  return __hiloint2double(from_lane(__double2hiint(v), lane), from_lane(__double2loint(v), lane));
}
__device__ __forceinline__ int64_t from_lane_i64(int64_t v, int lane) {
  const uint32_t lo = (uint32_t)from_lane((int)(uint32_t)v, lane), hi = (uint32_t)from_lane((int)(uint32_t)((uint64_t)v >> 32), lane);
  return (int64_t)(((uint64_t)hi << 32) | lo);
}

// The value of the lane `N` further on within the lane's row of 16 (DPP row_shl:N), `beyond` behind the row's end.
template <int N>
__device__ __forceinline__ double from_lane_behind(double x, double beyond) {
  const int lo = __builtin_amdgcn_update_dpp(__double2loint(beyond), __double2loint(x), 0x100 + N, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(__double2hiint(beyond), __double2hiint(x), 0x100 + N, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}

// Bytes (as a double) and contiguity of the tensor whose dim lane & 7 this lane holds (size x, stride y): what
// tensor_bytes_and_contiguity_of returns, in every lane, from the whole wavefront.  A dim's expected stride is the product
// of the sizes behind it: three steps of a scan over the lanes in doubles, exact while the product of all is below 2^53.
// Any other tensor (and one with an empty dim, where the two expected strides differ) goes dim by dim in integers.
// (As scalar integers the eight dims are 190 instructions one behind the other, on the one scalar unit of a compute unit,
// in every wavefront; 35 vector instructions now.  With a tile's compute costs through the checked reciprocals, us a pass: 1.8 M entries on
// (16, 8, 4) 15.6 -> 14.6, 5.9 M on (64, 4) 27.2 -> 26.2, 704 k on (6, 4, 2) 11.6 -> 11.2, 1.7 M on (32, 8) over packed tiles 8.42 -> 8.32.)
__device__ __forceinline__ void tensor_info_of_lanes(int rank, int itemsize, int64_t x, int64_t y, int lane, double &bytes, bool &contiguous) {
  const int dim = lane & 15;
  const bool live = dim < min(rank, APC_MAX_RANK);  // (lanes 8 .. 15 of a row hold no dim)
  const double size = live ? (double)x : 1.0;
  double product = size;
  product *= from_lane_behind<1>(product, 1.0);
  product *= from_lane_behind<2>(product, 1.0);
  product *= from_lane_behind<4>(product, 1.0);
  const double expected = from_lane_behind<1>(product, 1.0);
  const bool differs = size != 1.0 && (double)y != expected;
  contiguous = __ballot(differs) == 0;
  const double total = __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(product)),
                                        __builtin_amdgcn_readfirstlane(__double2loint(product))) * (double)itemsize;
  bytes = total;
  if (__ballot(!(size >= 1.0) || !(product < 0x1p53) || !(total < 0x1p53)) != 0) {  // (uniform)
    int64_t nbytes = itemsize, one = 1, most = 1;
    contiguous = true;
#pragma unroll 1
    for (int i = min(rank, APC_MAX_RANK) - 1; i >= 0; --i) {
      const int64_t xi = value_of_lane(x, i), yi = value_of_lane(y, i);
      nbytes *= xi;
      if (xi == 1) continue;
      if (yi != one && yi != most) contiguous = false;
      most *= xi > 1 ? xi : 1;
      one *= xi;
    }
    bytes = (double)nbytes;
  }
}

// Stages tile `tile` with `nthreads` (>= 64) cooperating threads (this thread is `tid`).  The
// caller synchronises before the stage is read.  Only global loads and LDS writes: no stores.
// A vector load waits behind every store the compute unit has in flight, so what staging costs under a store-bound
// kernel is the vector loads it issues: all of them at once, in one round, and each by one wavefront of the tile where one needs it.
// The first takes the producer specs and the image (three loads, four on 4-D meshes) and, DERIVE, the tensor (two), the last the consumer
// specs and their costs (three; DERIVE: nine, with what those are worked out of).  Every wavefront takes the copies' offsets, where there
// are some (one, RM two), and DERIVE in the general layout the tensor (two), whose states all of them work out; what is the same for
// all lanes comes through the scalar cache.  (When every wavefront loaded everything, twelve loads each, four more cost the one launch over 66 M
// entries in 80 layers 11 of 142 us.  us a pass, everything by every wavefront / by one: 20 M entries on (16, 8, 4) 62.6 / 61.4, 47 M in eight
// layers on (64, 4) 129.7 / 123.8, 5.9 M there 26.4 / 25.2, 1.8 M on (16, 8, 4) 14.5 / 13.4, 2.6 M on (12, 6) 11.5 / 11.4, 66 M in 80 layers
// 127.1 / 126.4; the other way 704 k on (6, 4, 2) 11.3 / 11.6.)
template <int M, bool DERIVE, bool RM>
__device__ __forceinline__ void stage_tile(const apc_params &p, const TableArgs &a, const apc_tile &tile,
                                           TileStage<M> &st, int tid, int nthreads, TileCopies &copies) {
  constexpr int NS = TermTable<M>::kStates, kComputed = kComputedArrays<M>, kPieces = kImagePieces<M>;
  const int rows = tile.counts & 0xFFFF, cols = tile.counts >> 16;
  const int t0 = tile.tensor;  // spec_tensor of the tile's first producer spec (checked by the host)
  const bool no_producer = (tile.flags & APC_EDGE_NO_PRODUCER) != 0;
  const bool terms_wanted = t0 >= 0 && !no_producer;
  bool mixed = !terms_wanted;
  const TermLayout &lay = a.lay;
  const int E = lay.exponents;  // wave-uniform; 0: general layout
  const int lane = tid & 63, wave = uniform_i32(tid >> 6);
  static_assert(APC_TILE_MAX_COLS <= 64 && APC_TILE_MAX_ROWS <= 64, "a wavefront for the specs of either side");
  const bool first_wave = wave == 0, last_wave = wave == (nthreads >> 6) - 1;
  const int t0c = t0 >= 0 ? t0 : 0;  // (row 0 when the tile has no tensor: unconditional loads, the values are not used then)
  // ---- the round of vector loads ------------------------------------------------------------
  // Lanes past the tile's specs load its first spec again.
  const bool has_col = first_wave && lane < cols, has_row = last_wave && lane < rows;
  const uint32_t at_col = has_col ? (uint32_t)lane : 0u, at_row = has_row ? (uint32_t)lane : 0u;
  u32x4 piece{}, piece2{};
  int col_tensor = 0, row_tensor = 0;
  uint32_t col_codes = 0, row_codes = 0;
  int64_t dim_size = 0, dim_stride = 0;
  if (first_wave) {
    struct __attribute__((packed, aligned(8))) Piece {
      u32x4 v;
    };
    const Piece *image = reinterpret_cast<const Piece *>(lay.image);
    piece = load_of_lane(image, (uint32_t)min(lane, kPieces - 1)).v;
    if (kPieces > 64) piece2 = load_of_lane(image, (uint32_t)min(lane + 64, kPieces - 1)).v;
    const int64_t sp = (int64_t)tile.src_begin + tile.col_begin;
    col_codes = load_of_lane(a.spec_codes + sp, at_col);
    col_tensor = load_of_lane(a.spec_tensor + sp, at_col);
  }
  if (DERIVE && (first_wave || E == 0)) {  // (general layout: every wavefront takes part in the states)
    dim_size = load_of_lane(a.shape + (int64_t)t0c * APC_MAX_RANK, (uint32_t)lane & (APC_MAX_RANK - 1));
    dim_stride = load_of_lane(a.stride + (int64_t)t0c * APC_MAX_RANK, (uint32_t)lane & (APC_MAX_RANK - 1));
  }
  double row_cpa = 0.0, gf_of_lane = 0.0, inv_gf_of_lane = 0.0;
  int64_t row_flops = 0, row_rw = 0;
  int row_dtype = 0, row_zero = 1, row_args = 1;
  if (last_wave) {
    const int64_t ts = (int64_t)tile.tgt_begin + tile.row_begin, sr = (int64_t)tile.strat_begin + tile.row_begin;
    row_codes = load_of_lane(a.spec_codes + ts, at_row);
    row_tensor = load_of_lane(a.spec_tensor + ts, at_row);
    if (!DERIVE) {
      if (a.per_arg) row_cpa = load_of_lane(a.per_arg + sr, at_row);
    } else {
      // (lane j holds the throughput of dtype code j & 7: fetched by the lanes that need it, below)
      gf_of_lane = load_of_lane(p.gpu_flops, (uint32_t)lane & (APC_MAX_DTYPES - 1));
      inv_gf_of_lane = load_of_lane(p.inv_gpu_flops, (uint32_t)lane & (APC_MAX_DTYPES - 1));
      row_flops = load_of_lane(a.flops + sr, at_row);
      row_rw = load_of_lane(a.rw_bytes + sr, at_row);
      row_dtype = load_of_lane(a.dtype + sr, at_row);
      row_zero = load_of_lane(a.zero_cost + sr, at_row);
      row_args = load_of_lane(a.num_args + sr, at_row);
    }
  }
  // (every wavefront its own copy of the identical edges' offsets, in lanes 0 .. dup_count - 1)
  copies.entry0 = copies.row0 = copies.row_out = 0;
  if (tile.dup_count > 0 && lane < tile.dup_count) {
    copies.entry0 = load_of_lane(a.dup_entry_begin + tile.dup_begin, (uint32_t)lane);
    if constexpr (RM) copies.row0 = load_of_lane(a.dup_row_begin + tile.dup_begin, (uint32_t)lane);
  }
  // ---- the scalar loads of the round (wave-uniform addresses), issued together ---------------------
  // The tile's tensor and the first matrix row of its edge.  The contiguity byte is read as the aligned word around it (which
  // lies in the byte's own page).
  if constexpr (RM) copies.row_out = uniform_load(a.edge_row_begin + tile.edge);
  bool contiguous = true;
  double fbytes = 0.0;
  if constexpr (!DERIVE) {
    const uint8_t *flag = a.tensor_contiguous + t0c;
    const uint32_t byte = (uint32_t)(reinterpret_cast<uintptr_t>(flag) & 3);
    const uint32_t word = uniform_load(reinterpret_cast<const uint32_t *>(flag - byte));
    const int64_t tensor_nbytes = uniform_load(a.tensor_bytes + t0c);
    fetch_arguments_now(word, tensor_nbytes);
    contiguous = ((word >> (8 * byte)) & 0xFFu) != 0;
    fbytes = (double)tensor_nbytes;
  } else {
    const int t_rank = uniform_load(a.rank + t0c), t_item = uniform_load(a.itemsize + t0c);
    fetch_arguments_now(t_rank, t_item);
    if (first_wave || E == 0) tensor_info_of_lanes(t_rank, t_item, dim_size, dim_stride, lane, fbytes, contiguous);
  }
  char *const image = reinterpret_cast<char *>(st.image);
  if (first_wave) {
    if (lane < kPieces) *reinterpret_cast<u32x4 *>(image + lane * 16) = piece;
    if (kPieces > 64 && lane < kPieces - 64) *reinterpret_cast<u32x4 *>(image + (lane + 64) * 16) = piece2;
  }
  const char *const arrays = image + kPairWords<M> * 4;  // (TermArrayConstants)
  // ---- term arrays --------------------------------------------------------------------------
  if (terms_wanted && E != 0 && first_wave) {
    // power-of-two mesh.  A lane per computed array takes the array's chain on the tensor's bytes; below a lane per (array,
    // exponent) the value.
    __builtin_amdgcn_wave_barrier();  // (LDS operations of one wavefront complete in order)
    if (lane < kComputed) {
      const TermArrayConstants &k = *reinterpret_cast<const TermArrayConstants *>(arrays + lane * sizeof(TermArrayConstants));
      st.chain[lane] = div_by(div_by(fbytes * k.hops, k.div1, k.inv_div1) * 1e6, k.div2, k.inv_div2);
    }
  }
  if (terms_wanted && E == 0) {
    // every collective / read-write term the tile can need, once per running-bytes state, in
    // the reference's operation order (collective_runtime_estimation.py:66-68, :86, :128;
    // torch _collective_utils.py:281-313; compute_estimation.py:302-314)
    double *const terms = st.terms;
    const auto bytes_at = [&](int level, int mask, int hist) {
      double shards = 1.0;  // exact: a product of mesh sizes (torch _dtensor_spec.py:555-561)
#pragma unroll
      for (int i = 0; i < M; ++i)
        if ((mask >> i) & 1) shards *= (double)p.mesh_size[i];
      double gb = fbytes / shards * 0x1p-30;  // / 1024 / 1024 / 1024
#pragma unroll
      for (int i = 0; i < M; ++i) {
        if (i < level && ((hist >> i) & 1)) {
          const double m = (double)p.mesh_size[i];
          gb = ((mask >> i) & 1) ? gb * m : div_by(gb, m, p.inv_mesh[i]);
        }
      }
      return gb;
    };
    const auto store_state = [&](int state, double gb, double ag, double rs, double ar) {
      const double rw = rw_time_r(gb * 2 * 1073741824.0, p);
      double *e = terms + __mul24(state, kGeneralStride / 8);
      e[kZerosArray] = 0.0;
      e[kInfArray] = __builtin_inf();
      e[kRw1Array] = rw;
      e[kRw1Array + 1] = 2.0 * rw;
      e[4] = ag;
      e[5] = rs;
      e[6] = ar;
      e[7] = rs * p.a2a_scale;
    };
    // On 3-D and 4-D meshes the last level apart, which has an all-gather and a read+write alone.
    constexpr bool kLastApart = M >= 3;
    constexpr int kFirst = kLastApart ? States<M>::kLast : NS, kHalf = States<M>::kHalf;
    for (int k = tid; k < kFirst; k += nthreads) {
      const bool flip_state = M == 2 && k == States<M>::kCount, last = !kLastApart && k >= States<M>::kLast && !flip_state;
      const int level = flip_state ? 0 : last ? M : 31 - __clz((k >> M) + 1);
      const int rem = flip_state ? 0 : last ? k - States<M>::kLast : k - (((1 << level) - 1) << M);
      const int mask = last ? kHalf | (rem >> (M - 1)) : rem >> level;
      const int hist = last ? kHalf | (rem & (kHalf - 1)) : rem & ((1 << level) - 1);
      double gb = bytes_at(level, mask, hist);
      if (flip_state) gb = div_by(gb, (double)p.mesh_size[1], p.inv_mesh[1]);
      double ag = 0.0, rs = 0.0, ar = 0.0, unused;
      if (level >= 1) rings_at<M>(gb, p, level - 1, ag, unused);
      if (level < M) rings_at<M>(gb, p, level, rs, ar);
      store_state(flip_state ? States<M>::kCount : States<M>::index(level, mask, hist), gb, ag, rs, ar);
    }
    if constexpr (kLastApart) {
      const int first = (tid + 8 * nthreads - 64 * ((kFirst + 63) / 64)) & (nthreads - 1);  // from the wavefronts that had fewer of the others
      for (int u = first; u < kHalf * kHalf; u += nthreads) {
        const int mask = kHalf | (u >> (M - 1)), hist = kHalf | (u & (kHalf - 1));
        const double gb = bytes_at(M, mask, hist);
        const double hops = (double)(p.mesh_size[M - 1] - 1);
        const double bw = div_by(div_by(gb * hops, (double)p.mesh_size[M - 1], p.inv_mesh[M - 1]), p.bw[M - 1], p.inv_bw[M - 1]);
        store_state(States<M>::index(M, mask, hist), gb, (p.base_latency + hops * p.lat[M - 1]) + bw * 1e6, 0.0, 0.0);
      }
    }
  }
  // ---- what the loads brought, to LDS ---------------------------------------------------------
  if (tid == 0) st.cont = contiguous;
  if (has_col) {
    uint32_t slots = 0, codes = col_codes, others = 0;
    int index = lay.index0;
#pragma unroll
    for (int i = 0; i < M; ++i) {
      const uint32_t cls = placement_class(col_codes, i), sharded = cls >> 1;
      slots += cls << (8 * i + 4);
      index += __mul24((int)sharded, lay.index_weight[i]);
      if (i + 1 < M) others += sharded << i;
      else index += __mul24((int)(sharded * others), lay.last_weight);
    }
    if (M == 2 && col_codes == 0x4040u) codes |= kFlipShift << 24;
    if (M < 4) slots |= (uint32_t)index << 24;
    if (col_tensor < 0) slots |= kNotASpec;
    if constexpr (M < 4) st.col[lane] = ColRecord<M>{codes, slots};
    else st.col[lane] = ColRecord<M>{codes, slots, (uint32_t)index, 0u};
    if (col_tensor != t0 || col_tensor < 0) mixed = true;
  }
  double row_cost = 0.0;
  if constexpr (DERIVE) {  // (every lane takes part in the exchange)
    if (last_wave) {
      const bool known = row_dtype >= 0 && row_dtype < APC_MAX_DTYPES;
      const double gf = from_lane(gf_of_lane, row_dtype & (APC_MAX_DTYPES - 1)), inv_gf = from_lane(inv_gf_of_lane, row_dtype & (APC_MAX_DTYPES - 1));
      row_cost = compute_cost_through_reciprocals(p, row_zero != 0, row_rw, row_flops, known ? gf : 0.0, known ? inv_gf : 0.0);
    }
  }
  if (has_row) {
    uint32_t slots = 0;
    bool all_shard = true;
#pragma unroll
    for (int i = 0; i < M; ++i) {
      const uint32_t t = (row_codes >> (8 * i)) & 0xFF;
      slots += (16u * i + placement_class(row_codes, i)) << (8 * i + 2);
      all_shard &= kind_of(t) == 2;
    }
    if (M == 2) {
      // (the producer adds the 16 of its class, Partial)
      const uint32_t flip = ((kFlipWord * 4u - 16u + (dim_of((row_codes >> 8) & 0xFF) != 0 ? 4u : 0u)) << 16) |
                            ((kFlipWord * 4u - 16u + 8u + (dim_of(row_codes & 0xFF) != 0 ? 4u : 0u)) << 24);
      slots |= all_shard ? flip : slots << 16;
    }
    if (row_tensor < 0) {  // a consumer spec that is not a DTensorSpec
      slots |= kNotASpec;
      mixed = true;
    }
    if (DERIVE) row_cpa = row_cost / (double)row_args;  // the value compute_costs_block writes for this strategy
    st.row[lane] = RowRecord{row_codes, slots, row_cpa};
  }
  // one flag per wavefront, written unconditionally: nothing to clear beforehand
  const bool wave_mixed = __ballot(mixed) != 0;
  if (lane == 0) st.mixed[wave] = wave_mixed ? 1 : 0;
  // ---- the values of the power-of-two layout's arrays ------------------------------------------
  if (terms_wanted && E != 0) {
    if (nthreads > 64) __syncthreads();
    else __builtin_amdgcn_wave_barrier();
    char *const terms = reinterpret_cast<char *>(st.terms);
    for (int t = tid; t < kComputed * E; t += nthreads) {
      // (24-bit multiplies: an integer multiply of 32 bits takes four times as long)
      const int arr = (int)((uint32_t)__umul24((uint32_t)t, lay.exponent_magic) >> 16);  // t / E
      const int j = t - __mul24(arr, E);  // the running bytes are bytes x 2^(j - L - 30)
      // (Constants out of LDS.  Read from the kernel arguments by a per-lane index inside this loop, `lat + ldexp(..)` was
      // compiled to `x + x` in the 4-D instantiations by hipcc 7.2: the placement-pair tests on 4-D power-of-two meshes show it.)
      const TermArrayConstants &k = *reinterpret_cast<const TermArrayConstants *>(arrays + __mul24(arr, (int)sizeof(TermArrayConstants)));
      double v = k.lat + __builtin_ldexp(st.chain[arr], j + k.shift);
      v = v > k.floor ? v : k.floor;
      v = v * k.scale;
      *reinterpret_cast<double *>(terms + __mul24(j, kPow2Stride) + (arr + 2) * 8) = v;
    }
    if (tid < 2 * E) {
      const int j = tid < E ? tid : tid - E;
      *reinterpret_cast<double *>(terms + __mul24(j, kPow2Stride) + (tid < E ? 0 : 8)) = tid < E ? 0.0 : __builtin_inf();
    }
  }
}


// The arguments an entry loop uses, in scalar registers before it begins.  (Left to the compiler, an argument is loaded
// where it is used, in every pass, and a scalar load in flight makes the wait for an LDS read a wait for everything.)
struct EntryConstants {
  double rescale, inv_rescale, transition;
  int32_t transition_scale, state_stride, level_stride;
};
__device__ __forceinline__ EntryConstants entry_constants(const apc_params &p, const TermLayout &lay) {
  EntryConstants k{p.rescale, lay.inv_rescale, (double)p.transition_scale, p.transition_scale, lay.state_stride, lay.level_stride};
  __asm__ volatile("" : "+s"(k.rescale), "+s"(k.inv_rescale), "+v"(k.transition), "+s"(k.transition_scale), "+s"(k.state_stride),
                   "+s"(k.level_stride));
  return k;
}

// Where a lane is in a tile: the addresses of its producer spec's record and of its consumer spec's, and the bytes to its
// entry from the tile's first one.  (Kept as what the loads and the store need: of a column and a row, every pass would shift
// and multiply again.)
struct TileWalk {
  lds_address col, row;
  uint32_t out;
};
struct TileSteps {  // of one pass; `wrap`: when the column passes the row's end
  uint32_t dcol, end, cols, drow, drow_wrap, dout, dout_wrap;
};
template <int M>
__device__ __forceinline__ TileWalk tile_walk(lds_address stage, int r, int c, int n_src) {
  return TileWalk{stage + cols_at<M>() + (uint32_t)c * (uint32_t)sizeof(ColRecord<M>),
                  stage + rows_at<M>() + (uint32_t)r * 16u,
                  (uint32_t)(__mul24(r, n_src) + c) * 8u};
}
// (dr, dc: rows and columns of a pass; uniform, as everything here)
template <int M>
__device__ __forceinline__ TileSteps tile_steps(lds_address stage, uint32_t dr, uint32_t dc, uint32_t cols, uint32_t n_src) {
  constexpr uint32_t kCol = (uint32_t)sizeof(ColRecord<M>);
  const uint32_t dout = (dr * n_src + dc) * 8u;
  return TileSteps{dc * kCol, stage + cols_at<M>() + cols * kCol, cols * kCol, dr * 16u, dr * 16u + 16u, dout, dout + (n_src - cols) * 8u};
}
template <bool WHOLE>  // whole rows: the entries of a tile are consecutive
__device__ __forceinline__ void advance(TileWalk &w, const TileSteps &s) {
  const uint32_t col = w.col + s.dcol;
  const bool wrap = col >= s.end;
  w.col = wrap ? col - s.cols : col;
  w.row += wrap ? s.drow_wrap : s.drow;
  w.out += WHOLE ? s.dout : wrap ? s.dout_wrap : s.dout;
}

// x / d for a wave-uniform 0 < d <= 64 and 0 <= x <= 8192: (x + 1/2) / d is at least 1/128 away from a whole number,
// its rounding and that of 1 / d in 24 bits are 2^-9 at most.  (An integer division is 20 instructions.)
__device__ __forceinline__ uint32_t small_quotient(uint32_t x, float inv_d) { return (uint32_t)(((float)x + 0.5f) * inv_d); }
// The same where x is uniform too, as a scalar.  (The conversion would be moved behind the read of the first lane, into a
// vector register again.)
__device__ __forceinline__ uint32_t uniform_quotient(uint32_t x, float inv_d) {
  uint32_t q = small_quotient(x, inv_d);
  __asm__("" : "+v"(q));
  return (uint32_t)uniform_i32((int)q);
}

// The byte offset of the lookup word of mesh dim I: byte I of `slots`, or `same` where the
// placements (byte I of the codes) are equal.  Two instructions that select bytes, where a compiler masks, compares,
// shifts and selects.  (s_nop 1: two cycles from a comparison's result to the select that reads it; the compiler does not look
// inside an asm statement.)
template <int I>
__device__ __forceinline__ uint32_t word_slot(uint32_t src, uint32_t tgt, uint32_t slots, uint32_t same) {
  uint32_t slot;
#define APC_WORD_SLOT(BYTE_)                                                                                            \
  __asm__("v_cmp_ne_u32_sdwa vcc, %1, %2 src0_sel:" BYTE_ " src1_sel:" BYTE_ "\n\ts_nop 1\n\t"                         \
          "v_cndmask_b32_sdwa %0, %3, %4, vcc dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:" BYTE_       \
          : "=v"(slot)                                                                                                  \
          : "v"(src), "v"(tgt), "v"(same), "v"(slots)                                                                   \
          : "vcc")
  if constexpr (I == 0) APC_WORD_SLOT("BYTE_0");
  else if constexpr (I == 1) APC_WORD_SLOT("BYTE_1");
  else if constexpr (I == 2) APC_WORD_SLOT("BYTE_2");
  else APC_WORD_SLOT("BYTE_3");
#undef APC_WORD_SLOT
  return slot;
}
template <int I, int M>
__device__ __forceinline__ void word_slots(uint32_t src, uint32_t tgt, uint32_t slots, uint32_t (&out)[M]) {
  out[I] = word_slot<I>(src, tgt, slots, 0u);  // (word 0: nothing to add)
  if constexpr (I + 1 < M) word_slots<I + 1>(src, tgt, slots, out);
}

// One entry of a tile whose producer specs all name one tensor.
// What bounds a table of large tiles: its stores, and under them the vector instructions (20 M entries on (16, 8, 4): stores alone 42 us, 23.2 M
// instructions, 91 thousand of a SIMD's cycles or 38 us, LDS 22 us, one launch 46.5 us where the output stays in the caches and 56.8 where it
// does not), which only partly run beside each other, so a pass counts both: 40 vector instructions on a 3-D mesh with the walk and the store (54 when columns, rows and loop were kept as numbers of a lane and the codes
// compared by mask), and a tile's staging, which two wavefronts share, about 330 (430; 250 since the words are the launch's).  us a pass: 20 M on (16, 8, 4) 57.0 ->
// 50.8, 5.3 M on (2, 4, 2, 2) 41.8 -> 39.4, 5.1 M on (3, 2, 2, 2) 53.2 -> 50.7, 2.6 M on (12, 6) 14.4 -> 13.4, 587 k on
// (6, 4, 2) 16.0 -> 15.4.  (Every copy's address in scalar registers, one instruction less a store, is 1 % slower.)
// Straight-line code: all lookups of an entry are independent of its fp additions, so they
// are issued together; no vector memory loads.
template <int M, bool CONT, bool RESCALE>
__device__ __forceinline__ void uniform_entry(const EntryConstants &k, lds_address stage, lds_address terms, const TileWalk &where, double &comm_o,
                                              double &total_o, int &trans_o) {
  typedef uint32_t col_words __attribute__((ext_vector_type(sizeof(ColRecord<M>) / 4)));
  const col_words col = lds_read<col_words>(where.col);
  const u32x4 raw = lds_read<u32x4>(where.row);
  const uint32_t src = col.x;
  const RowRecord row{raw.x, raw.y, __hiloint2double((int)raw.w, (int)raw.z)};
  const uint32_t x = src ^ row.codes;
  const bool differs = M == 2 ? (x & 0xFFFFu) != 0 : x != 0;
  // (2-D: a (Partial, Partial) producer's shift takes the slots of its order flip)
  const uint32_t slots = (M == 2 ? row.slots >> (src >> 24) : row.slots) + col.y;
  uint32_t index;
  if constexpr (M < 4) index = col.y >> 24;
  else index = col.z;
  // ---- integer part: which term at which running index each mesh dim adds -------------------
  uint32_t at = terms + __umul24(index, (uint32_t)k.state_stride);  // the running index' entry
  uint32_t slot[M], term_at[M], rw_at[M], nc_at[M];
  word_slots<0>(src, row.codes, slots, slot);
#pragma unroll
  for (int i = 0; i < M; ++i) {
    const uint32_t w = lds_read<uint32_t>(stage + words_at<M>() + slot[i]);
    term_at[i] = (w & 0xFFFFu) + at;
    rw_at[i] = term_at[i] + (uint32_t)(int32_t)(int8_t)(w >> 16);
    if (!CONT) nc_at[i] = at + (uint32_t)(kRw1Array * 8u + ((1u << i) - 1u) * (uint32_t)k.level_stride);  // (the state before the dim)
    at += (uint32_t)__mul24((int32_t)w >> 24, k.state_stride);  // (24-bit multiplies issue at full rate)
  }
  // ---- lookups ------------------------------------------------------------------------------
  double term[M], rw[M], nc[M];
#pragma unroll
  for (int i = 0; i < M; ++i) {
    term[i] = lds_read<double>(term_at[i]);
    rw[i] = lds_read<double>(rw_at[i]);
    if (!CONT) nc[i] = lds_read<double>(nc_at[i]);
  }
  // ---- additions in the reference's order (0.0 + t == t for these non-negative terms) ------------
  double cost = 0.0;
  // a fully replicated producer returns before the non-contiguity term (:56-62)
  bool cont = CONT || src == 0u;
#pragma unroll
  for (int i = 0; i < M; ++i) {
    if (!CONT) {
      const bool neq = ((x >> (8 * i)) & 0xFF) != 0;
      cost += (neq && !cont) ? nc[i] : 0.0;
      cont = cont || neq;
    }
    if (CONT && i == 0) cost = term[0];
    else cost += term[i];
    cost += rw[i];  // 0, 1 or 2 read+writes: (double)copies * rw, picked from the staged multiples
  }
  double comm = cost;  // (a banned transition added the +inf term)
  // :358-359; the quotient through the reciprocal is the division's (div_by), +inf stays +inf
  if (RESCALE) comm = comm < __builtin_inf() ? div_by(comm, k.rescale, k.inv_rescale) : comm;
  comm_o = comm;
  // :345-351, :368-372
  total_o = comm + row.cpa + (differs ? k.transition : 0.0);
  trans_o = differs ? k.transition_scale : 0;
}

// The three output streams of one tile: wave-uniform bases, so an entry's addresses are a
// scalar base plus a 32-bit lane offset (the host checks that a tile spans < 4 GiB).
struct TileOut {
  double *comm;
  uint8_t *trans;
  double *cost;
  int64_t entry_begin;  // first entry of the tile's edge (an identical edge's values sit at its own first entry)
};

// Which of the three per-entry output arrays a launch writes, as a compile-time choice of the
// kernel (no per-store checks, and the registers of streams that are not written are free):
// the planner's table build wants the assembled cost alone (what the ILP objective is summed
// from, optimize_sharding.py:650-655; comm and transition are fetched by a later launch only
// if a report asks for them), a caller that wants every array gets all three, any other subset
// is checked per store.
enum : int { kOutAny = 0, kOutAll = 1, kOutCost = 2 };

// Evaluates one entry and stores its values to its edge and to every identical edge; -> its assembled cost.  Called by every lane of
// the wavefront (`active`: this lane holds an entry), so that the copies' offsets are read from
// their lanes under uniform control flow.
template <int OUT>
__device__ __forceinline__ void store_values(const TileOut &o, int64_t delta, uint32_t off8, double comm, double total, int trans) {
  constexpr bool ALL = OUT == kOutAll, COST = OUT == kOutCost;
  if (ALL || (!COST && o.comm)) *reinterpret_cast<double *>(reinterpret_cast<char *>(o.comm + delta) + off8) = comm;
  if (ALL || (!COST && o.trans)) (o.trans + delta)[off8 / 8u] = (uint8_t)trans;
  if (ALL || COST || o.cost) *reinterpret_cast<double *>(reinterpret_cast<char *>(o.cost + delta) + off8) = total;
}
template <int OUT, typename Entry>
__device__ __forceinline__ double store_entry(const TileOut &o, int dup_count, const TileCopies &copies, bool active, const TileWalk &where,
                                              Entry entry) {
  double comm, total;
  int trans;
  if (active) {
    entry(where, comm, total, trans);
    store_values<OUT>(o, 0, where.out, comm, total, trans);
  }
  for (int d = 0; d < dup_count; ++d) {
    const int64_t delta = value_of_lane(copies.entry0, d) - o.entry_begin;
    if (active) store_values<OUT>(o, delta, where.out, comm, total, trans);
  }
  return total;
}

// A 32-bit value from the lane `N` further on within the lane's row of 16 (DPP row_shl:N); a
// lane whose source lies outside its row keeps its own value.
template <int N>
__device__ __forceinline__ int from_lane_ahead(int x) {
  return __builtin_amdgcn_update_dpp(x, x, 0x100 + N, 0xF, 0xF, false);
}
template <int N>
__device__ __forceinline__ double from_lane_ahead(double x) {
  const int lo = from_lane_ahead<N>(__double2loint(x)), hi = from_lane_ahead<N>(__double2hiint(x));
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double value_of_lane(double x, int lane) {  // lane: a constant
  const int lo = __builtin_amdgcn_readlane(__double2loint(x), lane), hi = __builtin_amdgcn_readlane(__double2hiint(x), lane);
  return __hiloint2double(hi, lo);
}

// Row minima of one pass, as the packed tiles take them.  The 64 lanes of a wavefront hold 64 consecutive entries
// of the tile (inactive lanes: +inf), row after row.  `c` is the lane's column, `cols` the row
// length.  First a segmented minimum by doubling inside every 16 lanes (data-parallel
// primitives: vector ALU only, the LDS pipe stays free for the entry loop's lookups): a lane
// then holds the minimum, and the first column that has it, of its row's entries from itself to
// the end of its 16 lanes.  Lanes 16, 32 and 48 hold such a part for a row that came in from the
// lanes before them: their values are read as scalars and joined, in lane order, by the lanes
// whose row reaches them.  On return a lane holds minimum and first argmin of its
// row's entries from itself to the row's end within the wavefront (the whole row for c == 0).
__device__ __forceinline__ void row_min_in_wave(bool active, double value, int c, int cols, int lane, double &m, int &mc) {
  m = active ? value : __builtin_inf();
  mc = c;
  const int in_row16 = lane & 15;
#define APC_ROW_MIN_STEP(N_)                                                            \
  if (N_ < cols) { /* (cols is wave-uniform) */                                         \
    const double om = from_lane_ahead<N_>(m);                                           \
    const int oc = from_lane_ahead<N_>(mc);                                             \
    /* that lane holds an entry of the same row; strict <: ties keep the lower column */ \
    if (in_row16 + N_ < 16 && c + N_ < cols && om < m) {                                \
      m = om;                                                                           \
      mc = oc;                                                                          \
    }                                                                                   \
  }
  APC_ROW_MIN_STEP(1)
  APC_ROW_MIN_STEP(2)
  APC_ROW_MIN_STEP(4)
  APC_ROW_MIN_STEP(8)
#undef APC_ROW_MIN_STEP
#define APC_ROW_MIN_JOIN(LANE_)                                              \
  {                                                                          \
    const double pm = value_of_lane(m, LANE_);                               \
    const int pc = __builtin_amdgcn_readlane(mc, LANE_);                     \
    if (LANE_ > lane && c + (LANE_ - lane) < cols && pm < m) {               \
      m = pm;                                                                \
      mc = pc;                                                               \
    }                                                                        \
  }
  if (cols > 1) {
    APC_ROW_MIN_JOIN(16)
    APC_ROW_MIN_JOIN(32)
    APC_ROW_MIN_JOIN(48)
  }
#undef APC_ROW_MIN_JOIN
}

// The minimum, and the lowest column that has it, over neighbouring lanes of a row of 16: one step of a butterfly.
template <int CTRL>
__device__ __forceinline__ void lower_of_lanes(double &m, int &mc) {
  const int lo = __double2loint(m), hi = __double2hiint(m);
  const double om = __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, CTRL, 0xF, 0xF, false), __builtin_amdgcn_update_dpp(lo, lo, CTRL, 0xF, 0xF, false));
  const int oc = __builtin_amdgcn_update_dpp(mc, mc, CTRL, 0xF, 0xF, false);
  const bool take = (om < m) | ((om == m) & (oc < mc));
  m = take ? om : m;
  mc = take ? oc : mc;
}

// The entry loop of a tile that holds whole rows, with the row minima.  Every wavefront walks rows of its own, some at a
// time: 64 consecutive entries a pass, evaluated (`entry`), stored, and kept in the wavefront's LDS; then 1 to 16 lanes a
// row read it back, the lanes of a row the columns in turn, and join their minima.  The rows of a wavefront need no
// barrier, and a value costs one write and one read of 8 bytes where a minimum taken across the lanes of every pass
// (neighbours in doubling distances, value and column) was 70 vector instructions a pass, more than the entry's own.
// (6.1 M entries on (64, 4) 50.4 -> 38.7 us, 27.4 without the minima.)  kRowMinValues: more rows are joined at once, fewer workgroups
// fit a compute unit.  512 / 384 / 320 / 256, later: those entries 28.2 / 26.6 / 26.1 / 26.2 us, 5.2 M on (12, 6) 27.2 / 25.0 / 25.1 /
// 24.7, 5.3 M in two layers on (64, 4) 21.2 / 20.0 / 20.1 / 19.3, 410 k on (32, 8) 11.0 / 10.3 / 10.2 / 9.0; 5.8 M in nineteen layers
// 18.3 / 17.5 / 17.8 / 18.5, 850 k on (8, 8, 8), which fit once anyway, 8.5 / 8.6 / 8.7 / 9.1.
template <int M, int OUT, typename Entry>
__device__ __forceinline__ void tile_entries_row_min(const TableArgs &a, lds_address stage, const TileView &v, const TileCopies &copies,
                                                     int tid, int nthreads, Entry entry) {
  const int lane = tid & 63, wave = uniform_i32(tid >> 6), waves = nthreads >> 6;
  constexpr bool RM = true;
  const lds_address values = stage + terms_at<M>() + term_bytes<M>(a.lay) + (uint32_t)kWaveScratchBytes<RM> * (uint32_t)wave;
  const int cols = v.cols;
  // bytes from row to row: an odd number of doubles, so that the lanes of consecutive rows read different banks
  const uint32_t row_bytes = (uint32_t)(cols | 1) * 8u;
  const float inv_cols = __builtin_amdgcn_rcpf((float)cols);
  const int at_once = min((int)uniform_quotient(kRowMinValues, __builtin_amdgcn_rcpf((float)(cols | 1))), 64);
  const int r0 = (int)small_quotient((uint32_t)lane, inv_cols), c0 = lane - __mul24(r0, cols);
  const uint32_t dr = uniform_quotient(64, inv_cols), dc = 64u - dr * (uint32_t)cols;
  const TileSteps steps = tile_steps<M>(stage, dr, dc, (uint32_t)cols, (uint32_t)cols);
  const int row_begin = (int)((uint32_t)(v.rows * wave) / (uint32_t)waves), row_end = (int)((uint32_t)(v.rows * (wave + 1)) / (uint32_t)waves);
  const int64_t tile_base = v.entry_begin + (int64_t)v.row_begin * v.n_src + v.col_begin;
  const TileOut out{a.comm_out ? a.comm_out + tile_base : nullptr, a.trans_out ? a.trans_out + tile_base : nullptr,
                    a.cost_out ? a.cost_out + tile_base : nullptr, v.entry_begin};
  // a value's place in `values`: its place in the output and, where the rows are padded, 8 bytes a row
  const uint32_t pad = (cols & 1) ? 31u : 1u;  // (a record of 16 bytes a row)
  for (int first = row_begin; first < row_end; first += at_once) {
    const int rows = min(at_once, row_end - first), n = rows * cols;
    TileWalk w = tile_walk<M>(stage, first + r0, c0, cols);
    const uint32_t to_values = values - (uint32_t)(first * cols) * 8u - ((stage + rows_at<M>() + (uint32_t)first * 16u) >> pad);
    for (int at = 0; at < n; at += 64) {
      const bool active = at + lane < n;
      const double total = store_entry<OUT>(out, v.dup_count, copies, active, w, entry);
      if (active) lds_write(w.out + (w.row >> pad) + to_values, total);
      advance<true>(w, steps);
    }
    __builtin_amdgcn_wave_barrier();  // (LDS operations of one wavefront complete in order)
    const int shift = rows <= 4 ? 4 : rows <= 8 ? 3 : rows <= 16 ? 2 : rows <= 32 ? 1 : 0;  // 2^shift lanes a row
    const int lanes = 1 << shift, row = lane >> shift, sub = lane & (lanes - 1);
    const lds_address line = values + (uint32_t)__umul24((uint32_t)min(row, rows - 1), row_bytes);
    const double head = lds_read<double>(line);
    double m = __builtin_inf();
    int mc = 0;
    for (int y = sub; y < cols; y += 4 * lanes) {
      int at[4];
      double value[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        at[u] = min(y + u * lanes, cols - 1);  // (past the row's end: its last value once more)
        value[u] = lds_read<double>(line + (uint32_t)at[u] * 8u);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (value[u] < m) {  // strict: ties keep the lower column
          m = value[u];
          mc = at[u];
        }
    }
    if (shift >= 1) lower_of_lanes<0xB1>(m, mc);   // quad_perm [1, 0, 3, 2]
    if (shift >= 2) lower_of_lanes<0x4E>(m, mc);   // quad_perm [2, 3, 0, 1]
    if (shift >= 3) lower_of_lanes<0x141>(m, mc);  // row_half_mirror
    if (shift >= 4) lower_of_lanes<0x140>(m, mc);  // row_mirror
    if (head != head) {  // (no value compares below a NaN in the first column)
      m = head;
      mc = 0;
    }
    __builtin_amdgcn_wave_barrier();
    // all lanes of a row have the result: each stores it to a copy (copy 0 is the tile's own edge, copy d > 0 the d-th identical one)
    const bool live = row < rows;
    for (int copy0 = 0; copy0 <= v.dup_count; copy0 += lanes) {
      const int copy = copy0 + sub;
      int64_t first_row = copies.row_out;
      if (v.dup_count > 0) {  // (uniform; every lane takes part)
        const int64_t of_copy = from_lane_i64(copies.row0, max(copy - 1, 0));
        first_row = copy == 0 ? first_row : of_copy;
      }
      if (live && copy <= v.dup_count) {
        const int64_t o = first_row + v.row_begin + first + row;
        a.row_min_out[o] = m;
        a.row_arg_out[o] = v.col_begin + mc;
      }
    }
  }
}

// The per-entry loop of a tile for `nthreads` threads (this one is `tid`): a flattened
// (row, column) walk, so a wavefront writes 64 consecutive entries.
// A full-width tile (WHOLE) is one contiguous run of entries: lanes are shifted so that every
// wavefront store starts on a 64-entry boundary of the output arrays (whole 128-byte lines
// of the fp64 streams) instead of straddling one more line than it fills.  Every lane of a
// wavefront makes the same number of passes (a lane in front of the tile's first entry idles
// in the first one), so the copies' offsets are read under uniform control flow.
template <int M, int OUT, bool WHOLE, typename Entry>
__device__ __forceinline__ void tile_entries_walk(const TableArgs &a, lds_address stage, const TileView &v, const TileCopies &copies,
                                                  int tid, int nthreads, Entry entry) {
  const int n = v.rows * v.cols;
  const float inv_cols = __builtin_amdgcn_rcpf((float)v.cols);
  const uint32_t dr = uniform_quotient((uint32_t)nthreads, inv_cols), dc = (uint32_t)nthreads - dr * (uint32_t)v.cols;
  const int n_src = WHOLE ? v.cols : v.n_src;
  const TileSteps steps = tile_steps<M>(stage, dr, dc, (uint32_t)v.cols, (uint32_t)n_src);
  const int64_t tile_base = v.entry_begin + (int64_t)v.row_begin * v.n_src + v.col_begin;
  const int shift = WHOLE ? (int)(tile_base & 63) : 0;
  const int lane = tid & 63;
  // (in front of the tile's first entry rows count backwards: 64 rows are more than the shift)
  const int r = (int)small_quotient((uint32_t)(tid - shift + 64 * v.cols), inv_cols) - 64;
  TileWalk w = tile_walk<M>(stage, r, tid - shift - __mul24(r, v.cols), n_src);
  const TileOut out{a.comm_out ? a.comm_out + tile_base : nullptr, a.trans_out ? a.trans_out + tile_base : nullptr,
                    a.cost_out ? a.cost_out + tile_base : nullptr, v.entry_begin};
  for (int at = uniform_i32(tid - lane) - shift; at < n; at += nthreads) {
    store_entry<OUT>(out, v.dup_count, copies, (uint32_t)(at + lane) < (uint32_t)n, w, entry);
    advance<WHOLE>(w, steps);
  }
}

// The generic entry: pass-through edges and edges whose producer specs name different tensors.
template <int M, bool DERIVE>
__device__ __forceinline__ void generic_entry(const apc_params &p, const TableArgs &a, const TileStage<M> &st, lds_address stage, const TileView &v,
                                              const TileWalk &where, double &comm, double &total, int &trans) {
  const int r = (int)((where.row - stage - rows_at<M>()) / 16u), c = (int)((where.col - stage - cols_at<M>()) / (uint32_t)sizeof(ColRecord<M>));
  const int64_t local = (int64_t)(v.row_begin + r) * v.n_src + (v.col_begin + c);
  const ColRecord<M> col = st.col[c];
  const uint32_t src = M == 2 ? col.codes & 0xFFFFu : col.codes;  // (without the flip's shift)
  const RowRecord row = st.row[r];
  const uint32_t tgt = row.codes;
  trans = 0;
  if ((v.flags & APC_EDGE_NO_PRODUCER) || (col.slots & 0xFFu) == kNotASpec || (row.slots & 0xFFu) == kNotASpec) {
    comm = a.pt_values[v.pt_begin + local];
  } else {
    trans = (src != tgt) ? p.transition_scale : 0;
    const int sten = a.spec_tensor[v.src_begin + v.col_begin + c];
    int64_t shards = 1;
#pragma unroll
    for (int i = 0; i < M; ++i)
      if (kind_of((src >> (8 * i)) & 0xFF) == 2) shards *= p.mesh_size[i];
    int64_t sten_bytes;
    bool sten_contiguous;
    tensor_info<DERIVE>(a, sten, sten_bytes, sten_contiguous);
    const double gb = (double)sten_bytes / (double)shards / 1024 / 1024 / 1024;
    comm = entry_cost<M>(src, tgt, gb, sten_contiguous, p);
  }
  if (v.flags & APC_EDGE_GRAD_RESCALE) comm = comm / p.rescale;
  total = comm + row.cpa + (double)trans;
}

// All entries of a staged tile.  Row minima are taken when the caller wants them and the tile
// holds whole rows (which the host arranges for every tile of a table before asking).
template <int M, bool DERIVE, bool RM, int OUT>
__device__ __forceinline__ void tile_entries(const apc_params &p, const TableArgs &a, const TileStage<M> &st, lds_address stage,
                                             const TileView &v, const TileCopies &copies, int tid, int nthreads) {
  int mixed = st.mixed[0];
  for (int w = 1; w < nthreads / 64; ++w) mixed |= st.mixed[w];
  const bool whole = v.cols == v.n_src, row_minima = RM && whole;
  const auto entries = [&](auto out, auto entry) {
    constexpr int kOut = decltype(out)::value;
    if constexpr (RM) {
      if (row_minima) {
        tile_entries_row_min<M, kOut>(a, stage, v, copies, tid, nthreads, entry);
        return;
      }
    }
    if (whole) tile_entries_walk<M, kOut, true>(a, stage, v, copies, tid, nthreads, entry);
    else tile_entries_walk<M, kOut, false>(a, stage, v, copies, tid, nthreads, entry);
  };
  if (uniform_i32(mixed)) {
    entries(std::integral_constant<int, kOutAny>{}, [&](const TileWalk &where, double &comm, double &total, int &trans) {
      generic_entry<M, DERIVE>(p, a, st, stage, v, where, comm, total, trans);
    });
    return;
  }
  const bool rescale = (v.flags & APC_EDGE_GRAD_RESCALE) != 0;
  const EntryConstants k = entry_constants(p, a.lay);
  const lds_address terms = stage + terms_at<M>();
#define APC_TILE_LOOP(CONT_, RESCALE_)                                                                                       \
  entries(std::integral_constant<int, OUT>{}, [&](const TileWalk &where, double &comm, double &total, int &trans) {          \
    uniform_entry<M, CONT_, RESCALE_>(k, stage, terms, where, comm, total, trans);                                                  \
  })
  if (uniform_i32(st.cont)) {
    if (rescale) { APC_TILE_LOOP(true, true); } else { APC_TILE_LOOP(true, false); }
  } else {
    if (rescale) { APC_TILE_LOOP(false, true); } else { APC_TILE_LOOP(false, false); }
  }
#undef APC_TILE_LOOP
}

// A tile record (64 bytes, wave-uniform) as one scalar load.
__device__ __forceinline__ apc_tile load_tile_record(const apc_tile *tiles, int64_t tile_id) {
  static_assert(sizeof(apc_tile) == sizeof(i32x16), "one 64-byte scalar load per record");
  const i32x16 raw = uniform_load(reinterpret_cast<const i32x16 *>(tiles + tile_id));
  apc_tile tile;
  __builtin_memcpy(&tile, &raw, sizeof(tile));
  return tile;
}

// A tile's record and the table addresses its wavefronts use, all fetched on entry under one wait
// (fetch_arguments_now): the record's address needs only arguments that arrive in registers.
template <bool DERIVE, bool RM, int OUT>
__device__ __forceinline__ apc_tile fetch_tile(const apc_tile *tiles, int64_t tile_id, const TableArgs &a) {
  const apc_tile tile = load_tile_record(tiles, tile_id);
  if constexpr (DERIVE && RM && OUT == kOutCost)
    fetch_arguments_now(tile.counts, a.lay.exponents, a.spec_codes, a.spec_tensor, a.dup_entry_begin, a.cost_out, a.rank, a.itemsize, a.shape,
                        a.stride, a.flops, a.rw_bytes, a.dtype, a.zero_cost, a.num_args, a.edge_row_begin, a.dup_row_begin,
                        a.row_min_out, a.row_arg_out);
  else if constexpr (DERIVE)
    fetch_arguments_now(tile.counts, a.lay.exponents, a.spec_codes, a.spec_tensor, a.dup_entry_begin, a.rank, a.itemsize, a.shape, a.stride,
                        a.flops, a.rw_bytes, a.dtype, a.zero_cost, a.num_args);
  else if constexpr (RM)
    fetch_arguments_now(tile.counts, a.lay.exponents, a.spec_codes, a.spec_tensor, a.dup_entry_begin, a.tensor_bytes, a.tensor_contiguous,
                        a.per_arg, a.edge_row_begin, a.dup_row_begin);
  else
    fetch_arguments_now(tile.counts, a.lay.exponents, a.spec_codes, a.spec_tensor, a.dup_entry_begin, a.tensor_bytes, a.tensor_contiguous,
                        a.per_arg);
  return tile;
}

template <int M, int kTileThreads, bool RM, int OUT>
__device__ __forceinline__ void redistribute_tile(const apc_params &p, const TableArgs &a, const apc_tile *tiles, int n_tiles,
                                                  int xcd_shift, TileStage<M> &stage, lds_address at) {
  const int tile_id = tile_of_block((int)blockIdx.x, n_tiles, xcd_shift);
  if (tile_id >= n_tiles) return;
  static_assert(kTileThreads == 64 || kTileThreads == 128 || kTileThreads == 256, "wavefronts per tile: 1, 2 or 4");
  static_assert(kTileThreads >= APC_TILE_MAX_COLS && kTileThreads >= APC_TILE_MAX_ROWS &&
                kTileThreads >= APC_TILE_MAX_DUPS, "one staging round covers a tile");
  const apc_tile tile = fetch_tile<false, RM, OUT>(tiles, tile_id, a);
  // a record the host validator would have rejected (more identical edges than lanes hold): skipped
  if ((unsigned)tile.dup_count > (unsigned)APC_TILE_MAX_DUPS) return;
  TileCopies copies;
  stage_tile<M, false, RM>(p, a, tile, stage, threadIdx.x, kTileThreads, copies);
  settle(copies);
  __syncthreads();
  tile_entries<M, false, RM, OUT>(p, a, stage, at, view_of(tile), copies, threadIdx.x, kTileThreads);
}

// Wavefronts per SIMD the tile kernels ask for: what the LDS of their larger, row-minimum
// instantiation leaves room for (one-wavefront workgroups and 4-D meshes hold more LDS per
// wavefront).  Asked for explicitly because the compiler sizes its register budget by the LDS
// use otherwise: the row-minimum kernel got 97 registers and 4 wavefronts on a 3-D mesh where 67
// registers do without spilling (stress table 2.94 -> 2.58 ms); the kernel without the minima
// gains 1 - 2 % (same box: stress 1.93 -> 1.88 ms, Llama-3-70B 251 -> 248 us).
constexpr int tile_waves_per_simd(int mesh_ndim, int threads, bool row_min) {
  if (mesh_ndim >= 4) return threads >= 256 ? 4 : threads >= 128 ? 3 : 2;
  if (threads < 128) return mesh_ndim <= 1 ? 7 : mesh_ndim == 2 ? 6 : 4;
  // (Asked for eight, the compiler allows itself 78 scalar registers instead of 94, and spills; with the 53 vector
  // registers that it takes, eight fit all the same.)
  return 7;
}

struct TilesBlock {
  apc_params p;
  TableArgs a;
};

template <int M, int kTileThreads, int OUT>
__global__ __launch_bounds__(kTileThreads) __attribute__((amdgpu_waves_per_eu(tile_waves_per_simd(M, kTileThreads, false), 8)))
void redistribute_tiles_kernel(APC_LAUNCH_PARAMS(TilesBlock, false)) {
  extern __shared__ __align__(16) unsigned char s_stage_bytes[];  // stage_lds_bytes<M, false>
  const TilesBlock &k = launch_block<false>(kept);
  redistribute_tile<M, kTileThreads, false, OUT>(k.p, k.a, static_cast<const apc_tile *>(work), n_tiles, xcd_shift,
                                                 *reinterpret_cast<TileStage<M> *>(s_stage_bytes), address_in_lds(s_stage_bytes));
}

// The same with the row minima.
template <int M, int kTileThreads, int OUT>
__global__ __launch_bounds__(kTileThreads)
__attribute__((amdgpu_waves_per_eu(tile_waves_per_simd(M, kTileThreads, true), 8)))
void redistribute_tiles_row_min_kernel(APC_LAUNCH_PARAMS(TilesBlock, false)) {
  extern __shared__ __align__(16) unsigned char s_stage_bytes[];  // stage_lds_bytes<M, true>
  const TilesBlock &k = launch_block<false>(kept);
  redistribute_tile<M, kTileThreads, true, OUT>(k.p, k.a, static_cast<const apc_tile *>(work), n_tiles, xcd_shift,
                                                *reinterpret_cast<TileStage<M> *>(s_stage_bytes), address_in_lds(s_stage_bytes));
}

// Every table of a pass in one launch: workgroups [0, tile_blocks) take the tiles of the
// redistribution-cost matrices (tile_blocks = n_tiles rounded up to the number of XCDs), the
// next spec_blocks the spec table, then the tensor table, then the compute costs, kThreads rows
// per workgroup.  No workgroup reads what another writes: a tile derives its tensor's byte
// count and contiguity and its consumer strategies' compute costs with the functions the
// table workgroups use (TableArgs), so the values are the same bits.  One launch instead of
// two spares a table of a few tens of MB one ramp-up and one drain of the chip, which at that
// size are a third of each kernel.
// (LDS is sized per launch for the layout in use: with the general layout's share held for every mesh, a
// workgroup of a 4-D launch held 45 KB of which a power-of-two mesh uses 10.  6.4 M entries on (2, 4, 2, 2) 46.2 -> 32.9 us,
// 9.4 M on (16, 8, 4) 64.6 -> 59.1, 901 k on (8, 8, 8) 14.9 -> 13.8; on 1-D and 2-D meshes, where the larger layout was held, 6.1 M
// on (64, 4) 29.5 -> 28.2, 41 k on (64,) 10.6 -> 9.6.)
// (On 1-D and 2-D meshes seven wavefronts per SIMD are asked for, what 72 vector registers leave room for: 7.6 M entries on (32, 8),
// 59 layers, 17.0 us with 5, 16.4 with 7, 2.6 M on (12, 6) 13.4 / 13.2, 6.1 M on (64, 4) with the minima the same.  On 3-D meshes without
// the minima too: the compiler then takes 94 scalar registers instead of 106, and with its 62 vector registers eight wavefronts are
// resident instead of seven, 20 M entries on (16, 8, 4) 60.1 -> 58.6 us; with the minima it takes 67, and spills for nothing.)
template <int M, bool RM>
static size_t build_tables_lds_bytes(const TermLayout &lay, int threads, bool spec_table) {
  const size_t stage = stage_lds_bytes<M, RM>(lay, threads);
  const size_t rows = spec_table ? (size_t)threads * (APC_MAX_RANK + 1) * sizeof(int64_t) : 0;  // (spec_tables_block)
  return stage > rows ? stage : rows;
}

struct BuildTablesBlock {
  apc_params p;
  TableArgs a;
  TensorTableArgs t;
  SpecTableArgs sp;
  ComputeCostArgs c;
  int64_t spec_blocks, tensor_blocks;
};

template <int M, int kThreads, bool RM, int OUT, bool KEPT>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(M <= 2 || (M == 3 && !RM) ? 7 : 1, 8)))
void build_tables_kernel(APC_LAUNCH_PARAMS(BuildTablesBlock, KEPT)) {
  const BuildTablesBlock &k = launch_block<KEPT>(kept);
  const apc_params &p = k.p;
  const TableArgs &a = k.a;
  const apc_tile *const tiles = static_cast<const apc_tile *>(work);
  extern __shared__ __align__(16) unsigned char s_raw[];  // build_tables_lds_bytes<M, RM>
  static_assert(kThreads == 64 || kThreads == 128 || kThreads == 256, "wavefronts per workgroup: 1, 2 or 4");
  const int64_t b = blockIdx.x;
  if (b < tile_blocks) {
    const int tile_id = tile_of_block((int)b, n_tiles, xcd_shift);
    if (tile_id >= n_tiles) return;
    TileStage<M> &stage = *reinterpret_cast<TileStage<M> *>(s_raw);
    const apc_tile tile = fetch_tile<true, RM, OUT>(tiles, tile_id, a);
    if ((unsigned)tile.dup_count > (unsigned)APC_TILE_MAX_DUPS) return;  // (see redistribute_tile)
    TileCopies copies;
    stage_tile<M, true, RM>(p, a, tile, stage, threadIdx.x, kThreads, copies);
    settle(copies);
    __syncthreads();
    tile_entries<M, true, RM, OUT>(p, a, stage, address_in_lds(s_raw), view_of(tile), copies, threadIdx.x, kThreads);
    return;
  }
  const int64_t tb = b - tile_blocks;
  if (tb < k.spec_blocks) spec_tables_block<kThreads>(tb, p, k.sp, reinterpret_cast<int64_t *>(s_raw));
  else if (tb < k.spec_blocks + k.tensor_blocks) tensor_tables_block<kThreads>(tb - k.spec_blocks, k.t);
  else compute_costs_block<kThreads>(tb - k.spec_blocks - k.tensor_blocks, p, k.c);
}

// ------------------------------------------------------------------------------------------
// Packed tiles: the planner's pass over a small table, every wavefront on its own.
//
// A table of a few million entries is bound by the latency of one workgroup: all workgroups are
// resident at once, stage and then store in step, and the chain of dependent loads in front of
// the first store decides the launch.  Here a workgroup's loads depend on nothing but its index
// (one fixed-size record per tile, copied out of the tables beforehand: apc_packed_tile), and
// nothing is staged in LDS: lane j of every wavefront holds producer spec j, consumer spec j and
// the compute cost / num_args of consumer strategy j; a wavefront walks whole matrix rows,
// fetches an entry's two specs from their lanes, evaluates the entry directly
// (collective_runtime_estimation.py:37-153 in the reference's operation order, divisions through
// the checked reciprocals), reduces the row minima across its lanes and stores values and minima to
// the tile's edge and to every identical edge.  No barrier, no second pass over the rows.
// ------------------------------------------------------------------------------------------
struct DimConstants {  // of one mesh dim, wave-uniform
  double n, inv_n, bw, inv_bw;
  double hops1, lat1;  // all-gather, reduce-scatter, all-to-all: n - 1 hops (torch _collective_utils.py:281-301)
  double hops2, lat2;  // all-reduce: 2 (n - 1) hops (:304-313)
};
template <int M>
struct FlatConstants {
  DimConstants dim[M];
};

template <int M>
__device__ __forceinline__ FlatConstants<M> flat_constants(const apc_params &p) {
  FlatConstants<M> k;
#pragma unroll
  for (int i = 0; i < M; ++i) {
    DimConstants &d = k.dim[i];
    d.n = (double)p.mesh_size[i];
    d.inv_n = p.inv_mesh[i];
    d.bw = p.bw[i];
    d.inv_bw = p.inv_bw[i];
    d.hops1 = (double)(p.mesh_size[i] - 1);
    d.hops2 = (double)(2 * (p.mesh_size[i] - 1));
    d.lat1 = p.base_latency + d.hops1 * p.lat[i];
    d.lat2 = p.base_latency + d.hops2 * p.lat[i];
  }
  return k;
}

// entry_cost without branches: every lane of a wavefront evaluates its own (producer spec,
// consumer spec) pair, whatever collectives the pair needs.  What a mesh dim adds is selected,
// not branched on: the ring term of the one collective the dim can need (none: + 0.0, which
// leaves a non-negative sum unchanged), 0, 1 or 2 read+write reshuffles ((double)copies x rw:
// 0.0, rw, 2.0 x rw).  FIRST = 1 (2-D meshes): dim 1 before dim 0 (:146-151).  CONT: the tensor
// is contiguous (no lane ever adds the non-contiguity term); else `contiguous`: whether the lane's is.  gb = bytes / num_shards / 1024^3.
template <int M, int FIRST, bool CONT>
__device__ __forceinline__ double entry_cost_flat(uint32_t srcp, uint32_t tgtp, double gb, const apc_params &p,
                                                  const FlatConstants<M> &k, bool contiguous = false) {
  double cost = 0.0;
  bool banned = false, cont = CONT || contiguous;
  bool tgt_partial = false;
#pragma unroll
  for (int s = 0; s < M; ++s) {
    const int i = (M == 2 && FIRST == 1) ? 1 - s : s;
    const DimConstants &d = k.dim[i];
    const uint32_t c = (srcp >> (8 * i)) & 0xFF, t = (tgtp >> (8 * i)) & 0xFF;
    const bool neq = c != t;
    const uint32_t ck = c >> 6, tk = t >> 6;
    tgt_partial |= tk == 1;
    const bool from_shard = neq && ck == 2, from_partial = neq && ck == 1;
    const bool is_ag = from_shard && tk == 0, is_a2a = from_shard && tk == 2;  // :83-113
    const bool is_ar = from_partial && tk == 0, is_rs = from_partial && tk == 2;  // :115-130
    banned |= neq && tk == 1 && ck != 1;  // :131-138
    if (!CONT) {  // :81-82: charged once, on the bytes before this dim
      const double rw_before = rw_time_r(gb * 2 * 1073741824.0, p);
      cost += (neq && !cont) ? rw_before : 0.0;
      cont = cont || neq;  // :141
    }
    const double x = is_ag ? gb * d.n : gb;  // an all-gather is charged on the gathered bytes (:86)
    const double hops = is_ar ? d.hops2 : d.hops1;
    const double ring0 = (is_ar ? d.lat2 : d.lat1) + div_by(div_by(x * hops, d.n, d.inv_n), d.bw, d.inv_bw) * 1e6;
    const double ring = is_a2a ? ring0 * p.a2a_scale : ring0;  // :22-32
    cost += (from_shard || from_partial) && tk != 1 ? ring : 0.0;
    const double rw = rw_time_r(x * 2 * 1073741824.0, p);
    const uint32_t cn = (c & 0x0F) != 0 ? 1u : 0u, tn = (t & 0x0F) != 0 ? 1u : 0u;
    const uint32_t copies = is_ag ? cn : is_a2a ? cn + tn : is_rs ? tn : 0u;
    cost += copies == 0u ? 0.0 : copies == 1u ? rw : 2.0 * rw;
    gb = is_ag ? x : is_rs ? div_by(gb, d.n, d.inv_n) : gb;  // :86, :128
  }
  if (srcp == 0u) return tgt_partial ? __builtin_inf() : 0.0;  // :56-62
  return banned ? __builtin_inf() : cost;
}

// The same entry on a mesh whose sizes are all powers of two (TermLayout::exponents != 0; "Term
// arrays" above): the running bytes are the tensor's bytes x 2^(j - L - 30) for an integer j a lane
// carries from dim to dim, and every term is one ldexp of a wave-uniform chain value: no division
// per entry.  R / B[d]: the chains of the read+write and of dim d's one-hop ring on the tensor's
// bytes (TermArrayConstants of arrays 2 and 4 + 3 d).
template <int M>
struct Pow2Constants {
  double R, B[M];
  double lat1[M], lat2[M];
  int lg[M], shift[M];  // log2 n_d; -L - 30 - log2 n_d
  int rw_shift;         // -L - 30 + 31
  double floor;         // launch floor of a read+write
};

template <int M, int FIRST, bool CONT>
__device__ __forceinline__ double entry_cost_pow2(uint32_t srcp, uint32_t tgtp, int j, double a2a_scale, const Pow2Constants<M> &k,
                                                  bool contiguous = false) {
  double cost = 0.0;
  bool banned = false, cont = CONT || contiguous, tgt_partial = false;
#pragma unroll
  for (int s = 0; s < M; ++s) {
    const int i = (M == 2 && FIRST == 1) ? 1 - s : s;
    const uint32_t c = (srcp >> (8 * i)) & 0xFF, t = (tgtp >> (8 * i)) & 0xFF;
    const bool neq = c != t;
    const uint32_t ck = c >> 6, tk = t >> 6;
    tgt_partial |= tk == 1;
    const bool from_shard = neq && ck == 2, from_partial = neq && ck == 1;
    const bool is_ag = from_shard && tk == 0, is_a2a = from_shard && tk == 2;
    const bool is_ar = from_partial && tk == 0, is_rs = from_partial && tk == 2;
    banned |= neq && tk == 1 && ck != 1;
    if (!CONT) {
      const double before = __builtin_ldexp(k.R, j + k.rw_shift);
      cost += (neq && !cont) ? (before > k.floor ? before : k.floor) : 0.0;
      cont = cont || neq;
    }
    const int jx = is_ag ? j + k.lg[i] : j;  // an all-gather is charged on the gathered bytes
    const double ring0 = (is_ar ? k.lat2[i] : k.lat1[i]) + __builtin_ldexp(k.B[i], jx + k.shift[i] + (is_ar ? 1 : 0));
    const double ring = is_a2a ? ring0 * a2a_scale : ring0;
    cost += (from_shard || from_partial) && tk != 1 ? ring : 0.0;
    const double rw0 = __builtin_ldexp(k.R, jx + k.rw_shift);
    const double rw = rw0 > k.floor ? rw0 : k.floor;
    const uint32_t cn = (c & 0x0F) != 0 ? 1u : 0u, tn = (t & 0x0F) != 0 ? 1u : 0u;
    const uint32_t copies = is_ag ? cn : is_a2a ? cn + tn : is_rs ? tn : 0u;
    cost += copies == 0u ? 0.0 : copies == 1u ? rw : 2.0 * rw;
    j = is_ag ? jx : is_rs ? j - k.lg[i] : j;
  }
  if (srcp == 0u) return tgt_partial ? __builtin_inf() : 0.0;
  return banned ? __builtin_inf() : cost;
}

// value -> *(double *)((char *)base + byte_offset) for a wave-uniform base: the address stays a
// scalar register pair plus a 32-bit lane offset (left to the compiler, the sum is re-associated
// into per-lane 64-bit arithmetic inside a loop over bases).  A store needs no wait before the
// wavefront ends, and a wait by count for an older load stays correct with younger stores in
// flight (loads return in order among themselves).
// (sc0 sc1: the store is written through to memory.  Left in the L2 until the kernel ends, the
// table's lines are written back after the last wavefront has finished, and a launch of this
// size waits for that: 10.0 -> 8.6 us on the Llama-3-8B table.)
// (s_nop 4: a vector-memory instruction may read a scalar register a vector instruction wrote,
// such as a value fetched from a lane, only five cycles later; the compiler inserts that wait
// for its own instructions and does not look inside an asm statement.)
__device__ __forceinline__ void store_at(double *base, uint32_t byte_offset, double value) {
  __asm__ volatile("s_nop 4\n\tglobal_store_dwordx2 %0, %1, %2 sc0 sc1" ::"v"(byte_offset), "v"(value), "s"(base) : "memory");
}

struct PackedArgs {
  // the wavefronts of the tiles read their own copy of the parameters: a value both kinds of
  // workgroup load from one place is loaded on entry, for all of them, before the first branch
  apc_params p;
  double *row_min_out;
  int32_t *row_arg_out;
  const double *pt_values;
  // the tensor table: a tile whose producer specs name several tensors reads it entry by entry
  const int32_t *rank, *itemsize;
  const int64_t *shape, *stride;
  double inv_rescale;  // 1.0 / params.rescale
  // every mesh size a power of two (term_layout): log2 of the sizes and of their product; else exponents = 0
  int32_t exponents, lg_total, lg[APC_MAX_MESH];
};

template <int M, bool POW2, bool ALONE>  // ALONE: a wavefront takes the tile, else those of the workgroup
__device__ __forceinline__ void packed_tile(const apc_packed_tile *T, double *cost_out, const PackedArgs &a) {
  const apc_params &p = a.p;
  const int tid = threadIdx.x, lane = tid & 63, wave = ALONE ? 0 : tid >> 6, waves = ALONE ? 1 : blockDim.x >> 6;
  // ---- the one round of loads: nothing here depends on another load ---------------------------
  const i32x16 h = uniform_load(reinterpret_cast<const i32x16 *>(T));
  const int64_t dim_size = T->tensor_shape[lane & (APC_MAX_RANK - 1)], dim_stride = T->tensor_stride[lane & (APC_MAX_RANK - 1)];
  TileCopies copies;
  copies.entry0 = T->dup_entry_begin[lane & (APC_PACKED_MAX_DUPS - 1)];
  copies.row0 = T->dup_row_begin[lane & (APC_PACKED_MAX_DUPS - 1)];
  copies.row_out = 0;
  const uint32_t col_code = T->col_codes[lane], row_code = T->row_codes[lane];
  const int col_tensor = T->col_tensor[lane], row_tensor = T->row_tensor[lane];
  const int64_t row_flops = T->row_flops[lane], row_rw = T->row_rw_bytes[lane];
  const int row_meta = T->row_meta[lane];
  // (lane j holds the throughput of dtype code j & 7: fetched by the lanes that need it, below)
  const double gf_of_lane = a.p.gpu_flops[lane & (APC_MAX_DTYPES - 1)], inv_gf_of_lane = a.p.inv_gpu_flops[lane & (APC_MAX_DTYPES - 1)];
  // (kernel arguments the wavefront needs first or in its store loops, under the same wait)
  fetch_arguments_now(h[0], a.row_min_out, a.row_arg_out, p.hbm_bw, p.inv_hbm_bw, p.rw_eff, p.inv_rw_eff,
                      p.launch_floor, p.compute_eff, p.inv_compute_eff, a.inv_rescale, p.rescale, p.a2a_scale, p.base_latency);
  const int rows = h[0], cols = h[1], flags = h[2], dup_count = h[3], t0 = h[4];
  if ((unsigned)rows > (unsigned)APC_TILE_MAX_ROWS || (unsigned)(cols - 1) >= (unsigned)APC_TILE_MAX_COLS ||
      (unsigned)dup_count > (unsigned)APC_PACKED_MAX_DUPS)
    return;  // a record the host validator would have rejected
  const int64_t entry_begin = ((int64_t)h[9] << 32) | (uint32_t)h[8], row_begin = ((int64_t)h[11] << 32) | (uint32_t)h[10];
  const int64_t pt_begin = ((int64_t)h[13] << 32) | (uint32_t)h[12];
  const uint32_t magic = (65536u + (uint32_t)cols - 1u) / (uint32_t)cols;  // x / cols = (x magic) >> 16 for x <= 64
  const int rows_per_pass = (int)((64u * magic) >> 16);
  if (wave * rows_per_pass >= rows) return;  // a wavefront without rows (a tile of fewer rows than the workgroup walks at once)
  // ---- per wavefront: the tensor's bytes, the rows' compute costs -------------------------------
  double fbytes;
  bool contiguous;
  tensor_info_of_lanes(h[5], h[6], dim_size, dim_stride, lane, fbytes, contiguous);
  const int dt = (int)(int8_t)(row_meta & 0xFF);
  const bool known_dtype = dt >= 0 && dt < APC_MAX_DTYPES;
  const double gf = from_lane(gf_of_lane, dt & (APC_MAX_DTYPES - 1)), inv_gf = from_lane(inv_gf_of_lane, dt & (APC_MAX_DTYPES - 1));
  const double cpa = compute_cost_through_reciprocals(p, ((row_meta >> 8) & 0xFF) != 0, row_rw, row_flops, known_dtype ? gf : 0.0,
                                                      known_dtype ? inv_gf : 0.0) /
                     (double)(row_meta >> 16);  // (lanes past the tile's rows: never read)
  settle(copies);
  FlatConstants<M> k;
  constexpr bool pow2 = POW2;
  Pow2Constants<M> k2;
  if constexpr (!POW2) k = flat_constants<M>(p);
  if constexpr (POW2) {  // the chains of TermArrayConstants arrays 2 (read+write) and 4 + 3 d (one-hop ring of dim d)
    k2.R = div_by(div_by(fbytes, p.hbm_bw, p.inv_hbm_bw) * 1e6, p.rw_eff, p.inv_rw_eff);
    k2.rw_shift = 1 - a.lg_total;
    k2.floor = p.launch_floor;
#pragma unroll
    for (int i = 0; i < M; ++i) {
      const double hops1 = (double)(p.mesh_size[i] - 1), hops2 = (double)(2 * (p.mesh_size[i] - 1));
      k2.B[i] = div_by(fbytes * hops1, p.bw[i], p.inv_bw[i]) * 1e6;
      k2.lat1[i] = p.base_latency + hops1 * p.lat[i];
      k2.lat2[i] = p.base_latency + hops2 * p.lat[i];
      k2.lg[i] = a.lg[i];
      k2.shift[i] = -a.lg_total - 30 - a.lg[i];
    }
  }
  // ---- whole rows: cols lanes per row, 64 / cols rows per pass, wavefront w the passes w, w + waves, ...
  const int r_local = (int)(((uint32_t)lane * magic) >> 16), c = lane - r_local * cols;
  const bool in_pass = r_local < rows_per_pass;
  // (for the stores of the row minima: lane -> (row of the pass, copy))
  const uint32_t magic_rows = (65536u + (uint32_t)rows_per_pass - 1u) / (uint32_t)rows_per_pass;
  const int copies_per_store = (int)((64u * magic_rows) >> 16);
  const int copy_slot = (int)(((uint32_t)lane * magic_rows) >> 16), q = lane - copy_slot * rows_per_pass;
  const int q_first_lane = q * cols;
  const bool rescale = (flags & APC_EDGE_GRAD_RESCALE) != 0, no_producer = (flags & APC_EDGE_NO_PRODUCER) != 0;
  const bool entry_by_entry = (flags & APC_PACKED_MIXED) != 0 || no_producer || t0 < 0;
  double *const cost_base = cost_out + entry_begin;
  for (int row0 = wave * rows_per_pass; row0 < rows; row0 += waves * rows_per_pass) {
    const int r = row0 + r_local;
    const bool active = in_pass && r < rows;
    const uint32_t src = (uint32_t)from_lane((int)col_code, c), tgt = (uint32_t)from_lane((int)row_code, r);
    const double row_cpa = from_lane(cpa, r);
    const uint32_t local = (uint32_t)(r * cols + c);
    double comm = 0.0;
    int trans = 0;
    if (!entry_by_entry) {
      const bool flip = M == 2 && src == 0x4040u && ((tgt >> 6) & 3u) == 2u && ((tgt >> 14) & 3u) == 2u;
      const bool some_flip = M == 2 && __ballot(flip && active) != 0;  // (Partial, Partial) -> all Shard walks dim 1 first (:146-151)
      if constexpr (pow2) {
        int j = a.lg_total;  // bytes / num_shards = bytes x 2^(j - L): exact on such a mesh
#pragma unroll
        for (int i = 0; i < M; ++i) j -= ((src >> (8 * i + 6)) & 3u) == 2u ? k2.lg[i] : 0;
        comm = contiguous ? entry_cost_pow2<M, 0, true>(src, tgt, j, p.a2a_scale, k2) : entry_cost_pow2<M, 0, false>(src, tgt, j, p.a2a_scale, k2);
        if (some_flip) {
          const double other = contiguous ? entry_cost_pow2<M, 1, true>(src, tgt, j, p.a2a_scale, k2)
                                          : entry_cost_pow2<M, 1, false>(src, tgt, j, p.a2a_scale, k2);
          comm = flip ? other : comm;
        }
      } else {
        double shards = 1.0;  // exact: a product of mesh sizes (torch _dtensor_spec.py:555-561)
#pragma unroll
        for (int i = 0; i < M; ++i) shards *= ((src >> (8 * i + 6)) & 3u) == 2u ? (double)p.mesh_size[i] : 1.0;
        const double gb = fbytes / shards * 0x1p-30;  // / 1024 / 1024 / 1024 (:66-68)
        comm = contiguous ? entry_cost_flat<M, 0, true>(src, tgt, gb, p, k) : entry_cost_flat<M, 0, false>(src, tgt, gb, p, k);
        if (some_flip) {
          const double other = contiguous ? entry_cost_flat<M, 1, true>(src, tgt, gb, p, k)
                                          : entry_cost_flat<M, 1, false>(src, tgt, gb, p, k);
          comm = flip ? other : comm;
        }
      }
      trans = src != tgt ? p.transition_scale : 0;  // optimize_sharding.py:345-351
      // :358-359; the quotient through the reciprocal is the division's (div_by), +inf stays +inf
      if (rescale) comm = comm < __builtin_inf() ? div_by(comm, p.rescale, a.inv_rescale) : comm;
    } else {
      // pass-through edges and tiles whose specs are not all DTensorSpecs on one tensor: the
      // rule-provided value, or the direct evaluation on the entry's own tensor
      const int sten = from_lane(col_tensor, c), tten = from_lane(row_tensor, r);
      if (active) {
        if (no_producer || sten < 0 || tten < 0) {
          comm = a.pt_values[pt_begin + local];
        } else {
          trans = src != tgt ? p.transition_scale : 0;
          int64_t shards = 1;
#pragma unroll
          for (int i = 0; i < M; ++i)
            if (kind_of((src >> (8 * i)) & 0xFF) == 2) shards *= p.mesh_size[i];
          int64_t sten_bytes;
          bool sten_contiguous;
          tensor_bytes_and_contiguity(a.rank[sten], a.itemsize[sten], a.shape + (int64_t)sten * APC_MAX_RANK,
                                      a.stride + (int64_t)sten * APC_MAX_RANK, sten_bytes, sten_contiguous);
          const double gb = (double)sten_bytes / (double)shards / 1024 / 1024 / 1024;
          comm = entry_cost<M>(src, tgt, gb, sten_contiguous, p);
        }
        if (rescale) comm = comm / p.rescale;
      }
    }
    const double total = comm + row_cpa + (double)trans;  // optimize_sharding.py:368-372
    // ---- the entry, to the tile's edge and to every identical edge ----------------------------------
    const uint32_t off8 = local * 8u;
    if (active) store_at(cost_base, off8, total);
    for (int d = 0; d < dup_count; ++d) {  // per copy: the offset out of its lane, scalar address arithmetic, the store
      double *const base = cost_out + value_of_lane(copies.entry0, d);
      if (active) store_at(base, off8, total);
    }
    // ---- the rows' minima ----------------------------------------------------------------------------
    double m;
    int mc;
    row_min_in_wave(active, total, c, cols, lane, m, mc);
    // A row's minimum sits in the row's first lane.  Stored to all copies at once: lane (q, copy) =
    // (lane mod rows per pass, lane / rows per pass) fetches row q's result and writes it to its
    // copy (copy 0 = the tile's own edge), 64 / rows-per-pass copies per store instruction.
    const double m_q = from_lane(m, q_first_lane);
    const int mc_q = from_lane(mc, q_first_lane);
    const bool row_live = row0 + q < rows;
    for (int copy0 = 0; copy0 <= dup_count; copy0 += copies_per_store) {
      const int copy = copy0 + copy_slot;
      const int64_t first_row = from_lane_i64(copies.row0, copy - 1);  // (every lane takes part)
      if (row_live && copy_slot < copies_per_store && copy <= dup_count) {
        const int64_t out = (copy == 0 ? row_begin : first_row) + row0 + q;
        // (plain stores: written through, these 8- and 4-byte pieces cost whole sectors of HBM
        // writes, 21.0 instead of 19.2 MB per launch, for 0.15 us)
        a.row_min_out[out] = m_q;
        a.row_arg_out[out] = mc_q;
      }
    }
  }
}

// ------------------------------------------------------------------------------------------
// The same pass over small tiles: kLanes (16 or 32) lanes take a tile, a wavefront four or two.  A tile costs a wavefront some 900
// instructions, eleven arrays to fetch and what the dispatcher does for it whether it has four entries or 256: from a few thousand tiles on
// that, and not latency, is the launch.  Everything that is wave-uniform above is a lane's own here: the record's words and the copies' offsets by
// DPP broadcasts within 16 lanes, each of which fetches them; a lane's row and column by quotients, and whole rows go round by round, though one round
// (1.5 us: a chain of bpermutes and fp64, few wavefronts to hide it) is what the host takes few lanes for (CostTables.packed_lanes).
// What a launch's constants cost: the compiler keeps 54 to 116 scalar registers in vector lanes (pow2 meshes; 62 to 180 on others), where the form
// with 256 lanes has 7 to 43 (11 to 81).  Four numbers of lanes are 64 forms of the kernel instead of 16.
// us a pass before (the faster of a workgroup a tile and of staged tiles) / now: 4 292 tiles of at most 16 entries on (64,) 6.5 / 4.2, 5 770 on (12, 6)
// 9.1 / 5.5, 2 908 on (3, 2, 2, 2) 10.2 / 5.8; with 32 lanes 4 644 of at most 25 on (16, 8, 4) 7.4 / 6.4, 4 693 on (3, 2, 2, 2) 15.1 / 9.5.
// ------------------------------------------------------------------------------------------
static_assert(APC_PACKED_MAX_DUPS == 16 && APC_MAX_RANK <= 16, "16 lanes hold a tile's dims, identical edges and the first words of its record");

// The value of lane N of the lane's row of 16 (DPP row_newbcast:N).
template <int N>
__device__ __forceinline__ int of_lane16(int x) {
  return __builtin_amdgcn_update_dpp(0, x, 0x150 + N, 0xF, 0xF, true);
}
template <int N>
__device__ __forceinline__ int64_t of_lane16(int64_t x) {
  return (int64_t)((uint64_t)(uint32_t)of_lane16<N>((int)((uint64_t)x >> 32)) << 32 | (uint32_t)of_lane16<N>((int)(uint32_t)x));
}
// The largest over the four tiles of a value that their 16 lanes share.
__device__ __forceinline__ int most_of_tiles(int x) {
  return max(max(__builtin_amdgcn_readlane(x, 0), __builtin_amdgcn_readlane(x, 16)),
             max(__builtin_amdgcn_readlane(x, 32), __builtin_amdgcn_readlane(x, 48)));
}

// tensor_info_of_lanes, every 16 lanes of their own tensor.
__device__ __forceinline__ void tensor_info_of_lanes16(int rank, int itemsize, int64_t x, int64_t y, int lane, double &bytes, bool &contiguous) {
  const int dim = lane & 15;
  const bool live = dim < min(rank, APC_MAX_RANK);
  const double size = live ? (double)x : 1.0;
  double product = size;
  product *= from_lane_behind<1>(product, 1.0);
  product *= from_lane_behind<2>(product, 1.0);
  product *= from_lane_behind<4>(product, 1.0);
  const double expected = from_lane_behind<1>(product, 1.0);
  const bool differs = size != 1.0 && (double)y != expected;
  const int shift = lane & 48;
  contiguous = ((__ballot(differs) >> shift) & 0xFFFF) == 0;
  const double total = __hiloint2double(of_lane16<0>(__double2hiint(product)), of_lane16<0>(__double2loint(product))) * (double)itemsize;
  bytes = total;
  const uint64_t odd = __ballot(!(size >= 1.0) || !(product < 0x1p53) || !(total < 0x1p53));
  if (odd != 0) {  // (uniform)
    int64_t nbytes = itemsize, one = 1, most = 1;
    bool dims_contiguous = true;
#pragma unroll 1
    for (int i = APC_MAX_RANK - 1; i >= 0; --i) {
      const int64_t xi = from_lane_i64(x, shift + i), yi = from_lane_i64(y, shift + i);  // (every lane takes part)
      if (i >= rank) continue;
      nbytes *= xi;
      if (xi == 1) continue;
      if (yi != one && yi != most) dims_contiguous = false;
      most *= xi > 1 ? xi : 1;
      one *= xi;
    }
    if (((odd >> shift) & 0xFFFF) != 0) {
      bytes = (double)nbytes;
      contiguous = dims_contiguous;
    }
  }
}

__device__ __forceinline__ void store_at(double *to, double value) {  // written through, as above
  __asm__ volatile("global_store_dwordx2 %0, %1, off sc0 sc1" ::"v"(to), "v"(value) : "memory");
}
// x / y for 0 <= x <= 32, 1 <= y <= 32: x + 0.5 is nowhere nearer to a multiple of y than half of one, the reciprocal as good as exact
__device__ __forceinline__ int small_quotient(int x, float inverse) { return (int)(((float)x + 0.5f) * inverse); }

template <int D>
__device__ __forceinline__ void store_copies16(int64_t entry0, double *cost_out, int64_t local, int dup_count, int most_dups, bool active, double total) {
  if constexpr (D < APC_PACKED_MAX_DUPS) {
    if (D >= most_dups) return;  // (uniform)
    double *const to = cost_out + (of_lane16<D>(entry0) + local);
    if (active && D < dup_count) store_at(to, total);
    store_copies16<D + 1>(entry0, cost_out, local, dup_count, most_dups, active, total);
  }
}

// `first`: the wavefront's first tile.  A tile of more rows or columns than lanes is left out and says so.
constexpr int kTooFewLanes = 2;  // in the error flag
template <int M, bool POW2, int kLanes>
__device__ __forceinline__ void packed_small_tiles(const apc_packed_tile *tiles, int first, int n_tiles, double *cost_out, const PackedArgs &a,
                                                   int32_t *const &error_flag) {
  const apc_params &p = a.p;
  const int lane = threadIdx.x & 63, sub = lane & (kLanes - 1), first_lane = lane & (64 - kLanes);
  const int tile = first + lane / kLanes;
  // ---- the one round of loads -------------------------------------------------------------------
  const char *const T = reinterpret_cast<const char *>(tiles + min(tile, n_tiles - 1));
  const char *const T4 = T + sub * 4, *const T8 = T + sub * 8, *const of_16 = T + (lane & 15) * 8, *const dims = T + (sub & (APC_MAX_RANK - 1)) * 8;
#define APC_OF(TYPE_, BASE_, FIELD_) (*reinterpret_cast<const TYPE_ *>((BASE_) + offsetof(apc_packed_tile, FIELD_)))
  const int h = *reinterpret_cast<const int32_t *>(T + (lane & 15) * 4);
  const int64_t dim_size = APC_OF(int64_t, dims, tensor_shape), dim_stride = APC_OF(int64_t, dims, tensor_stride);
  TileCopies copies;
  copies.entry0 = APC_OF(int64_t, of_16, dup_entry_begin);
  copies.row0 = APC_OF(int64_t, of_16, dup_row_begin);
  copies.row_out = 0;
  const uint32_t col_code = APC_OF(uint32_t, T4, col_codes), row_code = APC_OF(uint32_t, T4, row_codes);
  const int col_tensor = APC_OF(int32_t, T4, col_tensor), row_tensor = APC_OF(int32_t, T4, row_tensor);
  const int64_t row_flops = APC_OF(int64_t, T8, row_flops), row_rw = APC_OF(int64_t, T8, row_rw_bytes);
  const int row_meta = APC_OF(int32_t, T4, row_meta);
#undef APC_OF
  const double gf_of_lane = a.p.gpu_flops[lane & (APC_MAX_DTYPES - 1)], inv_gf_of_lane = a.p.inv_gpu_flops[lane & (APC_MAX_DTYPES - 1)];
  fetch_arguments_now(a.row_min_out, a.row_arg_out, p.hbm_bw, p.inv_hbm_bw, p.rw_eff, p.inv_rw_eff, p.launch_floor, p.compute_eff,
                      p.inv_compute_eff, a.inv_rescale, p.rescale, p.a2a_scale, p.base_latency);
  int rows = of_lane16<0>(h);
  const int cols = of_lane16<1>(h), flags = of_lane16<2>(h), dup_count = of_lane16<3>(h), t0 = of_lane16<4>(h);
  const bool refused = (unsigned)rows > (unsigned)kLanes || (unsigned)(cols - 1) >= (unsigned)kLanes || (unsigned)dup_count > (unsigned)APC_PACKED_MAX_DUPS;
  if (__ballot(refused && tile < n_tiles) != 0) {  // (uniform: the flag's address is fetched here)
    int32_t *const flag = error_flag;
    if (refused && tile < n_tiles && flag) *flag = kTooFewLanes;
  }
  if (tile >= n_tiles || refused) rows = 0;
  const int64_t entry_begin = (int64_t)((uint64_t)(uint32_t)of_lane16<9>(h) << 32 | (uint32_t)of_lane16<8>(h));
  const int64_t row_begin = (int64_t)((uint64_t)(uint32_t)of_lane16<11>(h) << 32 | (uint32_t)of_lane16<10>(h));
  // ---- the tensor's bytes, the rows' compute costs ------------------------------------------------
  double fbytes;
  bool contiguous;
  tensor_info_of_lanes16(of_lane16<5>(h), of_lane16<6>(h), dim_size, dim_stride, lane, fbytes, contiguous);
  const int dt = (int)(int8_t)(row_meta & 0xFF);
  const bool known_dtype = dt >= 0 && dt < APC_MAX_DTYPES;
  const double gf = from_lane(gf_of_lane, dt & (APC_MAX_DTYPES - 1)), inv_gf = from_lane(inv_gf_of_lane, dt & (APC_MAX_DTYPES - 1));
  const double cpa = compute_cost_through_reciprocals(p, ((row_meta >> 8) & 0xFF) != 0, row_rw, row_flops, known_dtype ? gf : 0.0,
                                                      known_dtype ? inv_gf : 0.0) /
                     (double)(row_meta >> 16);  // (lanes past the tile's rows: never read)
  settle(copies);
  FlatConstants<M> k;
  Pow2Constants<M> k2;
  if constexpr (!POW2) k = flat_constants<M>(p);
  if constexpr (POW2) {
    k2.R = div_by(div_by(fbytes, p.hbm_bw, p.inv_hbm_bw) * 1e6, p.rw_eff, p.inv_rw_eff);
    k2.rw_shift = 1 - a.lg_total;
    k2.floor = p.launch_floor;
#pragma unroll
    for (int i = 0; i < M; ++i) {
      const double hops1 = (double)(p.mesh_size[i] - 1), hops2 = (double)(2 * (p.mesh_size[i] - 1));
      k2.B[i] = div_by(fbytes * hops1, p.bw[i], p.inv_bw[i]) * 1e6;
      k2.lat1[i] = p.base_latency + hops1 * p.lat[i];
      k2.lat2[i] = p.base_latency + hops2 * p.lat[i];
      k2.lg[i] = a.lg[i];
      k2.shift[i] = -a.lg_total - 30 - a.lg[i];
    }
  }
  // ---- whole rows, `cols` lanes a row ---------------------------------------------------------------
  const float inv_cols = __builtin_amdgcn_rcpf((float)cols);
  const int rows_per_pass = rows > 0 ? small_quotient(kLanes, inv_cols) : 1;
  const int r_local = small_quotient(sub, inv_cols), c = sub - r_local * cols;
  const bool in_pass = r_local < rows_per_pass;
  // (the stores of the row minima: lane -> (row of the pass, copy))
  const float inv_rows = __builtin_amdgcn_rcpf((float)rows_per_pass);
  const int copies_per_store = small_quotient(kLanes, inv_rows);
  const int copy_slot = small_quotient(sub, inv_rows), q = sub - copy_slot * rows_per_pass;
  const int q_first_lane = first_lane + q * cols;
  const bool rescale = (flags & APC_EDGE_GRAD_RESCALE) != 0, no_producer = (flags & APC_EDGE_NO_PRODUCER) != 0;
  const bool entry_by_entry = (flags & APC_PACKED_MIXED) != 0 || no_producer || t0 < 0;
  const bool all_contiguous = __ballot(rows > 0 && !contiguous) == 0;
  const int most_dups = most_of_tiles(rows > 0 ? dup_count : 0), most_cols = most_of_tiles(rows > 0 ? cols : 1);
  for (int row0 = 0; __ballot(row0 < rows) != 0; row0 += rows_per_pass) {
    const int r = row0 + r_local;
    const bool active = in_pass && r < rows;
    const uint32_t src = (uint32_t)from_lane((int)col_code, first_lane + c), tgt = (uint32_t)from_lane((int)row_code, first_lane + (r & (kLanes - 1)));
    const double row_cpa = from_lane(cpa, first_lane + (r & (kLanes - 1)));
    const int64_t local = entry_begin + (r * cols + c);
    const bool flip = M == 2 && src == 0x4040u && ((tgt >> 6) & 3u) == 2u && ((tgt >> 14) & 3u) == 2u;
    const bool some_flip = M == 2 && __ballot(flip && active) != 0;  // (Partial, Partial) -> all Shard walks dim 1 first (:146-151)
    double comm;
    if constexpr (POW2) {
      int j = a.lg_total;  // bytes / num_shards = bytes x 2^(j - L)
#pragma unroll
      for (int i = 0; i < M; ++i) j -= ((src >> (8 * i + 6)) & 3u) == 2u ? k2.lg[i] : 0;
      comm = all_contiguous ? entry_cost_pow2<M, 0, true>(src, tgt, j, p.a2a_scale, k2) : entry_cost_pow2<M, 0, false>(src, tgt, j, p.a2a_scale, k2, contiguous);
      if (some_flip) {
        const double other = entry_cost_pow2<M, 1, false>(src, tgt, j, p.a2a_scale, k2, contiguous);
        comm = flip ? other : comm;
      }
    } else {
      double shards = 1.0;  // exact: a product of mesh sizes (torch _dtensor_spec.py:555-561)
#pragma unroll
      for (int i = 0; i < M; ++i) shards *= ((src >> (8 * i + 6)) & 3u) == 2u ? (double)p.mesh_size[i] : 1.0;
      const double gb = fbytes / shards * 0x1p-30;  // / 1024 / 1024 / 1024 (:66-68)
      comm = all_contiguous ? entry_cost_flat<M, 0, true>(src, tgt, gb, p, k) : entry_cost_flat<M, 0, false>(src, tgt, gb, p, k, contiguous);
      if (some_flip) {
        const double other = entry_cost_flat<M, 1, false>(src, tgt, gb, p, k, contiguous);
        comm = flip ? other : comm;
      }
    }
    int trans = src != tgt ? p.transition_scale : 0;  // optimize_sharding.py:345-351
    // :358-359; the quotient through the reciprocal is the division's (div_by), +inf stays +inf
    if (rescale) comm = comm < __builtin_inf() ? div_by(comm, p.rescale, a.inv_rescale) : comm;
    if (__ballot(active && entry_by_entry) != 0) {  // pass-through edges, and tiles whose specs are not all DTensorSpecs on one tensor
      const int sten = from_lane(col_tensor, first_lane + c), tten = from_lane(row_tensor, first_lane + (r & (kLanes - 1)));
      const int64_t pt_begin = (int64_t)((uint64_t)(uint32_t)of_lane16<13>(h) << 32 | (uint32_t)of_lane16<12>(h));  // (every lane takes part)
      if (active && entry_by_entry) {
        trans = 0;
        if (no_producer || sten < 0 || tten < 0) {
          comm = a.pt_values[pt_begin + (r * cols + c)];
        } else {
          trans = src != tgt ? p.transition_scale : 0;
          int64_t shards = 1;
#pragma unroll
          for (int i = 0; i < M; ++i)
            if (kind_of((src >> (8 * i)) & 0xFF) == 2) shards *= p.mesh_size[i];
          int64_t sten_bytes;
          bool sten_contiguous;
          tensor_bytes_and_contiguity(a.rank[sten], a.itemsize[sten], a.shape + (int64_t)sten * APC_MAX_RANK,
                                      a.stride + (int64_t)sten * APC_MAX_RANK, sten_bytes, sten_contiguous);
          const double gb = (double)sten_bytes / (double)shards / 1024 / 1024 / 1024;
          comm = entry_cost<M>(src, tgt, gb, sten_contiguous, p);
        }
        if (rescale) comm = comm / p.rescale;
      }
    }
    const double total = comm + row_cpa + (double)trans;  // optimize_sharding.py:368-372
    // ---- the entry, to the tile's edge and to every identical edge ------------------------------------
    if (active) store_at(cost_out + local, total);
    store_copies16<0>(copies.entry0, cost_out, local - entry_begin, dup_count, most_dups, active, total);
    // ---- the rows' minima (row_min_in_wave, within 16 lanes) -------------------------------------------
    double m = active ? total : __builtin_inf();
    int mc = c;
#define APC_ROW_MIN_STEP(N_)                                        \
  if (N_ < most_cols) {                                             \
    const double om = from_lane_ahead<N_>(m);                       \
    const int oc = from_lane_ahead<N_>(mc);                         \
    if ((sub & 15) + N_ < 16 && c + N_ < cols && om < m) {                 \
      m = om;                                                       \
      mc = oc;                                                      \
    }                                                               \
  }
    APC_ROW_MIN_STEP(1)
    APC_ROW_MIN_STEP(2)
    APC_ROW_MIN_STEP(4)
    APC_ROW_MIN_STEP(8)
#undef APC_ROW_MIN_STEP
    if constexpr (kLanes == 32) {
      const double pm = from_lane(m, first_lane + 16);
      const int pc = from_lane(mc, first_lane + 16);
      if (sub < 16 && c + 16 - sub < cols && pm < m) {
        m = pm;
        mc = pc;
      }
    }
    const double m_q = from_lane(m, q_first_lane);
    const int mc_q = from_lane(mc, q_first_lane);
    const bool row_live = row0 + q < rows && copy_slot < copies_per_store;
    for (int copy0 = 0; __ballot(row_live && copy0 <= dup_count) != 0; copy0 += copies_per_store) {
      const int copy = copy0 + copy_slot;
      const int64_t first_row = from_lane_i64(copies.row0, first_lane + ((copy - 1) & 15));  // (every lane takes part)
      if (row_live && copy <= dup_count) {
        const int64_t out = (copy == 0 ? row_begin : first_row) + row0 + q;
        a.row_min_out[out] = m_q;
        a.row_arg_out[out] = mc_q;
      }
    }
  }
}

struct PackedBlock {
  PackedArgs a;
  apc_params p;
  TensorTableArgs t;
  ComputeCostArgs c;
  int64_t tensor_blocks;
};

template <int M, bool POW2, bool KEPT, int LANES>  // LANES a tile
__global__ __launch_bounds__(kBlock) void build_tables_packed_kernel(APC_LAUNCH_PARAMS(PackedBlock, KEPT)) {
  const PackedBlock &k = launch_block<KEPT>(kept);
  const int64_t b = blockIdx.x;
  if (b < tile_blocks) {
    const apc_packed_tile *const tiles = static_cast<const apc_packed_tile *>(work);
    if constexpr (LANES == kBlock) {
      const int tile_id = tile_of_block((int)b, n_tiles, xcd_shift);
      if (tile_id >= n_tiles) return;
      packed_tile<M, POW2, false>(tiles + tile_id, cost_out, k.a);
    } else {
      constexpr int per_block = kBlock / LANES;
      const int n_groups = (n_tiles + per_block - 1) / per_block, group = tile_of_block((int)b, n_groups, xcd_shift);
      const int first = group * per_block + uniform_i32((int)threadIdx.x >> 6) * (64 / LANES);
      if (group >= n_groups || first >= n_tiles) return;
      if constexpr (LANES == 64) packed_tile<M, POW2, true>(tiles + first, cost_out, k.a);
      else packed_small_tiles<M, POW2, LANES>(tiles, first, n_tiles, cost_out, k.a, k.c.error_flag);
    }
    return;
  }
  const int64_t tb = b - tile_blocks;
  if (tb < k.tensor_blocks) tensor_tables_block<kBlock, true>(tb, k.t);
  else compute_costs_block<kBlock, true>(tb - k.tensor_blocks, k.p, k.c);
}

// ------------------------------------------------------------------------------------------
// a14: segmented min + first argmin.  G consecutive lanes share one segment (G = 4 .. 64,
// chosen by the host from the mean segment length), so short segments do not leave most of
// a wavefront idle.
// ------------------------------------------------------------------------------------------
// Which segments to reduce and where else each result goes (SELECTED instantiation): segment
// selected[i] is reduced and its result stored to itself and to copy_segments[copy_ptr[i] ..
// copy_ptr[i + 1]), segments the caller knows to hold the same values.
struct SegmentCopies {
  const int64_t *selected;
  const int64_t *copy_ptr;
  const int64_t *copy_segments;
};

template <int G, bool SELECTED>
__global__ __launch_bounds__(kBlock) void segmented_min_kernel(const double *__restrict__ values,
                                                               const int64_t *__restrict__ seg_ptr,
                                                               int64_t n_seg, double *__restrict__ mins,
                                                               int32_t *__restrict__ args, SegmentCopies copies) {
  const int sub = threadIdx.x & (G - 1);
  const int64_t slot = (int64_t)blockIdx.x * (kBlock / G) + (threadIdx.x / G);
  const bool live = slot < n_seg;  // (n_seg counts the selected segments when SELECTED)
  const int64_t seg = SELECTED ? (live ? copies.selected[slot] : 0) : slot;
  const int64_t lo = live ? seg_ptr[seg] : 0, hi = live ? seg_ptr[seg + 1] : 0;
  double best = INFINITY;
  int64_t arg = INT64_MAX;  // absolute index; INT64_MAX = none seen
  auto take = [&](double v, int64_t j) {
    if (arg == INT64_MAX || v < best) {
      best = v;
      arg = j;
    }
  };
  // A lane reads pairs of consecutive values (one 16-byte load; segments start at any 8-byte
  // offset, which global loads allow), four such loads in flight (two on a short remainder), taken in index order (first
  // minimum wins); the G lanes of a group sweep 2 G consecutive values per load.
  struct __attribute__((packed, aligned(8))) Pair {
    double x, y;
  };
  int64_t j = lo + 2 * sub;
  for (; j + 6 * G + 1 < hi; j += 8 * G) {
    const Pair a = *reinterpret_cast<const Pair *>(values + j);
    const Pair b = *reinterpret_cast<const Pair *>(values + j + 2 * G);
    const Pair c = *reinterpret_cast<const Pair *>(values + j + 4 * G);
    const Pair d = *reinterpret_cast<const Pair *>(values + j + 6 * G);
    take(a.x, j);
    take(a.y, j + 1);
    take(b.x, j + 2 * G);
    take(b.y, j + 2 * G + 1);
    take(c.x, j + 4 * G);
    take(c.y, j + 4 * G + 1);
    take(d.x, j + 6 * G);
    take(d.y, j + 6 * G + 1);
  }
  for (; j + 2 * G + 1 < hi; j += 4 * G) {
    const Pair a = *reinterpret_cast<const Pair *>(values + j);
    const Pair b = *reinterpret_cast<const Pair *>(values + j + 2 * G);
    take(a.x, j);
    take(a.y, j + 1);
    take(b.x, j + 2 * G);
    take(b.y, j + 2 * G + 1);
  }
  for (; j + 1 < hi; j += 2 * G) {
    const Pair a = *reinterpret_cast<const Pair *>(values + j);
    take(a.x, j);
    take(a.y, j + 1);
  }
  if (j < hi) take(values[j], j);
  // lexicographic (value, index) min inside the group; lanes that saw nothing lose
#pragma unroll
  for (int off = G / 2; off > 0; off >>= 1) {
    const double ob = __shfl_xor(best, off, 64);
    const int64_t oa = __shfl_xor(arg, off, 64);
    const bool take = (oa != INT64_MAX) && (arg == INT64_MAX || ob < best || (ob == best && oa < arg));
    if (take) {
      best = ob;
      arg = oa;
    }
  }
  if (live && sub == 0) {
    const int32_t rel = arg == INT64_MAX ? -1 : (int32_t)(arg - lo);
    mins[seg] = best;
    args[seg] = rel;
    if (SELECTED) {
      for (int64_t k = copies.copy_ptr[slot], end = copies.copy_ptr[slot + 1]; k < end; ++k) {
        const int64_t to = copies.copy_segments[k];
        mins[to] = best;
        args[to] = rel;
      }
    }
  }
}

// 8 XCDs; APC_XCD_SHIFT=0 restores the plain work order (tuning)
int xcd_shift() {
  static const int shift = [] {
    const char *env = getenv("APC_XCD_SHIFT");
    const int v = env ? atoi(env) : 3;
    return v < 0 ? 0 : v > 5 ? 5 : v;
  }();
  return shift;
}

// ------------------------------------------------------------------------------------------
// a14: optimistic cost of every (node, strategy): the sum over the node's edges of that
// consumer strategy's row minimum.  A plan pays, on every edge, at least the minimum of the
// row of the strategy its consumer takes, so min over a node's strategies, summed over the
// nodes, bounds the ILP objective from below, and the per-node argmin is the greedy choice a
// warm start begins from.  One thread per strategy; a node's edges are added in the order of
// edges_by_node (deterministic sum).
// ------------------------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void strategy_bounds_kernel(int64_t n_strategies,
                                                                 const int32_t *__restrict__ strat_node,
                                                                 const int64_t *__restrict__ node_strat_begin,
                                                                 const int64_t *__restrict__ node_edge_begin,
                                                                 const int32_t *__restrict__ edges_by_node,
                                                                 const int64_t *__restrict__ edge_row_begin,
                                                                 const double *__restrict__ row_min,
                                                                 double *__restrict__ bound) {
  const int64_t s = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (s >= n_strategies) return;
  const int n = strat_node[s];
  const int64_t k = s - node_strat_begin[n];
  double sum = 0.0;
  for (int64_t j = node_edge_begin[n]; j < node_edge_begin[n + 1]; ++j) sum += row_min[edge_row_begin[edges_by_node[j]] + k];
  bound[s] = sum;
}

// The bounds, the smallest of every node and the first strategy that has it: G consecutive lanes to a node, its
// strategies and their order those of segmented_min_kernel, so that the result is its result, NaN included.
// Bound by a chain of loads: a node's ranges, its edges, their first rows, the minima.  A lane has four edges and eight of its
// strategies in flight and goes through the chain once for them all; pair of strategies by pair and edge by edge that was a dozen round
// trips one behind the other.  us by rocprofv3, before / now: 8 320 nodes of some 12 strategies 13.3 / 7.4, 3 000 of 34 30.7 / 10.1,
// 2 500 of 30 27.9 / 10.0, 24 000 of 12 14.9 / 9.1, 2 000 of 15 17.3 / 7.6, 8 000 of 3 4.3 / 4.5.
// (Workgroups of one wavefront: more compute units take part.)
template <int G, int kPairs>  // kPairs: of a lane's strategies, in flight
__global__ __launch_bounds__(kBlock) void greedy_strategies_kernel(int64_t n_nodes, const int64_t *__restrict__ node_strat_begin,
                                                                   const int64_t *__restrict__ node_edge_begin,
                                                                   const int32_t *__restrict__ edges_by_node,
                                                                   const int64_t *__restrict__ edge_row_begin,
                                                                   const double *__restrict__ row_min, double *__restrict__ bound,
                                                                   double *__restrict__ node_min, int32_t *__restrict__ node_argmin) {
  const int sub = threadIdx.x & (G - 1);
  const int64_t n = (int64_t)blockIdx.x * (blockDim.x / G) + (threadIdx.x / G);
  const bool live = n < n_nodes;
  const int64_t lo = live ? node_strat_begin[n] : 0, hi = live ? node_strat_begin[n + 1] : 0;
  const int64_t e0 = live ? node_edge_begin[n] : 0, e1 = live ? node_edge_begin[n + 1] : 0;
  double best = INFINITY;
  int64_t arg = INT64_MAX;  // INT64_MAX = none seen
  auto take = [&](double v, int64_t j) {
    bound[j] = v;
    if (arg == INT64_MAX || v < best) {
      best = v;
      arg = j;
    }
  };
  constexpr int kEdges = 4;
  for (int64_t j = lo + 2 * sub; j < hi; j += 2 * G * kPairs) {
    double sum[2 * kPairs] = {};
    for (int64_t e = e0; e < e1; e += kEdges) {
      const double *row[kEdges];
      double v[kEdges][2 * kPairs] = {};
      int32_t edge[kEdges];
#pragma unroll
      for (int u = 0; u < kEdges; ++u)
        if (e + u < e1) edge[u] = edges_by_node[e + u];
#pragma unroll
      for (int u = 0; u < kEdges; ++u)
        if (e + u < e1) row[u] = row_min + edge_row_begin[edge[u]] - lo;
#pragma unroll
      for (int u = 0; u < kEdges; ++u)
        if (e + u < e1) {
#pragma unroll
          for (int k = 0; k < 2 * kPairs; ++k)
            if (const int64_t at = j + (k / 2) * 2 * G + (k & 1); at < hi) v[u][k] = row[u][at];
        }
#pragma unroll
      for (int u = 0; u < kEdges; ++u)
#pragma unroll
        for (int k = 0; k < 2 * kPairs; ++k) sum[k] = e + u < e1 ? sum[k] + v[u][k] : sum[k];
    }
#pragma unroll
    for (int k = 0; k < 2 * kPairs; ++k)
      if (const int64_t at = j + (k / 2) * 2 * G + (k & 1); at < hi) take(sum[k], at);
  }
#pragma unroll
  for (int off = G / 2; off > 0; off >>= 1) {
    const double ob = __shfl_xor(best, off, 64);
    const int64_t oa = __shfl_xor(arg, off, 64);
    if (oa != INT64_MAX && (arg == INT64_MAX || ob < best || (ob == best && oa < arg))) {
      best = ob;
      arg = oa;
    }
  }
  if (live && sub == 0) {
    node_min[n] = best;
    node_argmin[n] = arg == INT64_MAX ? -1 : (int32_t)(arg - lo);
  }
}

// Several arrays in one launch, kCopyUnit bytes of one a workgroup, in pieces of 16 bytes where both its ends allow it.  For what travels
// between device and pinned host memory together: bound by the bus, and behind it by what every copy of the runtime costs, some
// 10 us between two of them.  us until the stream has finished, the runtime's copies / this: five arrays of 4 KB 21 / 12, of 64 KB 50 / 18, of 1 MB 137 /
// 106; 84 MB to the host in parts of 2 MB with an event each 2 150 / 1 810 (one copy of all: 1 550).  (4, 16, 32 and 64 KB a
// workgroup: 1 770 / 1 810 to the host, 2 460 / 1 910 from it, larger ones as 16.)
constexpr int kCopyUnit = 16384;
struct CopyArrays {
  const char *from[APC_COPY_MAX_ARRAYS];
  char *to[APC_COPY_MAX_ARRAYS];
  int64_t bytes[APC_COPY_MAX_ARRAYS];
  int32_t first_block[APC_COPY_MAX_ARRAYS];
  int32_t n;
};
template <typename V>
__device__ __forceinline__ void copy_unit(const char *from, char *to, int n) {  // n bytes, at most kCopyUnit
  constexpr int kAhead = 4, kRound = kAhead * kBlock;  // loads a thread issues before it waits for the first
  const V *x = reinterpret_cast<const V *>(from);
  V *y = reinterpret_cast<V *>(to);
  const int whole = n / (int)sizeof(V), tid = threadIdx.x;
  for (int base = 0; base < whole; base += kRound) {
    V v[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u)
      if (const int i = base + u * kBlock + tid; i < whole) v[u] = x[i];
#pragma unroll
    for (int u = 0; u < kAhead; ++u)
      if (const int i = base + u * kBlock + tid; i < whole) y[i] = v[u];
  }
  if (const int i = whole * (int)sizeof(V) + tid; i < n) to[i] = from[i];  // (fewer than 16)
}
__global__ __launch_bounds__(kBlock) void copy_arrays_kernel(CopyArrays a) {
  const int lane = threadIdx.x & 63, b = (int)blockIdx.x;
  // the last array that begins at this workgroup or before (none is empty)
  const int k = uniform_i32(__popcll(__ballot(lane < a.n && a.first_block[min(lane, APC_COPY_MAX_ARRAYS - 1)] <= b))) - 1;
  if (k < 0) return;
  const int64_t at = (int64_t)(b - a.first_block[k]) * kCopyUnit;
  const int n = (int)min((int64_t)kCopyUnit, a.bytes[k] - at);
  const char *from = a.from[k] + at;
  char *to = a.to[k] + at;
  const uint32_t low = (uint32_t)(reinterpret_cast<uintptr_t>(from) | reinterpret_cast<uintptr_t>(to));
  if ((low & 15) == 0) copy_unit<u32x4>(from, to, n);
  else if ((low & 3) == 0) copy_unit<uint32_t>(from, to, n);
  else copy_unit<uint8_t>(from, to, n);
}

// First matrix row of every edge: one workgroup walks the edges in blocks of four a thread, four blocks at a time, whose sums are scanned
// across it behind one barrier.  Bound by the latency of the counts, which may be in host memory.  (us a call with its wait, a consecutive
// run of edges a thread / these / the host's sum and its transfer: 8 300 edges 19 / 18 / 25, 100 000 135 / 54 / 97, 1 000 000 2 116 / 430 / 1 110.)
constexpr int kScanThreads = 1024, kScanEdges = 4, kScanBlocks = 4;
__device__ __forceinline__ void edge_rows_of_workgroup(int64_t n_edges, const int32_t *__restrict__ n_tgt, int64_t *__restrict__ begin) {
  constexpr int kWaves = kScanThreads / 64;
  constexpr int64_t kBlockEdges = kScanThreads * kScanEdges;
  __shared__ int64_t s_wave[2][kScanBlocks][kWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  struct __attribute__((packed, aligned(4))) Counts {
    int32_t v[kScanEdges];
  };
  int64_t carry = 0;
  int buffer = 0;
  for (int64_t blocks = 0; blocks < n_edges; blocks += kScanBlocks * kBlockEdges, buffer ^= 1) {
    int32_t rows[kScanBlocks][kScanEdges];
#pragma unroll
    for (int b = 0; b < kScanBlocks; ++b) {
      const int64_t first = blocks + b * kBlockEdges + (int64_t)tid * kScanEdges;
      if (first + kScanEdges <= n_edges) {
        const Counts c = *reinterpret_cast<const Counts *>(n_tgt + first);
#pragma unroll
        for (int k = 0; k < kScanEdges; ++k) rows[b][k] = c.v[k];
      } else {
#pragma unroll
        for (int k = 0; k < kScanEdges; ++k) rows[b][k] = first + k < n_edges ? n_tgt[first + k] : 0;
      }
    }
    int64_t in_front[kScanBlocks];  // of this thread's edges, within its wavefront
#pragma unroll
    for (int b = 0; b < kScanBlocks; ++b) {
      int64_t sum = 0;
#pragma unroll
      for (int k = 0; k < kScanEdges; ++k) sum += rows[b][k];
      int64_t upto = sum;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int64_t o = __shfl_up(upto, off, 64);
        if (lane >= off) upto += o;
      }
      if (lane == 63) s_wave[buffer][b][wave] = upto;
      in_front[b] = upto - sum;
    }
    __syncthreads();  // (the other buffer is written again behind the next one)
#pragma unroll
    for (int b = 0; b < kScanBlocks; ++b) {
      int64_t at = carry + in_front[b];
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        const int64_t of_wave = s_wave[buffer][b][w];
        at += w < wave ? of_wave : 0;
        carry += of_wave;
      }
      const int64_t first = blocks + b * kBlockEdges + (int64_t)tid * kScanEdges;
#pragma unroll
      for (int k = 0; k < kScanEdges; ++k) {
        if (first + k < n_edges) begin[first + k] = at;
        at += rows[b][k];
      }
    }
  }
}
__global__ __launch_bounds__(kScanThreads) void edge_rows_kernel(int64_t n_edges, const int32_t *__restrict__ n_tgt, int64_t *__restrict__ begin) {
  edge_rows_of_workgroup(n_edges, n_tgt, begin);
}

// What the tiles of a report read, in one launch: the first rows of the edges by the first workgroup, the tensor table and the compute
// costs by the others, which are done before it is.  The flag of an unsupported dtype may be in host memory.  (us a report, as two launches with a
// fill of the flag in front and a copy of it behind / this way, in turn: 1.5 M entries on (64, 4) 276 / 241, 5.8 M on (16, 8, 4) 257 / 228, 530 k on
// (3, 2, 2, 2) 237 / 215; the faster greedy strategies above show by 0 to 6 us in the same calls.)
struct ReportInputsArgs {
  apc_params p;
  TensorTableArgs t;
  ComputeCostArgs c;
  int64_t n_edges;
  const int32_t *n_tgt;
  int64_t *row_begin;
  int64_t row_blocks, tensor_blocks;
};
__global__ __launch_bounds__(kScanThreads) void report_inputs_kernel(ReportInputsArgs a) {
  const int64_t b = (int64_t)blockIdx.x - a.row_blocks;
  if (b < 0) edge_rows_of_workgroup(a.n_edges, a.n_tgt, a.row_begin);
  else if (b < a.tensor_blocks) tensor_tables_block<kScanThreads>(b, a.t);
  else compute_costs_block<kScanThreads>(b - a.tensor_blocks, a.p, a.c);
}

// ------------------------------------------------------------------------------------------
// Whether the tables are well formed, where they are about to be read: a lane a spec and a tensor, a wavefront an edge and a tile, every
// index checked before it is used.  Bound by the launch and by the wait for its answer: 315 k specs, 15 104 edges and 4 000 tiles with 15 000
// copies are 8 MB of reads.  (The host takes 0.35 ms for the specs and edges, on eight threads, and as long for every 5 000 copies'
// offsets, one after the other.)
// ------------------------------------------------------------------------------------------
struct CheckTablesArgs {
  int32_t mesh_ndim;
  int64_t n_tensors, n_specs, n_edges, n_pt, n_strategies, n_tiles, n_dups;
  const int32_t *tensor_rank;
  const uint32_t *spec_codes;
  const int32_t *spec_tensor;
  const int32_t *src_begin, *n_src, *tgt_begin, *n_tgt, *flags, *strat_begin;
  const int64_t *pt_begin, *entry_begin;
  const apc_tile *tiles;
  const int64_t *dup_entry_begin;
  int64_t tensor_blocks, spec_blocks, edge_blocks;
  int32_t *malformed;
};
constexpr int kEmptyEdgesPassed = 64;  // in a row, in front of a copy's edge

__device__ bool spec_holds(const CheckTablesArgs &a, int64_t s) {
  const int t = a.spec_tensor[s];
  if (t < -1 || t >= a.n_tensors) return false;
  const uint32_t codes = a.spec_codes[s];
  if (a.mesh_ndim < 4 && (codes >> (8 * a.mesh_ndim)) != 0) return false;
  const int rank = t >= 0 ? a.tensor_rank[t] : APC_MAX_RANK + 16;  // (no DTensorSpec: a Shard of any dim passes)
  bool holds = true;
#pragma unroll
  for (int i = 0; i < APC_MAX_MESH; ++i) {
    const uint32_t c = (codes >> (8 * i)) & 0xFF;
    holds &= kind_of(c) != 3 && (kind_of(c) != 0 || c == 0) && (kind_of(c) != 2 || dim_of(c) < rank);
  }
  return holds;
}

// (uniform but for the lanes' share of the specs)
__device__ bool edge_holds(const CheckTablesArgs &a, int64_t e, int lane) {
  const int64_t ns = a.n_src[e], nt = a.n_tgt[e], sb = a.src_begin[e], tb = a.tgt_begin[e], st = a.strat_begin[e], pt = a.pt_begin[e];
  if (!(ns >= 0 && nt >= 0 && ns <= APC_MAX_STRATEGIES && nt <= APC_MAX_STRATEGIES && sb >= 0 && sb + ns <= a.n_specs && tb >= 0 &&
        tb + nt <= a.n_specs && st >= 0 && st + nt <= a.n_strategies && a.entry_begin[e + 1] - a.entry_begin[e] == ns * nt))
    return false;
  if (pt >= 0 && pt <= a.n_pt && ns * nt <= a.n_pt - pt) return true;
  // without pass-through values: a producer and a tensor behind every spec
  bool needs_pt = (a.flags[e] & APC_EDGE_NO_PRODUCER) != 0;
  for (int64_t j = lane; j < ns; j += 64) needs_pt |= a.spec_tensor[sb + j] < 0;
  for (int64_t j = lane; j < nt; j += 64) needs_pt |= a.spec_tensor[tb + j] < 0;
  return !needs_pt;
}

// (uniform but for a copy's offset a lane)
__device__ bool tile_holds(const CheckTablesArgs &a, int64_t t, int lane) {
  const apc_tile &tl = a.tiles[t];
  const int e = tl.edge, rows = tl.counts & 0xFFFF, cols = tl.counts >> 16;
  if (e < 0 || e >= a.n_edges) return false;
  const int ns = a.n_src[e], nt = a.n_tgt[e];
  if (rows < 1 || rows > APC_TILE_MAX_ROWS || tl.row_begin < 0 || (int64_t)tl.row_begin + rows > nt) return false;
  if (cols < 1 || cols > APC_TILE_MAX_COLS || tl.col_begin < 0 || (int64_t)tl.col_begin + cols > ns) return false;
  const int64_t sp = (int64_t)tl.src_begin + tl.col_begin;
  if (tl.src_begin != a.src_begin[e] || tl.n_src != ns || tl.tgt_begin != a.tgt_begin[e] || tl.flags != a.flags[e] ||
      tl.strat_begin != a.strat_begin[e] || tl.entry_begin != a.entry_begin[e] || tl.pt_begin != a.pt_begin[e])
    return false;
  if (sp < 0 || sp >= a.n_specs || tl.tensor != a.spec_tensor[sp]) return false;
  if (tl.dup_count < 0 || tl.dup_count > APC_TILE_MAX_DUPS || tl.dup_begin < 0 || (int64_t)tl.dup_begin + tl.dup_count > a.n_dups) return false;
  if (lane >= tl.dup_count) return true;
  // the start of another edge with a matrix of the same shape
  const int64_t offset = a.dup_entry_begin[tl.dup_begin + lane];
  int64_t lo = 0, hi = a.n_edges;  // the first edge that begins there, then past the edges without entries
  while (lo < hi) {
    const int64_t mid = (lo + hi) / 2;
    if (a.entry_begin[mid] < offset) lo = mid + 1;
    else hi = mid;
  }
  for (int passed = 0; lo < a.n_edges && (a.n_src[lo] == 0 || a.n_tgt[lo] == 0); ++lo)
    if (++passed > kEmptyEdgesPassed) return false;
  return lo < a.n_edges && a.entry_begin[lo] == offset && lo != e && a.n_src[lo] == ns && a.n_tgt[lo] == nt;
}

__global__ __launch_bounds__(kBlock) void check_tables_kernel(CheckTablesArgs a) {
  int64_t b = blockIdx.x;
  const int64_t row = threadIdx.x, item = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  bool holds = true;
  if (b < a.tensor_blocks) {
    const int64_t t = b * kBlock + row;
    if (t < a.n_tensors) holds = a.tensor_rank[t] >= 0 && a.tensor_rank[t] <= APC_MAX_RANK;
    if (t == 0) holds &= a.entry_begin[0] == 0;
  } else if ((b -= a.tensor_blocks) < a.spec_blocks) {
    const int64_t s = b * kBlock + row;
    if (s < a.n_specs) holds = spec_holds(a, s);
  } else if ((b -= a.spec_blocks) < a.edge_blocks) {
    const int64_t e = b * (kBlock / 64) + item;
    if (e < a.n_edges) holds = edge_holds(a, e, lane);
  } else {
    const int64_t t = (b - a.edge_blocks) * (kBlock / 64) + item;
    if (t < a.n_tiles) holds = tile_holds(a, t, lane);
  }
  if (__ballot(!holds) != 0 && lane == 0) *a.malformed = 1;
}

// ------------------------------------------------------------------------------------------
// Identical edges of tables on the device (apc_edge_classes): a wavefront an edge hashes what its matrix depends on and enters the hash
// into a table, whose slot keeps the smallest edge; then it compares itself with that edge.  Two launches, bound by latency: 15 104 edges with
// 326 k specs, 54 us with the workspaces cleared and the wait for the result, 0.2 ms with the host's strategy table sent in front.  (The host
// hashes, enters and compares in 0.7 ms on eight threads.)
// ------------------------------------------------------------------------------------------
struct EdgeClassArgs {
  int64_t n_specs, n_strategies, n_edges, n_pt, n_slots;
  const uint32_t *spec_codes;
  const int32_t *spec_tensor;
  const int64_t *flops, *rw_bytes;
  const int8_t *dtype;
  const uint8_t *zero_cost;
  const int32_t *num_args;
  const int32_t *src_begin, *n_src, *tgt_begin, *n_tgt, *flags, *strat_begin;
  const int64_t *pt_begin;
  const double *pt_values;
  unsigned long long *keys;
  int32_t *first, *slots;
  int64_t *first_same;
};

// The multiply-and-fold step of the host's hash (Hash128), with its constants.
__device__ __forceinline__ uint64_t fold(uint64_t x, uint64_t y) { return (x * y) ^ __umul64hi(x, y); }
// One value of an edge at its place: a sum over all of them does not depend on the order they are added in.
__device__ __forceinline__ uint64_t hash_of(uint64_t value, int64_t place, int array) {
  return fold(value ^ 0x0CC4A61194F81761ull, ((uint64_t)place * 16 + (uint64_t)array) * 0x5815A7BE0543C11Dull + 0x261DC1F2B8A998C9ull);
}

struct EdgeRanges {
  int64_t ns, nt, sb, tb, st, pt;
  bool inside;
};
__device__ __forceinline__ EdgeRanges ranges_of(const EdgeClassArgs &a, int64_t e) {
  EdgeRanges r{a.n_src[e], a.n_tgt[e], a.src_begin[e], a.tgt_begin[e], a.strat_begin[e], a.pt_begin[e], true};
  r.inside = r.ns >= 0 && r.nt >= 0 && r.sb >= 0 && r.tb >= 0 && r.st >= 0 && r.sb + r.ns <= a.n_specs && r.tb + r.nt <= a.n_specs &&
             r.st + r.nt <= a.n_strategies && (r.pt < 0 || (r.ns * r.nt <= a.n_pt && r.pt <= a.n_pt - r.ns * r.nt));
  return r;
}

__global__ __launch_bounds__(kBlock) void edge_hashes_kernel(EdgeClassArgs a) {
  const int64_t e = (int64_t)blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (e >= a.n_edges) return;
  const EdgeRanges r = ranges_of(a, e);
  if (!r.inside) {  // (uniform)
    if (lane == 0) a.slots[e] = -1;
    return;
  }
  uint64_t sum = 0;
  for (int64_t j = lane; j < r.ns; j += 64) {
    sum += hash_of(a.spec_codes[r.sb + j], j, 0);
    sum += hash_of((uint32_t)a.spec_tensor[r.sb + j], j, 1);
  }
  for (int64_t j = lane; j < r.nt; j += 64) {
    sum += hash_of(((uint64_t)a.spec_codes[r.tb + j] << 32) | (uint32_t)a.spec_tensor[r.tb + j], j, 2);
    sum += hash_of((uint64_t)a.flops[r.st + j], j, 3);
    sum += hash_of((uint64_t)a.rw_bytes[r.st + j], j, 4);
    sum += hash_of(((uint64_t)(uint32_t)a.num_args[r.st + j] << 16) | ((uint64_t)(uint8_t)a.dtype[r.st + j] << 8) | a.zero_cost[r.st + j], j, 5);
  }
  if (r.pt >= 0)
    for (int64_t j = lane; j < r.ns * r.nt; j += 64) sum += hash_of((uint64_t)__double_as_longlong(a.pt_values[r.pt + j]), j, 6);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sum += (uint64_t)__shfl_xor((unsigned long long)sum, off, 64);
  if (lane != 0) return;
  sum += hash_of(((uint64_t)r.ns << 32) | (uint64_t)r.nt, (uint32_t)a.flags[e], r.pt >= 0 ? 7 : 8);
  unsigned long long key = fold(sum, 0x70B7ED67FC9B5C43ull);
  if (key == 0) key = 1;  // (0: an empty slot)
  int64_t at = (int64_t)(key & (unsigned long long)(a.n_slots - 1)), slot = -1;
  for (int64_t probe = 0; probe < a.n_slots; ++probe, at = (at + 1) & (a.n_slots - 1)) {  // (half of them stay empty)
    const unsigned long long there = atomicCAS(a.keys + at, 0ull, key);
    if (there != 0ull && there != key) continue;
    atomicMin(a.first + at, (int)e);
    slot = at;
    break;
  }
  a.slots[e] = (int32_t)slot;
}

__global__ __launch_bounds__(kBlock) void edge_classes_kernel(EdgeClassArgs a) {
  const int64_t e = (int64_t)blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (e >= a.n_edges) return;
  const int slot = a.slots[e];
  const int64_t f = slot < 0 ? e : a.first[slot];
  bool same = f >= 0 && f < e;
  if (same) {  // (uniform)
    const EdgeRanges x = ranges_of(a, f), y = ranges_of(a, e);
    same = x.ns == y.ns && x.nt == y.nt && a.flags[f] == a.flags[e] && (x.pt >= 0) == (y.pt >= 0) && x.inside && y.inside;
    if (same) {
      for (int64_t j = lane; j < x.ns; j += 64)
        same &= a.spec_codes[x.sb + j] == a.spec_codes[y.sb + j] && a.spec_tensor[x.sb + j] == a.spec_tensor[y.sb + j];
      for (int64_t j = lane; j < x.nt; j += 64)
        same &= a.spec_codes[x.tb + j] == a.spec_codes[y.tb + j] && a.spec_tensor[x.tb + j] == a.spec_tensor[y.tb + j] &&
                a.flops[x.st + j] == a.flops[y.st + j] && a.rw_bytes[x.st + j] == a.rw_bytes[y.st + j] &&
                a.num_args[x.st + j] == a.num_args[y.st + j] && a.dtype[x.st + j] == a.dtype[y.st + j] &&
                a.zero_cost[x.st + j] == a.zero_cost[y.st + j];
      if (x.pt >= 0)
        for (int64_t j = lane; j < x.ns * x.nt; j += 64)
          same &= __double_as_longlong(a.pt_values[x.pt + j]) == __double_as_longlong(a.pt_values[y.pt + j]);
    }
  }
  same = __ballot(!same) == 0;
  if (lane == 0) a.first_same[e] = same ? f : e;
}

// ------------------------------------------------------------------------------------------
// Packed records out of tables on the device: a wavefront a tile, lane j producer spec j, consumer spec j and its strategy.  1 138 tiles
// are 3.1 MB: 50 us with the rows of the edges in front and the wait for the answer, 0.2 ms with the host's strategy table sent.  (The host
// copies them together in 0.28 ms and sends them in 0.3.)
// ------------------------------------------------------------------------------------------
struct PackArgs {
  TensorTableArgs t;
  int64_t n_specs, n_strategies, n_edges, n_tiles, n_dups;
  const uint32_t *spec_codes;
  const int32_t *spec_tensor;
  const int64_t *flops, *rw_bytes;
  const int8_t *dtype;
  const uint8_t *zero_cost;
  const int32_t *num_args;
  const int64_t *edge_row_begin;
  const apc_tile *tiles;
  const int64_t *dup_entry_begin, *dup_row_begin;
  apc_packed_tile *packed;
  int32_t *refused;
};

__global__ __launch_bounds__(kBlock) void pack_tiles_kernel(PackArgs a) {
  static_assert(APC_TILE_MAX_COLS == 64 && APC_TILE_MAX_ROWS == 64 && APC_PACKED_MAX_DUPS <= 64 && APC_MAX_RANK <= 64, "a lane each");
  const int64_t id = (int64_t)blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (id >= a.n_tiles) return;
  const apc_tile tl = a.tiles[id];
  const int rows = tl.counts & 0xFFFF, cols = tl.counts >> 16, rb = tl.row_begin, n_dups = tl.dup_count;
  const int64_t first = (int64_t)rb * cols, sb = tl.src_begin, tb = (int64_t)tl.tgt_begin + rb, st = (int64_t)tl.strat_begin + rb;
  bool holds = tl.edge >= 0 && tl.edge < a.n_edges && rows >= 1 && rows <= APC_TILE_MAX_ROWS && cols >= 1 && cols <= APC_TILE_MAX_COLS &&
               tl.col_begin == 0 && cols == tl.n_src && rb >= 0 && sb >= 0 && sb + cols <= a.n_specs && tb >= 0 && tb + rows <= a.n_specs &&
               st >= 0 && st + rows <= a.n_strategies && tl.tensor < a.t.n && n_dups >= 0 && n_dups <= APC_PACKED_MAX_DUPS &&
               tl.dup_begin >= 0 && (int64_t)tl.dup_begin + n_dups <= a.n_dups;
  const bool col = holds && lane < cols, row = holds && lane < rows;
  uint32_t col_codes = 0, row_codes = 0;
  int32_t col_tensor = 0, row_tensor = 0, meta = 0;
  int64_t flops = 0, rw_bytes = 0;
  if (col) {
    col_codes = a.spec_codes[sb + lane];
    col_tensor = a.spec_tensor[sb + lane];
  }
  if (row) {
    row_codes = a.spec_codes[tb + lane];
    row_tensor = a.spec_tensor[tb + lane];
    flops = a.flops[st + lane];
    rw_bytes = a.rw_bytes[st + lane];
    const int num_args = a.num_args[st + lane];
    holds = num_args >= 1 && num_args <= 0x7FFF;
    meta = (int32_t)((uint32_t)(uint8_t)a.dtype[st + lane] | (a.zero_cost[st + lane] != 0 ? 1u << 8 : 0u) | ((uint32_t)num_args << 16));
  }
  if (__ballot(!holds) != 0) {
    if (lane == 0) *a.refused = 1;
    return;
  }
  const bool mixed = __ballot((col && (col_tensor < 0 || col_tensor != tl.tensor)) || (row && row_tensor < 0)) != 0;
  apc_packed_tile &pk = a.packed[id];
  pk.col_codes[lane] = col_codes;
  pk.col_tensor[lane] = col_tensor;
  pk.row_codes[lane] = row_codes;
  pk.row_tensor[lane] = row_tensor;
  pk.row_flops[lane] = flops;
  pk.row_rw_bytes[lane] = rw_bytes;
  pk.row_meta[lane] = meta;
  if (lane < APC_MAX_RANK) {
    const int64_t at = (int64_t)tl.tensor * APC_MAX_RANK + lane;
    pk.tensor_shape[lane] = tl.tensor >= 0 ? a.t.shape[at] : 0;
    pk.tensor_stride[lane] = tl.tensor >= 0 ? a.t.stride[at] : 0;
  }
  if (lane < APC_PACKED_MAX_DUPS) {
    pk.dup_entry_begin[lane] = lane < n_dups ? a.dup_entry_begin[tl.dup_begin + lane] + first : 0;
    pk.dup_row_begin[lane] = lane < n_dups ? a.dup_row_begin[tl.dup_begin + lane] + rb : 0;
  }
  if (lane == 0) {
    pk.rows = rows;
    pk.cols = cols;
    pk.flags = tl.flags | (mixed ? APC_PACKED_MIXED : 0);
    pk.dup_count = n_dups;
    pk.tensor = tl.tensor;
    pk.tensor_rank = tl.tensor >= 0 ? a.t.rank[tl.tensor] : 0;
    pk.tensor_itemsize = tl.tensor >= 0 ? a.t.itemsize[tl.tensor] : 0;
    pk.edge = tl.edge;
    pk.entry_begin = tl.entry_begin + first;
    pk.row_begin = a.edge_row_begin[tl.edge] + rb;
    pk.pt_begin = tl.pt_begin < 0 ? -1 : tl.pt_begin + first;
    pk.reserved = 0;
  }
}

// ------------------------------------------------------------------------------------------
// The ILP objective, summed on the device.  Entries of linked nodes share an ILP variable
// (optimize_sharding.py:211-231) and the objective coefficient of a variable is the sum of the
// costs of its entries, added one by one in entry order starting from 0
// (optimize_sharding.py:650-655: opt_target[va] += cost over ds.values()); a cost that is not
// finite counts as inf_replacement and forces the variable to 0 (:522-536).  Variables are
// numbered group by group: a group is a set of edges with matrices of the same shape whose
// entries share variables position by position (one edge when nothing is linked); variable
// group_var_begin[g] + k sums entry k of every member edge, members in ascending entry order.
// One workgroup per group (gridDim.y workgroups share a group, each taking every gridDim.y-th
// run of kBlock variables): which group a variable belongs to is never searched for, what a
// group needs (its first variable, its size, its member list) is the same for every lane and is
// fetched once, and neighbouring lanes read neighbouring entries of each member.  The member
// list goes through LDS, so the loads a thread has in flight are costs and nothing else:
// kObjectiveMembersAhead members of one variable, or kObjectiveAhead variables of a group with a
// single member; the additions of a variable stay in member order.
// ------------------------------------------------------------------------------------------
constexpr int kObjectiveAhead = 8;          // variables of a single-member group a thread has in flight
constexpr int kObjectiveMembersAhead = 8;   // members of a variable a thread has in flight

__global__ __launch_bounds__(kBlock) void cost_objective_kernel(const int64_t *__restrict__ group_var_begin,
                                                                const int64_t *__restrict__ group_member_begin,
                                                                const int64_t *__restrict__ member_entry_begin,
                                                                const double *__restrict__ cost, double inf_replacement,
                                                                double *__restrict__ objective,
                                                                uint8_t *__restrict__ forced_zero) {
  __shared__ int64_t s_first_entry[kBlock];
  const int tid = threadIdx.x;
  const int64_t g = blockIdx.x;
  const int64_t var0 = uniform_load(group_var_begin + g), size = uniform_load(group_var_begin + g + 1) - var0;
  const int64_t member0 = uniform_load(group_member_begin + g), n_members = uniform_load(group_member_begin + g + 1) - member0;
  const int64_t begin = (int64_t)blockIdx.y * kBlock, stride = (int64_t)gridDim.y * kBlock;
  if (begin >= size) return;
  const double inf = __builtin_inf();
  auto put = [&](int64_t k, double sum, bool forced) {
    objective[var0 + k] = sum;
    forced_zero[var0 + k] = forced ? 1 : 0;
  };
  if (n_members == 1) {  // nothing is linked: one entry per variable, kObjectiveAhead variables of a thread in flight
    const int64_t first = uniform_load(member_entry_begin + member0);
    for (int64_t base = begin; base < size; base += kObjectiveAhead * stride) {
      double c[kObjectiveAhead];
#pragma unroll
      for (int i = 0; i < kObjectiveAhead; ++i) {
        const int64_t k = base + i * stride + tid;
        c[i] = k < size ? cost[first + k] : 0.0;
      }
#pragma unroll
      for (int i = 0; i < kObjectiveAhead; ++i) {
        const int64_t k = base + i * stride + tid;
        if (k >= size) continue;
        const bool bad = !(__builtin_fabs(c[i]) < inf);  // inf or nan: math.isfinite is false
        put(k, 0.0 + (bad ? inf_replacement : c[i]), bad);
      }
    }
    return;
  }
  for (int64_t base = begin; base < size; base += stride) {  // (the same trips for every thread of the workgroup)
    const int64_t k = base + tid;
    const bool active = k < size;
    double sum = 0.0;
    bool forced = false;
    for (int64_t chunk = 0; chunk < n_members; chunk += kBlock) {
      const int in_chunk = (int)(n_members - chunk < kBlock ? n_members - chunk : kBlock);
      if (n_members > kBlock || base == begin) {  // (a list of at most kBlock members is staged once)
        __syncthreads();
        if (tid < in_chunk) s_first_entry[tid] = member_entry_begin[member0 + chunk + tid];
        __syncthreads();
      }
      for (int at = 0; at < in_chunk; at += kObjectiveMembersAhead) {
        double c[kObjectiveMembersAhead];
#pragma unroll
        for (int i = 0; i < kObjectiveMembersAhead; ++i) c[i] = active && at + i < in_chunk ? cost[s_first_entry[at + i] + k] : 0.0;
#pragma unroll
        for (int i = 0; i < kObjectiveMembersAhead; ++i) {
          if (at + i < in_chunk) {
            const bool bad = !(__builtin_fabs(c[i]) < inf);
            forced |= bad;
            sum += bad ? inf_replacement : c[i];
          }
        }
      }
    }
    if (active) put(k, sum, forced);
  }
}

// ------------------------------------------------------------------------------------------
// a14 put to work: min-sum diffusion over the planning program's labelling form.  A class
// (linked nodes) has a unary cost vector; an edge between two classes has a cost matrix
// (rows = labels of class edge_i, columns = labels of class edge_j, +inf = forbidden pair).
// A node update takes, for every incident matrix, the minima of the rows (or columns) the
// class labels out of the matrix and into the class, then hands their sum back to the
// incident matrices in equal shares.  Every update leaves the cost of every labelling unchanged
// and never lowers  sum_classes min unary + sum_edges min matrix,  a lower bound of the
// program's optimum; min-marginals read off the reparametrised costs prune the program.
// One workgroup per class of one colour (classes of a colour share no edge, so they update
// together); the sweep is the sequence of colours.  Arithmetic in a fixed order (the sum over
// incident edges in incidence order, one division, one subtraction and one addition per
// matrix element): the same bits as the CPU restatement.
// ------------------------------------------------------------------------------------------
constexpr int kDiffusionMaxLabels = 2048;

struct DiffusionArgs {
  const int32_t *nodes;  // the classes of this launch
  const int64_t *label_begin, *inc_begin;
  const int32_t *inc_edge;
  const uint8_t *inc_side;
  const int64_t *edge_begin;
  const int32_t *edge_i, *edge_j;
  double *theta, *unary;
};

__device__ __forceinline__ double wave_min(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const double o = __shfl_xor(v, off, 64);
    v = o < v ? o : v;
  }
  return v;
}

// The update of one class against the matrices where they lie: one pass over every incident
// matrix for the minima, one for the shares, the matrices taken one after the other.  The path
// of a class whose matrices do not fit the staging arrays of the kernel below.
__device__ void diffusion_update_in_memory(const DiffusionArgs &a, double *s_tot, int64_t l0, int n_labels, int64_t t0,
                                           int64_t t1) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  constexpr int kWaves = kBlock / 64;
  const double inf = __builtin_inf();
  for (int x = tid; x < n_labels; x += kBlock) s_tot[x] = a.unary[l0 + x];
  __syncthreads();
  // pull: the minimum of every row / column of the class out of each incident matrix
  for (int64_t t = t0; t < t1; ++t) {
    const int k = a.inc_edge[t];
    double *m = a.theta + a.edge_begin[k];
    const int ej = a.edge_j[k];
    const int nj = (int)(a.label_begin[ej + 1] - a.label_begin[ej]);
    if (a.inc_side[t] == 0) {  // the class labels the rows: one wavefront per row
      for (int x = wave; x < n_labels; x += kWaves) {
        double *row = m + (int64_t)x * nj;
        double d = inf;
        for (int y = lane; y < nj; y += 64) {
          const double v = row[y];
          d = v < d ? v : d;
        }
        d = wave_min(d);
        if (d < inf)
          for (int y = lane; y < nj; y += 64) row[y] -= d;
        if (lane == 0) s_tot[x] += d;
      }
    } else {  // the class labels the columns: one thread per column
      const int ei = a.edge_i[k];
      const int ni = (int)(a.label_begin[ei + 1] - a.label_begin[ei]);
      for (int y = tid; y < n_labels; y += kBlock) {
        double d = inf;
        for (int x = 0; x < ni; ++x) {
          const double v = m[(int64_t)x * n_labels + y];
          d = v < d ? v : d;
        }
        if (d < inf)
          for (int x = 0; x < ni; ++x) m[(int64_t)x * n_labels + y] -= d;
        s_tot[y] += d;
      }
    }
    __syncthreads();
  }
  // share: an equal part of the total for every incident matrix; a label without a finite
  // pair on some edge can never be taken: +inf everywhere
  const double degree = (double)(t1 - t0);
  for (int x = tid; x < n_labels; x += kBlock) {
    const double tot = s_tot[x];
    const bool finite = tot < inf;
    s_tot[x] = finite ? tot / degree : inf;
    a.unary[l0 + x] = finite ? 0.0 : inf;
  }
  __syncthreads();
  for (int64_t t = t0; t < t1; ++t) {
    const int k = a.inc_edge[t];
    double *m = a.theta + a.edge_begin[k];
    if (a.inc_side[t] == 0) {
      const int ej = a.edge_j[k];
      const int nj = (int)(a.label_begin[ej + 1] - a.label_begin[ej]);
      for (int x = wave; x < n_labels; x += kWaves) {
        double *row = m + (int64_t)x * nj;
        const double share = s_tot[x];
        for (int y = lane; y < nj; y += 64) row[y] = share < inf ? row[y] + share : inf;
      }
    } else {
      const int ei = a.edge_i[k];
      const int ni = (int)(a.label_begin[ei + 1] - a.label_begin[ei]);
      for (int y = tid; y < n_labels; y += kBlock) {
        const double share = s_tot[y];
        for (int x = 0; x < ni; ++x) {
          double *p = m + (int64_t)x * n_labels + y;
          *p = share < inf ? *p + share : inf;
        }
      }
    }
  }
}

// One workgroup per class.  A planning program's classes are small (tens of labels, a handful
// of incident matrices of a few hundred elements), so an update is a chain of dependent memory
// round trips and nothing else; the kernel keeps that chain as short as the data allows: the
// incidence list in one round, every incident matrix into LDS in one round of independent
// loads (the elements of all matrices numbered through, a thread finds the matrix of an
// element by bisecting the staged offsets), minima, totals and shares out of LDS, and every
// element stored once.  Element by element the arithmetic is that of the path above, in the
// same order: (v - d) where the row has a finite minimum, then + share or +inf.
// (48 KB of LDS in all, so that a compute unit holds three classes: the largest class of the planning programs
// measured has 3 856 elements and 256 pairs)
constexpr int kDiffusionStagedElements = 4096;  // doubles of LDS for the incident matrices of a class
constexpr int kDiffusionStagedDegree = 64;      // incident matrices of a class
constexpr int kDiffusionStagedPairs = 1024;     // (incident matrix, label) pairs of a class
static_assert(kDiffusionStagedElements >= kDiffusionMaxLabels, "the update in memory keeps its totals where the matrices are staged");

__global__ __launch_bounds__(kBlock) void diffusion_node_update_kernel(DiffusionArgs a) {
  __shared__ double s_m[kDiffusionStagedElements];
  __shared__ double s_d[kDiffusionStagedPairs];
  __shared__ double s_share[kDiffusionStagedPairs];  // (a staged class has at most kDiffusionStagedPairs labels)
  double *s_tot = s_m;                               // the update in memory stages no matrix: its totals lie there
  __shared__ int64_t s_base[kDiffusionStagedDegree];
  __shared__ int s_off[kDiffusionStagedDegree + 1];
  __shared__ int s_other[kDiffusionStagedDegree];
  __shared__ int s_side[kDiffusionStagedDegree];
  const int c = a.nodes[blockIdx.x];
  const int64_t l0 = a.label_begin[c];
  const int n_labels = (int)(a.label_begin[c + 1] - l0);
  const int64_t t0 = a.inc_begin[c], t1 = a.inc_begin[c + 1];
  if (t1 == t0) return;
  if (n_labels > kDiffusionMaxLabels || n_labels < 0) return;  // (the host entry point refuses such a class)
  const int tid = threadIdx.x;
  const int64_t degree64 = t1 - t0;
  if (degree64 > kDiffusionStagedDegree || degree64 * n_labels > kDiffusionStagedPairs) {
    diffusion_update_in_memory(a, s_tot, l0, n_labels, t0, t1);
    return;
  }
  const int degree = (int)degree64;
  const double inf = __builtin_inf();
  // the incidence list: edge, side, where its matrix starts and how many labels the class at
  // its other end has; the unary vector rides along in the same round
  double unary = 0.0;
  if (tid < n_labels) unary = a.unary[l0 + tid];  // (n_labels <= kStagedPairs / degree; labels beyond kBlock below)
  int size = 0;
  if (tid < degree) {
    const int k = a.inc_edge[t0 + tid];
    const int side = a.inc_side[t0 + tid];
    const int other_class = side == 0 ? a.edge_j[k] : a.edge_i[k];
    const int other = (int)(a.label_begin[other_class + 1] - a.label_begin[other_class]);
    s_base[tid] = a.edge_begin[k];
    s_other[tid] = other;
    s_side[tid] = side;
    size = other * n_labels;
  }
  if (tid < 64) {  // degree <= 64: the offsets of the matrices in LDS, a scan within the first wavefront
    int incl = size;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int o = __shfl_up(incl, off, 64);
      if (tid >= off) incl += o;
    }
    if (tid < degree) s_off[tid + 1] = incl;
    if (tid == 0) s_off[0] = 0;
  }
  __syncthreads();
  const int total = s_off[degree];
  if (total > kDiffusionStagedElements || total < 0) {  // uniform: every thread reads the same word
    diffusion_update_in_memory(a, s_tot, l0, n_labels, t0, t1);
    return;
  }
  auto matrix_of = [&](int g) {  // the incident matrix that holds staged element g: the last t with s_off[t] <= g
    int lo = 0, hi = degree - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (s_off[mid] <= g) lo = mid; else hi = mid - 1;
    }
    return lo;
  };
  constexpr int kAhead = 4;  // loads a thread issues before it waits for the first
  for (int base = 0; base < total; base += kAhead * kBlock) {
    double v[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int g = base + u * kBlock + tid;
      v[u] = 0.0;
      if (g < total) {
        const int t = matrix_of(g);
        v[u] = a.theta[s_base[t] + (g - s_off[t])];
      }
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int g = base + u * kBlock + tid;
      if (g < total) s_m[g] = v[u];
    }
  }
  __syncthreads();
  // pull: one thread per (incident matrix, label of the class)
  const int pairs = degree * n_labels;
  for (int q = tid; q < pairs; q += kBlock) {
    const int t = q / n_labels, x = q - t * n_labels;
    const int other = s_other[t];
    // rows of the class are contiguous runs of `other` elements; its columns are strided by n_labels
    const int first = s_off[t] + (s_side[t] == 0 ? x * other : x);
    const int step = s_side[t] == 0 ? 1 : n_labels;
    double d = inf;
    for (int y = 0; y < other; ++y) {
      const double v = s_m[first + y * step];
      d = v < d ? v : d;
    }
    if (d < inf)
      for (int y = 0; y < other; ++y) s_m[first + y * step] -= d;
    s_d[q] = d;
  }
  __syncthreads();
  // totals in incidence order, one division: the share every incident matrix gets back
  for (int x = tid; x < n_labels; x += kBlock) {
    double tot = x == tid && tid < n_labels ? unary : a.unary[l0 + x];
    for (int t = 0; t < degree; ++t) tot += s_d[t * n_labels + x];
    const bool finite = tot < inf;
    s_share[x] = finite ? tot / (double)degree : inf;
    a.unary[l0 + x] = finite ? 0.0 : inf;
  }
  __syncthreads();
  for (int g = tid; g < total; g += kBlock) {
    const int t = matrix_of(g);
    const int e = g - s_off[t];
    const int x = s_side[t] == 0 ? e / s_other[t] : e % n_labels;
    const double share = s_share[x];
    a.theta[s_base[t] + e] = share < inf ? s_m[g] + share : inf;
  }
}

// ------------------------------------------------------------------------------------------
// The same sweeps with the matrices resident on the chip.  A sweep of a planning program touches a
// few hundred matrices of a few hundred elements; as one launch per colour it is a chain of 480
// launches for 160 sweeps, each of which waits for the one before, reads its matrices and writes them
// back: 7.6 us a launch on a two-dimensional mesh (34 000 elements), 134 us on a three-dimensional one
// (977 000 elements), where a class's matrices no longer fit the staging arrays.  Here every workgroup keeps a run of
// consecutive matrices in its LDS over all sweeps, and what moves between workgroups is the minima of
// classes whose matrices lie in several of them.
//   A step (one colour of one sweep) of a workgroup: the minima of its rows (columns) of that colour, a
//   row by 1 to 16 lanes -> barrier -> the same lanes take their class's total, in incidence order, and
//   update the elements they still hold in registers -> barrier, in front of which the next step's rows
//   are fetched.  Element by element the arithmetic and its order are those of the launches above.
//   Exchange: a slot per (incidence, label) in memory holds a minimum as two 64-bit words, each half of
//   the value under the sweep's number, written and read by relaxed device-scope atomics: a reader
//   that sees the number it waits for in both words has the value, so no flag, fence or cache
//   maintenance is needed.  Two sets of slots in turn: a workgroup is at most one update of a class
//   ahead of the others that hold matrices of it, because it needs their minima for its next one.
//   Progress: all workgroups have to be resident (one per compute unit, at most
//   APC_SWEEP_MAX_WORKGROUPS of 256; a second such kernel may hold the rest).  A wait that lasts longer
//   than `wait_ticks` ends the kernel: the status word is set, every workgroup leaves at its own next
//   wait, and the caller, whose inputs are untouched, takes the launches above instead.
// Bound by latency: 0.8 us a step of a workgroup alone (LDS round trips and two barriers in a chain; one
// wavefront per SIMD, so every instruction is on it), 1.4 - 1.7 us with an exchange.  160 sweeps, against one
// launch per colour: 36 509 elements, three colours, 84 workgroups 3.65 -> 0.85 ms; 1 016 497 elements, 212
// workgroups of 1024 threads 64 -> 1.39 ms.
// ------------------------------------------------------------------------------------------
// The plan of one workgroup, int32 words, 16-byte aligned:
//   [0] first element of theta, [1] elements, [2] rows, [3] incidences, [4] steps (the colours it has rows of)
//   rows         8 words each, colour by colour: first element | count << 16, step | label within its class << 16,
//                slot or -1, first incidence | degree << 16; then where the minima of its class's first four
//                incidences at this label are: a row here, or 0x40000000 | a slot, or (none) the row behind the last,
//                which holds 0.0
//   per row      its label's position in `unary`; | 0x80000000 where this row stores it
//   incidences   of classes with more than four: as above, of label 0
//   steps        the first row of each; behind the last: the number of rows
// A row and its class's total belong to G consecutive lanes, the same ones in every sweep.
constexpr int kResidentInverses = 64;  // reciprocals of the degrees below this many are kept

struct ResidentArgs {
  const int32_t *plan;
  const int64_t *plan_begin;
  const double *theta, *unary;
  double *theta_out, *unary_out;
  uint64_t *slots;
  int64_t n_slots;
  uint64_t wait_ticks;
  int32_t *status;
  int n_sweeps;
};

__global__ __launch_bounds__(kBlock) void resident_sweeps_begin_kernel(uint64_t *slots, int64_t n_words, const double *unary,
                                                                       double *unary_out, int64_t n_labels, int32_t *status) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n_words) slots[i] = 0;
  if (i < n_labels) unary_out[i] = unary[i];
  if (i == 0) *status = 0;
}

__device__ __forceinline__ void publish_minimum(uint64_t *slot, double d, uint32_t number) {
  const uint64_t tag = (uint64_t)number << 32;
  __hip_atomic_store(slot, tag | (uint32_t)__double2loint(d), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(slot + 1, tag | (uint32_t)__double2hiint(d), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The smaller of two numbers in one instruction (a comparison and two selects otherwise).
__device__ __forceinline__ double min_of(double a, double b) {
  double m;
  __asm__("v_min_f64 %0, %1, %2" : "=v"(m) : "v"(a), "v"(b));
  return m;
}

// The minimum over `lanes` (uniform; 1, 2, 4, 8 or 16) consecutive lanes, in every lane: within a row of 16,
// vector ALU only.
template <int CTRL>
__device__ __forceinline__ double min_with_dpp(double d) {
  const int lo = __double2loint(d), hi = __double2hiint(d);
  return min_of(d, __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, CTRL, 0xF, 0xF, false),
                                    __builtin_amdgcn_update_dpp(lo, lo, CTRL, 0xF, 0xF, false)));
}
__device__ __forceinline__ double min_over_lanes(double d, int lanes) {
  if (lanes >= 2) d = min_with_dpp<0xB1>(d);    // quad_perm [1, 0, 3, 2]
  if (lanes >= 4) d = min_with_dpp<0x4E>(d);    // quad_perm [2, 3, 0, 1]
  if (lanes >= 8) d = min_with_dpp<0x141>(d);   // row_half_mirror
  if (lanes >= 16) d = min_with_dpp<0x140>(d);  // row_mirror
  return d;
}

struct ResidentLds {
  int4 *row;
  double *m, *d, *un, *inv;
  int *inc, *steps, *abort;
};

// A lane's row of a step; nothing a step writes, so it is fetched while the step before runs.
struct ResidentRow {
  int4 r, ref;
  int q;      // -1: no row
  int lanes;  // lanes per row (uniform): as many as keep the workgroup busy, at most 16
};

template <int T>
__device__ __forceinline__ ResidentRow resident_row(const ResidentLds &l, int begin, int end, int tid) {
  const int rb = uniform_i32(begin), re = uniform_i32(end), rows = re - rb;
  const int shift = rows * 16 <= T ? 4 : rows * 8 <= T ? 3 : rows * 4 <= T ? 2 : rows * 2 <= T ? 1 : 0;
  ResidentRow x;
  x.lanes = 1 << shift;
  x.q = rb + (tid >> shift);
  const int q = min(x.q, re - 1);  // (a step has rows)
  x.r = l.row[2 * q];
  x.ref = l.row[2 * q + 1];
  if (x.q >= re) x.q = -1;
  return x;
}

// The minimum of an incidence at a label: here, or (`slot`) waited for.
struct PendingMinima {
  double e[4];
  int ref[4];
};

// Waits for the minima that other workgroups publish; false when the wait expired.
__device__ __forceinline__ bool await_minima(const uint64_t *slots, uint32_t number, uint64_t wait_ticks, PendingMinima &p) {
  int pending = 0;
#pragma unroll
  for (int u = 0; u < 4; ++u) pending |= (p.ref[u] & 0x40000000) ? 1 << u : 0;
  const uint64_t began = wall_clock64();
  while (pending) {
    uint64_t lo[4], hi[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (pending & (1 << u)) {
        const uint64_t *slot = slots + 2 * (int64_t)(p.ref[u] & 0x3FFFFFFF);
        lo[u] = __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        hi[u] = __hip_atomic_load(slot + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if ((pending & (1 << u)) && (uint32_t)(lo[u] >> 32) == number && (uint32_t)(hi[u] >> 32) == number) {
        p.e[u] = __hiloint2double((int)(uint32_t)hi[u], (int)(uint32_t)lo[u]);
        pending &= ~(1 << u);
      }
    if (pending && wall_clock64() - began > wait_ticks) return false;
  }
  return true;
}

// One step of a workgroup, `x` its rows; on return those of the next step.  False: a wait expired in the
// workgroup (every thread returns the same).
template <int T>
__device__ __forceinline__ bool resident_step(const ResidentLds &l, const ResidentArgs &a, uint64_t *slots, uint32_t number, int n_rows,
                                              ResidentRow &x, int next_step, int tid) {
  // Elements of a row that a lane holds between its minimum and its update.  A lane past the row's end
  // holds its last element once more: the same value, stored again.
  constexpr int kHeld = 4;
  const double inf = __builtin_inf();
  const int lanes = uniform_i32(x.lanes), sub = tid & (lanes - 1);
  const int last = (int)((uint32_t)x.r.x >> 16) - 1, stride = x.r.y & 0xFFFF, label = (int)((uint32_t)x.r.y >> 16);
  const int degree = (int)((uint32_t)x.r.w >> 16);
  const bool live = x.q >= 0;
  double *const m = l.m + (x.r.x & 0xFFFF);
  int at[kHeld];
  double v[kHeld];
#pragma unroll
  for (int u = 0; u < kHeld; ++u) {
    at[u] = __mul24(min(sub + u * lanes, last), stride);
    v[u] = m[at[u]];
  }
  const int expired_before = *l.abort;  // (written between the two barriers of a step, read outside of them)
  const double unary = l.un[max(x.q, 0)], inv = l.inv[min(degree, kResidentInverses - 1)];
  const int next_begin = l.steps[next_step], next_end = l.steps[next_step + 1];
  double d = min_of(min_of(v[0], v[1]), min_of(v[2], v[3]));
  for (int y = sub + kHeld * lanes; y <= last; y += lanes) d = min_of(m[__mul24(y, stride)], d);
  if (uniform_i32(expired_before)) return false;
  d = min_over_lanes(d, lanes);
  if (sub == 0 && live) {
    l.d[x.q] = d;
    if (x.r.z >= 0) publish_minimum(slots + 2 * (int64_t)x.r.z, d, number);
  }
  const ResidentRow next = resident_row<T>(l, next_begin, next_end, tid);
  __syncthreads();
  if (live) {
    PendingMinima p;
    p.ref[0] = x.ref.x;
    p.ref[1] = x.ref.y;
    p.ref[2] = x.ref.z;
    p.ref[3] = x.ref.w;
    bool expired = false;
    auto add = [&](double tot) {
      int remote = 0;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        p.e[u] = l.d[(p.ref[u] & 0x40000000) ? n_rows : p.ref[u]];
        remote |= p.ref[u];
      }
      if (remote & 0x40000000) expired = !await_minima(slots, number, a.wait_ticks, p);
#pragma unroll
      for (int u = 0; u < 4; ++u) tot += p.e[u];  // (none: + 0.0)
      return tot;
    };
    double tot = add(unary);
    for (int t = 4; t < degree && !expired; t += 4) {
#pragma unroll
      for (int u = 0; u < 4; ++u) p.ref[u] = t + u < degree ? l.inc[(x.r.w & 0xFFFF) + t + u] + label : n_rows;
      tot = add(tot);
    }
    if (expired) *l.abort = 1;
    const bool finite = tot < inf;  // (then every minimum of the class is finite)
    // (the quotient through the reciprocal is the division's: div_by)
    double share = div_by(tot, (double)degree, inv);
    if (degree >= kResidentInverses) share = tot / (double)degree;
    if (sub == 0) l.un[x.q] = finite ? 0.0 : inf;
#pragma unroll
    for (int u = 0; u < kHeld; ++u) m[at[u]] = finite ? (v[u] - d) + share : inf;  // (a label that can never be taken: +inf)
    for (int y = sub + kHeld * lanes; y <= last; y += lanes) {
      double *const e = m + __mul24(y, stride);
      *e = finite ? (*e - d) + share : inf;
    }
  }
  x = next;
  __syncthreads();
  return true;
}

// ------------------------------------------------------------------------------------------
// The same sweeps by teams: a matrix belongs to a team of 1, 2, 4, 8 or 16 wavefronts of a workgroup, which updates its rows
// and its columns in turn and waits for nothing but the classes at its two ends.  (Above, a workgroup holds a run of
// matrices and steps through the colours behind barriers: every step of it is as long as its slowest exchange.)
//   A minimum lies in a place of two 64-bit words, each half of the value under the sweep's number: in LDS for the
//   workgroup's teams, and in memory too where a matrix of the class lies in another workgroup.  A reader that
//   sees the number in both words has the value: no barrier, no fence.  Two sets of places in turn, as above.
//   What a lane needs of the plan stays in its registers over all sweeps.  All labels of a class have an incidence's minima at the
//   same kind of place, so how many places are read, and which of them in memory, is uniform: scalar branches.
//   The wavefronts of a team share its matrix: each counts its finished updates, and waits for the others' counts before it
//   reads.  (The LDS operations of one wavefront complete in order.)
//   Classes with more than four matrices: the next four places are on their way while the first four are waited for.
// Lanes beyond a wavefront's rows repeat its last row: the same values, to the same addresses.
// Bound by latency: an update is three round trips through LDS and some 200 instructions in a chain, 0.4 - 0.5 us, and an exchange
// through memory 0.4 - 0.65 us more; a sweep is as long as the longest cycle of classes, three updates and more around a class
// with many.  us a sweep, before (runs) and now: 358 matrices of at most 24 labels 5.5 -> 3.5, of at most 124 8.5 -> 6.7, 794 of 40
// in five colours 14.7 -> 9.4, 1 098 of 12 6.0 -> 3.9, 1 428 of 64 12.0 -> 7.8.  Runs stay where one workgroup holds them all, which
// exchanges nothing (27 matrices of at most 3 labels 2.7 against 3.3, 38 of 6 2.3 against 2.6), and where the matrices are too many, or small and
// of two colours (apc_sweep_plan_host).  Chains without hubs, which are two steps a sweep, gain least: 358 of at most 24 labels 3.2 / 3.2, 794 of 40
// 4.5 / 4.2, 1 428 of 64 13.8 / 6.8.
// Tried: any wavefront waiting per lane instead of uniformly, with the plan's rows read from LDS for every step (16 % slower than the
// barriers); waiting wavefronts at the priority of the others (13 % slower); sleeping between two looks (no difference).
// ------------------------------------------------------------------------------------------
// The plan of a workgroup: as above, with [3] incidences of classes with more than four, [4] 0, [5] APC_SWEEP_TEAMS; the rows
// team by team, the side of the lower colour first; behind the incidences, instead of steps,
//   wavefronts   APC_SWEEP_MAX_WAVES x 4 words: first row, rows of the first side | rows of the second << 16,
//                team | wavefront of the team << 8 | wavefronts of the team << 16 (0: idle), 0
struct TeamLds {
  double *m;
  uint64_t *places;  // [row][set][2]
  uint32_t *finished;
  int *inc, *abort;
  uint32_t looks;  // the clock is read at every (looks + 1)th: it takes longer than the LDS
  mutable int sweeps;  // of this wavefront: no more where it has given up
};

__device__ __forceinline__ void keep_order() { __asm__ volatile("" ::: "memory"); }

// One side of a team's matrix, as a lane sees it.
struct TeamSide {
  uint32_t at[4], last;  // LDS addresses of the lane's first elements, and of the row's last one
  lds_address own;       // its row's place
  uint32_t slot;         // its place in memory, bytes
  uint32_t ref[4];       // the places of its class's first four incidences: LDS addresses, or bytes in memory
  double unary;
  bool finite;
  int label;
  // uniform
  uint32_t step;  // bytes from an element of the lane to its next
  int rounds;     // of four elements, beyond the first
  int lanes, degree, inc;
  int far;     // which of the first four incidences lie in memory
  int shared;  // the own row has a place there
  int idle;
  double inverse;
};

// (a uniform number that the compiler has to test where it is used: hoisted out of the sweeps, the outcomes of all tests
// took more scalar registers than there are, and came back through vector registers)
__device__ __forceinline__ int here(int v) {
  v = uniform_i32(v);
  __asm__ volatile("" : "+s"(v));
  return v;
}
__device__ __forceinline__ uint64_t half_under(uint32_t number, int half) { return (uint64_t)number << 32 | (uint32_t)half; }

// A wait that lasts too long is given up: the workgroup's results are then not used.  The wavefront ends its sweep with whatever it finds and
// leaves; those that wait for it find the flag at their next look at the clock and do the same, and other workgroups, whose waits began
// when this one's did, give up themselves.  (1 000 000 sweeps given up at their first wait, ms when wavefronts went on to the last sweep / now: 149
// matrices in 20 workgroups 2 850 / 0.02, a class with 70 matrices 16 300 / 0.05; a sweep that nothing is given up in takes as long as before.)
struct Patience {
  uint64_t began;
  uint32_t tries;
};
__device__ __forceinline__ bool give_up(Patience &w, const TeamLds &l, uint64_t wait_ticks) {
  if ((++w.tries & l.looks) != 0) return false;
  const uint64_t now = (uint64_t)wall_clock64();
  if (w.tries == l.looks + 1) w.began = now;
  if (uniform_i32(__hip_atomic_load(l.abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) == 0 && now - w.began < wait_ticks) return false;
  __hip_atomic_store(l.abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  l.sweeps = 0;
  return true;
}

struct Halves {
  uint64_t lo, hi;
  __device__ __forceinline__ bool of(uint32_t number) const { return (uint32_t)(lo >> 32) == number && (uint32_t)(hi >> 32) == number; }
  __device__ __forceinline__ double value() const { return __hiloint2double((int)(uint32_t)hi, (int)(uint32_t)lo); }
};
__device__ __forceinline__ Halves near_place(uint32_t ref) {
  const APC_LDS uint64_t *p = (const APC_LDS uint64_t *)(uintptr_t)ref;
  return Halves{__hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP),
                __hip_atomic_load(p + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)};
}
__device__ __forceinline__ Halves far_place(const uint64_t *slots, uint32_t ref) {
  const uint64_t *p = reinterpret_cast<const uint64_t *>(reinterpret_cast<const char *>(slots) + ref);
  return Halves{__hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), __hip_atomic_load(p + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)};
}

// The minima of N incidences that all lie in LDS, added to `tot` in order.  (Where there are fewer, the last places are the own
// row's: read, and not added.)
template <int N>
__device__ __forceinline__ void add_near(const TeamLds &l, uint32_t number, uint64_t wait_ticks, const uint32_t (&ref)[4], int n, double &tot) {
  Halves h[N];
  Patience wait{0, 0};
  for (;;) {
#pragma unroll
    for (int u = 0; u < N; ++u) h[u] = near_place(ref[u]);
    bool there = true;
#pragma unroll
    for (int u = 0; u < N; ++u) there = there & h[u].of(number);
    if (__all(there) || give_up(wait, l, wait_ticks)) break;
  }
#pragma unroll
  for (int u = 0; u < N; ++u)
    if (u < N / 2 || u < here(n)) tot += h[u].value();
}

// Four incidences (or the last n) of a class, those of `far` in memory.
struct Four {
  uint32_t ref[4];
  int n, far;
  Halves f[4];
  __device__ __forceinline__ void fetch_far(const uint64_t *slots) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if ((here(far) >> u) & 1) f[u] = far_place(slots, ref[u]);
  }
  // Their minima, added to `tot` in order; the far ones are on their way.
  __device__ __forceinline__ void add(const TeamLds &l, const uint64_t *slots, uint32_t number, uint64_t wait_ticks, double &tot) {
    Halves h[4];
    if (const int near = here(((1 << n) - 1) & ~far)) {
      Patience wait{0, 0};
      for (;;) {
        bool there = true;
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if ((here(near) >> u) & 1) h[u] = near_place(ref[u]);
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if ((here(near) >> u) & 1) there = there & h[u].of(number);
        if (__all(there) || give_up(wait, l, wait_ticks)) break;
      }
    }
    if (here(far)) {
      Patience wait{0, 0};
      for (;;) {
        bool there = true;
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if ((here(far) >> u) & 1) there = there & f[u].of(number);
        if (__all(there) || give_up(wait, l, wait_ticks)) break;
        fetch_far(slots);
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (u < here(n)) tot += (here(far) >> u) & 1 ? f[u].value() : h[u].value();
  }
};

// The update of one side.
__device__ __forceinline__ void team_update(const TeamLds &l, const ResidentArgs &a, TeamSide &x, uint32_t number, int waves, uint32_t *finished,
                                            uint32_t updates, int lane) {
  const double inf = __builtin_inf();
  if (here(waves) > 1) {
    Patience wait{0, 0};
    while ((int32_t)((uint32_t)uniform_i32((int)__hip_atomic_load(finished, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) - updates * (uint32_t)waves) < 0)
      if (give_up(wait, l, a.wait_ticks)) break;
    keep_order();
  }
  if (!here(x.idle)) {
    double v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = lds_read<double>(x.at[u]);
    double d = min_of(min_of(v[0], v[1]), min_of(v[2], v[3]));
    uint32_t at = x.at[0];
    for (int i = here(x.rounds); i > 0; --i) {
      double w[4];
      at += 4 * x.step;
#pragma unroll
      for (int u = 0; u < 4; ++u) w[u] = lds_read<double>(min(at + u * x.step, x.last));
      d = min_of(d, min_of(min_of(w[0], w[1]), min_of(w[2], w[3])));
    }
    d = min_over_lanes(d, here(x.lanes));
    const uint64_t lo = half_under(number, __double2loint(d)), hi = half_under(number, __double2hiint(d));
    if ((lane & (x.lanes - 1)) == 0) {
      if (here(x.shared)) {
        uint64_t *slot = reinterpret_cast<uint64_t *>(reinterpret_cast<char *>(a.slots) + x.slot);
        __hip_atomic_store(slot, lo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(slot + 1, hi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      APC_LDS uint64_t *p = (APC_LDS uint64_t *)(uintptr_t)x.own;
      __hip_atomic_store(p, lo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      __hip_atomic_store(p + 1, hi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    __builtin_amdgcn_s_setprio(0);  // (who waits steps back)
    double tot = x.unary;
    const int degree = here(x.degree);
    if (degree <= 2 && here(x.far) == 0) {
      add_near<2>(l, number, a.wait_ticks, x.ref, degree, tot);
    } else if (degree <= 4 && here(x.far) == 0) {
      add_near<4>(l, number, a.wait_ticks, x.ref, degree, tot);
    } else {
      Four now{{x.ref[0], x.ref[1], x.ref[2], x.ref[3]}, min(degree, 4), x.far, {}};
      now.fetch_far(a.slots);  // (on their way while the LDS is read)
      for (int t = 4;; t += 4) {
        Four next;
        if (t < degree) {
          int place[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) place[u] = l.inc[x.inc + min(t + u, degree - 1)];
          next.n = min(degree - t, 4);
          next.far = 0;
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const bool is_far = (uniform_i32(place[u]) & 0x40000000) != 0;
            next.far |= is_far && u < next.n ? 1 << u : 0;
            next.ref[u] = ((uint32_t)(place[u] & 0x3FFFFFFF) + x.label) * 32u + (x.own & 16u) + (is_far ? 0u : address_in_lds(l.places));
          }
          next.fetch_far(a.slots);
        }
        now.add(l, a.slots, number, a.wait_ticks, tot);
        if (t >= degree) break;
        now = next;
      }
    }
    __builtin_amdgcn_s_setprio(3);
    const bool finite = tot < inf;  // (then every minimum of the class is finite)
    const double share = div_by(tot, (double)degree, x.inverse);  // (the division's quotient)
    x.unary = 0.0;  // (or +inf, where the row's elements are)
    x.finite = finite;
#pragma unroll
    for (int u = 0; u < 4; ++u) lds_write(x.at[u], finite ? (v[u] - d) + share : inf);  // (a label that can never be taken: +inf)
    at = x.at[0];
    for (int i = here(x.rounds); i > 0; --i) {
      double w[4];
      uint32_t to[4];
      at += 4 * x.step;
#pragma unroll
      for (int u = 0; u < 4; ++u) to[u] = min(at + u * x.step, x.last);
#pragma unroll
      for (int u = 0; u < 4; ++u) w[u] = lds_read<double>(to[u]);
#pragma unroll
      for (int u = 0; u < 4; ++u) lds_write(to[u], finite ? (w[u] - d) + share : inf);
    }
    // the other set of places
#pragma unroll
    for (int u = 0; u < 4; ++u) x.ref[u] ^= 16u;
    x.own ^= 16u;
    x.slot ^= 16u;
  }
  keep_order();
  if (here(waves) > 1 && lane == 0) __hip_atomic_fetch_add(finished, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

__device__ __forceinline__ void team_side(TeamSide &x, const TeamLds &l, const ResidentArgs &a, const int4 *rows, const int32_t *labels, int first, int n, int tid,
                                          int threads) {
  const int shift = n * 16 <= threads ? 4 : n * 8 <= threads ? 3 : n * 4 <= threads ? 2 : n * 2 <= threads ? 1 : 0;
  x.lanes = 1 << shift;
  x.idle = uniform_i32((tid & ~63) >> shift >= n);
  const int q = first + min(tid >> shift, n - 1), sub = tid & (x.lanes - 1);
  const int4 r = rows[2 * q], ref = rows[2 * q + 1];
  const uint32_t places = address_in_lds(l.places);
  const uint32_t m = address_in_lds(l.m) + 8u * (uint32_t)(r.x & 0xFFFF);
  const int count = uniform_i32((int)((uint32_t)r.x >> 16)), stride = uniform_i32(r.y & 0xFFFF) * 8;
  x.last = m + (uint32_t)((count - 1) * stride);
  x.step = (uint32_t)(x.lanes * stride);
#pragma unroll
  for (int u = 0; u < 4; ++u) x.at[u] = min(m + (uint32_t)((sub + u * x.lanes) * stride), x.last);
  x.rounds = (count + 4 * x.lanes - 1) / (4 * x.lanes) - 1;
  x.own = (lds_address)(places + 32u * (uint32_t)q);
  x.shared = uniform_i32(r.z) >= 0;
  x.slot = (uint32_t)max(r.z, 0) * 32u;
  x.label = (int)((uint32_t)r.y >> 16);
  x.inc = uniform_i32(r.w & 0xFFFF);
  x.degree = uniform_i32((int)((uint32_t)r.w >> 16));
  x.far = 0;
  const int refs[4] = {ref.x, ref.y, ref.z, ref.w};
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const bool far = (uniform_i32(refs[u]) & 0x40000000) != 0;
    x.far |= far ? 1 << u : 0;
    x.ref[u] = u >= x.degree ? x.own : (uint32_t)(refs[u] & 0x3FFFFFFF) * 32u + (far ? 0u : places);
  }
  x.inverse = x.degree > 0 ? 1.0 / (double)x.degree : 0.0;
  const int32_t label = labels[q];
  x.unary = a.unary[label & 0x7FFFFFFF];
  x.finite = true;
}

template <int T>
__device__ __forceinline__ void team_sweeps(const ResidentArgs &a, unsigned char *s_bytes) {
  const int tid = threadIdx.x;
  // Workgroups go to the XCDs in turn; those of one XCD take consecutive parts of the plan, which share most classes (a number
  // is there after 0.4 us within an XCD, 0.5 - 0.65 between two).
  const unsigned xcd = blockIdx.x % 8u, share = gridDim.x / 8u, rest = gridDim.x % 8u;
  const int32_t *plan = a.plan + a.plan_begin[xcd * share + min(xcd, rest) + blockIdx.x / 8u];
  const int64_t first = plan[0];
  const int n_el = plan[1], n_rows = plan[2], n_inc = plan[3];
  // the layout of LDS (apc_sweep_plan_host counts the same bytes)
  TeamLds l;
  l.places = reinterpret_cast<uint64_t *>(s_bytes);
  l.m = reinterpret_cast<double *>(l.places + 4 * n_rows);
  l.inc = reinterpret_cast<int *>(l.m + n_el);
  l.finished = reinterpret_cast<uint32_t *>(l.inc + n_inc);
  l.abort = reinterpret_cast<int *>(l.finished + APC_SWEEP_MAX_WAVES);
  l.looks = a.wait_ticks == 0 ? 0 : 15;
  l.sweeps = a.n_sweeps;
  const int4 *rows = reinterpret_cast<const int4 *>(plan + 8);
  const int32_t *labels = reinterpret_cast<const int32_t *>(rows + 2 * n_rows);
  const int32_t *incs = labels + n_rows;
  const int32_t *wave = incs + n_inc + 4 * uniform_i32(tid >> 6);
  const int first_row = uniform_i32(wave[0]), n_first = uniform_i32(wave[1]) & 0xFFFF, n_second = (int)((uint32_t)uniform_i32(wave[1]) >> 16);
  const uint32_t team = (uint32_t)uniform_i32(wave[2]);
  const int waves = (int)(team >> 16), of_team = 64 * (int)((team >> 8) & 0xFF) + (tid & 63);
  TeamSide x, y;
  if (waves > 0) {
    team_side(x, l, a, rows, labels, first_row, n_first, of_team, 64 * waves);
    team_side(y, l, a, rows, labels, first_row + n_first, n_second, of_team, 64 * waves);
  }
  for (int i = tid; i < 4 * n_rows; i += T) l.places[i] = 0;
  for (int i = tid; i < n_el; i += T) l.m[i] = a.theta[first + i];
  for (int i = tid; i < n_inc; i += T) l.inc[i] = incs[i];
  if (tid < APC_SWEEP_MAX_WAVES) l.finished[tid] = 0;
  if (tid == 0) *l.abort = 0;
  __syncthreads();
  if (waves > 0) {
    uint32_t *const finished = l.finished + (team & 0xFF);
    uint32_t updates = 0;
    __builtin_amdgcn_s_setprio(3);
    for (int sweep = 0; sweep < l.sweeps; ++sweep, updates += 2) {
      team_update(l, a, x, (uint32_t)sweep + 1, waves, finished, updates, tid & 63);
      team_update(l, a, y, (uint32_t)sweep + 1, waves, finished, updates + 1, tid & 63);
    }
    __builtin_amdgcn_s_setprio(0);
  }
  __syncthreads();
  if (*l.abort) {
    if (tid == 0) __hip_atomic_store(a.status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return;
  }
  for (int i = tid; i < n_el; i += T) a.theta_out[first + i] = l.m[i];
  if (waves > 0 && a.n_sweeps > 0) {
    const auto store = [&](const TeamSide &s) {
      if (s.idle || ((tid & 63) & (s.lanes - 1)) != 0) return;
      const int32_t label = labels[(s.own - address_in_lds(l.places)) / 32u];
      if (label < 0) a.unary_out[label & 0x7FFFFFFF] = s.finite ? 0.0 : __builtin_inf();
    };
    store(x);
    store(y);
  }
}

template <int T>
__global__ __launch_bounds__(T) void diffusion_resident_kernel(ResidentArgs a) {
  extern __shared__ __align__(32) unsigned char s_bytes[];
  const int tid = threadIdx.x;
  const bool teams = a.plan[a.plan_begin[0] + 5] == APC_SWEEP_TEAMS;
  if (teams ? T == 256 : T == 512) {  // (uniform; no plan of apc_sweep_plan_host)
    if (tid == 0) __hip_atomic_store(a.status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return;
  }
  if constexpr (T != 256) {
    if (teams) {
      team_sweeps<T>(a, s_bytes);
      return;
    }
  }
  const int32_t *plan = a.plan + a.plan_begin[blockIdx.x];
  const int64_t first = plan[0];
  const int n_el = plan[1], n_rows = plan[2], n_inc = plan[3], n_steps = plan[4];
  // the layout of LDS (apc_sweep_plan_host counts the same bytes)
  ResidentLds l;
  l.row = reinterpret_cast<int4 *>(s_bytes);
  l.m = reinterpret_cast<double *>(l.row + 2 * n_rows);
  l.d = l.m + n_el;  // (one more than rows: 0.0)
  l.un = l.d + n_rows + 1;
  l.inv = l.un + n_rows;
  l.inc = reinterpret_cast<int *>(l.inv + kResidentInverses);
  l.steps = l.inc + n_inc;
  l.abort = l.steps + n_steps + 1;
  const int4 *rows = reinterpret_cast<const int4 *>(plan + 8);
  const int32_t *labels = reinterpret_cast<const int32_t *>(rows + 2 * n_rows);
  const int32_t *incs = labels + n_rows;  // (the steps follow)
  for (int i = tid; i < 2 * n_rows; i += T) l.row[i] = rows[i];
  for (int i = tid; i < n_rows; i += T) l.un[i] = a.unary[labels[i] & 0x7FFFFFFF];
  for (int i = tid; i < n_el; i += T) l.m[i] = a.theta[first + i];
  for (int i = tid; i < n_inc + n_steps + 1; i += T) l.inc[i] = incs[i];
  for (int i = tid; i < kResidentInverses; i += T) l.inv[i] = i > 0 ? 1.0 / (double)i : 0.0;
  if (tid == 0) {
    *l.abort = 0;
    l.d[n_rows] = 0.0;
  }
  __syncthreads();
  ResidentRow x = resident_row<T>(l, l.steps[0], l.steps[1], tid);
  for (int sweep = 0; sweep < a.n_sweeps; ++sweep) {
    const uint32_t number = (uint32_t)sweep + 1;
    uint64_t *slots = a.slots + (sweep & 1) * 2 * a.n_slots;
    for (int step = 0; step < n_steps; ++step)
      if (!resident_step<T>(l, a, slots, number, n_rows, x, step + 1 < n_steps ? step + 1 : 0, tid)) {  // (uniform)
        if (tid == 0) __hip_atomic_store(a.status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return;
      }
  }
  if (*l.abort) {  // (set in the very last step, behind whose barrier this is)
    if (tid == 0) __hip_atomic_store(a.status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return;
  }
  for (int i = tid; i < n_el; i += T) a.theta_out[first + i] = l.m[i];
  for (int i = tid; i < n_rows; i += T) {
    const int32_t label = labels[i];
    if (label < 0) a.unary_out[label & 0x7FFFFFFF] = l.un[i];
  }
}

inline unsigned blocks_for(int64_t n, int per_block) { return (unsigned)((n + per_block - 1) / per_block); }

template <int G>
void launch_segmented_min(const double *values, const int64_t *seg_ptr, int64_t n_seg, double *mins, int32_t *args,
                          const SegmentCopies *copies, hipStream_t stream) {
  if (copies)
    hipLaunchKernelGGL((segmented_min_kernel<G, true>), dim3(blocks_for(n_seg, kBlock / G)), dim3(kBlock), 0, stream,
                       values, seg_ptr, n_seg, mins, args, *copies);
  else
    hipLaunchKernelGGL((segmented_min_kernel<G, false>), dim3(blocks_for(n_seg, kBlock / G)), dim3(kBlock), 0, stream,
                       values, seg_ptr, n_seg, mins, args, SegmentCopies{nullptr, nullptr, nullptr});
}

int check_width(int width) {
  if (width < 2 || width > APC_MAX_RANK || (width & 1))
    return fail(-1, "shape_width %d must be even and in [2, %d]", width, APC_MAX_RANK);
  return 0;
}

}  // namespace

int apc_internal::check_params(const apc_params *p) {
  if (!p) return fail(-1, "params is NULL");
  if (p->mesh_ndim < 1 || p->mesh_ndim > APC_MAX_MESH)
    return fail(-1, "mesh_ndim %d outside [1, %d]", p->mesh_ndim, APC_MAX_MESH);
  for (int i = 0; i < p->mesh_ndim; ++i) {
    if (p->mesh_size[i] < 1) return fail(-1, "mesh_size[%d] = %d must be >= 1", i, p->mesh_size[i]);
    // the kernels divide through these reciprocals: they must be the correctly rounded ones
    if (p->inv_mesh[i] != 1.0 / (double)p->mesh_size[i] || p->inv_bw[i] != 1.0 / p->bw[i])
      return fail(-1, "inv_mesh[%d] / inv_bw[%d] are not 1.0 / mesh_size, 1.0 / bw", i, i);
  }
  if (p->inv_hbm_bw != 1.0 / p->hbm_bw || p->inv_rw_eff != 1.0 / p->rw_eff || p->inv_compute_eff != 1.0 / p->compute_eff)
    return fail(-1, "inv_hbm_bw / inv_rw_eff / inv_compute_eff are not 1.0 / hbm_bw, 1.0 / rw_eff, 1.0 / compute_eff");
  for (int i = 0; i < APC_MAX_DTYPES; ++i)
    if (p->inv_gpu_flops[i] != (p->gpu_flops[i] != 0.0 ? 1.0 / p->gpu_flops[i] : 0.0))
      return fail(-1, "inv_gpu_flops[%d] is not 1.0 / gpu_flops[%d] (0 for an unsupported dtype)", i, i);
  return 0;
}

extern "C" {

int apc_version(void) { return APC_ABI_VERSION; }

const char *apc_last_error(void) { return g_err; }

int apc_tensor_tables(int64_t n, const int32_t *rank, const int32_t *itemsize, const int64_t *shape,
                      const int64_t *stride, int64_t *bytes, uint8_t *cont, void *stream) {
  if (n < 0) return fail(-1, "n_tensors < 0");
  if (n == 0) return 0;
  if (!rank || !itemsize || !shape || !stride || !bytes || !cont) return fail(-1, "apc_tensor_tables: NULL array");
  hipLaunchKernelGGL(tensor_tables_kernel, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0, (hipStream_t)stream,
                     TensorTableArgs{n, rank, itemsize, shape, stride, bytes, cont});
  return check_launch("apc_tensor_tables");
}

int apc_spec_tables(const apc_params *params, int64_t n, const uint32_t *codes, const int32_t *tensor,
                    const int32_t *rank, const int32_t *itemsize, const int64_t *shape, const int64_t *stride,
                    int64_t *shards, int64_t *lshape, int64_t *lstride, int32_t shape_width, int64_t *lnumel,
                    int64_t *lbytes, void *stream) {
  if (int rc = check_params(params)) return rc;
  if (int rc = check_width(shape_width)) return rc;
  if (n < 0) return fail(-1, "n_specs < 0");
  if (n == 0) return 0;
  if (!codes || !tensor || !rank || !itemsize || !shape || !stride || !shards || !lshape || !lstride || !lnumel ||
      !lbytes)
    return fail(-1, "apc_spec_tables: NULL array");
  hipLaunchKernelGGL(spec_tables_kernel, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0, (hipStream_t)stream, *params,
                     SpecTableArgs{n, codes, tensor, rank, itemsize, shape, stride, shards, lshape, lstride, lnumel,
                                   lbytes, shape_width});
  return check_launch("apc_spec_tables");
}

int apc_compute_costs(const apc_params *params, int64_t n, const int64_t *flops, const int64_t *rw_bytes,
                      const int8_t *dtype, const uint8_t *zero_cost, const int32_t *num_args, double *compute,
                      double *per_arg, int32_t *error_flag, void *stream) {
  if (int rc = check_params(params)) return rc;
  if (n < 0) return fail(-1, "n_strategies < 0");
  if (n == 0) return 0;
  if (!flops || !rw_bytes || !dtype || !zero_cost || !num_args) return fail(-1, "apc_compute_costs: NULL input");
  hipLaunchKernelGGL(compute_costs_kernel, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0, (hipStream_t)stream,
                     *params,
                     ComputeCostArgs{n, flops, rw_bytes, dtype, zero_cost, num_args, compute, per_arg, error_flag});
  return check_launch("apc_compute_costs");
}

int apc_strategy_inputs(int64_t n_strategies, const int32_t *strat_node, int64_t n_nodes, const int64_t *node_strat_begin,
                        const int32_t *node_kind, const int8_t *node_dtype, const int64_t *node_const_bytes,
                        const int64_t *node_row_begin, const int32_t *byte_rows, const int32_t *node_flop_rows,
                        const int64_t *local_shape, int32_t shape_width, const int64_t *local_bytes, int64_t *flops,
                        int64_t *rw_bytes, int8_t *dtype_code, uint8_t *zero_cost, void *stream) {
  if (n_strategies < 0 || n_nodes < 0) return fail(-1, "apc_strategy_inputs: negative count");
  if (n_strategies == 0) return 0;
  if (int rc = check_width(shape_width)) return rc;
  if (!strat_node || !node_strat_begin || !node_kind || !node_dtype || !node_const_bytes || !node_row_begin ||
      !node_flop_rows || !local_shape || !local_bytes || !flops || !rw_bytes || !dtype_code || !zero_cost)
    return fail(-1, "apc_strategy_inputs: NULL array");
  hipLaunchKernelGGL(strategy_inputs_kernel, dim3(blocks_for(n_strategies, kBlock)), dim3(kBlock), 0, (hipStream_t)stream,
                     StrategyInputArgs{n_strategies, strat_node, node_strat_begin, node_kind, node_dtype, node_const_bytes,
                                       node_row_begin, byte_rows, node_flop_rows, local_shape, shape_width, local_bytes, flops,
                                       rw_bytes, dtype_code, zero_cost});
  return check_launch("apc_strategy_inputs");
}

}  // extern "C"

// Enqueues a table kernel, or (`to.keep`) records the launch for apc_run_kept.
struct LaunchTo {
  void *stream;
  apc_kept_launch *keep;
};

// The launch that apc_keep_next_launch asked this thread to record (taken by the next table launch, whatever becomes of it).
static thread_local apc_kept_launch *g_keep_next = nullptr;
static LaunchTo launch_to(void *stream) {
  const LaunchTo to{stream, g_keep_next};
  g_keep_next = nullptr;
  return to;
}

static int enqueue_kept(const apc_kept_launch &k, const void *block, void *stream) {
  void *args[] = {const_cast<void **>(&k.work), const_cast<int32_t *>(&k.n_tiles), const_cast<int32_t *>(&k.xcd_shift),
                  const_cast<int64_t *>(&k.tile_blocks), const_cast<double **>(&k.cost_out), &block, const_cast<int64_t *>(k.block)};
  (void)hipLaunchKernel(block ? k.kernel : k.kernel_by_value, dim3(k.grid), dim3(k.threads), args, k.lds_bytes, (hipStream_t)stream);
  return check_launch(k.what);
}

// A table kernel, and its form without arguments by value where it has one.
template <typename Block>
struct TableKernel {
  void (*by_value)(APC_LAUNCH_PARAMS(Block, false));
  void (*kept)(APC_LAUNCH_PARAMS(Block, true)) = nullptr;
};

template <typename Block>
static int launch_table_kernel(const char *what, const LaunchTo &to, const TableKernel<Block> &kernel, unsigned grid, int threads,
                               size_t lds, const void *work, int n_tiles, int xcd_shift, int64_t tile_blocks, double *cost_out,
                               const Block &block) {
  static_assert(sizeof(Block) <= APC_KEPT_BLOCK_BYTES, "the arguments fit a kept launch");
  static_assert(std::is_trivially_copyable<Block>::value, "the arguments travel as bytes");
  if (!to.keep) {
    hipLaunchKernelGGL(kernel.by_value, dim3(grid), dim3(threads), lds, (hipStream_t)to.stream, work, n_tiles, xcd_shift, tile_blocks, cost_out,
                       (const Block *)nullptr, BlockByValue<Block, false>{block});
    return check_launch(what);
  }
  apc_kept_launch &k = *to.keep;
  k.kernel = kernel.kept ? reinterpret_cast<const void *>(kernel.kept) : reinterpret_cast<const void *>(kernel.by_value);
  k.kernel_by_value = reinterpret_cast<const void *>(kernel.by_value);
  k.what = what;
  k.grid = grid;
  k.threads = (uint32_t)threads;
  k.lds_bytes = (uint32_t)lds;
  k.block_bytes = (uint32_t)sizeof(Block);
  k.work = const_cast<void *>(work);
  k.n_tiles = n_tiles;
  k.xcd_shift = xcd_shift;
  k.tile_blocks = tile_blocks;
  k.cost_out = cost_out;
  std::memcpy(k.block, &block, sizeof(Block));
  return 0;
}

// Row minima need their index arrays and, when some tile serves identical edges, those edges' rows.
static int check_row_minima(const apc_row_minima *rows, const int64_t *dup_entry_begin, const char *who) {
  if (!rows) return 0;
  if (!rows->edge_row_begin || !rows->row_min || !rows->row_argmin) return fail(-1, "%s: NULL row-minimum array", who);
  if (dup_entry_begin && !rows->dup_row_begin) return fail(-1, "%s: identical edges need dup_row_begin", who);
  return 0;
}

// The compile-time output mode of a launch (kOut*).  The specialised modes exist for 2-D and
// 3-D meshes (the planned graphs); other mesh ranks check their output pointers per store.
static int out_mode(int mesh_ndim, const double *comm_out, const uint8_t *trans_out, const double *cost_out) {
  if (mesh_ndim != 2 && mesh_ndim != 3) return kOutAny;
  if (comm_out && trans_out && cost_out) return kOutAll;
  if (cost_out && !comm_out && !trans_out) return kOutCost;
  return kOutAny;
}

// Threads of a tile's workgroup.  More wavefronts stage and drain a tile sooner, fewer leave more tiles resident per
// compute unit, so what counts is whether the tiles fill the chip and how many values one stores (n_entries
// counts the copies written for identical edges too: work per tile either way).
//   At most kTilesInOneRound tiles, all of them resident at once: four wavefronts (829 tiles of 387 values, (32, 8),
//   one launch: 9.5 / 7.4 / 7.1 us with one / two / four; 968 tiles of 1 800 values 21.6 / 14.8 / 12.0).
//   `many_states`: four (a tile stages the 304 states of a 4-D mesh: 9 852 tiles of 22 values 101 / 73 / 58 us).  With
//   power-of-two sizes it stages the exponents' 14 arrays, as on other meshes: 2 218 tiles of 390 values - / 9.0 / 11.8, 1 540 of 560
//   15.2 / 10.0 / 9.9, 8 747 of 609 - / 31.3 / 37.3.
//   Else by the values per tile: two from `two`, four from `four`.  The launch over the tables' own copies (512, 2048):
//   1 800 values, (8, 8, 8), 169 / 154 / 179 us; 3 236 values there - / 173 / 131; 2 390 values, (32, 8), - / 32.9 / 29.2.  The launch
//   of all tables, whose tiles derive what the other reads (64, on 3-D meshes always, with kTilesOfManyRounds 512; 2304): (32, 8), 398 values 18.5 /
//   17.2 / 21.0, 2 166 in 6 850 tiles - / 46.5 / 44.9, 2 178 in 10 836 - / 70.3 / 70.7, (16, 8, 4) - / 68.5 / 72.4, then 2 435 in 5 890, (32, 8), - / 43.7 / 40.8,
//   2 412 in 9 235 - / 65.5 / 63.3, 2 951 in 10 165 - / 82.2 / 75.2, (16, 8, 4), 2 348 in 2 840 - / 16.3 / 16.5, 2 923 in 5 098 - / 44.1 / 41.0, 22 values 13.9 / 15.7 / 24.5; (8, 8, 8), 22 values
//   17.1 / 16.1 / 24.1 us; 36 157 tiles of 149 values 46.8 / 59.4 / 96.7 there, 46.7 / 56.5 / 94.9 on (16, 8, 4), 4 123 of 139
//   on (8, 8, 8) 16.6 / 14.3 / 17.8.
//   ... and (a 20th of the tiles, 256 at most, and 256 where matrices of fewer entries have copies, 512 where they have 64 at most; 300) from the
//   second round of its workgroups on one wavefront takes the tiles that store less than that (few rounds end with the largest tiles, which
//   one wavefront takes longest over; a second one has no part in 64 entries, however many copies they are stored to): us with one / two,
//   2 081 tiles of 191 values, (16, 8, 4), 7.8 / 6.4, (2, 4, 2, 2) 8.9 / 6.8, 2 650 of 166, (8, 8, 8), 8.0 / 7.4, 3 093 of 222, (32, 8), 9.8 / 8.2, (12, 6)
//   10.0 / 9.2; the other way 2 548 of 95, (12, 6), 7.0 / 7.8, 3 334 of 146, (8, 8, 8), 8.0 / 8.9, 4 017 of 99, (64, 4), 7.4 / 8.9, (2, 4, 2, 2) 8.3 / 9.6; about
//   equal 3 900 of 171, (8, 8, 8) 10.3 / 9.6, (12, 6) 10.0 / 10.6, 4 872 of 217, (16, 8, 4) 11.8 / 11.7, (64, 4) 11.2 / 11.4, 6 533 of 161, (8, 8, 8), 9.9 / 9.9; 16
//   copies of 8 in 2 582, (64,), 7.3 / 8.9, 12 of 18 in 2 582, (12, 6), 8.1 / 9.4, 16 9.0 / 10.1, (32, 8) 8.4 / 9.3,
//   (2, 4, 2, 2) 9.0 / 10.0, 16 of 17 in 4 478, (8, 8, 8), 10.8 / 13.2;
//   4 694 tiles of 129 values, (16, 8, 4), 9.4 / 10.8, 10 834 of 246, (8, 8, 8), 14.8 / 16.3, 8 566 of 207 12.6 / 13.3, 10 278 of 159, (32, 8),
//   12.3 / 13.3, 9 426 of 200, (2, 4, 2, 2), 14.5 / 15.7, 10 278 of 266, (6,), 13.5 / 14.7, 2 906 of 5, (64,), 5.5 / 6.4; the other way 6 950 of 273,
//   (32, 8), 13.9 / 11.3, 6 335 of 287, (16, 8, 4), 12.3 / 11.7, 9 425 of 420 18.0 / 17.1.  Not with the 72 states of a 3-D mesh to
//   stage: 6 333 of 202, (6, 4, 2), 14.0 / 13.3, 9 425 of 255 18.6 / 18.1, 8 967 of 17 13.3 / 13.1.
//   Small tiles fill the chip sooner: from kSmallTilesInOneRound on, two for those of less than kSmallTile values (1 181 tiles of
//   338 values, (8, 8, 8), 6.6 with two / 7.5 with four, 1 265 of 330, (12, 6), 7.0 / 8.0; the other way 880 of 480 7.9 / 7.1, 812 of
//   490 7.5 / 6.7, 1 270 of 710 11.7 / 8.7).
constexpr int64_t kTilesInOneRound = 1280;  // five workgroups of four wavefronts to a compute unit
constexpr int64_t kSmallTilesInOneRound = 1024, kSmallTile = 448;
constexpr int64_t kTilesOfTwoRounds = 2048, kTilesOfSomeRounds = 8192, kTilesPerValueOfOne = 20, kSideOfOne = 4;
constexpr int64_t kTilesOfManyRounds = 16384;  // (of one wavefront: 32 workgroups to a compute unit, twice)

static int tile_threads(int64_t n_tiles, int64_t n_entries, bool many_states, int64_t two, int64_t four) {
  int threads = 256;
  const int64_t per_tile = n_tiles > 0 ? n_entries / n_tiles : 0;
  if ((n_tiles > kTilesInOneRound || (n_tiles > kSmallTilesInOneRound && per_tile < kSmallTile)) && !many_states) {
    threads = per_tile >= four ? 256 : per_tile >= two ? 128 : 64;
  }
  if (const char *env = getenv("APC_TILE_THREADS")) threads = atoi(env);  // tuning override
  return threads >= 256 ? 256 : threads >= 128 ? 128 : 64;
}

static int input_tables_impl(const apc_params *params, int64_t n_tensors, const int32_t *rank, const int32_t *itemsize,
                     const int64_t *shape, const int64_t *stride, int64_t *tensor_bytes, uint8_t *tensor_contiguous,
                     int64_t n_specs, const uint32_t *spec_codes, const int32_t *spec_tensor, int64_t *num_shards,
                     int64_t *local_shape, int64_t *local_stride, int32_t shape_width, int64_t *local_numel,
                     int64_t *local_bytes, int64_t n_strategies, const int64_t *flops, const int64_t *rw_bytes,
                     const int8_t *dtype, const uint8_t *zero_cost, const int32_t *num_args, double *compute,
                     double *per_arg, int32_t *error_flag, const LaunchTo &to) {
  if (int rc = check_params(params)) return rc;
  if (n_tensors < 0 || n_specs < 0 || n_strategies < 0) return fail(-1, "apc_input_tables: negative count");
  if (n_tensors > 0 && (!rank || !itemsize || !shape || !stride || !tensor_bytes || !tensor_contiguous))
    return fail(-1, "apc_input_tables: NULL tensor array");
  // the five spec-table outputs may all be NULL: the spec table is then skipped
  const bool spec_table = num_shards || local_shape || local_stride || local_numel || local_bytes;
  if (spec_table)
    if (int rc = check_width(shape_width)) return rc;
  if (spec_table && n_specs > 0 && (!spec_codes || !spec_tensor || !rank || !itemsize || !shape || !stride ||
                                    !num_shards || !local_shape || !local_stride || !local_numel || !local_bytes))
    return fail(-1, "apc_input_tables: the spec table needs all five of its outputs");
  if (n_strategies > 0 && (!flops || !rw_bytes || !dtype || !zero_cost || !num_args))
    return fail(-1, "apc_input_tables: NULL strategy array");
  const int64_t sb = spec_table ? blocks_for(n_specs, kBlock) : 0, tb = blocks_for(n_tensors, kBlock),
                cb = blocks_for(n_strategies, kBlock);
  if (sb + tb + cb == 0) return 0;
  if (sb + tb + cb > INT32_MAX) return fail(-1, "apc_input_tables: too many rows for one launch");
  const InputTablesBlock block{*params,
                               {n_tensors, rank, itemsize, shape, stride, tensor_bytes, tensor_contiguous},
                               {n_specs, spec_codes, spec_tensor, rank, itemsize, shape, stride, num_shards, local_shape, local_stride,
                                local_numel, local_bytes, shape_width},
                               {n_strategies, flops, rw_bytes, dtype, zero_cost, num_args, compute, per_arg, error_flag},
                               sb,
                               tb};
  return launch_table_kernel("apc_input_tables", to, TableKernel<InputTablesBlock>{input_tables_kernel<false>, input_tables_kernel<true>}, (unsigned)(sb + tb + cb), kBlock, 0, nullptr, 0, 0, 0, nullptr, block);
}

static int redistribute_tables_impl(const apc_params *params, const int64_t *tensor_bytes,
                                    const uint8_t *tensor_contiguous, const uint32_t *spec_codes,
                                    const int32_t *spec_tensor, const double *pt_values, const double *per_arg,
                                    int64_t n_tiles, const apc_tile *tiles, const int64_t *dup_entry_begin,
                                    int64_t n_entries, double *comm_out, uint8_t *trans_out, double *cost_out,
                                    const apc_row_minima *rows, const LaunchTo &to) {
  if (int rc = check_params(params)) return rc;
  if (n_tiles < 0 || n_tiles > (1 << 30)) return fail(-1, "n_tiles %lld out of range", (long long)n_tiles);
  if (n_tiles == 0) return 0;
  if (int rc = check_row_minima(rows, dup_entry_begin, "apc_redistribute_tables_row_min")) return rc;
  if (n_entries < 0) return fail(-1, "n_entries < 0");
  if (!tensor_bytes || !tensor_contiguous || !spec_codes || !spec_tensor || !tiles)
    return fail(-1, "apc_redistribute_tables: NULL table");
  if (cost_out && !per_arg) return fail(-1, "cost_out needs compute_cost_per_arg");
  TableArgs a{tensor_bytes, tensor_contiguous, spec_codes, spec_tensor, pt_values, per_arg,
              tiles,        dup_entry_begin,   comm_out,   trans_out,   cost_out,
              nullptr,      nullptr,           nullptr,    nullptr,     nullptr, nullptr, nullptr, nullptr, nullptr,
              rows ? rows->edge_row_begin : nullptr, rows ? rows->dup_row_begin : nullptr,
              rows ? rows->row_min : nullptr, rows ? rows->row_argmin : nullptr, term_layout(*params)};
  const int nt = (int)n_tiles, xs = xcd_shift();
  const int64_t grid = ((n_tiles + (1 << xs) - 1) >> xs) << xs;  // rounded up for tile_of_block
  const char *const what = rows ? "apc_redistribute_tables_row_min" : "apc_redistribute_tables";
  const int threads = tile_threads(n_tiles, n_entries, params->mesh_ndim == 4 && a.lay.exponents == 0, 512, 2048);
  const int om = out_mode(params->mesh_ndim, comm_out, trans_out, cost_out);
#define APC_LAUNCH_T(KERNEL_, M_, OUT_)                                                                               \
  const int wg = threads >= 256 ? 256 : threads >= 128 ? 128 : 64;                                                     \
  const size_t lds = rows ? stage_lds_bytes<M_, true>(a.lay, wg) : stage_lds_bytes<M_, false>(a.lay, wg);              \
  const TableKernel<TilesBlock> kernel{wg == 256 ? KERNEL_<M_, 256, OUT_> : wg == 128 ? KERNEL_<M_, 128, OUT_> : KERNEL_<M_, 64, OUT_>}; \
  return launch_table_kernel(what, to, kernel, (unsigned)grid, wg, lds, tiles, nt, xs, grid, cost_out, TilesBlock{*params, a})
#define APC_LAUNCH_K(KERNEL_, M_)                                   \
  if (om == kOutAll) { APC_LAUNCH_T(KERNEL_, M_, kOutAll); }        \
  else if (om == kOutCost) { APC_LAUNCH_T(KERNEL_, M_, kOutCost); } \
  else { APC_LAUNCH_T(KERNEL_, M_, kOutAny); }
#define APC_LAUNCH_ANY(KERNEL_, M_) { APC_LAUNCH_T(KERNEL_, M_, kOutAny); }
  if (rows) {
    switch (params->mesh_ndim) {
      case 1: APC_LAUNCH_ANY(redistribute_tiles_row_min_kernel, 1); break;
      case 2: APC_LAUNCH_K(redistribute_tiles_row_min_kernel, 2); break;
      case 3: APC_LAUNCH_K(redistribute_tiles_row_min_kernel, 3); break;
      default: APC_LAUNCH_ANY(redistribute_tiles_row_min_kernel, 4); break;
    }
  } else {
    switch (params->mesh_ndim) {
      case 1: APC_LAUNCH_ANY(redistribute_tiles_kernel, 1); break;
      case 2: APC_LAUNCH_K(redistribute_tiles_kernel, 2); break;
      case 3: APC_LAUNCH_K(redistribute_tiles_kernel, 3); break;
      default: APC_LAUNCH_ANY(redistribute_tiles_kernel, 4); break;
    }
  }
#undef APC_LAUNCH_T
#undef APC_LAUNCH_K
#undef APC_LAUNCH_ANY
}

// (kept: of the outputs a planner's pass has)
template <int M, int kThreads, bool RM, int OUT>
static TableKernel<BuildTablesBlock> build_tables_forms() {
  if constexpr (OUT == kOutCost || M == 1 || M == 4)
    return {build_tables_kernel<M, kThreads, RM, OUT, false>, build_tables_kernel<M, kThreads, RM, OUT, true>};
  else
    return {build_tables_kernel<M, kThreads, RM, OUT, false>};
}

static int build_tables_impl(const apc_params *params, int64_t n_tensors, const int32_t *rank, const int32_t *itemsize,
                     const int64_t *shape, const int64_t *stride, int64_t *tensor_bytes, uint8_t *tensor_contiguous,
                     int64_t n_specs, const uint32_t *spec_codes, const int32_t *spec_tensor, int64_t *num_shards,
                     int64_t *local_shape, int64_t *local_stride, int32_t shape_width, int64_t *local_numel,
                     int64_t *local_bytes, int64_t n_strategies, const int64_t *flops, const int64_t *rw_bytes,
                     const int8_t *dtype, const uint8_t *zero_cost, const int32_t *num_args, double *compute,
                     double *per_arg, int32_t *error_flag, const double *pt_values, int64_t n_tiles, const apc_tile *tiles,
                     const int64_t *dup_entry_begin, int64_t n_entries, double *comm_out, uint8_t *trans_out,
                     double *cost_out, const apc_row_minima *rows, const LaunchTo &to) {
  if (int rc = check_params(params)) return rc;
  if (n_tiles > 0)
    if (int rc = check_row_minima(rows, dup_entry_begin, "apc_build_tables_row_min")) return rc;
  if (n_tensors < 0 || n_specs < 0 || n_strategies < 0 || n_entries < 0) return fail(-1, "apc_build_tables: negative count");
  if (n_tiles < 0 || n_tiles > (1 << 30)) return fail(-1, "n_tiles %lld out of range", (long long)n_tiles);
  if (n_tensors > 0 && (!rank || !itemsize || !shape || !stride || !tensor_bytes || !tensor_contiguous))
    return fail(-1, "apc_build_tables: NULL tensor array");
  const bool spec_table = num_shards || local_shape || local_stride || local_numel || local_bytes;
  if (spec_table)
    if (int rc = check_width(shape_width)) return rc;
  if (spec_table && n_specs > 0 && (!spec_codes || !spec_tensor || !num_shards || !local_shape || !local_stride ||
                                    !local_numel || !local_bytes))
    return fail(-1, "apc_build_tables: the spec table needs all five of its outputs");
  if (n_strategies > 0 && (!flops || !rw_bytes || !dtype || !zero_cost || !num_args))
    return fail(-1, "apc_build_tables: NULL strategy array");
  if (n_tiles > 0 && (!spec_codes || !spec_tensor || !tiles || !rank || !itemsize || !shape || !stride))
    return fail(-1, "apc_build_tables: NULL table");
  // (a tile without a tensor still loads row 0 of the tensor table: unconditional loads)
  if (n_tiles > 0 && n_tensors == 0) return fail(-1, "apc_build_tables: tiles need a tensor table with at least one row");
  const int xs = xcd_shift();
  const TermLayout lay = term_layout(*params);
  const bool many_states = params->mesh_ndim == 4 && lay.exponents == 0;
  // (about the side of a matrix: a spec is a row of one and, where it is a node's, a column of its readers')
  const int64_t side = n_specs > 0 ? 8 * n_entries / (5 * n_specs) : 0, a_20th = n_tiles / kTilesPerValueOfOne;
  const int64_t two = n_tiles > kTilesOfManyRounds                       ? 512
                      : params->mesh_ndim == 3 && lay.exponents == 0 ? 0
                      : n_tiles > kTilesOfSomeRounds                  ? 300
                      : n_tiles > kTilesOfTwoRounds                   ? (side <= kSideOfOne ? 512 : side * side < a_20th ? 256 : std::min<int64_t>(256, a_20th))
                      : params->mesh_ndim == 3                       ? 0
                                                                     : 64;
  const int threads = tile_threads(n_tiles, n_entries, many_states, two, 2304);
  const int64_t tile_blocks = ((n_tiles + (1 << xs) - 1) >> xs) << xs;
  const int64_t sb = spec_table ? blocks_for(n_specs, threads) : 0, tb = blocks_for(n_tensors, threads),
                cb = blocks_for(n_strategies, threads);
  const int64_t blocks = tile_blocks + sb + tb + cb;
  if (blocks == 0) return 0;
  if (blocks > INT32_MAX) return fail(-1, "apc_build_tables: too many rows for one launch");
  // the tiles read neither the tensor table nor the compute costs (written by this launch)
  TableArgs a{nullptr, nullptr, spec_codes, spec_tensor, pt_values, nullptr, tiles, dup_entry_begin,
              comm_out, trans_out, cost_out, rank, itemsize, shape, stride, flops, rw_bytes, dtype, zero_cost, num_args,
              rows ? rows->edge_row_begin : nullptr, rows ? rows->dup_row_begin : nullptr,
              rows ? rows->row_min : nullptr, rows ? rows->row_argmin : nullptr, lay};
  const TensorTableArgs ta{n_tensors, rank, itemsize, shape, stride, tensor_bytes, tensor_contiguous};
  const SpecTableArgs sa{n_specs, spec_codes, spec_tensor, rank, itemsize, shape, stride, num_shards,
                         local_shape, local_stride, local_numel, local_bytes, shape_width};
  const ComputeCostArgs ca{n_strategies, flops, rw_bytes, dtype, zero_cost, num_args, compute, per_arg, error_flag};
  const char *const what = rows ? "apc_build_tables_row_min" : "apc_build_tables";
  const int nt = (int)n_tiles;
  const int om = out_mode(params->mesh_ndim, comm_out, trans_out, cost_out);
#define APC_LAUNCH_ALL_T(M_, RM_, OUT_)                                                                                 \
  const size_t lds = build_tables_lds_bytes<M_, RM_>(a.lay, threads, spec_table);                                      \
  const auto kernel = threads == 256   ? build_tables_forms<M_, 256, RM_, OUT_>()                                       \
                      : threads == 128 ? build_tables_forms<M_, 128, RM_, OUT_>() : build_tables_forms<M_, 64, RM_, OUT_>(); \
  return launch_table_kernel(what, to, kernel, (unsigned)blocks, threads, lds, tiles, nt, xs, tile_blocks, cost_out,  \
                             BuildTablesBlock{*params, a, ta, sa, ca, sb, tb})
#define APC_LAUNCH_ALL_RM(M_, RM_)                                   \
  if (om == kOutAll) { APC_LAUNCH_ALL_T(M_, RM_, kOutAll); }         \
  else if (om == kOutCost) { APC_LAUNCH_ALL_T(M_, RM_, kOutCost); }  \
  else { APC_LAUNCH_ALL_T(M_, RM_, kOutAny); }
#define APC_LAUNCH_ALL(M_)                    \
  if (rows) { APC_LAUNCH_ALL_RM(M_, true); } else { APC_LAUNCH_ALL_RM(M_, false); }
#define APC_LAUNCH_ALL_ANY(M_)                \
  if (rows) { APC_LAUNCH_ALL_T(M_, true, kOutAny); } else { APC_LAUNCH_ALL_T(M_, false, kOutAny); }
  switch (params->mesh_ndim) {
    case 1: APC_LAUNCH_ALL_ANY(1); break;
    case 2: APC_LAUNCH_ALL(2); break;
    case 3: APC_LAUNCH_ALL(3); break;
    default: APC_LAUNCH_ALL_ANY(4); break;
  }
#undef APC_LAUNCH_ALL_T
#undef APC_LAUNCH_ALL_RM
#undef APC_LAUNCH_ALL
#undef APC_LAUNCH_ALL_ANY
}

extern "C" {

int apc_keep_next_launch(apc_kept_launch *out) {
  if (!out) return fail(-1, "apc_keep_next_launch: NULL");
  out->kernel = nullptr;
  g_keep_next = out;
  return 0;
}

int apc_run_kept(const apc_kept_launch *kept, const void *device_block, void *stream) {
  if (!kept) return fail(-1, "apc_run_kept: NULL");
  if (!kept->kernel) return 0;  // (nothing to launch)
  if ((reinterpret_cast<uintptr_t>(device_block) & 63) != 0) return fail(-1, "apc_run_kept: the block must be 64-byte aligned");
  return enqueue_kept(*kept, device_block, stream);
}

int apc_input_tables(const apc_params *params, int64_t n_tensors, const int32_t *rank, const int32_t *itemsize,
                     const int64_t *shape, const int64_t *stride, int64_t *tensor_bytes, uint8_t *tensor_contiguous,
                     int64_t n_specs, const uint32_t *spec_codes, const int32_t *spec_tensor, int64_t *num_shards,
                     int64_t *local_shape, int64_t *local_stride, int32_t shape_width, int64_t *local_numel,
                     int64_t *local_bytes, int64_t n_strategies, const int64_t *flops, const int64_t *rw_bytes,
                     const int8_t *dtype, const uint8_t *zero_cost, const int32_t *num_args, double *compute,
                     double *per_arg, int32_t *error_flag, void *stream) {
  return input_tables_impl(params, n_tensors, rank, itemsize, shape, stride, tensor_bytes, tensor_contiguous, n_specs, spec_codes,
                           spec_tensor, num_shards, local_shape, local_stride, shape_width, local_numel, local_bytes, n_strategies,
                           flops, rw_bytes, dtype, zero_cost, num_args, compute, per_arg, error_flag, launch_to(stream));
}

int apc_redistribute_tables(const apc_params *params, const int64_t *tensor_bytes, const uint8_t *tensor_contiguous,
                            const uint32_t *spec_codes, const int32_t *spec_tensor, const double *pt_values,
                            const double *per_arg, int64_t n_tiles, const apc_tile *tiles,
                            const int64_t *dup_entry_begin, int64_t n_entries, double *comm_out, uint8_t *trans_out,
                            double *cost_out, void *stream) {
  return redistribute_tables_impl(params, tensor_bytes, tensor_contiguous, spec_codes, spec_tensor, pt_values, per_arg,
                                  n_tiles, tiles, dup_entry_begin, n_entries, comm_out, trans_out, cost_out, nullptr,
                                  launch_to(stream));
}

int apc_redistribute_tables_row_min(const apc_params *params, const int64_t *tensor_bytes,
                                    const uint8_t *tensor_contiguous, const uint32_t *spec_codes,
                                    const int32_t *spec_tensor, const double *pt_values, const double *per_arg,
                                    int64_t n_tiles, const apc_tile *tiles, const int64_t *dup_entry_begin,
                                    int64_t n_entries, double *comm_out, uint8_t *trans_out, double *cost_out,
                                    const apc_row_minima *rows, void *stream) {
  const LaunchTo to = launch_to(stream);
  if (!rows) return fail(-1, "apc_redistribute_tables_row_min: NULL rows");
  return redistribute_tables_impl(params, tensor_bytes, tensor_contiguous, spec_codes, spec_tensor, pt_values, per_arg,
                                  n_tiles, tiles, dup_entry_begin, n_entries, comm_out, trans_out, cost_out, rows, to);
}

#define APC_BUILD_TABLES_PARAMS                                                                                         \
  const apc_params *params, int64_t n_tensors, const int32_t *rank, const int32_t *itemsize, const int64_t *shape,      \
      const int64_t *stride, int64_t *tensor_bytes, uint8_t *tensor_contiguous, int64_t n_specs,                        \
      const uint32_t *spec_codes, const int32_t *spec_tensor, int64_t *num_shards, int64_t *local_shape,                \
      int64_t *local_stride, int32_t shape_width, int64_t *local_numel, int64_t *local_bytes, int64_t n_strategies,     \
      const int64_t *flops, const int64_t *rw_bytes, const int8_t *dtype, const uint8_t *zero_cost,                     \
      const int32_t *num_args, double *compute, double *per_arg, int32_t *error_flag, const double *pt_values,          \
      int64_t n_tiles, const apc_tile *tiles, const int64_t *dup_entry_begin, int64_t n_entries, double *comm_out,      \
      uint8_t *trans_out, double *cost_out
#define APC_BUILD_TABLES_ARGS                                                                                           \
  params, n_tensors, rank, itemsize, shape, stride, tensor_bytes, tensor_contiguous, n_specs, spec_codes, spec_tensor,  \
      num_shards, local_shape, local_stride, shape_width, local_numel, local_bytes, n_strategies, flops, rw_bytes,      \
      dtype, zero_cost, num_args, compute, per_arg, error_flag, pt_values, n_tiles, tiles, dup_entry_begin, n_entries,  \
      comm_out, trans_out, cost_out

int apc_build_tables(APC_BUILD_TABLES_PARAMS, void *stream) {
  return build_tables_impl(APC_BUILD_TABLES_ARGS, nullptr, launch_to(stream));
}

int apc_build_tables_row_min(APC_BUILD_TABLES_PARAMS, const apc_row_minima *rows, void *stream) {
  const LaunchTo to = launch_to(stream);
  if (!rows) return fail(-1, "apc_build_tables_row_min: NULL rows");
  return build_tables_impl(APC_BUILD_TABLES_ARGS, rows, to);
}
#undef APC_BUILD_TABLES_PARAMS
#undef APC_BUILD_TABLES_ARGS

}  // extern "C"

// Lanes per segment: about a tenth of the mean length, so that a lane has several
// independent loads in flight (measured best on both benchmark tables; APC_SEGMIN_GROUP
// overrides, for tuning).
static int segment_lanes(int64_t n_values, int64_t n_seg) {
  const double mean = (double)n_values / (double)n_seg;
  int g = 2;
  while (g < 64 && g * 12 <= mean) g *= 2;
  if (const char *env = getenv("APC_SEGMIN_GROUP")) g = atoi(env);
  return g;
}

static int segmented_min_impl(const double *values, const int64_t *seg_ptr, int64_t n_seg, int64_t n_values, double *mins,
                              int32_t *args, const SegmentCopies *copies, const char *who, void *stream) {
  if (n_seg < 0 || n_values < 0) return fail(-1, "negative count");
  if (n_seg == 0) return 0;
  if (!seg_ptr || !mins || !args || (!values && n_values > 0)) return fail(-1, "%s: NULL array", who);
  if (n_seg > (int64_t)INT32_MAX * 4) return fail(-1, "n_segments %lld too large", (long long)n_seg);
  hipStream_t s = (hipStream_t)stream;
  const int g = segment_lanes(n_values, n_seg);
  switch (g) {
    case 1: launch_segmented_min<1>(values, seg_ptr, n_seg, mins, args, copies, s); break;
    case 2: launch_segmented_min<2>(values, seg_ptr, n_seg, mins, args, copies, s); break;
    case 4: launch_segmented_min<4>(values, seg_ptr, n_seg, mins, args, copies, s); break;
    case 8: launch_segmented_min<8>(values, seg_ptr, n_seg, mins, args, copies, s); break;
    case 16: launch_segmented_min<16>(values, seg_ptr, n_seg, mins, args, copies, s); break;
    case 32: launch_segmented_min<32>(values, seg_ptr, n_seg, mins, args, copies, s); break;
    case 64: launch_segmented_min<64>(values, seg_ptr, n_seg, mins, args, copies, s); break;
    default: return fail(-1, "segment group width %d is not a power of two up to 64", g);
  }
  return check_launch(who);
}

extern "C" {

int apc_segmented_min(const double *values, const int64_t *seg_ptr, int64_t n_seg, int64_t n_values, double *mins,
                      int32_t *args, void *stream) {
  return segmented_min_impl(values, seg_ptr, n_seg, n_values, mins, args, nullptr, "apc_segmented_min", stream);
}

int apc_segmented_min_copies(const double *values, const int64_t *seg_ptr, int64_t n_selected, const int64_t *selected,
                             const int64_t *copy_ptr, const int64_t *copy_segments, int64_t n_values_selected,
                             double *mins, int32_t *args, void *stream) {
  if (n_selected > 0 && (!selected || !copy_ptr)) return fail(-1, "apc_segmented_min_copies: NULL selection");
  const SegmentCopies copies{selected, copy_ptr, copy_segments};
  return segmented_min_impl(values, seg_ptr, n_selected, n_values_selected, mins, args, &copies,
                            "apc_segmented_min_copies", stream);
}

int apc_strategy_bounds(int64_t n_strategies, const int32_t *strat_node, const int64_t *node_strat_begin,
                        const int64_t *node_edge_begin, const int32_t *edges_by_node, const int64_t *edge_row_begin,
                        const double *row_min, double *bound, void *stream) {
  if (n_strategies < 0) return fail(-1, "negative count");
  if (n_strategies == 0) return 0;
  if (!strat_node || !node_strat_begin || !node_edge_begin || !edge_row_begin || !row_min || !bound)
    return fail(-1, "apc_strategy_bounds: NULL array");  // (edges_by_node may be NULL when no node has an edge)
  if ((n_strategies + kBlock - 1) / kBlock > INT32_MAX) return fail(-1, "n_strategies %lld too large", (long long)n_strategies);
  hipLaunchKernelGGL(strategy_bounds_kernel, dim3(blocks_for(n_strategies, kBlock)), dim3(kBlock), 0, (hipStream_t)stream,
                     n_strategies, strat_node, node_strat_begin, node_edge_begin, edges_by_node, edge_row_begin, row_min,
                     bound);
  return check_launch("apc_strategy_bounds");
}

int apc_greedy_strategies(int64_t n_nodes, int64_t n_strategies, const int64_t *node_strat_begin, const int64_t *node_edge_begin,
                          const int32_t *edges_by_node, const int64_t *edge_row_begin, const double *row_min, double *bound,
                          double *node_min, int32_t *node_argmin, void *stream) {
  if (n_nodes < 0 || n_strategies < 0) return fail(-1, "apc_greedy_strategies: negative count");
  if (n_nodes == 0) return 0;
  // (edges_by_node may be NULL when no node has an edge, the arrays of strategies when there is none)
  if (!node_strat_begin || !node_edge_begin || !node_min || !node_argmin || (n_strategies > 0 && !bound))
    return fail(-1, "apc_greedy_strategies: NULL array");
  if (n_nodes > (int64_t)INT32_MAX * 4) return fail(-1, "n_nodes %lld too large", (long long)n_nodes);
  const int g = segment_lanes(n_strategies, n_nodes), threads = n_nodes <= INT32_MAX ? 64 : kBlock;
  const bool few = n_strategies <= 2 * g * n_nodes;  // a lane has a pair
#define APC_GREEDY(G_)                                                                                                       \
  case G_:                                                                                                                   \
    hipLaunchKernelGGL((few ? greedy_strategies_kernel<G_, 1> : greedy_strategies_kernel<G_, 4>), dim3(blocks_for(n_nodes, threads / G_)), dim3(threads), 0, \
                       (hipStream_t)stream, n_nodes, node_strat_begin, node_edge_begin, edges_by_node, edge_row_begin,        \
                       row_min, bound, node_min, node_argmin);                                                               \
    break
  switch (g) {
    APC_GREEDY(1);
    APC_GREEDY(2);
    APC_GREEDY(4);
    APC_GREEDY(8);
    APC_GREEDY(16);
    APC_GREEDY(32);
    APC_GREEDY(64);
    default: return fail(-1, "segment group width %d is not a power of two up to 64", g);
  }
#undef APC_GREEDY
  return check_launch("apc_greedy_strategies");
}

int apc_edge_rows(int64_t n_edges, const int32_t *edge_n_tgt, int64_t *edge_row_begin, void *stream) {
  if (n_edges < 0) return fail(-1, "apc_edge_rows: n_edges < 0");
  if (n_edges == 0) return 0;
  if (!edge_n_tgt || !edge_row_begin) return fail(-1, "apc_edge_rows: NULL array");
  hipLaunchKernelGGL(edge_rows_kernel, dim3(1), dim3(kScanThreads), 0, (hipStream_t)stream, n_edges, edge_n_tgt, edge_row_begin);
  return check_launch("apc_edge_rows");
}

int apc_report_inputs(const apc_params *params, int64_t n_tensors, const int32_t *rank, const int32_t *itemsize, const int64_t *shape,
                      const int64_t *stride, int64_t *tensor_bytes, uint8_t *tensor_contiguous, int64_t n_strategies, const int64_t *flops,
                      const int64_t *rw_bytes, const int8_t *dtype, const uint8_t *zero_cost, const int32_t *num_args, double *compute,
                      double *per_arg, int32_t *error_flag, int64_t n_edges, const int32_t *edge_n_tgt, int64_t *edge_row_begin, void *stream) {
  if (int rc = check_params(params)) return rc;
  if (n_tensors < 0 || n_strategies < 0 || n_edges < 0) return fail(-1, "apc_report_inputs: negative count");
  if (n_tensors > 0 && (!rank || !itemsize || !shape || !stride || !tensor_bytes || !tensor_contiguous))
    return fail(-1, "apc_report_inputs: NULL tensor array");
  if (n_strategies > 0 && (!flops || !rw_bytes || !dtype || !zero_cost || !num_args)) return fail(-1, "apc_report_inputs: NULL strategy array");
  if (n_edges > 0 && (!edge_n_tgt || !edge_row_begin)) return fail(-1, "apc_report_inputs: NULL edge array");
  const int64_t rb = n_edges > 0 ? 1 : 0, tb = blocks_for(n_tensors, kScanThreads), cb = blocks_for(n_strategies, kScanThreads);
  if (rb + tb + cb == 0) return 0;
  if (rb + tb + cb > INT32_MAX) return fail(-1, "apc_report_inputs: too many rows for one launch");
  const ReportInputsArgs a{*params, {n_tensors, rank, itemsize, shape, stride, tensor_bytes, tensor_contiguous},
                           {n_strategies, flops, rw_bytes, dtype, zero_cost, num_args, compute, per_arg, error_flag},
                           n_edges, edge_n_tgt, edge_row_begin, rb, tb};
  hipLaunchKernelGGL(report_inputs_kernel, dim3((unsigned)(rb + tb + cb)), dim3(kScanThreads), 0, (hipStream_t)stream, a);
  return check_launch("apc_report_inputs");
}

int apc_copy_arrays(int64_t n, const void *const *from_host, void *const *to_host, const int64_t *bytes_host, void *stream) {
  if (n < 0 || n > APC_COPY_MAX_ARRAYS) return fail(-1, "apc_copy_arrays: %lld arrays, at most %d", (long long)n, APC_COPY_MAX_ARRAYS);
  if (n > 0 && (!from_host || !to_host || !bytes_host)) return fail(-1, "apc_copy_arrays: NULL array");
  CopyArrays a{};
  int64_t blocks = 0;
  for (int64_t k = 0; k < n; ++k) {
    if (bytes_host[k] < 0) return fail(-1, "apc_copy_arrays: array %lld has a negative size", (long long)k);
    if (bytes_host[k] == 0) continue;
    if (!from_host[k] || !to_host[k]) return fail(-1, "apc_copy_arrays: array %lld is NULL", (long long)k);
    if (bytes_host[k] > (int64_t)INT32_MAX * kCopyUnit || (blocks + (bytes_host[k] + kCopyUnit - 1) / kCopyUnit) > INT32_MAX)
      return fail(-1, "apc_copy_arrays: too many bytes for one launch");
    a.from[a.n] = static_cast<const char *>(from_host[k]);
    a.to[a.n] = static_cast<char *>(to_host[k]);
    a.bytes[a.n] = bytes_host[k];
    a.first_block[a.n++] = (int32_t)blocks;
    blocks += (bytes_host[k] + kCopyUnit - 1) / kCopyUnit;
  }
  if (blocks == 0) return 0;
  hipLaunchKernelGGL(copy_arrays_kernel, dim3((unsigned)blocks), dim3(kBlock), 0, (hipStream_t)stream, a);
  return check_launch("apc_copy_arrays");
}

int apc_check_tables(const apc_params *params, int32_t with_rows, int64_t n_tensors, const int32_t *tensor_rank, int64_t n_specs,
                     const uint32_t *spec_codes, const int32_t *spec_tensor, int64_t n_edges, const int32_t *edge_src_begin,
                     const int32_t *edge_n_src, const int32_t *edge_tgt_begin, const int32_t *edge_n_tgt, const int32_t *edge_flags,
                     const int64_t *edge_pt_begin, const int64_t *edge_entry_begin, const int32_t *edge_strat_begin, int64_t n_pt,
                     int64_t n_strategies, int64_t n_tiles, const apc_tile *tiles, int64_t n_dups, const int64_t *dup_entry_begin,
                     int32_t *malformed, void *stream) {
  if (int rc = check_params(params)) return rc;
  if (n_tensors < 0 || n_specs < 0 || n_edges < 0 || n_pt < 0 || n_strategies < 0 || n_tiles < 0 || n_dups < 0)
    return fail(-1, "apc_check_tables: negative count");
  if (!malformed || !edge_entry_begin || (n_tensors > 0 && !tensor_rank) || (n_specs > 0 && (!spec_codes || !spec_tensor)) ||
      (n_edges > 0 && (!edge_src_begin || !edge_n_src || !edge_tgt_begin || !edge_n_tgt || !edge_flags || !edge_pt_begin || !edge_strat_begin)) ||
      (n_tiles > 0 && !tiles) || (n_dups > 0 && !dup_entry_begin))
    return fail(-1, "apc_check_tables: NULL array");
  CheckTablesArgs a{};
  a.mesh_ndim = params->mesh_ndim;
  a.n_tensors = n_tensors, a.n_specs = n_specs, a.n_edges = n_edges, a.n_pt = n_pt, a.n_strategies = n_strategies;
  a.n_tiles = n_tiles, a.n_dups = n_dups;
  a.tensor_rank = tensor_rank, a.spec_codes = spec_codes, a.spec_tensor = spec_tensor;
  a.src_begin = edge_src_begin, a.n_src = edge_n_src, a.tgt_begin = edge_tgt_begin, a.n_tgt = edge_n_tgt, a.flags = edge_flags;
  a.strat_begin = edge_strat_begin, a.pt_begin = edge_pt_begin, a.entry_begin = edge_entry_begin;
  a.tiles = tiles, a.dup_entry_begin = dup_entry_begin, a.malformed = malformed;
  constexpr int64_t kItems = kBlock / 64;
  if (with_rows) {
    a.tensor_blocks = std::max<int64_t>(1, (n_tensors + kBlock - 1) / kBlock);  // (one for the first entry at least)
    a.spec_blocks = (n_specs + kBlock - 1) / kBlock;
    a.edge_blocks = (n_edges + kItems - 1) / kItems;
  }
  const int64_t blocks = a.tensor_blocks + a.spec_blocks + a.edge_blocks + (n_tiles + kItems - 1) / kItems;
  if (blocks == 0) return 0;
  if (blocks > INT32_MAX) return fail(-1, "apc_check_tables: too many workgroups");
  hipLaunchKernelGGL(check_tables_kernel, dim3((unsigned)blocks), dim3(kBlock), 0, (hipStream_t)stream, a);
  return check_launch("apc_check_tables");
}

int apc_edge_classes(int64_t n_specs, const uint32_t *spec_codes, const int32_t *spec_tensor, int64_t n_strategies, const int64_t *flops,
                     const int64_t *rw_bytes, const int8_t *dtype_code, const uint8_t *zero_cost, const int32_t *num_args, int64_t n_edges,
                     const int32_t *edge_src_begin, const int32_t *edge_n_src, const int32_t *edge_tgt_begin, const int32_t *edge_n_tgt,
                     const int32_t *edge_flags, const int64_t *edge_pt_begin, const int32_t *edge_strat_begin, int64_t n_pt,
                     const double *pt_values, int64_t n_slots, uint64_t *keys, int32_t *first, int32_t *slots, int64_t *first_same,
                     void *stream) {
  if (n_specs < 0 || n_strategies < 0 || n_edges < 0 || n_pt < 0) return fail(-1, "apc_edge_classes: negative count");
  if (n_edges == 0) return 0;
  if (n_edges > INT32_MAX / 4 || n_slots < 2 * n_edges || n_slots > INT32_MAX || (n_slots & (n_slots - 1)) != 0)
    return fail(-1, "apc_edge_classes: %lld slots for %lld edges: a power of two, at least twice as many", (long long)n_slots, (long long)n_edges);
  if (!edge_src_begin || !edge_n_src || !edge_tgt_begin || !edge_n_tgt || !edge_flags || !edge_pt_begin || !edge_strat_begin || !keys ||
      !first || !slots || !first_same || (n_specs > 0 && (!spec_codes || !spec_tensor)) || (n_pt > 0 && !pt_values) ||
      (n_strategies > 0 && (!flops || !rw_bytes || !dtype_code || !zero_cost || !num_args)))
    return fail(-1, "apc_edge_classes: NULL array");
  EdgeClassArgs a{};
  a.n_specs = n_specs, a.n_strategies = n_strategies, a.n_edges = n_edges, a.n_pt = n_pt, a.n_slots = n_slots;
  a.spec_codes = spec_codes, a.spec_tensor = spec_tensor, a.flops = flops, a.rw_bytes = rw_bytes, a.dtype = dtype_code;
  a.zero_cost = zero_cost, a.num_args = num_args;
  a.src_begin = edge_src_begin, a.n_src = edge_n_src, a.tgt_begin = edge_tgt_begin, a.n_tgt = edge_n_tgt, a.flags = edge_flags;
  a.strat_begin = edge_strat_begin, a.pt_begin = edge_pt_begin, a.pt_values = pt_values;
  a.keys = reinterpret_cast<unsigned long long *>(keys), a.first = first, a.slots = slots, a.first_same = first_same;
  const dim3 grid((unsigned)((n_edges + kBlock / 64 - 1) / (kBlock / 64)));
  hipLaunchKernelGGL(edge_hashes_kernel, grid, dim3(kBlock), 0, (hipStream_t)stream, a);
  if (int rc = check_launch("apc_edge_classes")) return rc;
  hipLaunchKernelGGL(edge_classes_kernel, grid, dim3(kBlock), 0, (hipStream_t)stream, a);
  return check_launch("apc_edge_classes");
}

int apc_pack_tiles(int64_t n_tensors, const int32_t *tensor_rank, const int32_t *tensor_itemsize, const int64_t *tensor_shape,
                   const int64_t *tensor_stride, int64_t n_specs, const uint32_t *spec_codes, const int32_t *spec_tensor,
                   int64_t n_strategies, const int64_t *flops, const int64_t *rw_bytes, const int8_t *dtype_code,
                   const uint8_t *zero_cost, const int32_t *num_args, int64_t n_edges, const int64_t *edge_row_begin, int64_t n_tiles,
                   const apc_tile *tiles, int64_t n_dups, const int64_t *dup_entry_begin, const int64_t *dup_row_begin,
                   apc_packed_tile *packed, int32_t *refused, void *stream) {
  if (n_tensors < 0 || n_specs < 0 || n_strategies < 0 || n_edges < 0 || n_tiles < 0 || n_dups < 0)
    return fail(-1, "apc_pack_tiles: negative count");
  if (n_tiles == 0) return 0;
  if (!tiles || !packed || !refused || !spec_codes || !spec_tensor || !edge_row_begin || !flops || !rw_bytes || !dtype_code || !zero_cost ||
      !num_args || (n_dups > 0 && (!dup_entry_begin || !dup_row_begin)) ||
      (n_tensors > 0 && (!tensor_rank || !tensor_itemsize || !tensor_shape || !tensor_stride)))
    return fail(-1, "apc_pack_tiles: NULL array");
  const int64_t blocks = (n_tiles + kBlock / 64 - 1) / (kBlock / 64);
  if (blocks > INT32_MAX) return fail(-1, "apc_pack_tiles: too many workgroups");
  PackArgs a{};
  a.t.n = n_tensors, a.t.rank = tensor_rank, a.t.itemsize = tensor_itemsize, a.t.shape = tensor_shape, a.t.stride = tensor_stride;
  a.n_specs = n_specs, a.n_strategies = n_strategies, a.n_edges = n_edges, a.n_tiles = n_tiles, a.n_dups = n_dups;
  a.spec_codes = spec_codes, a.spec_tensor = spec_tensor, a.flops = flops, a.rw_bytes = rw_bytes, a.dtype = dtype_code;
  a.zero_cost = zero_cost, a.num_args = num_args, a.edge_row_begin = edge_row_begin, a.tiles = tiles;
  a.dup_entry_begin = dup_entry_begin, a.dup_row_begin = dup_row_begin, a.packed = packed, a.refused = refused;
  hipLaunchKernelGGL(pack_tiles_kernel, dim3((unsigned)blocks), dim3(kBlock), 0, (hipStream_t)stream, a);
  return check_launch("apc_pack_tiles");
}

int apc_cost_objective(int64_t n_vars, int64_t n_groups, const int64_t *group_var_begin, const int64_t *group_member_begin,
                       const int64_t *member_entry_begin, const double *cost, double inf_replacement, double *objective,
                       uint8_t *forced_zero, void *stream) {
  if (n_vars < 0 || n_groups < 0) return fail(-1, "apc_cost_objective: negative count");
  if (n_vars == 0) return 0;
  if (n_groups == 0) return fail(-1, "apc_cost_objective: %lld variables and no group", (long long)n_vars);
  if (!group_var_begin || !group_member_begin || !member_entry_begin || !cost || !objective || !forced_zero)
    return fail(-1, "apc_cost_objective: NULL array");
  if (n_groups > INT32_MAX) return fail(-1, "apc_cost_objective: %lld groups, at most %d are launched", (long long)n_groups, INT32_MAX);
  // a program of few groups spreads each over several workgroups (those beyond a group's size
  // leave at once); with thousands of groups the device is full as it is
  // (and no more shares than twice what a group of average size fills)
  const int64_t average_runs = (n_vars / n_groups + kBlock - 1) / kBlock;
  const int64_t shares = n_groups >= 4096 ? 1 : std::min<int64_t>({64, (4096 + n_groups - 1) / n_groups, 2 * std::max<int64_t>(1, average_runs)});
  hipLaunchKernelGGL(cost_objective_kernel, dim3((unsigned)n_groups, (unsigned)shares), dim3(kBlock), 0, (hipStream_t)stream,
                     group_var_begin, group_member_begin, member_entry_begin, cost, inf_replacement, objective, forced_zero);
  return check_launch("apc_cost_objective");
}

int apc_diffusion_sweeps(int32_t n_sweeps, int32_t n_colors, const int64_t *color_begin_host, const int32_t *color_nodes,
                         int64_t n_classes, const int64_t *label_begin, const int64_t *inc_begin, const int32_t *inc_edge,
                         const uint8_t *inc_side, const int64_t *edge_begin, const int32_t *edge_i, const int32_t *edge_j,
                         int32_t max_labels, double *theta, double *unary, void *stream) {
  if (n_sweeps < 0 || n_colors < 0 || n_classes < 0) return fail(-1, "apc_diffusion_sweeps: negative count");
  if (n_sweeps == 0 || n_colors == 0 || n_classes == 0) return 0;
  if (max_labels > kDiffusionMaxLabels)
    return fail(-1, "apc_diffusion_sweeps: a class has %d labels, at most %d are staged", max_labels, kDiffusionMaxLabels);
  if (!color_begin_host || !color_nodes || !label_begin || !inc_begin || !edge_begin || !theta || !unary)
    return fail(-1, "apc_diffusion_sweeps: NULL array");
  if (color_begin_host[0] != 0 || color_begin_host[n_colors] != n_classes)
    return fail(-1, "apc_diffusion_sweeps: the colours must partition the classes");
  for (int32_t s = 0; s < n_sweeps; ++s) {
    for (int32_t c = 0; c < n_colors; ++c) {
      const int64_t n = color_begin_host[c + 1] - color_begin_host[c];
      if (n < 0 || n > INT32_MAX) return fail(-1, "apc_diffusion_sweeps: colour %d has %lld classes", c, (long long)n);
      if (n == 0) continue;
      hipLaunchKernelGGL(diffusion_node_update_kernel, dim3((unsigned)n), dim3(kBlock), 0, (hipStream_t)stream,
                         DiffusionArgs{color_nodes + color_begin_host[c], label_begin, inc_begin, inc_edge, inc_side,
                                       edge_begin, edge_i, edge_j, theta, unary});
    }
    if (int rc = check_launch("apc_diffusion_sweeps")) return rc;
  }
  return 0;
}

int apc_diffusion_sweeps_resident(int32_t n_sweeps, int64_t n_workgroups, const int32_t *plan, const int64_t *plan_begin,
                                  int64_t n_slots, int64_t lds_bytes, int32_t threads,
                                  int64_t n_labels, const double *theta, const double *unary,
                                  double *theta_out, double *unary_out, uint64_t *slots, uint64_t wait_ticks, int32_t *status,
                                  void *stream) {
  if (n_sweeps < 0 || n_slots < 0 || n_labels < 0) return fail(-1, "apc_diffusion_sweeps_resident: negative count");
  if (n_workgroups < 1 || n_workgroups > APC_SWEEP_MAX_WORKGROUPS)
    return fail(-1, "apc_diffusion_sweeps_resident: %lld workgroups, 1 .. %d can be resident", (long long)n_workgroups, APC_SWEEP_MAX_WORKGROUPS);
  if (lds_bytes < 1 || lds_bytes > APC_SWEEP_LDS_BYTES)
    return fail(-1, "apc_diffusion_sweeps_resident: %lld bytes of LDS, at most %d", (long long)lds_bytes, APC_SWEEP_LDS_BYTES);
  if (threads != 256 && threads != 512 && threads != 1024)
    return fail(-1, "apc_diffusion_sweeps_resident: workgroups of 256, 512 or 1024 threads (%d)", threads);
  if (!plan || !plan_begin || !theta || !unary || !theta_out || !unary_out || !status || (n_slots > 0 && !slots))
    return fail(-1, "apc_diffusion_sweeps_resident: NULL array");
  if (theta == theta_out || unary == unary_out) return fail(-1, "apc_diffusion_sweeps_resident: the outputs are arrays of their own");
  hipStream_t s = (hipStream_t)stream;
  const int64_t words = 4 * n_slots;  // two sets of two words
  const int64_t n = std::max<int64_t>({words, n_labels, 1});
  hipLaunchKernelGGL(resident_sweeps_begin_kernel, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0, s, slots, words, unary, unary_out, n_labels, status);
  // at least half a compute unit's LDS plus a little: one workgroup per compute unit
  const size_t lds = (size_t)std::max<int64_t>((lds_bytes + 15) / 16 * 16, 84 * 1024);
  const void *kernel = threads == 256   ? reinterpret_cast<const void *>(diffusion_resident_kernel<256>)
                       : threads == 512 ? reinterpret_cast<const void *>(diffusion_resident_kernel<512>)
                                        : reinterpret_cast<const void *>(diffusion_resident_kernel<1024>);
  hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return fail(-3, "apc_diffusion_sweeps_resident: %s", hipGetErrorString(e));
  const ResidentArgs a{plan, plan_begin, theta, unary, theta_out, unary_out, slots, n_slots, wait_ticks, status, n_sweeps};
  if (threads == 256) hipLaunchKernelGGL(diffusion_resident_kernel<256>, dim3((unsigned)n_workgroups), dim3(256), lds, s, a);
  else if (threads == 512) hipLaunchKernelGGL(diffusion_resident_kernel<512>, dim3((unsigned)n_workgroups), dim3(512), lds, s, a);
  else hipLaunchKernelGGL(diffusion_resident_kernel<1024>, dim3((unsigned)n_workgroups), dim3(1024), lds, s, a);
  return check_launch("apc_diffusion_sweeps_resident");
}

}  // extern "C"

// ------------------------------------------------------------------------------------------
// An entry point that allocates nothing and needs no caller-provided staging: the cost
// matrices straight from the tensor and strategy tables.  The staging tables the tile kernel
// reads (bytes and contiguity per tensor, compute cost / num_args per strategy; what
// apc_input_tables writes into caller arrays for apc_redistribute_tables) live in a file-scope
// device array of fixed size.  Every device holds its own copy of the array at its own address,
// looked up once per device; calls on one device share it, so calls that overlap on a device race.
// ------------------------------------------------------------------------------------------
constexpr int64_t kStaticMaxTensors = 1 << 16;     // 8 B + 1 B each
constexpr int64_t kStaticMaxStrategies = 1 << 21;  // 8 B each (compute cost / num_args)
constexpr size_t kStaticBytesOff = 0;
constexpr size_t kStaticPerArgOff = kStaticBytesOff + (size_t)kStaticMaxTensors * sizeof(int64_t);
constexpr size_t kStaticContigOff = kStaticPerArgOff + (size_t)kStaticMaxStrategies * sizeof(double);
constexpr size_t kStaticScratchBytes = kStaticContigOff + (size_t)kStaticMaxTensors;  // 17.1 MB
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

constexpr int kMaxDevices = 64;
static void *g_scratch_of_device[kMaxDevices];  // the array's device address, per device (0 = not looked up yet)

// The address of this device's copy of `scratch` (the array's name is only a host-side handle).
static int scratch_of_current_device(unsigned char **out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(-3, "hipGetDevice: %s", hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDevices) return fail(-1, "device %d outside [0, %d)", dev, kMaxDevices);
  void *p = __atomic_load_n(&g_scratch_of_device[dev], __ATOMIC_ACQUIRE);
  if (!p) {
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) return fail(-3, "hipGetSymbolAddress(scratch) on device %d: %s", dev, hipGetErrorString(e));
    __atomic_store_n(&g_scratch_of_device[dev], p, __ATOMIC_RELEASE);  // (every thread finds the same address)
  }
  *out = static_cast<unsigned char *>(p);
  return 0;
}

extern "C" {

int apc_redistribute_tables_static(const apc_params *params, int64_t n_tensors, const int32_t *rank, const int32_t *itemsize,
                                   const int64_t *shape, const int64_t *stride, int64_t n_strategies, const int64_t *flops,
                                   const int64_t *rw_bytes, const int8_t *dtype, const uint8_t *zero_cost,
                                   const int32_t *num_args, const uint32_t *spec_codes, const int32_t *spec_tensor,
                                   const double *pt_values, int64_t n_tiles, const apc_tile *tiles,
                                   const int64_t *dup_entry_begin, int64_t n_entries, double *comm_out, uint8_t *trans_out,
                                   double *cost_out, void *stream) {
  if (n_tensors < 0 || n_strategies < 0) return fail(-1, "apc_redistribute_tables_static: negative count");
  if (n_tensors > kStaticMaxTensors)
    return fail(-1, "apc_redistribute_tables_static: %lld tensors, the static staging holds %lld (use apc_input_tables + "
                "apc_redistribute_tables with caller-allocated staging)", (long long)n_tensors, (long long)kStaticMaxTensors);
  if (n_strategies > kStaticMaxStrategies)
    return fail(-1, "apc_redistribute_tables_static: %lld strategies, the static staging holds %lld (use apc_input_tables + "
                "apc_redistribute_tables with caller-allocated staging)", (long long)n_strategies,
                (long long)kStaticMaxStrategies);
  unsigned char *base = nullptr;
  if (int rc = scratch_of_current_device(&base)) return rc;
  int64_t *tensor_bytes = reinterpret_cast<int64_t *>(base + kStaticBytesOff);
  double *per_arg = reinterpret_cast<double *>(base + kStaticPerArgOff);
  uint8_t *tensor_contiguous = base + kStaticContigOff;
  // staging tables into the static array (no spec table, no per-strategy compute cost, no error
  // flag: a strategy with flops and an unsupported dtype shows as NaN costs), then the tiles;
  // both launches on the caller's stream, so the second sees what the first wrote
  const LaunchTo now{stream, nullptr};
  if (int rc = input_tables_impl(params, n_tensors, rank, itemsize, shape, stride, tensor_bytes, tensor_contiguous, 0, nullptr,
                                 nullptr, nullptr, nullptr, nullptr, 2, nullptr, nullptr, n_strategies, flops, rw_bytes, dtype,
                                 zero_cost, num_args, nullptr, per_arg, nullptr, now))
    return rc;
  return redistribute_tables_impl(params, tensor_bytes, tensor_contiguous, spec_codes, spec_tensor, pt_values, per_arg, n_tiles,
                                  tiles, dup_entry_begin, n_entries, comm_out, trans_out, cost_out, nullptr, now);
}

}  // extern "C"

// ------------------------------------------------------------------------------------------
// Packed tiles: launch.
// ------------------------------------------------------------------------------------------
static_assert(sizeof(apc_packed_tile) == 2752 && sizeof(apc_packed_tile) % 64 == 0, "apc_packed_tile layout");
static_assert(offsetof(apc_packed_tile, entry_begin) == 32 && offsetof(apc_packed_tile, tensor_shape) == 64,
              "the header is the record's first 64 bytes");

static int build_tables_packed_impl(const apc_params *params, int64_t n_tensors, const int32_t *rank, const int32_t *itemsize,
                            const int64_t *shape, const int64_t *stride, int64_t *tensor_bytes, uint8_t *tensor_contiguous,
                            int64_t n_strategies, const int64_t *flops, const int64_t *rw_bytes, const int8_t *dtype,
                            const uint8_t *zero_cost, const int32_t *num_args, double *compute, double *per_arg,
                            int32_t *error_flag, const double *pt_values, int64_t n_tiles, const apc_packed_tile *packed,
                            int64_t n_entries, double *cost_out, double *row_min, int32_t *row_argmin, int lanes,
                                    const LaunchTo &to) {
  if (int rc = check_params(params)) return rc;
  if (lanes != 16 && lanes != 32 && lanes != 64 && lanes != kBlock)
    return fail(-1, "apc_build_tables_packed: 16, 32, 64 or %d lanes a tile (got %d)", kBlock, lanes);
  if (n_tensors < 0 || n_strategies < 0 || n_entries < 0) return fail(-1, "apc_build_tables_packed: negative count");
  if (n_tiles < 0 || n_tiles > (1 << 30)) return fail(-1, "n_tiles %lld out of range", (long long)n_tiles);
  if (n_tensors > 0 && (!rank || !itemsize || !shape || !stride || !tensor_bytes || !tensor_contiguous))
    return fail(-1, "apc_build_tables_packed: NULL tensor array");
  if (n_strategies > 0 && (!flops || !rw_bytes || !dtype || !zero_cost || !num_args))
    return fail(-1, "apc_build_tables_packed: NULL strategy array");
  if (n_tiles > 0 && (!packed || !cost_out || !row_min || !row_argmin))
    return fail(-1, "apc_build_tables_packed: NULL tile records or outputs");
  if ((reinterpret_cast<uintptr_t>(packed) & 63) != 0) return fail(-1, "apc_build_tables_packed: packed tiles must be 64-byte aligned");
  const int xs = xcd_shift();
  const int64_t groups = blocks_for(n_tiles, kBlock / lanes);
  const int64_t tile_blocks = ((groups + (1 << xs) - 1) >> xs) << xs;
  const int64_t tb = blocks_for(n_tensors, kBlock), cb = blocks_for(n_strategies, kBlock);
  const int64_t blocks = tile_blocks + tb + cb;
  if (blocks == 0) return 0;
  if (blocks > INT32_MAX) return fail(-1, "apc_build_tables_packed: too many rows for one launch");
  const TermLayout lay = term_layout(*params);
  PackedArgs a{*params, row_min, row_argmin, pt_values, rank, itemsize, shape, stride, 1.0 / params->rescale, lay.exponents,
               lay.lg_total, {0, 0, 0, 0}};
  for (int i = 0; i < APC_MAX_MESH; ++i) a.lg[i] = lay.lg[i];
  const TensorTableArgs ta{n_tensors, rank, itemsize, shape, stride, tensor_bytes, tensor_contiguous};
  const ComputeCostArgs ca{n_strategies, flops, rw_bytes, dtype, zero_cost, num_args, compute, per_arg, error_flag};
  const PackedBlock block{a, *params, ta, ca, tb};
  using K = TableKernel<PackedBlock>;
#define APC_PACKED_FORM(M_, POW2_, LANES_) \
  K { build_tables_packed_kernel<M_, POW2_, false, LANES_>, build_tables_packed_kernel<M_, POW2_, true, LANES_> }
#define APC_PACKED_FORMS(M_, POW2_) \
  (lanes == 16 ? APC_PACKED_FORM(M_, POW2_, 16) : lanes == 32 ? APC_PACKED_FORM(M_, POW2_, 32) : lanes == 64 ? APC_PACKED_FORM(M_, POW2_, 64) : APC_PACKED_FORM(M_, POW2_, kBlock))
#define APC_LAUNCH_PACKED(M_)                                                                                                         \
  return launch_table_kernel("apc_build_tables_packed", to, lay.exponents ? APC_PACKED_FORMS(M_, true) : APC_PACKED_FORMS(M_, false), \
                             (unsigned)blocks, kBlock, 0, packed, (int)n_tiles, xs, tile_blocks, cost_out, block)
  switch (params->mesh_ndim) {
    case 1: APC_LAUNCH_PACKED(1);
    case 2: APC_LAUNCH_PACKED(2);
    case 3: APC_LAUNCH_PACKED(3);
    default: APC_LAUNCH_PACKED(4);
  }
#undef APC_LAUNCH_PACKED
#undef APC_PACKED_FORMS
#undef APC_PACKED_FORM
}

extern "C" {

int apc_build_tables_packed(const apc_params *params, int64_t n_tensors, const int32_t *rank, const int32_t *itemsize,
                            const int64_t *shape, const int64_t *stride, int64_t *tensor_bytes, uint8_t *tensor_contiguous,
                            int64_t n_strategies, const int64_t *flops, const int64_t *rw_bytes, const int8_t *dtype,
                            const uint8_t *zero_cost, const int32_t *num_args, double *compute, double *per_arg,
                            int32_t *error_flag, const double *pt_values, int64_t n_tiles, const apc_packed_tile *packed,
                            int64_t n_entries, double *cost_out, double *row_min, int32_t *row_argmin, void *stream) {
  return build_tables_packed_impl(params, n_tensors, rank, itemsize, shape, stride, tensor_bytes, tensor_contiguous, n_strategies,
                                  flops, rw_bytes, dtype, zero_cost, num_args, compute, per_arg, error_flag, pt_values, n_tiles, packed,
                                  n_entries, cost_out, row_min, row_argmin, kBlock, launch_to(stream));
}

int apc_build_tables_packed_small(const apc_params *params, int64_t n_tensors, const int32_t *rank, const int32_t *itemsize,
                            const int64_t *shape, const int64_t *stride, int64_t *tensor_bytes, uint8_t *tensor_contiguous,
                            int64_t n_strategies, const int64_t *flops, const int64_t *rw_bytes, const int8_t *dtype,
                            const uint8_t *zero_cost, const int32_t *num_args, double *compute, double *per_arg,
                            int32_t *error_flag, const double *pt_values, int64_t n_tiles, const apc_packed_tile *packed,
                            int64_t n_entries, double *cost_out, double *row_min, int32_t *row_argmin, int32_t lanes_per_tile, void *stream) {
  return build_tables_packed_impl(params, n_tensors, rank, itemsize, shape, stride, tensor_bytes, tensor_contiguous, n_strategies,
                                  flops, rw_bytes, dtype, zero_cost, num_args, compute, per_arg, error_flag, pt_values, n_tiles, packed,
                                  n_entries, cost_out, row_min, row_argmin, lanes_per_tile, launch_to(stream));
}

}  // extern "C"

// ------------------------------------------------------------------------------------------
// Measurement aids (no counterpart in the reference): what a launch costs on this system
// before it does any work, and what the store path gives a kernel that does nothing but write.
// A benchmark prices the table launches against both.
// ------------------------------------------------------------------------------------------
namespace {

__global__ void calibrate_empty_kernel() {}

// Workgroup b writes doubles [b * per_workgroup, (b + 1) * per_workgroup) of out (clipped to n),
// 16 bytes per lane and store instruction, consecutive lanes consecutive addresses.
// THROUGH: the stores are written through to memory (store_through), as the packed pass writes.
template <bool THROUGH>
__global__ __launch_bounds__(kBlock) void calibrate_fill_kernel(double *__restrict__ out, int64_t n, int64_t per_workgroup,
                                                                double value) {
  typedef double pair_t __attribute__((ext_vector_type(2)));
  const int64_t begin = (int64_t)blockIdx.x * per_workgroup;
  const int64_t end = begin + per_workgroup < n ? begin + per_workgroup : n;
  const pair_t v = {value, value};
  int64_t i = begin + 2 * (int64_t)threadIdx.x;
  for (; i + 1 < end; i += 2 * kBlock) {
    if (THROUGH) {
      __asm__ volatile("global_store_dwordx4 %0, %1, off sc0 sc1" ::"v"(out + i), "v"(v) : "memory");
    } else {
      *reinterpret_cast<pair_t *>(out + i) = v;
    }
  }
  if (i < end) {
    if (THROUGH) store_through(out + i, value);
    else out[i] = value;
  }
}

}  // namespace

extern "C" {

int apc_calibrate_launch(int64_t n_workgroups, int32_t threads, void *stream) {
  if (n_workgroups < 1 || n_workgroups > INT32_MAX || threads < 1 || threads > 1024)
    return fail(-1, "apc_calibrate_launch: %lld workgroups of %d threads", (long long)n_workgroups, threads);
  hipLaunchKernelGGL(calibrate_empty_kernel, dim3((unsigned)n_workgroups), dim3((unsigned)threads), 0, (hipStream_t)stream);
  return check_launch("apc_calibrate_launch");
}

int apc_calibrate_fill(double *out, int64_t n, int64_t per_workgroup, double value, int32_t write_through, void *stream) {
  if (n < 0 || per_workgroup < 2 || (per_workgroup & 1)) return fail(-1, "apc_calibrate_fill: n >= 0, per_workgroup even and >= 2");
  if (n == 0) return 0;
  if (!out) return fail(-1, "apc_calibrate_fill: NULL array");
  if ((reinterpret_cast<uintptr_t>(out) & 15) != 0) return fail(-1, "apc_calibrate_fill: out must be 16-byte aligned");
  const int64_t blocks = (n + per_workgroup - 1) / per_workgroup;
  if (blocks > INT32_MAX) return fail(-1, "apc_calibrate_fill: too many workgroups");
  if (write_through)
    hipLaunchKernelGGL(calibrate_fill_kernel<true>, dim3((unsigned)blocks), dim3(kBlock), 0, (hipStream_t)stream, out, n,
                       per_workgroup, value);
  else
    hipLaunchKernelGGL(calibrate_fill_kernel<false>, dim3((unsigned)blocks), dim3(kBlock), 0, (hipStream_t)stream, out, n,
                       per_workgroup, value);
  return check_launch("apc_calibrate_fill");
}

}  // extern "C"
