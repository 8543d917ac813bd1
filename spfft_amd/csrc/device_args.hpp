// Device-side helpers shared by the kernels that take FastArgs: argument
// tables in device memory, 32-bit addressing and the LDS barrier.
#pragma once

#include <hip/hip_runtime.h>

#include "fast_kernels.hpp"

namespace spfft {
namespace dev {

// Element `i` of an array smaller than 4 GiB, addressed with a 32-bit byte
// offset (lets the compiler use a scalar base and one offset register).
template <typename X>
__device__ __forceinline__ X at32(const X* base, int i) {
  const unsigned off = static_cast<unsigned>(i) * static_cast<unsigned>(sizeof(X));
  return *reinterpret_cast<const X*>(reinterpret_cast<const char*>(base) + off);
}

// Arguments read from a device table hold generic pointers, so the compiler
// would access them with flat instructions (which share the LDS counter and
// serialise against LDS traffic). Rebasing each pointer on a kernel argument
// (a global pointer) keeps the address and lets the accesses be global ones.
// A null pointer stays null (no offset is formed from it).
template <typename P>
__device__ __forceinline__ P* rebase(const char* anchor, P* p) {
  if (p == nullptr) return nullptr;
  return (P*)(anchor + (reinterpret_cast<const char*>(p) - anchor));
}
template <typename T>
__device__ __forceinline__ FastArgs<T> on_global(FastArgs<T> a, const void* table) {
  const char* g = static_cast<const char*>(table);
  a.zbuf = rebase(g, a.zbuf);
  a.in = rebase(g, a.in);
  a.out = rebase(g, a.out);
  a.stickCell = rebase(g, a.stickCell);
  a.columnSticks = rebase(g, a.columnSticks);
  a.trig = rebase(g, static_cast<const char*>(a.trig));
  a.stickBegin = rebase(g, a.stickBegin);
  a.colX = rebase(g, a.colX);
  a.stickAt = rebase(g, a.stickAt);
  a.zEntries = rebase(g, a.zEntries);
  a.zInfo = rebase(g, a.zInfo);
  a.xCol = rebase(g, a.xCol);
  a.resSticks = rebase(g, a.resSticks);
  a.resBegin = rebase(g, a.resBegin);
  a.resYM = rebase(g, a.resYM);
  a.ybuf = rebase(g, a.ybuf);
  a.twX = rebase(g, a.twX);
  a.twY = rebase(g, a.twY);
  a.twZ = rebase(g, a.twZ);
  return a;
}

// Workgroup barrier for LDS data: waits for this wave's LDS operations only.
// __syncthreads() releases at workgroup scope for all memory, which waits for
// every global load and store in flight (loads issued ahead of the barrier
// would land before it). No kernel here passes data between waves through
// global memory.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Before and after the streaming stores of one of two branches: the compiler
// would hoist or sink the stores of both into one plain store.
__device__ __forceinline__ void apart() { asm volatile(""); }

// Streaming store (no cache allocation on the way to HBM): for results that no
// later kernel of the chain reads while they could still be cached.
template <typename T>
__device__ __forceinline__ void store_stream(T* p, T v) {
  __builtin_nontemporal_store(v, p);
}
template <typename T>
__device__ __forceinline__ void store_stream(Cx<T>* p, Cx<T> v) {
  __builtin_nontemporal_store(v.re, &p->re);
  __builtin_nontemporal_store(v.im, &p->im);
}

template <typename T>
__device__ __forceinline__ T load_stream(const T* p) {
  return __builtin_nontemporal_load(p);
}
template <typename T>
__device__ __forceinline__ Cx<T> load_stream(const Cx<T>* p) {
  return Cx<T>{__builtin_nontemporal_load(&p->re), __builtin_nontemporal_load(&p->im)};
}

}  // namespace dev

}  // namespace spfft
