// Stand-in for the HIP runtime header in a CPU build of the kernel sources, in
// which every buffer load and store is checked against its resource
// (test_kernel_bounds.py).  The threads of a workgroup take turns from barrier
// to barrier; cross-lane operations return the lane's own value, products add
// nothing, buffer loads return zeros, and what is left is the control flow and
// the address arithmetic, which depend on the launch arguments and the thread
// index alone.
#pragma once
#include <cmath>
#include <cstddef>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <vector>

#include <ucontext.h>

#define __global__
#define __device__
#define __host__
#define __forceinline__ inline
#define __shared__ static
#define __restrict__
#define __launch_bounds__(...)

typedef void* hipStream_t;
struct dim3 {
    unsigned x, y, z;
    dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {}
};
inline dim3 threadIdx, blockIdx, blockDim, gridDim;
struct uint2 { unsigned x, y; };
struct uint4 { unsigned x, y, z, w; };
struct int4 { int x, y, z, w; };
inline uint2 make_uint2(unsigned x, unsigned y) { return {x, y}; }
inline int4 make_int4(int x, int y, int z, int w) { return {x, y, z, w}; }

inline int min(int a, int b) { return a < b ? a : b; }
inline int max(int a, int b) { return a < b ? b : a; }
inline unsigned min(unsigned a, unsigned b) { return a < b ? a : b; }
inline unsigned max(unsigned a, unsigned b) { return a < b ? b : a; }
inline long long min(long long a, long long b) { return a < b ? a : b; }
inline unsigned long long min(unsigned long long a, unsigned long long b) { return a < b ? a : b; }

inline int __shfl(int v, int, int) { return v; }
inline int __shfl_xor(int v, int, int) { return v; }
inline int __shfl_up(int v, int, int) { return v; }
inline int __mul24(int a, int b) { return a * b; }
inline unsigned __umul24(unsigned a, unsigned b) { return a * b; }
inline int __clz(int x) { return x ? __builtin_clz((unsigned)x) : 32; }

namespace bounds {
typedef int i4 __attribute__((ext_vector_type(4)));
typedef int i2 __attribute__((ext_vector_type(2)));
typedef unsigned u2 __attribute__((ext_vector_type(2)));
struct Rsrc {
    const void* base;
    unsigned n;
};
inline long accesses = 0, bad = 0;
// No access may need the range check to take the scalar offset into account
// (it is specified for the vector offset): either the vector offset alone lies
// past the end, or the whole access lies inside; and the scalar offset alone
// never passes the end.
inline void check(const Rsrc& r, int voff, int soff, unsigned bytes) {
    accesses++;
    const unsigned long long v = (unsigned)voff, s = (unsigned)soff;
    if (s <= r.n && (v >= r.n || v + s + bytes <= r.n)) return;
    if (bad++ < 3)
        std::printf("out of range: vector offset %llu, scalar offset %llu, %u bytes of %u (block %u, thread %u)\n", v, s, bytes,
                    r.n, blockIdx.x, threadIdx.x);
}
inline i4 load128(const Rsrc& r, int v, int s, int) { check(r, v, s, 16); return (i4){0, 0, 0, 0}; }
inline u2 load64(const Rsrc& r, int v, int s, int) { check(r, v, s, 8); return (u2){0, 0}; }
inline int load32(const Rsrc& r, int v, int s, int) { check(r, v, s, 4); return 0; }
template <class P>
void load_lds(const Rsrc& r, P, int bytes, int v, int s, int, int) { check(r, v, s, (unsigned)bytes); }
template <unsigned BYTES, class T>
void store(const T&, const Rsrc& r, int v, int s, int) { check(r, v, s, BYTES); }
template <class Op>
i4 mfma(Op, Op, i4 c, int, int, int) { return c; }
inline u2 swap2(unsigned a, unsigned b) { return (u2){a, b}; }
// the running workgroup: a context per thread, and whether it has ended
inline ucontext_t scheduler, *current;
inline bool ended;
inline void barrier() { swapcontext(current, &scheduler); }
template <class K>
void thread_main(unsigned lo, unsigned hi) {
    (*(K*)(((uintptr_t)hi << 32) | lo))();
    ended = true;
    setcontext(&scheduler);
}
template <class K>
void launch(dim3 grid, dim3 block, K kernel) {
    constexpr size_t STACK = 128 << 10;
    static const std::unique_ptr<char[]> stacks(new char[1024 * STACK]);
    std::vector<ucontext_t> ctx(block.x);
    std::vector<unsigned> live;
    gridDim = grid;
    blockDim = block;
    for (unsigned b = 0; b < grid.x * grid.y; b++) {
        blockIdx = dim3(b % grid.x, b / grid.x);
        live.clear();
        for (unsigned t = 0; t < block.x; t++) {
            getcontext(&ctx[t]);
            ctx[t].uc_stack.ss_sp = &stacks[t * STACK];
            ctx[t].uc_stack.ss_size = STACK;
            ctx[t].uc_link = nullptr;
            const uintptr_t k = (uintptr_t)&kernel;
            makecontext(&ctx[t], (void (*)())thread_main<K>, 2, (unsigned)k, (unsigned)(k >> 32));
            live.push_back(t);
        }
        while (!live.empty()) {
            std::vector<unsigned> next;
            for (unsigned t : live) {
                threadIdx = dim3(t);
                current = &ctx[t];
                ended = false;
                swapcontext(&scheduler, current);
                if (!ended) next.push_back(t);
            }
            live.swap(next);
        }
    }
}
}  // namespace bounds

inline void __syncthreads() { bounds::barrier(); }

#define hipLaunchKernelGGL(K, G, B, SH, S, ...) bounds::launch(G, B, [&] { (K)(__VA_ARGS__); })
#define __amdgpu_buffer_rsrc_t bounds::Rsrc
#define __builtin_amdgcn_make_buffer_rsrc(P, STRIDE, N, FLAGS) (bounds::Rsrc{(P), (unsigned)(N)})
#define __builtin_amdgcn_raw_buffer_load_b128 bounds::load128
#define __builtin_amdgcn_raw_buffer_load_b64 bounds::load64
#define __builtin_amdgcn_raw_buffer_load_b32 bounds::load32
#define __builtin_amdgcn_raw_ptr_buffer_load_lds bounds::load_lds
#define __builtin_amdgcn_raw_buffer_store_b128 bounds::store<16>
#define __builtin_amdgcn_raw_buffer_store_b64 bounds::store<8>
#define __builtin_amdgcn_raw_buffer_store_b8 bounds::store<1>
#define __builtin_amdgcn_mfma_i32_16x16x64_i8 bounds::mfma
#define __builtin_amdgcn_mfma_i32_16x16x32_i8 bounds::mfma
#define __builtin_amdgcn_sdot4(A, B, C, CLAMP) (C)
#define __builtin_amdgcn_readfirstlane(X) ((int)(X))
#define __builtin_amdgcn_readlane(X, L) ((int)(X))
#define __builtin_amdgcn_update_dpp(OLD, X, A, B, C, D) ((int)(X))
#define __builtin_amdgcn_perm(A, B, S) ((unsigned)(A))
#define __builtin_amdgcn_permlane32_swap(A, B, C, D) bounds::swap2(A, B)
#define __builtin_amdgcn_permlane16_swap(A, B, C, D) bounds::swap2(A, B)
#define __builtin_amdgcn_ballot_w64(X) ((void)(X), 1ull)
#define __builtin_amdgcn_sqrtf(X) std::sqrt(X)
#define __builtin_amdgcn_rcpf(X) (1.0f / (X))
#define __builtin_amdgcn_sched_barrier(X)
#define __builtin_amdgcn_sched_group_barrier(A, B, C)
#define __builtin_amdgcn_s_waitcnt(X)
#define __builtin_amdgcn_s_setprio(X)
#define __builtin_amdgcn_s_barrier() bounds::barrier()
#define __builtin_amdgcn_fence(...)
