// What the device headers of one workgroup's routines need to compile for the
// host, a workgroup's lanes being fibers.
#pragma once
#include <cmath>
#include <cstdint>
#include <cstring>

#define __host__
#define __device__
#define __forceinline__ inline

struct HostIndex { unsigned x, y, z; };
struct HostLane { HostIndex thread, block_dim; };
HostLane &host_lane();
#define threadIdx (host_lane().thread)
#define blockDim (host_lane().block_dim)

void host_barrier(int line);                          // barriers are told apart by their source line
uint64_t host_exchange(uint64_t value, int source);   // the value of lane `source` of this wave
uint64_t host_ballot(bool p);
#define __syncthreads() host_barrier(__LINE__)
#define __ballot(p) host_ballot(p)
inline int __popcll(unsigned long long x) { return __builtin_popcountll(x); }
inline int __ffsll(long long x) { return __builtin_ffsll(x); }
int host_lane_id();
template <typename T> T __shfl(T v, int source, int) {
    uint64_t u = 0;
    std::memcpy(&u, &v, sizeof(T));
    u = host_exchange(u, source);
    std::memcpy(&v, &u, sizeof(T));
    return v;
}
template <typename T> T __shfl_xor(T v, int mask, int width) { return __shfl(v, host_lane_id() ^ mask, width); }

// in routines of the headers that the tests do not call
#define __HIP_MEMORY_SCOPE_AGENT 0
#define __hip_atomic_load(p, order, scope) (*(p))
#define __builtin_amdgcn_s_sleep(n) ((void)0)
#define __builtin_amdgcn_fence(order, scope) ((void)0)
