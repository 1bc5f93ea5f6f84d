// A workgroup of 64-lane waves on the CPU, for tests of device code: what the
// headers of suitesparse_amd/csrc use of <hip/hip_runtime.h>.
//
// Every lane is a fiber.  A wave's lanes meet at each cross-lane operation
// (readlane, ballot, MFMA, wave barrier), as its lockstep execution orders them;
// between two workgroup barriers the waves run one after the other, each to the
// barrier before the next starts, in an order that the test chooses.  A read
// and a write of one LDS entry by two waves without a barrier between them give
// one result in one order and another in the reverse of it.
#pragma once
#include <limits.h>
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <ucontext.h>

#include <algorithm>
#include <functional>
#include <type_traits>
#include <vector>

#define __device__
#define __host__
#define __global__
#define __shared__ static
#define __forceinline__ inline
#define __launch_bounds__(...)

using std::max;
using std::min;
using std::isnan;

struct Dim3 { unsigned x, y, z; };
inline Dim3 threadIdx{0, 0, 0}, blockIdx{0, 0, 0}, blockDim{256, 1, 1}, gridDim{1, 1, 1};

namespace emu {

enum State { RUN, WAVE, BARRIER, DONE };
constexpr int THREADS = 256;

struct Lane {
    ucontext_t ctx;
    std::vector<char> stack;
    State state;
    unsigned ops;                         // cross-lane operations so far: which exchange buffer is in use
    bool released;                        // a device-scope release since the last cross-lane operation
};

inline Lane lanes[THREADS];
inline ucontext_t host;
inline int cur = 0;
inline std::function<void()> body;
struct Slot { double a, b; };
inline Slot slots[THREADS / 64][2][64];

inline void yield(State s) {
    lanes[cur].state = s;
    swapcontext(&lanes[cur].ctx, &host);
}

inline void entry() {
    body();
    lanes[cur].state = DONE;
    swapcontext(&lanes[cur].ctx, &host);
}

// every lane's (a, b), once all 64 have come here
inline const Slot *exchange(double a, double b = 0) {
    lanes[cur].released = false;
    const int w = cur >> 6, l = cur & 63, q = lanes[cur].ops++ & 1;
    slots[w][q][l] = Slot{a, b};
    yield(WAVE);
    return slots[w][q];
}

// run `f` in a workgroup, its waves in the given order between barriers
inline void run(const int (&order)[THREADS / 64], const std::function<void()> &f) {
    body = f;
    for (int t = 0; t < THREADS; t++) {
        Lane &L = lanes[t];
        L.stack.resize(256 << 10);
        L.state = RUN;
        L.ops = 0;
        L.released = false;
        getcontext(&L.ctx);
        L.ctx.uc_stack.ss_sp = L.stack.data();
        L.ctx.uc_stack.ss_size = L.stack.size();
        L.ctx.uc_link = &host;
        makecontext(&L.ctx, (void (*)())entry, 0);
    }
    for (;;) {
        for (int w : order) {
            Lane *W = lanes + 64 * w;
            while (W[0].state == RUN) {
                for (int l = 0; l < 64; l++) {
                    cur = 64 * w + l;
                    threadIdx.x = cur;
                    swapcontext(&host, &lanes[cur].ctx);
                }
                for (int l = 1; l < 64; l++)
                    if (W[l].state != W[0].state) {
                        printf("wave %d: lanes 0 and %d part at a cross-lane operation\n", w, l);
                        exit(2);
                    }
                if (W[0].state == WAVE)
                    for (int l = 0; l < 64; l++) W[l].state = RUN;
            }
        }
        for (int t = 1; t < THREADS; t++)
            if (lanes[t].state != lanes[0].state) {
                printf("waves 0 and %d part at a barrier\n", t >> 6);
                exit(2);
            }
        if (lanes[0].state == DONE) return;
        for (Lane &L : lanes) L.state = RUN;
    }
}

// A release at a barrier or by one wave orders that wave's own stores only: a
// flag that says to other workgroups that this one's stores are done needs a
// device-scope release of every wave before it.
inline int unreleased_flags = 0;          // flags stored while a lane had none

inline void fence(int order, const char *scope) {
    if (order == __ATOMIC_RELEASE && !strcmp(scope, "agent")) lanes[cur].released = true;
}

template <typename T>
void atomic_store(T *p, T v, int order, int scope) {
    if (scope == 1 && order == __ATOMIC_RELEASE)
        for (const Lane &L : lanes) unreleased_flags += !L.released;
    *p = v;
}

inline int readlane(int v, int k) { return (int)exchange(v)[k].a; }

inline unsigned long long ballot(bool p) {
    const Slot *s = exchange(p);
    unsigned long long m = 0;
    for (int l = 0; l < 64; l++) m |= (unsigned long long)(s[l].a != 0) << l;
    return m;
}

// D(m, n) += sum_k A(m, k) B(k, n): lane l gives A(l % 16, l / 16) and
// B(l / 16, l % 16), and holds D(row(l, v), l % 16)
template <typename T, typename V>
V mfma16x16x4(T a, T b, V c) {
    const int l = cur & 63;
    const Slot *s = exchange(a, b);
    for (int v = 0; v < 4; v++) {
        const int m = std::is_same<T, double>::value ? (l >> 4) + 4 * v : 4 * (l >> 4) + v;
        for (int k = 0; k < 4; k++) c[v] += (T)s[m + 16 * k].a * (T)s[(l & 15) + 16 * k].b;
    }
    return c;
}

template <typename V, typename H>
V not_emulated(H, H, V c) {
    abort();
    return c;
}

}  // namespace emu

#define __syncthreads() emu::yield(emu::BARRIER)
#define __ballot(p) emu::ballot(p)
#define __threadfence()
#define __builtin_amdgcn_readlane(v, k) emu::readlane(v, k)
#define __builtin_amdgcn_readfirstlane(v) emu::readlane(v, 0)
#define __builtin_amdgcn_wave_barrier() (void)emu::exchange(0)
#define __builtin_amdgcn_fence(order, scope) emu::fence(order, scope)
#define __builtin_amdgcn_sched_barrier(x)
#define __builtin_amdgcn_s_setprio(x)
#define __builtin_amdgcn_s_sleep(x)
#define __builtin_amdgcn_rsq(x) (1.0 / sqrt(x))
#define __builtin_amdgcn_rsqf(x) (1.0f / sqrtf(x))
#define __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, x, y, z) emu::mfma16x16x4<double>(a, b, c)
#define __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, x, y, z) emu::mfma16x16x4<float>(a, b, c)
#define __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, x, y, z) emu::not_emulated(a, b, c)
#define __HIP_MEMORY_SCOPE_AGENT 1
#define __HIP_MEMORY_SCOPE_WORKGROUP 0
#define __hip_atomic_store(p, v, order, scope) emu::atomic_store(p, v, order, scope)
#define __hip_atomic_load(p, order, scope) (*(p))
#define __hip_atomic_fetch_add(p, v, order, scope) (*(p) += (v))

template <typename T> T unsafeAtomicAdd(T *p, T v) { T o = *p; *p += v; return o; }
inline int atomicAdd(int *p, int v) { int o = *p; *p += v; return o; }
inline int atomicMin(int *p, int v) { int o = *p; *p = min(o, v); return o; }

inline int __double2loint(double v) { int64_t u; memcpy(&u, &v, 8); return (int)u; }
inline int __double2hiint(double v) { int64_t u; memcpy(&u, &v, 8); return (int)(u >> 32); }
inline double __hiloint2double(int hi, int lo) {
    uint64_t u = (uint64_t)(uint32_t)hi << 32 | (uint32_t)lo;
    double v;
    memcpy(&v, &u, 8);
    return v;
}
inline int __float_as_int(float v) { int u; memcpy(&u, &v, 4); return u; }
inline float __int_as_float(int u) { float v; memcpy(&v, &u, 4); return v; }
