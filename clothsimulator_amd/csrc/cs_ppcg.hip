// cs_ppcg.hip — PCG of whole systems in one launch, the matrix held in registers.
//
// A separately launched iteration (cs_pcg.hip) of a system of 16,641 rows or fewer takes 13-14 us,
// nearly all of it latency: two kernel boundaries, and in each kernel a chain of dependent loads.
// The chip's registers hold the matrices of 131,072 rows: here a thread owns one row for the whole
// solve and keeps its 3x3 blocks (RS of them), its columns as 16-bit offsets, and its r, x, z, d, q
// in registers.  An iteration then moves only vectors: a thread publishes its z and d and gathers
// its neighbours'.
//
// A system is solved by a group of workgroups, T rows each, that meet twice an iteration: when
// z and the partials of r.z and r.r are out, and when the partial of d.q is.  The meeting is an
// all-reduce: each workgroup stores (epoch, value) words to its slots, every workgroup polls all
// slots of its group, and forms the sums in the order of the separate launches: the solve gives
// their bits, whatever it shares a launch with (1.0 us for 2 workgroups, 1.4 us for 17, 2.9 us for 256; a
// cooperative-groups grid barrier took 700 us for 1,536 because every wave wrote its L2 back).
// No L2 write-back is needed: what others read is stored with agent-scope atomic stores, which
// write through.  Groups are independent, so one launch solves many systems.
//
// The whole solve is in the kernel: start, iterations, the check of the true residual with FP64 row
// sums and the continuations from it, as pcg_solve's.  The workgroups of a group wait for each
// other, so they must all be resident: launches are cooperative and no larger than the device
// holds at once.  One process at a time gets a device's cooperative queue: where the launch is
// refused, and if a wait (each is bounded in time) runs out, the solve is made with separate launches, and
// so are the context's next ones for a while (OneLaunch).
//
// The preconditioner is part of the kernel: block Jacobi in the update; the learned factor's two
// sweeps; or the multigrid cycle with the rows of each coarse level spread over the group's waves, a
// meeting per phase (restriction, pre-smoothing with residual, post-smoothing) instead of a launch.
//
// Measured, solves with their set-up in ms (iterations), separate launches -> here:
//   rows, regular grid   block Jacobi             learned factor          multigrid
//   289                  1.08 -> 0.29 (81)        0.88 -> 0.57 (31)       0.96 -> 0.68 (19)
//   1,089                1.39 -> 0.57 (104)       1.43 -> 0.90 (56)       0.94 -> 0.69 (24)
//   16,641               4.32 -> 2.34 (318)       3.49 -> 2.55 (141)      2.38 -> 1.87 (39)
//   65,536               7.90 -> 3.78 (400)       8.16 -> 5.73 (242)      3.96 -> 3.20 (48)
//   131,044              23.4 -> 14.8 (1,074)     (launched)              (launched)
//   rows, irregular mesh (17 to 20 blocks a row, those beyond the registers' 14 streamed)
//   1,089                1.81 -> 0.82 (127)       1.99 -> 1.46 (69)       1.48 -> 1.07 (35)
//   16,641               5.42 -> 3.13 (356)       6.17 -> 4.50 (190)      3.70 -> 2.67 (45)
//   65,536               8.74 -> 4.65 (400)       10.8 -> 9.68 (270)      6.03 -> 5.05 (61)
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstring>
#include <type_traits>

#include "cs_kernels.hpp"
#include "cs_math.hpp"

namespace cs {

namespace {

enum { PRE_JACOBI = 0, PRE_LEARNED = 1, PRE_AMG = 2 };
constexpr int RESTARTS = 4;                      // continuations from the true residual, as pcg_solve
constexpr unsigned long long WAIT_TICKS = 200000000ull;  // 2 s of the 100 MHz wall clock; a wait's bound

// One level of a cloth's multigrid hierarchy (cs_amg.hip); agg, mptr, midx lead to the next level.
struct PLev {
    int n, pad;
    const int *rp, *ci, *agg, *mptr, *midx;
    const float *val, *Dinv;
    float *b, *x, *t;  // right-hand side, pre-smoothed iterate, residual and then result
};
constexpr int MAXL = 12;
constexpr int BOTTOM = 512;  // nodes of the level solved by a dense operator, at most

struct PSys {
    int nn, nslices, G, contacts;
    const int *sliceOff, *sliceW, *cols, *cRowPtr, *cCol;
    const float *vals, *cVal, *Minv, *b, *bc;
    float* x;
    float4 *z, *d;      // z: nn, d: two generations of nn
    uint64_t* slots;    // 2 generations x 2 values x (G * T / BLK) words (epoch << 32 | value), zero at launch
    PcgScalars* out;
    // learned factor: bf16 blocks in the value layout, diagonal slot and length of each row, y = G r
    const int *diagSlot, *rowLen;
    const uint16_t* Gf;
    float4* y;
    // multigrid: levels 0 .. bottom, the bottom's dense operator (3 n rows) and result, level 0's A P
    int bottom, pad2;
    const float* op;
    float* eBottom;
    const int *apSliceOff, *apSliceW, *apCols;
    const float* apVals;
    int loseWg, loseAt;  // (testing) a wait of workgroup loseWg counts as run out at this meeting, 0: none
    PLev L[MAXL];
};

// The pointers in the global address space (cs_math.hpp, G1)
struct PSysG {
    int nn, nslices, G, contacts;
    const G1<int> *sliceOff, *sliceW, *cols, *cRowPtr, *cCol;
    const G1<float> *vals, *cVal, *Minv, *b, *bc;
    G1<float>* x;
    G1<f4n> *z, *d;
    G1<uint64_t>* slots;
    PcgScalars* out;
    const G1<int> *diagSlot, *rowLen;
    const G1<uint16_t>* Gf;
    G1<f4n>* y;
};
__device__ __forceinline__ PSysG gview(const PSys& c) {
    PSysG g;
    g.nn = c.nn;
    g.nslices = c.nslices;
    g.G = c.G;
    g.contacts = c.contacts;
    g.sliceOff = g1(c.sliceOff); g.sliceW = g1(c.sliceW); g.cols = g1(c.cols);
    g.cRowPtr = g1(c.cRowPtr); g.cCol = g1(c.cCol);
    g.vals = g1(c.vals); g.cVal = g1(c.cVal); g.Minv = g1(c.Minv); g.b = g1(c.b); g.bc = g1(c.bc);
    g.x = g1(c.x);
    g.z = (G1<f4n>*)c.z;
    g.d = (G1<f4n>*)c.d;
    g.slots = g1(c.slots);
    g.out = c.out;
    g.diagSlot = g1(c.diagSlot);
    g.rowLen = g1(c.rowLen);
    g.Gf = g1(c.Gf);
    g.y = (G1<f4n>*)c.y;
    return g;
}

// A level's pointers in the global address space
struct PLevG {
    int n;
    const G1<int> *rp, *ci, *agg, *mptr, *midx;
    const G1<float> *val, *Dinv;
    G1<float> *b, *x, *t;
};
__device__ __forceinline__ PLevG gview(const PLev& c) {
    PLevG g;
    g.n = c.n;
    g.rp = g1(c.rp); g.ci = g1(c.ci); g.agg = g1(c.agg); g.mptr = g1(c.mptr); g.midx = g1(c.midx);
    g.val = g1(c.val); g.Dinv = g1(c.Dinv);
    g.b = g1(c.b); g.x = g1(c.x); g.t = g1(c.t);
    return g;
}

__device__ __forceinline__ void put64(G1<uint64_t>* p, uint64_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t get64(const G1<uint64_t>* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// publishes a row's vector for the other workgroups
__device__ __forceinline__ void put3(G1<f4n>* p, V3f a) {
    G1<uint64_t>* q = (G1<uint64_t>*)p;
    put64(q, (uint64_t)__float_as_uint(a.y) << 32 | __float_as_uint(a.x));
    put64(q + 1, __float_as_uint(a.z));
}

// the same into an array of three floats a row
__device__ __forceinline__ void put3f(G1<float>* p, V3f a) {
    __hip_atomic_store(p, a.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(p + 1, a.y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(p + 2, a.z, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Element at a 32-bit byte offset from a uniform base: one scalar base and one offset register
// per access (systems here stay far below 4 GB).
template <class V> __device__ __forceinline__ G1<V>& at(G1<V>* base, unsigned byte) {
    return *(G1<V>*)((G1<char>*)base + byte);
}
template <class V> __device__ __forceinline__ const G1<V>& at(const G1<V>* base, unsigned byte) {
    return *(const G1<V>*)((const G1<char>*)base + byte);
}
// A value the compiler cannot see through: addresses formed from it are recomputed at each use
// (formed ahead of the iterations they would not fit the registers).
__device__ __forceinline__ int opaque(int q) {
    asm volatile("" : "+v"(q));
    return q;
}
typedef float f3n __attribute__((ext_vector_type(3)));

constexpr int BLK = 256;     // rows of one partial sum

// A workgroup's waits, in LDS (registers are short)
struct Wait {
    unsigned long long ticks;  // bound of one
    unsigned ranOut;           // the meeting at which one ran out (they count from 1)
};

struct Group {
    G1<uint64_t>* slots;
    float* lds;  // 2 * (T / 64 + 4) floats
    Wait* wait;
    int G, wg;
    unsigned epoch;
};

// Sums v over the group; every thread of every workgroup gets the same sums.  The order of the sum is
// that of the separate launches (cs_pcg.hip) and depends on the rows alone, not on T or on how many
// systems share the launch: a partial per 256 rows (64 by a shuffle tree, four of those pairwise),
// partials t, t + 256, .. to lane t of 256, and those 256 as the rows of a partial.  On return all
// stores that any thread of the group made before the call are visible to every thread.  False if the
// wait ran out (the same in every thread of the workgroup).  PUBLISH false: only the sums are
// exchanged; stores made before become visible at the next meeting with PUBLISH.
template <int T, int NS, bool PUBLISH = true, bool LOCAL = false>
__device__ __forceinline__ bool meet(Group& g, float (&v)[NS]) {
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr int NW = T / 64, NB = T / BLK;  // waves, partials per workgroup
#pragma unroll
    for (int s = 0; s < NS; s++)
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v[s] += __shfl_xor(v[s], o, 64);
    if (lane == 0)
#pragma unroll
        for (int s = 0; s < NS; s++) g.lds[NW * s + wave] = v[s];
    if (PUBLISH) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's published vectors are out
    __syncthreads();
    auto partial = [&](int s, int b) {
        const float* w = g.lds + NW * s + 4 * b;
        return (w[0] + w[1]) + (w[2] + w[3]);
    };
    if (g.G == 1) {
#pragma unroll
        for (int s = 0; s < NS; s++) {
            v[s] = partial(s, 0);
#pragma unroll
            for (int b = 1; b < NB; b++) v[s] += partial(s, b);
        }
        if (PUBLISH && !LOCAL && tid == 0) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        __syncthreads();
        return true;
    }
    const unsigned ep = ++g.epoch;
    const int n = g.G * NB;  // slots per value
    G1<uint64_t>* gen = g.slots + (ep & 1) * 2 * n;
    if (tid < NS * NB) {
        const int s = tid / NB, b = tid % NB;
        put64(&at(gen, 8u * (s * n + g.wg * NB + b)), (uint64_t)ep << 32 | __float_as_uint(partial(s, b)));
    }
    // the 256 lanes are four waves' worth; a wave polls its lanes' slots
    float* sums = g.lds + 2 * NW;
    unsigned long long since = 0;
    for (int c = wave; c < 4; c += NW) {
        float a[NS];
#pragma unroll
        for (int s = 0; s < NS; s++) a[s] = 0.0f;
        for (int t = 64 * c + lane; t < n; t += BLK) {
            uint64_t w[NS];
            bool late = false;
            for (int spin = 0;; spin++) {
                bool all = true;
#pragma unroll
                for (int s = 0; s < NS; s++) {
                    w[s] = get64(&at(gen, 8u * (s * n + opaque(t))));
                    all = all && (unsigned)(w[s] >> 32) == ep;
                }
                if (all) break;
                if (late) {
                    g.wait->ranOut = ep;
                    break;
                }
                if ((spin & 1023) == 1023) {
                    const unsigned long long now = wall_clock64();
                    if (since == 0) since = now;
                    late = now - since > g.wait->ticks;  // the words are read once more after the deadline
                }
            }
#pragma unroll
            for (int s = 0; s < NS; s++) a[s] += __uint_as_float((unsigned)w[s]);
        }
        if (64 * c < n)
#pragma unroll
            for (int s = 0; s < NS; s++)
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) a[s] += __shfl_xor(a[s], o, 64);
        if (lane == 0)
#pragma unroll
            for (int s = 0; s < NS; s++) sums[4 * s + c] = a[s];
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < NS; s++) v[s] = (sums[4 * s] + sums[4 * s + 1]) + (sums[4 * s + 2] + sums[4 * s + 3]);
    const bool ok = g.wait->ranOut != ep;
    // vectors cached from before the meeting are dropped (one wave: the caches are the CU's and
    // the XCD's), before any thread goes on to gather
    if (PUBLISH && tid == 0) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    __syncthreads();
    return ok;
}

template <class P> __device__ __forceinline__ V3f ld3v(P p, int i) { return mk(p[3 * i], p[3 * i + 1], p[3 * i + 2]); }
__device__ __forceinline__ V3f v3(float4 a) { return mk(a.x, a.y, a.z); }
__device__ __forceinline__ V3f v3(f4n a) { return mk(a.x, a.y, a.z); }
__device__ __forceinline__ V3f v3(f3n a) { return mk(a.x, a.y, a.z); }
__device__ __forceinline__ V3f mul3(const float (&m)[9], V3f a) {
    return mk(m[0] * a.x + m[1] * a.y + m[2] * a.z, m[3] * a.x + m[4] * a.y + m[5] * a.z,
              m[6] * a.x + m[7] * a.y + m[8] * a.z);
}
// (as acc3 of cs_pcg.hip: the same operations in the same order give the same bits)
__device__ __forceinline__ void acc3(V3f& y, const float (&a)[9], V3f v) {
    y.x += a[0] * v.x + a[1] * v.y + a[2] * v.z;
    y.y += a[3] * v.x + a[4] * v.y + a[5] * v.z;
    y.z += a[6] * v.x + a[7] * v.y + a[8] * v.z;
}

// The recursive stop of a continuation (cs_pcg.hip, continuation_stop)
__device__ __forceinline__ float continuation_stop(float tol2bb, int restarts) {
    return restarts >= 1 ? 0.25f * tol2bb : tol2bb;
}

// 3x3 block c of a block-CSR value array: 36 B in three loads (the memory unit handles a wave's 64
// scattered lines once per load, so nine loads of 4 B cost three times as much)
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ void ldblk(const G1<float>* v, unsigned k, float (&o)[9]) {
    const G1<char>* b = (const G1<char>*)v + 36u * k;
    const f4u p = *(const G1<f4u>*)b, q = *(const G1<f4u>*)(b + 16);
    o[0] = p.x; o[1] = p.y; o[2] = p.z; o[3] = p.w;
    o[4] = q.x; o[5] = q.y; o[6] = q.z; o[7] = q.w;
    o[8] = *(const G1<float>*)(b + 32);
}

// ---- rows of the coarse levels (block CSR), the operations and order of cs_amg.hip's kernels

// sum of t over the members of aggregate I (ascending)
__device__ __forceinline__ V3f restricted(int I, const G1<int>* mptr, const G1<int>* midx, const G1<float>* t) {
    V3f s = mk(0.0f, 0.0f, 0.0f);
    const int k0 = at(mptr, 4u * I), k1 = at(mptr, 4u * I + 4u);
    for (int k = k0; k < k1; k += 8) {  // eight members' loads at a time, summed in order
        V3f m[8];
#pragma unroll
        for (int u = 0; u < 8; u++) m[u] = ld3v(&at(t, 12u * at(midx, 4u * min(k + u, k1 - 1))), 0);
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (k + u < k1) s = s + m[u];
    }
    return s;
}

// f(block, column) gives the operand of each block of row i; the sum over the blocks in order, the
// loads of NB blocks in flight together
template <int NB, class F>
__device__ __forceinline__ V3f blockrow(int i, const G1<int>* rp, const G1<int>* ci, const G1<float>* val, F&& f) {
    V3f y = mk(0.0f, 0.0f, 0.0f);
    const int k0 = at(rp, 4u * i), k1 = at(rp, 4u * i + 4u);
    for (int k = k0; k < k1; k += NB) {
        float a[NB][9];
        V3f w[NB];
#pragma unroll
        for (int u = 0; u < NB; u++) {
            const int kk = min(k + u, k1 - 1);
            ldblk(val, kk, a[u]);
            w[u] = f(at(ci, 4u * kk));
        }
#pragma unroll
        for (int u = 0; u < NB; u++)
            if (k + u < k1) acc3(y, a[u], w[u]);
    }
    return y;
}

// x = w D^-1 b (formed on the fly for the gathered rows) and t = b - A x
__device__ __forceinline__ void presmoothed(int i, const G1<int>* rp, const G1<int>* ci, const G1<float>* val,
                                            const G1<float>* Dinv, const G1<float>* b, V3f& x, V3f& t) {
    auto pre = [&](int j) {
        float o[9];
        ldblk(Dinv, j, o);
        return AMG_OMEGA * mul3(o, ld3v(&at(b, 12u * j), 0));
    };
    const V3f y = blockrow<3>(i, rp, ci, val, pre);
    x = pre(i);
    t = ld3v(&at(b, 12u * i), 0) - y;
}

// x' + w D^-1 (b - A x'), x' = x + e_agg
__device__ __forceinline__ V3f postsmoothed(int i, const G1<int>* rp, const G1<int>* ci, const G1<float>* val,
                                            const G1<float>* Dinv, const G1<int>* agg, const G1<float>* e,
                                            const G1<float>* b, const G1<float>* x) {
    auto pro = [&](int j) { return ld3v(&at(x, 12u * j), 0) + ld3v(&at(e, 12u * at(agg, 4u * j)), 0); };
    const V3f y = blockrow<3>(i, rp, ci, val, pro);
    float o[9];
    ldblk(Dinv, i, o);
    return pro(i) + AMG_OMEGA * mul3(o, ld3v(&at(b, 12u * i), 0) - y);
}

// a gathered neighbour's z and previous d
struct Pair {
    V3f z, d;
};
// a block's products with them, as floats of the products' LDS array and back
__device__ __forceinline__ V3f times(const float (&o)[9], V3f v) { return mul3(o, v); }
__device__ __forceinline__ Pair times(const float (&o)[9], Pair w) { return Pair{mul3(o, w.z), mul3(o, w.d)}; }
__device__ __forceinline__ void toLds(float* p, V3f v) {
    p[0] = v.x;
    p[1] = v.y;
    p[2] = v.z;
}
__device__ __forceinline__ void toLds(float* p, Pair w) {
    toLds(p, w.z);
    toLds(p + 3, w.d);
}
__device__ __forceinline__ void fromLds(const float* p, V3f& v) { v = mk(p[0], p[1], p[2]); }
__device__ __forceinline__ void fromLds(const float* p, Pair& w) {
    fromLds(p, w.z);
    fromLds(p + 3, w.d);
}
// One row per thread, T rows per workgroup, one 64-row slice per wave; RS slots of a row in
// registers (interior rows of a grid have 13), any further ones read from memory every iteration;
// the gathers of GR slots are in flight together.  LOCAL: the system has one workgroup, whose
// vectors are exchanged through LDS.  PRE: the preconditioner, as in the separate launches.
template <int T, int RS, int GR, bool LOCAL, int PRE>
__global__ void __launch_bounds__(T, 2)  // 256 registers: the runtime refuses cooperative kernels of more
    k_ppcg(const PSys* __restrict__ tab, const int2* __restrict__ map, float tol2, int maxit,
           unsigned long long ticks) {
    constexpr int NW = T / 64, NF = 3, CN = 3, CAP = LOCAL ? 2048 : 5120;
    __shared__ float red[2 * (NW + 4)];
    __shared__ Wait wait;
    __shared__ float prod[6 * CAP];  // products of contact blocks
    __shared__ float4 zl[LOCAL ? T : 1], dl[LOCAL ? T : 1];
    constexpr bool NET = PRE == PRE_LEARNED;
    __shared__ float lb[PRE == PRE_AMG ? 3 * BOTTOM : 1];  // the bottom level's right-hand side
    const int2 m2 = map[blockIdx.x];
    const int id = __builtin_amdgcn_readfirstlane(m2.x), wg = __builtin_amdgcn_readfirstlane(m2.y);
    if (id < 0) return;
    const PSys& P = tab[id];
    const PSysG S = gview(P);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nn = S.nn;
    Group g;
    g.slots = S.slots;
    g.lds = red;
    g.wait = &wait;
    g.G = S.G;
    g.wg = wg;
    g.epoch = 0;
    if (tid == 0) {
        wait.ticks = ticks;
        wait.ranOut = P.loseWg == wg ? P.loseAt : 0;
    }
    // A workgroup whose wait ran out leaves the solve without its rows of x.  The others learn of it at
    // their next meeting, but after the last one there is none: the host reads it from the record.
    auto lost = [&]() {
        if (tid == 0) S.out->lost = 1;
    };

    const V3f zero = mk(0.0f, 0.0f, 0.0f);
    const int i = wg * T + tid, ic = min(i, nn - 1);
    const bool live = i < nn;
    // a slice past the last reads the last one's blocks, masked to zero (no branches around loads)
    const int sl = min(wg * NW + wave, S.nslices - 1);
    const int W = S.sliceW[sl];
    const G1<int>* cb = S.cols + (size_t)S.sliceOff[sl] * SLICE;
    const G1<float>* vb = S.vals + (size_t)S.sliceOff[sl] * 9 * SLICE;
    float a[RS][9];
    int rel[(RS + 1) / 2];  // two 16-bit column offsets each
#pragma unroll
    for (int k = 0; k < RS; k++)
#pragma unroll
        for (int c = 0; c < 9; c++) a[k][c] = at(vb, 4u * ((min(k, W - 1) * 9 + c) * SLICE + lane));
#pragma unroll
    for (int k = 0; k < RS; k++)
#pragma unroll
        for (int c = 0; c < 9; c++) {
            asm volatile("" : "+v"(a[k][c]));
            a[k][c] = k < W && live ? a[k][c] : 0.0f;
            asm volatile("" : "+v"(a[k][c]));  // masked here and now, not where it is first used
        }
#pragma unroll
    for (int k = 0; k < (RS + 1) / 2; k++) {
        int lo = at(cb, 4u * (min(2 * k, W - 1) * SLICE + lane)) - i;
        int hi = at(cb, 4u * (min(2 * k + 1, W - 1) * SLICE + lane)) - i;
        asm volatile("" : "+v"(lo), "+v"(hi));
        lo = 2 * k < W && live ? lo : 0;
        hi = 2 * k + 1 < W && live ? hi : 0;
        rel[k] = (lo & 0xffff) | (hi << 16);
    }

    auto row = [&]() { return opaque(ic); };
    auto zAt = [&](int j) { return LOCAL ? v3(zl[j]) : v3(at((const G1<f3n>*)S.z, 16u * j)); };
    auto dAt = [&](const G1<f4n>* dp, int j) { return LOCAL ? v3(dl[j]) : v3(at((const G1<f3n>*)dp, 16u * j)); };
    // The operand of a product is formed as it is gathered, gat(column); put(block, operand) adds it to
    // the row, add(product) adds a product.  A row's contacts, one thread and two blocks at a time:
    auto contactsOfRow = [&](auto& gat, auto& put) {
        if (!S.contacts || !live) return;
        const int c1 = at(S.cRowPtr, 4u * row() + 4u);
        for (int k = at(S.cRowPtr, 4u * row()); k < c1; k += 2) {
            float o[2][9];
            decltype(gat(0)) w[2];
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const int kk = min(k + u, c1 - 1);
                ldblk(S.cVal, kk, o[u]);
                w[u] = gat(at(S.cCol, 4u * kk));
            }
#pragma unroll
            for (int u = 0; u < 2; u++)
                if (k + u < c1) put(o[u], w[u]);
        }
    };
    // The contact blocks of the workgroup's rows: a row has none or dozens, and a thread that walks its
    // own holds up its wave, so the threads share the blocks evenly, CN in flight each and neighbours in
    // the matrix side by side, and a row's thread adds its products from LDS in order.  Solves, each row
    // walked by its thread -> shared: 129x129 drape block Jacobi 8.6 -> 7.9 ms, multigrid 5.7 -> 5.4;
    // 201x201 fold learned, before its sweeps were grouped, 19.7 -> 17.6 (18.9 with 2,048 products of LDS);
    // few contacts: the same.
    const int e0 = S.contacts ? S.cRowPtr[min(wg * T, nn)] : 0, e1 = S.contacts ? S.cRowPtr[min(wg * T + T, nn)] : 0;
    auto contacts = [&](auto& gat, auto&& add) {
        using W = decltype(gat(0));
        constexpr int WF = sizeof(W) / sizeof(float);
        if (e0 == e1) return;
        const int r0 = at(S.cRowPtr, 4u * row()), r1 = at(S.cRowPtr, 4u * row() + 4u);
        for (int base = e0; base < e1; base += CAP) {
            const int end = min(base + CAP, e1);
            if (base > e0) __syncthreads();
            for (int k = base + tid; k < end; k += CN * T) {
                float o[CN][9];
                W w[CN];
#pragma unroll
                for (int u = 0; u < CN; u++) {
                    const int kk = min(k + u * T, end - 1);
                    ldblk(S.cVal, kk, o[u]);
                    w[u] = gat(at(S.cCol, 4u * kk));
                }
#pragma unroll
                for (int u = 0; u < CN; u++)
                    if (k + u * T < end) toLds(prod + WF * (k + u * T - base), times(o[u], w[u]));
            }
            __syncthreads();
            if (live) {
                const int k1 = min(r1, end);
                for (int k = max(r0, base); k < k1; k += 4) {
                    W v[4];
#pragma unroll
                    for (int u = 0; u < 4; u++) fromLds(prod + WF * (min(k + u, k1 - 1) - base), v[u]);
#pragma unroll
                    for (int u = 0; u < 4; u++)
                        if (k + u < k1) add(v[u]);
                }
            }
        }
    };
    // slots k0.. of the row from memory
    auto streamed = [&](int k0, auto& gat, auto& put) {
#pragma unroll 2
        for (int k = k0; k < W; k++) {
            float o[9];
            const int j = at(cb, 4u * (k * SLICE + lane));
#pragma unroll
            for (int c = 0; c < 9; c++) o[c] = at(vb, 4u * ((k * 9 + c) * SLICE + lane));
            put(o, gat(live ? j : ic));
        }
    };
    // the pattern's slots in order, then the contacts
    auto sweep = [&](auto& gat, auto& put, auto&& add) {
        const int q = row();
#pragma unroll
        for (int k = 0; k < (RS + 1) / 2; k++) asm volatile("" : "+v"(rel[k]));  // columns unpacked here, not kept
        auto col = [&](int k) { return q + ((k & 1) ? rel[k >> 1] >> 16 : (int)(short)(rel[k >> 1] & 0xffff)); };
#pragma unroll
        for (int k0 = 0; k0 < RS; k0 += GR) {
            decltype(gat(0)) w[GR];
#pragma unroll
            for (int u = 0; u < GR; u++)
                if (k0 + u < RS) w[u] = gat(col(k0 + u));
#pragma unroll
            for (int u = 0; u < GR; u++)
                if (k0 + u < RS) put(a[k0 + u], w[u]);
        }
        streamed(RS, gat, put);
        contacts(gat, add);
    };
    auto putZ = [&](V3f v) {
        if (LOCAL) zl[tid] = st4(v);
        else if (live) put3(&at(S.z, 16u * row()), v);
    };
    auto rhs = [&](int k) { return ld3v(&at(S.b, 12u * k), 0) + ld3v(&at(S.bc, 12u * k), 0); };

    float m[9];
    V3f x = zero, d = zero, q = zero, z = zero, r = live ? rhs(row()) : zero;
    float v1[1], v2[2], rz = 0.0f, rzOld = 1.0f, rr = 0.0f, stop2bb = -1.0f;
    int it = 0, first = 0;

    // y = G u (lower slots and the diagonal) and w = G^T u (diagonal transposed, upper slots hold the
    // transposed lower blocks), u gathered from p: k_lpc_lower and k_lpc_upper
    const int kd = NET ? S.diagSlot[ic] : 0, rl = NET ? S.rowLen[ic] : 0;
    auto factor = [&](int k, float (&o)[9]) {
        const G1<uint16_t>* gb = S.Gf + (size_t)S.sliceOff[sl] * 9 * SLICE;
#pragma unroll
        for (int c = 0; c < 9; c++) o[c] = __uint_as_float((unsigned)at(gb, 2u * ((k * 9 + c) * SLICE + lane)) << 16);
    };
    // Slots k0 .. k1 - 1 of a row, which differ from lane to lane: a latency per NF of them, the last ones
    // included (a loop unrolled by 4 walked the remainder one at a time, and on irregular meshes, rows of
    // 17 to 20 blocks, lost to the separate launches: 65,536 rows 13.3 against 10.8 ms a solve, now 9.7;
    // a disc whose centre has 48 neighbours, 961 rows: 20.2 against 13.1 ms, now 9.7; regular grid, 16,641
    // rows: 3.2 ms, now 2.6; 2 or 4 in flight: the same within 5 %).
    auto factored = [&](const G1<f4n>* p, int k0, int k1, V3f& y) {
        for (int k = k0; k < k1; k += NF) {
            float o[NF][9];
            V3f w[NF];
#pragma unroll
            for (int u = 0; u < NF; u++) {
                const int kk = min(k + u, k1 - 1);
                factor(kk, o[u]);
                w[u] = v3(at((const G1<f3n>*)p, 16u * at(cb, 4u * (kk * SLICE + lane))));
            }
#pragma unroll
            for (int u = 0; u < NF; u++)
                if (k + u < k1) acc3(y, o[u], w[u]);
        }
    };
    auto lower = [&](const G1<f4n>* p) {
        V3f y = zero;
        factored(p, 0, kd + 1, y);
        return y;
    };
    auto upper = [&](const G1<f4n>* p, V3f own) {
        float o[9];
        factor(kd, o);
        V3f y = mk(o[0] * own.x + o[3] * own.y + o[6] * own.z, o[1] * own.x + o[4] * own.y + o[7] * own.z,
                   o[2] * own.x + o[5] * own.y + o[8] * own.z);
        factored(p, kd + 1, rl, y);
        return y;
    };
    auto putF = [&](G1<f4n>* p, V3f v) {
        if (live) put3(&at(p, 16u * row()), v);
    };
    // G^T G u for u published in S.z by every thread
    auto sweeps = [&](V3f& out) {
        const V3f y = live ? lower(S.z) : zero;
        putF(S.y, y);
        float none[1] = {0.0f};
        if (!meet<T, 1>(g, none)) return false;
        out = live ? upper(S.y, y) : zero;
        return true;
    };

    // z = M^-1 r, rz and rr of the current r; the stop test of the next iteration comes as soon as rr
    // is known, and z is then left alone.  False: a wait ran out.
    bool stop = false;
    auto precondition = [&](bool test) {
        auto stopped = [&]() {  // on the tolerance, the budget, or a non-finite r.r (NaN fails every comparison)
            stop = test && (rr <= stop2bb || it >= maxit || !(rr <= FLT_MAX));
            return stop;
        };
        if (PRE == PRE_JACOBI) {
            z = mul3(m, r);
            putZ(z);
            v2[0] = dot(r, z);
            v2[1] = dot(r, r);
            if (!meet<T, 2, true, LOCAL>(g, v2)) return false;
            rz = v2[0];
            rr = v2[1];
            stopped();
            return true;
        }
        V3f xs = zero;
        if (PRE == PRE_AMG) {
            const V3f mr = mul3(m, r);
            xs = mk(AMG_OMEGA * mr.x, AMG_OMEGA * mr.y, AMG_OMEGA * mr.z);
            putF(S.z, xs);
        } else {
            putF(S.z, r);
        }
        v1[0] = dot(r, r);
        if (!meet<T, 1>(g, v1)) return false;
        rr = v1[0];
        if (stopped()) return true;
        if (PRE == PRE_LEARNED) {
            if (!sweeps(z)) return false;
        } else {
            float none[1];
            // level 0: t = r - A xs
            V3f t = zero;
            auto gat = [&](int j) { return zAt(j); };
            auto put = [&](const float (&o)[9], V3f v) { acc3(t, o, v); };
            sweep(gat, put, [&](V3f v) { t = t + v; });
            t = r - t;
            if (live) put3f(&at(gview(P.L[0]).t, 12u * row()), t);
            none[0] = 0.0f;
            if (!meet<T, 1>(g, none)) return false;
            // down: restriction, then pre-smoothing and residual; rows in 64s over the workgroups
            const int gr = (wave * g.G + wg) * 64 + lane, gs = g.G * T;
            const int bottom = P.bottom;
            for (int l = 1; l < bottom; l++) {
                const PLevG F = gview(P.L[l - 1]), L = gview(P.L[l]);
                for (int k = gr; k < L.n; k += gs) put3f(&at(L.b, 12u * k), restricted(k, F.mptr, F.midx, F.t));
                none[0] = 0.0f;
                if (!meet<T, 1>(g, none)) return false;
                for (int k = gr; k < L.n; k += gs) {
                    V3f xk, tk;
                    presmoothed(k, L.rp, L.ci, L.val, L.Dinv, L.b, xk, tk);
                    put3f(&at(L.x, 12u * k), xk);
                    put3f(&at(L.t, 12u * k), tk);
                }
                none[0] = 0.0f;
                if (!meet<T, 1>(g, none)) return false;
            }
            // the bottom: every workgroup restricts its whole right-hand side, a wave per row of the operator
            {
                const PLevG F = gview(P.L[bottom - 1]);
                const int n = P.L[bottom].n, dim = 3 * n;
                for (int k = tid; k < n; k += T) {
                    const V3f b = restricted(k, F.mptr, F.midx, F.t);
                    lb[3 * k] = b.x;
                    lb[3 * k + 1] = b.y;
                    lb[3 * k + 2] = b.z;
                }
                __syncthreads();
                const G1<float>* op = g1(P.op);
                G1<float>* e = g1(P.eBottom);
                // a wave's rows of the operator, RU of them in flight together
                auto rows = [&](auto ru) {
                    constexpr int RU = decltype(ru)::value;
                    for (int k = (wave * g.G + wg) * RU; k < dim; k += NW * g.G * RU) {
                        float s[RU];
#pragma unroll
                        for (int u = 0; u < RU; u++) s[u] = 0.0f;
#pragma unroll 4
                        for (int c = lane; c < dim; c += 64) {
                            const float v = lb[c];
#pragma unroll
                            for (int u = 0; u < RU; u++) s[u] += at(op, 4u * (min(k + u, dim - 1) * dim + c)) * v;
                        }
#pragma unroll
                        for (int u = 0; u < RU; u++) {
#pragma unroll
                            for (int o = 32; o > 0; o >>= 1) s[u] += __shfl_xor(s[u], o, 64);
                            if (lane == 0 && k + u < dim)
                                __hip_atomic_store(&at(e, 4u * (k + u)), s[u], __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT);
                        }
                    }
                };
                if (dim <= NW * g.G) rows(std::integral_constant<int, 1>{});
                else if (dim <= 2 * NW * g.G) rows(std::integral_constant<int, 2>{});
                else if (dim <= 3 * NW * g.G) rows(std::integral_constant<int, 3>{});
                else rows(std::integral_constant<int, 4>{});
                none[0] = 0.0f;
                if (!meet<T, 1>(g, none)) return false;
            }
            // up: prolongation and post-smoothing, a level's result into its t
            const G1<float>* e = g1(P.eBottom);
            for (int l = bottom - 1; l >= 1; l--) {
                const PLevG L = gview(P.L[l]);
                for (int k = gr; k < L.n; k += gs)
                    put3f(&at(L.t, 12u * k), postsmoothed(k, L.rp, L.ci, L.val, L.Dinv, L.agg, e, L.b, L.x));
                e = L.t;
                none[0] = 0.0f;
                if (!meet<T, 1>(g, none)) return false;
            }
            // level 0: the residual after the correction is t - (A P) e
            const PLevG L = gview(P.L[0]);
            V3f y = zero;
            if (live) {
                const int WA = P.apSliceW[sl];
                const G1<int>* ac = g1(P.apCols) + (size_t)P.apSliceOff[sl] * SLICE;
                const G1<float>* av = g1(P.apVals) + (size_t)P.apSliceOff[sl] * 9 * SLICE;
#pragma unroll 4
                for (int k = 0; k < WA; k++) {
                    float o[9];
#pragma unroll
                    for (int c = 0; c < 9; c++) o[c] = at(av, 4u * ((k * 9 + c) * SLICE + lane));
                    acc3(y, o, ld3v(&at(e, 12u * at(ac, 4u * (k * SLICE + lane))), 0));
                }
                xs = xs + ld3v(&at(e, 12u * at(L.agg, 4u * row())), 0);
            }
            auto gatE = [&](int j) { return ld3v(&at(e, 12u * at(L.agg, 4u * j)), 0); };
            contacts(gatE, [&](V3f v) { y = y + v; });
            y = t - y;
            ldblk(S.Minv, row(), m);
            const V3f my = mul3(m, y);
            z = live ? mk(xs.x + AMG_OMEGA * my.x, xs.y + AMG_OMEGA * my.y, xs.z + AMG_OMEGA * my.z) : zero;
        }
        putF(S.z, z);
        v1[0] = live ? dot(r, z) : 0.0f;
        if (!meet<T, 1>(g, v1)) return false;
        rz = v1[0];
        return true;
    };

    // x = 0, r = b
    ldblk(S.Minv, row(), m);
    if (!precondition(false)) return lost();
    const float bb = rr, tol2bb = tol2 * bb;
    stop2bb = tol2bb;
    stop = bb <= tol2bb || maxit <= 0;
    for (int restarts = 0;; restarts++) {
        for (first = it; !stop;) {
            q = zero;
            if (it == first) {
                auto gat = [&](int j) { return zAt(j); };
                auto put = [&](const float (&o)[9], V3f w) { acc3(q, o, w); };
                sweep(gat, put, [&](V3f v) { q = q + v; });
                d = z;
            } else {
                const float beta = rz / rzOld;
                const G1<f4n>* dprev = S.d + (1 - (it & 1)) * nn;
                auto gat = [&](int j) { return Pair{zAt(j), dAt(dprev, j)}; };
                V3f t = zero;  // q = A z + beta (A d_prev)
                auto put = [&](const float (&o)[9], Pair w) {
                    acc3(q, o, w.z);
                    acc3(t, o, w.d);
                };
                sweep(gat, put, [&](Pair v) {
                    q = q + v.z;
                    t = t + v.d;
                });
                d = mk(z.x + beta * d.x, z.y + beta * d.y, z.z + beta * d.z);
                q = mk(q.x + beta * t.x, q.y + beta * t.y, q.z + beta * t.z);
            }
            if (LOCAL) {
                __syncthreads();  // every gather of the previous d is done
                dl[tid] = st4(d);
            } else if (live) {
                put3(&at(S.d + (it & 1) * nn, 16u * row()), d);
            }
            v1[0] = live ? dot(d, q) : 0.0f;
            if (PRE == PRE_JACOBI || PRE == PRE_AMG) ldblk(S.Minv, row(), m);  // ahead of the meeting
            if (!meet<T, 1, false, LOCAL>(g, v1)) return lost();
            const float alpha = rz / v1[0];
            if (live) {
                x = x + alpha * d;
                r = r - alpha * q;
            }
            it++;
            rzOld = rz;
            if (!precondition(true)) return lost();
        }
        // the true residual b - A x with every row sum in FP64, the matrix from memory (once per stop)
        putZ(x);
        v1[0] = 0.0f;
        if (!meet<T, 1, true, LOCAL>(g, v1)) return lost();
        if (live) {
            double y0 = 0.0, y1 = 0.0, y2 = 0.0;
            auto put = [&](const float (&o)[9], V3f xj) {
                y0 += (double)o[0] * xj.x + (double)o[1] * xj.y + (double)o[2] * xj.z;
                y1 += (double)o[3] * xj.x + (double)o[4] * xj.y + (double)o[5] * xj.z;
                y2 += (double)o[6] * xj.x + (double)o[7] * xj.y + (double)o[8] * xj.z;
            };
            streamed(0, zAt, put);
            contactsOfRow(zAt, put);
            const V3f b = ld3v(&at(S.b, 12u * row()), 0), bc = ld3v(&at(S.bc, 12u * row()), 0);
            r = mk((float)((double)b.x + (double)bc.x - y0), (float)((double)b.y + (double)bc.y - y1),
                   (float)((double)b.z + (double)bc.z - y2));
        }
        v1[0] = dot(r, r);
        if (!meet<T, 1, true, LOCAL>(g, v1)) return lost();
        rr = v1[0];
        if (rr <= tol2bb || it >= maxit || !(rr <= FLT_MAX) || restarts == RESTARTS) break;
        // continue from it, the direction restarted from its preconditioned residual
        stop2bb = continuation_stop(tol2bb, restarts);
        stop = false;
        ldblk(S.Minv, row(), m);
        if (!precondition(false)) return lost();
    }
    if (live) {
        G1<float>* o = &at(S.x, 12u * row());
        o[0] = x.x;
        o[1] = x.y;
        o[2] = x.z;
    }
    if (wg == 0 && tid == 0) {
        S.out->rr = rr;
        S.out->bb = bb;
        S.out->tol2bb = tol2bb;
        S.out->iters = it;
        S.out->done = 1;
    }
}

// A system's launch table entry: its group has G workgroups, its slots start at `slots`.
// dense: the multigrid's bottom is the small levels' operator, otherwise the coarsest level's inverse
PSys describe(const ClothSys& S, int pre, bool dense, int G, uint64_t* slots, PcgScalars* out) {
    PSys p{};
    p.nn = S.nn;
    p.nslices = S.nslices;
    p.G = G;
    p.contacts = S.nContact;
    p.sliceOff = S.sliceOff.ptr<int>();
    p.sliceW = S.sliceW.ptr<int>();
    p.cols = S.cols.ptr<int>();
    p.cRowPtr = S.cRowPtr.ptr<int>();
    p.cCol = S.nContact > 0 ? S.cCol.ptr<int>() : p.cRowPtr;
    p.vals = S.vals.ptr<float>();
    p.cVal = S.nContact > 0 ? S.cVal.ptr<float>() : p.vals;
    p.Minv = S.Minv.ptr<float>();
    p.b = S.b.ptr<float>();
    p.bc = S.bc.ptr<float>();
    p.x = S.x.ptr<float>();
    p.z = S.z.ptr<float4>();
    p.d = S.d.ptr<float4>();
    p.slots = slots;
    p.out = out;
    if (pre == PRE_LEARNED) {
        p.diagSlot = S.diagSlot.ptr<int>();
        p.rowLen = S.rowLen.ptr<int>();
        p.Gf = S.lpc.G.ptr<uint16_t>();
        p.y = S.lpc.y.ptr<float4>();
    }
    if (pre == PRE_AMG) {
        const AmgSys& A = S.amg;
        p.bottom = dense ? A.smallL0 : A.nl - 1;
        p.op = dense ? A.smallOp.ptr<float>() : A.inv.ptr<float>();
        p.eBottom = A.L[p.bottom].t.ptr<float>();
        p.apSliceOff = A.apSliceOff.ptr<int>();
        p.apSliceW = A.apSliceW.ptr<int>();
        p.apCols = A.apCols.ptr<int>();
        p.apVals = A.apVals.ptr<float>();
        for (int l = 0; l <= p.bottom; l++) {
            const AmgLevel& L = A.L[l];
            PLev& q = p.L[l];
            q.n = L.n;
            q.rp = L.rp.ptr<int>();
            q.ci = L.ci.ptr<int>();
            q.agg = L.agg.ptr<int>();
            q.mptr = L.mptr.ptr<int>();
            q.midx = L.midx.ptr<int>();
            q.val = L.val.ptr<float>();
            q.Dinv = L.Dinv.ptr<float>();
            q.b = L.b.ptr<float>();
            q.x = L.x.ptr<float>();
            q.t = L.t.ptr<float>();
        }
    }
    return p;
}

// Workgroups of T threads of kernel f the device holds at once, a multiple of 8 (0: no cooperative
// launch): by the 512 vector registers a lane of a SIMD has for all its waves and by the LDS of a
// CU (hipOccupancyMaxActiveBlocksPerMultiprocessor counts 256 registers).
int resident(cs_ctx* C, const void* f, int T) {
    int coop = 0, cus = 0, lds = 0;
    hipFuncAttributes fa;
    CS_HIP(hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, C->device));
    CS_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, C->device));
    CS_HIP(hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, C->device));
    CS_HIP(hipFuncGetAttributes(&fa, f));
    if (!coop || fa.numRegs <= 0) return 0;
    const int waves = std::min(8, 512 / ((fa.numRegs + 7) & ~7));  // per SIMD
    int per = waves * 4 / (T / 64);
    if (fa.sharedSizeBytes > 0) per = std::min(per, (int)(lds / fa.sharedSizeBytes));
    return (per * cus) & ~7;
}

template <int PRE> const void* kernel_of(int T) {
    // (a further gather in flight spills; the learned kernel of 512 threads spills 7 registers with 4)
    constexpr int GR = PRE == PRE_LEARNED ? 4 : 7;
    return T == 512 ? (const void*)k_ppcg<512, 14, 4, false, PRE> : (const void*)k_ppcg<256, 14, GR, false, PRE>;
}
const void* kernel_of(int T, bool local, int pre) {
    if (local) return (const void*)k_ppcg<512, 14, 4, true, PRE_JACOBI>;
    return pre == PRE_JACOBI ? kernel_of<PRE_JACOBI>(T)
         : pre == PRE_LEARNED ? kernel_of<PRE_LEARNED>(T) : kernel_of<PRE_AMG>(T);
}

struct Round {
    int off, n;  // its blocks in the map
};
struct Plan {
    bool fits = false;
    int T = 0;
    const void* f = nullptr;
    std::vector<int> G;  // workgroups per system
    std::vector<Round> rounds;
    std::vector<int2> map;  // block -> (system, workgroup), -1: none
};

// The launches for the systems of `cloths`; fits = false when one has more rows than the device holds
// at once, a column more than 32,767 away from its row or too deep a hierarchy, or when the
// separate launches are faster.
Plan plan_for(cs_ctx* C, const std::vector<int>& cloths, int pre, bool dense) {
    Plan p;
    const int n = (int)cloths.size();
    bool local = pre == PRE_JACOBI;
    int most = 0;
    for (int c : cloths) {
        const ClothSys& S = C->sys[c];
        if (S.bandwidth > 32767) return p;
        if (pre == PRE_AMG) {
            const int bottom = dense ? S.amg.smallL0 : S.amg.nl - 1;
            if (bottom >= MAXL || S.amg.L[bottom].n > BOTTOM) return p;
        }
        local = local && S.nn <= 512;
        most = std::max(most, S.nn);
    }
    // Large lone systems stream their factor or their coarse levels from memory either way.  Multigrid: 97,969
    // rows 4.16 ms a solve against 4.44 launched, 115,600 rows 4.81 against 4.63, 131,044 rows 5.00 against
    // 4.75.  Learned: 65,536 rows 5.7 against 8.2; the line was drawn before its sweeps were grouped, and
    // systems without contacts now gain beyond it too (90,000 rows 8.0 against 9.8, 131,044 rows 11.3 against
    // 12.1); folded ones have not been measured there.
    if ((pre == PRE_LEARNED && most > 65536) || (pre == PRE_AMG && most > 98304)) return p;
    // more rows than the launches hold
    long rows = 0;
    for (int c : cloths) rows += 512l * cdiv(C->sys[c].nn, 512);
    const int launches = pre == PRE_JACOBI ? 2 : 1;
    if (rows > launches * 131072l) return p;
    // Rows per workgroup: one workgroup and LDS for systems of 512 rows; otherwise a lone system is spread
    // over more CUs by 256, until the meeting of many workgroups costs more.  Solves with 256 and 512, block
    // Jacobi: 1,089 rows 0.57 and 0.68 ms, 8,281 rows 1.59 and 1.63, 16,641 rows 2.31 and 2.22, 24,336 rows
    // 2.87 and 2.68, 28,900 rows 3.26 and 2.93, 65,536 rows 4.98 and 3.78; learned 24,336 rows 3.25 and 3.16,
    // 28,900 rows 3.62 and 3.36; multigrid 2.37 and 2.16, 2.74 and 2.44: between 12,000 rows and the line the
    // two are within 9 %.  A batch fills the CUs anyway (32 cloths, 170,000 rows: 24.6 ms with 256, 15.9
    // with 512).
    const int T = p.T = local || n > 1 || most > 96 * 256 ? 512 : 256;
    p.f = kernel_of(T, local, pre);
    const int cap = resident(C, p.f, T);
    std::vector<int>& G = p.G;
    std::vector<int> order(n);
    G.resize(n);
    for (int k = 0; k < n; k++) {
        const ClothSys& S = C->sys[cloths[k]];
        G[k] = cdiv(S.nn, T);
        if (pre == PRE_AMG && dense) {
            // workgroups without rows join the group where the bottom's dense operator is more than
            // 128 KB a workgroup (4,225 rows on 17 workgroups and an operator of 8.4 MB: 4.9 ms a
            // solve, 3.5 with 72) or more than four rows a wave
            const int dim = 3 * S.amg.L[S.amg.smallL0].n;
            G[k] = std::max(G[k], std::max(cdiv((long)dim * dim * 4, 128 << 10), cdiv(dim, 4 * (T / 64))));
        }
        order[k] = k;
        if (((G[k] + 7) & ~7) > cap) return p;
    }
    // Launches of as many groups as fit, largest systems first (they iterate longest).  Workgroups are
    // dealt to the 8 XCDs round-robin; a group of a batch goes to the least loaded XCD, whose L2 its
    // vectors then share; a lone system of up to 8 workgroups too (1,089 rows: 4.6 against 5.0 us), a
    // larger one is split into eighths (4,225 rows: 5.2 against 6.3 us on one XCD).  Beyond two
    // launches the separate kernels win: they stream all matrices at once, while here each launch
    // waits out its slowest system (340,000 rows in 48 cloths: 37.6 against 40 ms; 170,000 in 32:
    // 15.9 against 22.5).
    std::sort(order.begin(), order.end(), [&](int a, int b) { return G[a] != G[b] ? G[a] > G[b] : a < b; });
    for (size_t at = 0; at < order.size();) {
        std::vector<int2> xcd[8];
        size_t deep = 0;
        if (n == 1) {
            const int per = G[0] <= 8 ? 8 : (G[0] + 7) / 8;
            for (int w = 0; w < G[0]; w++) xcd[w / per].push_back(make_int2(0, w));
            for (auto& v : xcd) deep = std::max(deep, v.size());
            at = 1;
        }
        for (; at < order.size(); at++) {
            const int k = order[at];
            int x = 0;
            for (int y = 1; y < 8; y++)
                if (xcd[y].size() < xcd[x].size()) x = y;
            // a group deeper than an XCD's share runs over all of them
            if (xcd[x].size() + G[k] <= (size_t)cap / 8) {
                for (int w = 0; w < G[k]; w++) xcd[x].push_back(make_int2(k, w));
            } else if (deep == 0 && G[k] > cap / 8) {
                for (int w = 0; w < G[k]; w++) xcd[w % 8].push_back(make_int2(k, w));
            } else {
                break;
            }
            for (auto& v : xcd) deep = std::max(deep, v.size());
        }
        p.rounds.push_back({(int)p.map.size(), (int)(8 * deep)});
        for (size_t d = 0; d < deep; d++)
            for (int y = 0; y < 8; y++) p.map.push_back(d < xcd[y].size() ? xcd[y][d] : make_int2(-1, 0));
    }
    p.fits = (int)p.rounds.size() <= launches;
    return p;
}

// Results per entry of `cloths`, as pcg_solve.  False, the entries of x undefined, when a launch is refused
// or any workgroup gave up.
bool run_plan(cs_ctx* C, const Plan& p, const std::vector<int>& cloths, int pre, bool dense, int* iters, float* relres,
              int* converged) {
    const int n = (int)cloths.size(), T = p.T;
    const std::vector<int>& G = p.G;
    const std::vector<int2>& map = p.map;
    hipStream_t s = C->stream;
    std::vector<size_t> so(n);
    size_t words = 0;
    for (int k = 0; k < n; k++) {
        so[k] = words;
        words += 4 * (size_t)G[k] * (T / BLK);
    }
    uint64_t* slots = C->ppSlots.as<uint64_t>(words);
    PcgScalars* out = C->bScal.as<PcgScalars>(n);
    std::vector<PSys> tab(n);
    const cs_launch_fault& fault = C->ppFault;
    for (int k = 0; k < n; k++) {
        tab[k] = describe(C->sys[cloths[k]], pre, dense, G[k], slots + so[k], out + k);
        tab[k].loseWg = fault.lose_wg;
        tab[k].loseAt = fault.lose_at;
    }
    PSys* dtab = C->ppTab.as<PSys>(n);
    int2* dmap = C->ppMap.as<int2>(map.size());
    PcgScalars* h = static_cast<PcgScalars*>(pinned_batch(C, sizeof(PcgScalars) * n));
    CS_HIP(hipMemcpyAsync(dtab, tab.data(), sizeof(PSys) * n, hipMemcpyHostToDevice, s));
    CS_HIP(hipMemcpyAsync(dmap, map.data(), sizeof(int2) * map.size(), hipMemcpyHostToDevice, s));
    fill_u64(slots, 0, (long)words, s);
    fill_u32(reinterpret_cast<uint32_t*>(out), 0u, (long)n * (sizeof(PcgScalars) / 4), s);
    float tol2 = C->P.pcg_rel_tol * C->P.pcg_rel_tol;
    int maxit = C->P.pcg_max_iters;
    unsigned long long ticks = fault.wait_s > 0.0f ? (unsigned long long)(fault.wait_s * 1e8f) : WAIT_TICKS;
    for (const Round& r : p.rounds) {
        const PSys* ct = dtab;
        const int2* cm = dmap + r.off;
        void* args[] = {(void*)&ct, (void*)&cm, (void*)&tol2, (void*)&maxit, (void*)&ticks};
        const hipError_t e = fault.refuse ? hipErrorCooperativeLaunchTooLarge
                                          : hipLaunchCooperativeKernel(p.f, dim3(r.n), dim3(T), args, 0, s);
        if (e != hipSuccess) {
            // too large, or another process holds the device's cooperative queue
            (void)hipGetLastError();
            CS_HIP(hipStreamSynchronize(s));
            C->ppOnce.refused();
            return false;
        }
    }
    CS_HIP(hipMemcpyAsync(h, out, sizeof(PcgScalars) * n, hipMemcpyDeviceToHost, s));
    CS_HIP(hipStreamSynchronize(s));
    for (int k = 0; k < n; k++)
        if (!h[k].done || h[k].lost) {
            C->ppOnce.ranOut();
            return false;
        }
    for (int k = 0; k < n; k++) {
        iters[k] = h[k].iters;
        relres[k] = h[k].bb > 0.0f ? sqrtf(h[k].rr / h[k].bb) : 0.0f;
        converged[k] = h[k].rr <= h[k].tol2bb;
        C->sys[cloths[k]].solved = converged[k] != 0;
    }
    C->ppLaunches += (int)p.rounds.size();
    return true;
}

bool allowed(const cs_ctx* C) {
    return !(C->P.flags & (CS_FLAG_TIME_KERNELS | CS_FLAG_GRAPH_CYCLES));
}

}  // namespace

bool ppcg_solve(cs_ctx* C, int c, bool amg, bool learned, int* iters, float* relres, int* converged) {
    C->ppLaunches = 0;
    // the cycle with the learned smoother would meet 13 times an iteration: measured slower at every size
    if (!allowed(C) || (amg && learned)) return false;
    const int pre = amg ? PRE_AMG : learned ? PRE_LEARNED : PRE_JACOBI;
    const std::vector<int> one{c};
    const Plan p = plan_for(C, one, pre, true);
    if (!p.fits || !C->ppOnce.attempt() || !run_plan(C, p, one, pre, true, iters, relres, converged)) return false;
    C->ppOnce.worked();
    return true;
}

bool ppcg_solve_batch(cs_ctx* C, bool amg, int* iters, float* relres, int* converged) {
    C->ppLaunches = 0;
    if (!allowed(C)) return false;
    std::vector<int> part[2];  // block Jacobi, multigrid
    const std::vector<int>* usable = amg ? &bamg_build(C) : nullptr;
    for (int c = 0; c < C->nCloths; c++) part[usable && (*usable)[c] ? 1 : 0].push_back(c);
    Plan plan[2];
    for (int k = 0; k < 2; k++) {
        if (part[k].empty()) continue;
        plan[k] = plan_for(C, part[k], k ? PRE_AMG : PRE_JACOBI, false);
        if (!plan[k].fits) return false;
    }
    if (!C->ppOnce.attempt()) return false;
    if (amg) bamg_prepare(C);
    for (int k = 0; k < 2; k++) {
        if (part[k].empty()) continue;
        const int n = (int)part[k].size();
        std::vector<int> it(n), cv(n);
        std::vector<float> rel(n);
        if (!run_plan(C, plan[k], part[k], k ? PRE_AMG : PRE_JACOBI, false, it.data(), rel.data(), cv.data())) {
            C->ppLaunches = 0;
            return false;
        }
        for (int j = 0; j < n; j++) {
            iters[part[k][j]] = it[j];
            relres[part[k][j]] = rel[j];
            converged[part[k][j]] = cv[j];
        }
    }
    C->ppOnce.worked();
    return true;
}

}  // namespace cs
