// cs_noalloc.hip — cs_solve_bsr_noalloc: block-Jacobi PCG on a system held in the caller's
// device memory, allocating nothing.
//
// The same algorithm and stop rule as the block-Jacobi solve of cs_solve (x = 0, r = b,
// z = d = M^-1 r; per iteration q = A d, alpha = r.z / d.q, x += alpha d, r -= alpha q, stop when
// r.r <= tol^2 b.b or at max_iters, z = M^-1 r, beta = r.z_new / r.z, d = z + beta d; a stop
// confirmed by the true residual b - A x in FP64, else continued from it), on a
// block-CSR matrix (3x3 row-major blocks, every row holding its diagonal block) instead of the
// context's sliced ELL.  Every temporary (M^-1, r, z, d, q, partial sums, scalars) lives in
// `scratch`, one file-scope device array of fixed size: each GPU holds its own copy for the
// life of the process, and every call on that GPU reuses it, so calls that overlap on one GPU
// race.
//
// The iterations run in one cooperative launch (k_na_loop), a row per thread, its first blocks in
// registers; where that launch is refused, or a wait in it runs out, and for a while after (OneLaunch), as
// separate launches with one scalar record read back every NA_CHUNK iterations.  Both give the same bits.
#include <cfloat>
#include <mutex>

#include "cs_common.hpp"
#include "cs_math.hpp"
#include "../../include/clothsim.h"

namespace cs {

namespace {

constexpr int NA_MAX = CS_NOALLOC_MAX_NODES;
constexpr int NA_TB = 256;                    // threads per workgroup, one row each
constexpr int NA_MAXB = NA_MAX / NA_TB;       // workgroups (partial-sum slots) at most
constexpr int NA_CHUNK = 16;                  // iterations between host reads
// Blocks of a row at most in the one launch (k_na_loop), which sends wider ones to the separate launches: they
// walk a lone long row faster (a hub row of 200 blocks 3.6 ms a solve against 2.8 in one launch, of 1,000
// blocks 11.1 against 12.6; 1,000 rows of 301 blocks 4.8 against 5.9).
constexpr int NA_WIDE = 256;
constexpr int NA_RESTARTS = 4;                // continuations from the true residual at most

struct NaScal {
    float bb, rz, rr, alpha, beta, tol2bb;
    int done, iters, maxit, bad;
    int lost;  // a workgroup of k_na_loop gave up waiting: x is incomplete
    int wide;  // a row has more than NA_WIDE blocks
};

// float offsets into the scratch array
constexpr size_t NA_MINV = 0;
constexpr size_t NA_R = NA_MINV + 9 * (size_t)NA_MAX;
constexpr size_t NA_Z = NA_R + 3 * (size_t)NA_MAX;
constexpr size_t NA_D = NA_Z + 3 * (size_t)NA_MAX;
constexpr size_t NA_Q = NA_D + 3 * (size_t)NA_MAX;
constexpr size_t NA_PART = NA_Q + 3 * (size_t)NA_MAX;  // 2 floats per workgroup
constexpr size_t NA_SCAL = NA_PART + 2 * (size_t)NA_MAXB;
constexpr size_t NA_SLOTS = NA_SCAL + 64;                    // 2 generations x 2 values x NA_MAXB 64-bit words
constexpr size_t NA_FLOATS = NA_SLOTS + 8 * (size_t)NA_MAXB;
static_assert(sizeof(NaScal) <= 64 * sizeof(float), "scalar record");

// The temporaries of every call on this GPU (about 5.5 MB).  Host code never passes this name
// to a kernel: it stands for the device array only in device code; the host uses the address
// hipGetSymbolAddress returns for the current device.
__device__ __align__(256) float scratch[NA_FLOATS];

struct NaPtr {
    float *Minv, *r, *z, *d, *q, *part;
    NaScal* sc;
    uint64_t* slots;
    unsigned long long ticks;  // bound of a wait of k_na_loop
    int loseWg, loseAt;        // (testing) a wait of workgroup loseWg counts as run out at this meeting, 0: none
};

NaPtr carve(float* base) {
    NaPtr p{};
    p.Minv = base + NA_MINV;
    p.r = base + NA_R;
    p.z = base + NA_Z;
    p.d = base + NA_D;
    p.q = base + NA_Q;
    p.part = base + NA_PART;
    p.sc = reinterpret_cast<NaScal*>(base + NA_SCAL);
    p.slots = reinterpret_cast<uint64_t*>(base + NA_SLOTS);
    return p;
}

__device__ __forceinline__ void mul3(const float* M, const float* v, float* o) {
    o[0] = M[0] * v[0] + M[1] * v[1] + M[2] * v[2];
    o[1] = M[3] * v[0] + M[4] * v[1] + M[5] * v[2];
    o[2] = M[6] * v[0] + M[7] * v[1] + M[8] * v[2];
}

// Fixed-order workgroup sum of two values (wave shuffles, then the waves in order).
__device__ void wg_sum2(float a, float b, float* out) {
    __shared__ float lds[2][NA_TB / 64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        a += __shfl_xor(a, o, 64);
        b += __shfl_xor(b, o, 64);
    }
    if (lane == 0) { lds[0][w] = a; lds[1][w] = b; }
    __syncthreads();
    if (threadIdx.x == 0) {
        float s0 = 0.0f, s1 = 0.0f;
        for (int k = 0; k < NA_TB / 64; k++) { s0 += lds[0][k]; s1 += lds[1][k]; }
        out[0] = s0;
        out[1] = s1;
    }
}

// M^-1 from the diagonal blocks, x = 0, r = b, z = d = M^-1 b; partials b.b and r.z.  A row
// without its diagonal block or with a column outside [0, n) raises `bad`: the set-up reduction
// then ends the solve before any SpMV, and the call returns CS_E_ARG.
__global__ void __launch_bounds__(NA_TB) k_na_init(int n, const int* __restrict__ rp, const int* __restrict__ ci,
                                                   const float* __restrict__ vals, const float* __restrict__ b,
                                                   float* __restrict__ x, NaPtr P) {
    const int i = blockIdx.x * NA_TB + threadIdx.x;
    float bb = 0.0f, rz = 0.0f;
    if (i < n) {
        int diag = -1;
        if (rp[i + 1] - rp[i] > NA_WIDE) P.sc->wide = 1;
        bool cols_ok = true;  // a column outside [0, n) would make the SpMV read outside the scratch vectors
        for (int k = rp[i]; k < rp[i + 1]; k++) {
            const int j = ci[k];
            cols_ok = cols_ok && j >= 0 && j < n;
            if (j == i && diag < 0) diag = k;
        }
        if (!cols_ok) P.sc->bad = 1;
        float a[9], m[9];
        if (diag >= 0) {
            for (int c = 0; c < 9; c++) a[c] = vals[(size_t)diag * 9 + c];
            inv3(a, m);
        } else {
            P.sc->bad = 1;  // the caller's matrix lacks a diagonal block
            for (int c = 0; c < 9; c++) m[c] = (c % 4 == 0) ? 1.0f : 0.0f;
        }
        for (int c = 0; c < 9; c++) P.Minv[(size_t)i * 9 + c] = m[c];
        float bi[3] = {b[3 * i], b[3 * i + 1], b[3 * i + 2]}, zi[3];
        mul3(m, bi, zi);
        for (int c = 0; c < 3; c++) {
            x[3 * i + c] = 0.0f;
            P.r[3 * i + c] = bi[c];
            P.z[3 * i + c] = zi[c];
            P.d[3 * i + c] = zi[c];
            bb += bi[c] * bi[c];
            rz += bi[c] * zi[c];
        }
    }
    wg_sum2(bb, rz, P.part + 2 * blockIdx.x);
}

// One workgroup: the partial sums in workgroup order.  mode 0: b.b and r.z of the start;
// mode 1: alpha = r.z / d.q; mode 2: r.r and the new r.z, the stop test and beta.
__global__ void __launch_bounds__(NA_TB) k_na_reduce(int nb, int mode, float tol2, int maxit, NaPtr P) {
    NaScal* sc = P.sc;
    if (mode != 0 && sc->done) return;
    float a = 0.0f, b = 0.0f;
    for (int k = threadIdx.x; k < nb; k += NA_TB) {
        a += P.part[2 * k];
        b += P.part[2 * k + 1];
    }
    __shared__ float tot[2];
    wg_sum2(a, b, tot);
    __syncthreads();
    if (threadIdx.x != 0) return;
    if (mode == 0) {
        sc->bb = tot[0];
        sc->rr = tot[0];
        sc->rz = tot[1];
        sc->tol2bb = tol2 * tot[0];
        sc->iters = 0;
        sc->maxit = maxit;
        sc->done = sc->bad || tot[0] <= tol2 * tot[0] || maxit <= 0;
    } else if (mode == 1) {
        sc->alpha = sc->rz / tot[0];
    } else {
        sc->rr = tot[0];
        sc->iters += 1;
        if (tot[0] <= sc->tol2bb || sc->iters >= sc->maxit || !(tot[0] <= FLT_MAX)) {  // NaN: breakdown
            sc->done = 1;
            return;
        }
        sc->beta = tot[1] / sc->rz;
        sc->rz = tot[1];
    }
}

// q = A d, partial d.q
__global__ void __launch_bounds__(NA_TB) k_na_spmv(int n, const int* __restrict__ rp, const int* __restrict__ ci,
                                                   const float* __restrict__ vals, NaPtr P) {
    if (P.sc->done) return;
    const int i = blockIdx.x * NA_TB + threadIdx.x;
    float dq = 0.0f;
    if (i < n) {
        float acc[3] = {0.0f, 0.0f, 0.0f};
        for (int k = rp[i]; k < rp[i + 1]; k++) {
            const int j = ci[k];
            const float* A = vals + (size_t)k * 9;
            const float dj[3] = {P.d[3 * j], P.d[3 * j + 1], P.d[3 * j + 2]};
            float t[3];
            mul3(A, dj, t);
            acc[0] += t[0];
            acc[1] += t[1];
            acc[2] += t[2];
        }
        for (int c = 0; c < 3; c++) {
            P.q[3 * i + c] = acc[c];
            dq += P.d[3 * i + c] * acc[c];
        }
    }
    wg_sum2(dq, 0.0f, P.part + 2 * blockIdx.x);
}

// x += alpha d, r -= alpha q, z = M^-1 r; partials r.r and r.z
__global__ void __launch_bounds__(NA_TB) k_na_update(int n, float* __restrict__ x, NaPtr P) {
    if (P.sc->done) return;
    const int i = blockIdx.x * NA_TB + threadIdx.x;
    float rr = 0.0f, rz = 0.0f;
    if (i < n) {
        const float alpha = P.sc->alpha;
        float ri[3], zi[3];
        for (int c = 0; c < 3; c++) {
            x[3 * i + c] += alpha * P.d[3 * i + c];
            ri[c] = P.r[3 * i + c] - alpha * P.q[3 * i + c];
            P.r[3 * i + c] = ri[c];
        }
        mul3(P.Minv + (size_t)i * 9, ri, zi);
        for (int c = 0; c < 3; c++) {
            P.z[3 * i + c] = zi[c];
            rr += ri[c] * ri[c];
            rz += ri[c] * zi[c];
        }
    }
    wg_sum2(rr, rz, P.part + 2 * blockIdx.x);
}

// d = z + beta d
__global__ void __launch_bounds__(NA_TB) k_na_dir(int n, NaPtr P) {
    if (P.sc->done) return;
    const int i = blockIdx.x * NA_TB + threadIdx.x;
    if (i >= n) return;
    const float beta = P.sc->beta;
    for (int c = 0; c < 3; c++) P.d[3 * i + c] = P.z[3 * i + c] + beta * P.d[3 * i + c];
}

// The true residual r = b - A x with FP64 row sums, z = M^-1 r and d = z (the direction
// restarted from it); partials r.r and r.z.
__global__ void __launch_bounds__(NA_TB) k_na_true(int n, const int* __restrict__ rp, const int* __restrict__ ci,
                                                   const float* __restrict__ vals, const float* __restrict__ b,
                                                   const float* __restrict__ x, NaPtr P) {
    const int i = blockIdx.x * NA_TB + threadIdx.x;
    float rr = 0.0f, rz = 0.0f;
    if (i < n) {
        double y[3] = {b[3 * i], b[3 * i + 1], b[3 * i + 2]};
        for (int k = rp[i]; k < rp[i + 1]; k++) {
            const int j = ci[k];
            const float* A = vals + (size_t)k * 9;
            for (int u = 0; u < 3; u++)
                y[u] -= (double)A[3 * u] * x[3 * j] + (double)A[3 * u + 1] * x[3 * j + 1] +
                        (double)A[3 * u + 2] * x[3 * j + 2];
        }
        const float ri[3] = {(float)y[0], (float)y[1], (float)y[2]};
        float zi[3];
        mul3(P.Minv + (size_t)i * 9, ri, zi);
        for (int c = 0; c < 3; c++) {
            P.r[3 * i + c] = ri[c];
            P.z[3 * i + c] = zi[c];
            P.d[3 * i + c] = zi[c];
            rr += ri[c] * ri[c];
            rz += ri[c] * zi[c];
        }
    }
    wg_sum2(rr, rz, P.part + 2 * blockIdx.x);
}

// Accept when the true residual meets the tolerance (or the budget is spent); otherwise reopen
// the loop with r.z of the replaced residual.
__global__ void __launch_bounds__(NA_TB) k_na_recheck(int nb, NaPtr P) {
    float a = 0.0f, b = 0.0f;
    for (int k = threadIdx.x; k < nb; k += NA_TB) {
        a += P.part[2 * k];
        b += P.part[2 * k + 1];
    }
    __shared__ float tot[2];
    wg_sum2(a, b, tot);
    __syncthreads();
    if (threadIdx.x != 0) return;
    NaScal* sc = P.sc;
    sc->rr = tot[0];
    sc->rz = tot[1];
    sc->done = (tot[0] <= sc->tol2bb || sc->iters >= sc->maxit || !(tot[0] <= FLT_MAX)) ? 1 : 0;
}

__global__ void k_na_clear(NaScal* sc) {
    if (threadIdx.x == 0) *sc = NaScal{};
}

// ---- the iterations in one launch ------------------------------------------
// Separate launches take 20 us an iteration, five of them (8,100 rows of up to 11 blocks), all latency.  Here
// an iteration is two meetings of the workgroups: for d.q, and for r.r and r.z, with which the new z
// becomes visible; each thread forms its neighbours' d = z + beta d itself.
// 8,100 rows of up to 11 blocks: a solve of 144 iterations 2.88 ms in separate launches, 1.44 here.  (One
// register spills, 8 B of scratch a lane.)
constexpr int NA_RS = 14;                                      // blocks of a row in registers
constexpr int NA_NT = 2;                                       // further blocks in flight together
constexpr unsigned long long NA_WAIT_TICKS = 200000000ull;     // 2 s of the 100 MHz wall clock; a wait's bound

typedef float f3u __attribute__((ext_vector_type(3), aligned(4)));

__device__ __forceinline__ void put1(float* p, float v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Sums v over the workgroups in the order of k_na_reduce; every thread gets them.  Each workgroup
// stores (epoch, partial) words, every workgroup polls all of them.  Stores that a thread made with
// put1 before the call are visible to all threads after it.  False if the wait ran out; *ranOut (LDS) is the
// meeting at which one did (they count from 1).
template <int NS>
__device__ bool na_meet(float (&v)[NS], int nb, unsigned ep, const NaPtr& P, unsigned* ranOut) {
    __shared__ float w0[2][NA_TB / 64], w1[2][NA_TB / 64];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
#pragma unroll
    for (int s = 0; s < NS; s++) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v[s] += __shfl_xor(v[s], o, 64);
        if (lane == 0) w0[s][w] = v[s];
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's stores are out
    __syncthreads();
    uint64_t* gen = P.slots + (ep & 1) * 2 * NA_MAXB;
    if (t < NS) {
        float p = 0.0f;
        for (int k = 0; k < NA_TB / 64; k++) p += w0[t][k];
        __hip_atomic_store(gen + t * NA_MAXB + blockIdx.x, (uint64_t)ep << 32 | __float_as_uint(p), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }
    float a[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) a[s] = 0.0f;
    if (t < nb) {
        unsigned long long since = 0;
        uint64_t word[NS];
        bool late = false;
        for (int spin = 0;; spin++) {
            bool all = true;
#pragma unroll
            for (int s = 0; s < NS; s++) {
                word[s] = __hip_atomic_load(gen + s * NA_MAXB + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                all = all && (unsigned)(word[s] >> 32) == ep;
            }
            if (all) break;
            if (late) {
                *ranOut = ep;
                break;
            }
            if ((spin & 1023) == 1023) {
                const unsigned long long now = wall_clock64();
                if (since == 0) since = now;
                late = now - since > P.ticks;  // the words are read once more after the deadline
            }
        }
#pragma unroll
        for (int s = 0; s < NS; s++) a[s] += __uint_as_float((unsigned)word[s]);
    }
#pragma unroll
    for (int s = 0; s < NS; s++) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) a[s] += __shfl_xor(a[s], o, 64);
        if (lane == 0) w1[s][w] = a[s];
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < NS; s++) {
        v[s] = 0.0f;
        for (int k = 0; k < NA_TB / 64; k++) v[s] += w1[s][k];
    }
    const bool ok = *ranOut != ep;
    if (t == 0) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");  // vectors cached before the meeting are dropped
    __syncthreads();
    return ok;
}

// The iterations from P's r, z = d and scalars to a stop.  nb = gridDim.x <= NA_MAXB workgroups, all
// resident; the slots are zero at launch.  A workgroup whose wait runs out leaves without its rows of x
// and says so in P's record: after the last meeting no other would notice.
__global__ void __launch_bounds__(NA_TB, 2) k_na_loop(int n, const int* __restrict__ rp, const int* __restrict__ ci,
                                                      const float* __restrict__ vals, float* __restrict__ x, NaPtr P) {
    __shared__ unsigned ranOut;
    if (P.sc->done || P.sc->wide) return;
    if (threadIdx.x == 0) ranOut = P.loseWg == (int)blockIdx.x ? P.loseAt : 0;
    auto lost = [&]() {
        if (threadIdx.x == 0) P.sc->lost = 1;
    };
    const int i = blockIdx.x * NA_TB + threadIdx.x, ic = min(i, n - 1), nb = gridDim.x;
    const bool live = i < n;
    const int k0 = rp[ic], k1 = live ? rp[ic + 1] : k0;
    const float tol2bb = P.sc->tol2bb;
    const int maxit = P.sc->maxit;
    float rz = P.sc->rz, rr = P.sc->rr, beta = 0.0f;
    int it = P.sc->iters;
    const int first = it;
    float a[NA_RS][9], m[9], xi[3], r[3], z[3], d[3], q[3];
    unsigned short col[NA_RS];  // n <= 65,536
#pragma unroll
    for (int k = 0; k < NA_RS; k++) {
        const bool in = k0 + k < k1;
        const int kk = in ? k0 + k : rp[ic];  // (every row has its diagonal block)
        col[k] = (unsigned short)(in ? ci[kk] : ic);
#pragma unroll
        for (int c = 0; c < 9; c++) {
            const float v = vals[(size_t)kk * 9 + c];
            a[k][c] = in ? v : 0.0f;
        }
    }
#pragma unroll
    for (int c = 0; c < 9; c++) m[c] = P.Minv[(size_t)ic * 9 + c];
#pragma unroll
    for (int c = 0; c < 3; c++) {
        xi[c] = x[3 * ic + c];
        r[c] = live ? P.r[3 * ic + c] : 0.0f;
        z[c] = live ? P.z[3 * ic + c] : 0.0f;
        d[c] = 0.0f;
    }
    unsigned ep = 0;
    __syncthreads();
    for (;; ) {
        // q = A d, d = z + beta d
        const float *dp = it & 1 ? P.d : P.q;
        float* dn = it & 1 ? P.q : P.d;
        auto dir = [&](int j, float (&o)[3]) {
#pragma unroll
            for (int c = 0; c < 3; c++) {
                const float zj = P.z[3 * j + c];
                o[c] = it == first ? zj : zj + beta * dp[3 * j + c];
            }
        };
#pragma unroll
        for (int c = 0; c < 3; c++) {
            q[c] = 0.0f;
            d[c] = it == first ? z[c] : z[c] + beta * d[c];
        }
        auto add = [&](const float* A, const float* v) {
            float t[3];
            mul3(A, v, t);
            q[0] += t[0];
            q[1] += t[1];
            q[2] += t[2];
        };
#pragma unroll
        for (int g = 0; g < NA_RS; g += 7) {
            float w[7][3];
#pragma unroll
            for (int u = 0; u < 7; u++) dir(col[g + u], w[u]);
#pragma unroll
            for (int u = 0; u < 7; u++) add(a[g + u], w[u]);
        }
        // further blocks, NA_NT in flight together, a row's vector in one load: bound by the loads a lone lane
        // issues (30,000 rows of 101 blocks: 25.6 ms in separate launches, 29.0 here with scalar loads one block
        // at a time, 20.7 now), which the blocks in registers are not (there the wider loads spill and lose 10 %)
        for (int k = k0 + NA_RS; k < k1; k += NA_NT) {
            float A[NA_NT][9], w[NA_NT][3];
#pragma unroll
            for (int u = 0; u < NA_NT; u++) {
                const int kk = min(k + u, k1 - 1), j = ci[kk];
#pragma unroll
                for (int c = 0; c < 9; c++) A[u][c] = vals[(size_t)kk * 9 + c];
                const f3u zj = *(const f3u*)(P.z + 3 * j);
                f3u dj = zj;
                if (it != first) dj = *(const f3u*)(dp + 3 * j);
#pragma unroll
                for (int c = 0; c < 3; c++) w[u][c] = it == first ? zj[c] : zj[c] + beta * dj[c];
            }
#pragma unroll
            for (int u = 0; u < NA_NT; u++)
                if (k + u < k1) add(A[u], w[u]);
        }
        float v1[1] = {0.0f};
        if (live)
#pragma unroll
            for (int c = 0; c < 3; c++) {
                put1(dn + 3 * i + c, d[c]);
                v1[0] += d[c] * q[c];
            }
        if (!na_meet<1>(v1, nb, ++ep, P, &ranOut)) return lost();
        const float alpha = rz / v1[0];
        float v2[2] = {0.0f, 0.0f};
#pragma unroll
        for (int c = 0; c < 3; c++) {
            xi[c] += alpha * d[c];
            r[c] = live ? r[c] - alpha * q[c] : 0.0f;
        }
        mul3(m, r, z);
        if (live)
#pragma unroll
            for (int c = 0; c < 3; c++) {
                put1(P.z + 3 * i + c, z[c]);
                v2[0] += r[c] * r[c];
                v2[1] += r[c] * z[c];
            }
        if (!na_meet<2>(v2, nb, ++ep, P, &ranOut)) return lost();
        rr = v2[0];
        it++;
        if (rr <= tol2bb || it >= maxit || !(rr <= FLT_MAX)) break;  // NaN: breakdown
        beta = v2[1] / rz;
        rz = v2[1];
    }
    if (live)
#pragma unroll
        for (int c = 0; c < 3; c++) x[3 * i + c] = xi[c];
    if (i == 0) {
        P.sc->rr = rr;
        P.sc->rz = rz;
        P.sc->iters = it;
        P.sc->done = 1;
    }
}

__global__ void k_na_clear_slots(uint64_t* slots) {
    slots[blockIdx.x * NA_TB + threadIdx.x] = 0;
}

// The scratch address on each device, looked up once per device with that device current, and whether the
// device's next call attempts the one launch (both paths give the same bits).
std::mutex gNaMutex;
struct NaDevice {
    float* base = nullptr;
    OneLaunch once;
} gNaDevice[64];

NaDevice& current_device() {
    int dev = 0;
    CS_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= 64) throw StatusError(CS_E_NO_DEVICE, "device index out of range");
    std::lock_guard<std::mutex> lock(gNaMutex);
    if (!gNaDevice[dev].base) {
        void* p = nullptr;
        CS_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        gNaDevice[dev].base = static_cast<float*>(p);
    }
    return gNaDevice[dev];
}

// The iterations in one launch.  False: refused (another process holds the device's cooperative
// queue, or the device has too few CUs), nothing was done.
bool loop_at_once(hipStream_t s, int nb, int n, const int* rp, const int* ci, const float* vals, float* x, NaPtr P,
                  bool refuse) {
    if (refuse) return false;
    hipLaunchKernelGGL(k_na_clear_slots, dim3(4 * NA_MAXB / NA_TB), dim3(NA_TB), 0, s, P.slots);
    CS_LAUNCH_CHECK();
    void* args[] = {(void*)&n, (void*)&rp, (void*)&ci, (void*)&vals, (void*)&x, (void*)&P};
    if (hipLaunchCooperativeKernel((const void*)k_na_loop, dim3(nb), dim3(NA_TB), args, 0, s) == hipSuccess) return true;
    (void)hipGetLastError();
    return false;
}

int solve_noalloc(hipStream_t s, int n, const int* rp, const int* ci, const float* vals, const float* b, float* x,
                  float tol, int maxit, int* iters, float* relres, const cs_launch_fault& fault, int* launches) {
    NaDevice& dev = current_device();
    auto locked = [&](auto&& f) {
        std::lock_guard<std::mutex> lock(gNaMutex);
        return f(dev.once);
    };
    NaPtr P = carve(dev.base);
    P.ticks = fault.wait_s > 0.0f ? (unsigned long long)(fault.wait_s * 1e8f) : NA_WAIT_TICKS;
    P.loseWg = fault.lose_wg;
    P.loseAt = fault.lose_at;
    const int nb = cdiv(n, NA_TB);
    NaScal h{};
    auto start = [&]() {
        // the scalar record starts cleared: `bad` is only ever raised by the set-up kernel
        hipLaunchKernelGGL(k_na_clear, dim3(1), dim3(64), 0, s, P.sc);
        CS_LAUNCH_CHECK();
        hipLaunchKernelGGL(k_na_init, dim3(nb), dim3(NA_TB), 0, s, n, rp, ci, vals, b, x, P);
        CS_LAUNCH_CHECK();
        hipLaunchKernelGGL(k_na_reduce, dim3(1), dim3(NA_TB), 0, s, nb, 0, tol * tol, maxit, P);
        CS_LAUNCH_CHECK();
    };
    auto read = [&]() {
        CS_HIP(hipMemcpyAsync(&h, P.sc, sizeof(NaScal), hipMemcpyDeviceToHost, s));
        CS_HIP(hipStreamSynchronize(s));
    };
    start();
    bool once = locked([](OneLaunch& o) { return o.attempt(); });
    int restart = 0;
    // The loop stops on its recursive residual; as in cs_solve, only the true residual (FP64 row
    // sums) accepts the result, otherwise the loop goes on from it, at most NA_RESTARTS times.
    for (;; restart++) {
        if (once) {
            once = loop_at_once(s, nb, n, rp, ci, vals, x, P, fault.refuse != 0);
            read();
            if (!once) {
                locked([](OneLaunch& o) { o.refused(); });
            } else if (h.lost || !(h.done || h.wide)) {  // a wait ran out: from the start
                locked([](OneLaunch& o) { o.ranOut(); });
                once = false;
                restart = 0;
                start();
            } else {
                locked([](OneLaunch& o) { o.worked(); });
                once = h.done;  // not done: rows too wide, the solve is as it was
            }
        }
        if (!once)
            for (int done = 0; done <= maxit; done += NA_CHUNK) {
                read();
                if (h.done) break;
                for (int k = 0; k < NA_CHUNK; k++) {
                    hipLaunchKernelGGL(k_na_spmv, dim3(nb), dim3(NA_TB), 0, s, n, rp, ci, vals, P);
                    hipLaunchKernelGGL(k_na_reduce, dim3(1), dim3(NA_TB), 0, s, nb, 1, 0.0f, 0, P);
                    hipLaunchKernelGGL(k_na_update, dim3(nb), dim3(NA_TB), 0, s, n, x, P);
                    hipLaunchKernelGGL(k_na_reduce, dim3(1), dim3(NA_TB), 0, s, nb, 2, 0.0f, 0, P);
                    hipLaunchKernelGGL(k_na_dir, dim3(nb), dim3(NA_TB), 0, s, n, P);
                }
                CS_LAUNCH_CHECK();
            }
        if (!once) read();
        if (h.bad) return CS_E_ARG;
        if (!h.done) throw StatusError(CS_E_HIP, "no-allocation PCG: the device never reported its stop");
        hipLaunchKernelGGL(k_na_true, dim3(nb), dim3(NA_TB), 0, s, n, rp, ci, vals, b, x, P);
        hipLaunchKernelGGL(k_na_recheck, dim3(1), dim3(NA_TB), 0, s, nb, P);
        CS_LAUNCH_CHECK();
        read();
        if (h.done || restart == NA_RESTARTS) break;
    }
    if (iters) *iters = h.iters;
    if (relres) *relres = h.bb > 0.0f ? sqrtf(h.rr / h.bb) : 0.0f;
    if (launches) *launches = once ? 1 + restart : 0;
    return h.rr <= h.tol2bb ? CS_OK : CS_E_NOT_CONVERGED;
}

}  // namespace

}  // namespace cs

extern "C" cs_status cs_solve_bsr_noalloc(void* stream, int n_nodes, const int* row_ptr, const int* col_idx,
                                          const float* vals, const float* b, float* x, float rel_tol, int max_iters,
                                          int* iters, float* rel_residual) {
    return cs_solve_bsr_noalloc_test(stream, n_nodes, row_ptr, col_idx, vals, b, x, rel_tol, max_iters, iters,
                                     rel_residual, nullptr, nullptr);
}

extern "C" cs_status cs_solve_bsr_noalloc_test(void* stream, int n_nodes, const int* row_ptr, const int* col_idx,
                                               const float* vals, const float* b, float* x, float rel_tol,
                                               int max_iters, int* iters, float* rel_residual,
                                               const cs_launch_fault* fault, int* launches) {
    if (n_nodes > CS_NOALLOC_MAX_NODES) return CS_E_CAPACITY;
    if (n_nodes < 1 || !row_ptr || !col_idx || !vals || !b || !x || !(rel_tol > 0.0f) || !(rel_tol < 1.0f) ||
        max_iters < 0)
        return CS_E_ARG;
    try {
        return static_cast<cs_status>(cs::solve_noalloc(static_cast<hipStream_t>(stream), n_nodes, row_ptr, col_idx,
                                                        vals, b, x, rel_tol, max_iters, iters, rel_residual,
                                                        fault ? *fault : cs_launch_fault{}, launches));
    } catch (const cs::StatusError& e) {
        return static_cast<cs_status>(e.status);
    } catch (const std::exception&) {
        return CS_E_HIP;
    }
}
