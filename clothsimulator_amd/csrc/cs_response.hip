// cs_response.hip — impact response: the augmented-Lagrangian gradient solve of
// CollisionOptimization (src/optimization/CollisionOptimization.cu:3-145,
// src/optimization/Optimization.cu:98-181), kept to reference semantics.
//
//   minimise   1/2 invMass sum_u m_u |x_u - x1_u|^2
//   subject to c_i = sum_j w_ij n_i . x_ij - thickness >= 0       (one per impact)
// mu = 1e3, clampViolation(x, +1) = min(x, 0), backtracking factor 0.7,
// <= 100 iterations, stops on s < 1e-12 or |f - ft| < 1e-10.
//
// The impact nodes are de-duplicated by a stable radix sort of (node, slot),
// which also gives every node the list of its constraint slots in ascending
// order, so gradients are gathered (no atomics).  The whole iteration, line
// search included, runs in one workgroup: the reference's host round trip per
// line-search evaluation is gone.  Up to LDS_SLOTS constraint slots the solve
// stays in registers and LDS (k_opt_solve_lds); above, k_opt_solve keeps
// them in memory.  Both add in the same order and give the same bits.
#include "cs_kernels.hpp"
#include "cs_math.hpp"

namespace cs {

namespace {

constexpr int OB = 1024;

// The constraints c_i = sum_j w_ij n_i . x_ij - thickness as the two stages store them: impacts
// (4 nodes, FP64 record fields) and separation constraints (6 nodes: the two faces' points).
struct ImpView {
    static constexpr int K = 4;
    const cs_impact_rec* r;
    __device__ int node(int i, int j) const { return r[i].nodes[j]; }
    __device__ float w(int i, int j) const { return (float)r[i].w[j]; }
    __device__ V3f n(int i) const { return mk((float)r[i].n[0], (float)r[i].n[1], (float)r[i].n[2]); }
};
struct SepView {
    static constexpr int K = 6;
    const SepRec* r;
    __device__ int node(int i, int j) const { return r[i].nodes[j]; }
    __device__ float w(int i, int j) const { return r[i].w[j]; }
    __device__ V3f n(int i) const { return mk(r[i].n[0], r[i].n[1], r[i].n[2]); }
};

template <class View>
__global__ void k_opt_collect(int m, View V, int deform, int NC, int N, uint64_t* __restrict__ keys,
                              uint32_t* __restrict__ vals) {
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= m) return;
    int nd = V.node(s / View::K, s % View::K);
    keys[s] = (deform == 1 || nd < NC) ? (uint64_t)nd : (uint64_t)N;
    vals[s] = (uint32_t)s;
}

__global__ void k_opt_heads(int m, int N, const uint64_t* __restrict__ keys, uint32_t* __restrict__ flag) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= m) return;
    flag[k] = (keys[k] < (uint64_t)N && (k == 0 || keys[k - 1] != keys[k])) ? 1u : 0u;
}

__global__ void k_opt_map(int m, int N, const uint64_t* __restrict__ keys, const uint32_t* __restrict__ vals,
                          const uint32_t* __restrict__ flag, const uint32_t* __restrict__ pos, int* __restrict__ nodes,
                          int* __restrict__ start, int* __restrict__ end, int* __restrict__ slotMap) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= m) return;
    uint64_t key = keys[k];
    if (key >= (uint64_t)N) return;
    int u = (int)(pos[k] + flag[k]) - 1;
    slotMap[vals[k]] = u;
    if (flag[k]) { nodes[u] = (int)key; start[u] = k; }
    if (k + 1 == m || keys[k + 1] != key) end[u] = k + 1;
}

template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}

// The sum over a wavefront, in every lane.  The pairs are those of shuffles by 32, 16, 8, 4, 2, 1:
// after the step by 8 a row holds equal values 8 lanes apart, so a rotation by 4 reads the partner
// of the shuffle by 4, and so on down.
__device__ __forceinline__ float wave_sum(float v) {
    auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(h[0]) + __uint_as_float(h[1]);
    auto q = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(q[0]) + __uint_as_float(q[1]);
    v = dpp_add<0x128>(v);  // row_ror:8
    v = dpp_add<0x124>(v);
    v = dpp_add<0x122>(v);
    return dpp_add<0x121>(v);
}

// Sums of two values over the workgroup (the wavefronts in order) with one barrier of its own; the
// caller has another between two sums (part is read after the barrier).
template <int T>
__device__ __forceinline__ float2 wg_sum2(float a, float b, float2* part) {
    a = wave_sum(a);
    b = wave_sum(b);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = make_float2(a, b);
    __syncthreads();
    float2 s = make_float2(0.0f, 0.0f);
#pragma unroll
    for (int w = 0; w < T / 64; w++) {
        s.x += part[w].x;
        s.y += part[w].y;
    }
    return s;
}

template <class View>
struct OptArgs {
    int nC;
    const uint32_t* nNptr;  // unique node count (scan total)
    View V;
    const int* nodes;
    const int* start;
    const int* end;
    const int* slotMap;
    const uint32_t* sortedSlots;
    float4* x;
    const float4* x1;
    const float* mass;  // per node: the objective's weight (mass for impacts, area for separation)
    int NC;
    float obstacleMass, thickness;  // obstacle nodes' weight
    // k_opt_solve's working set.  Per node: position, gradient, target and weight.  pos: node u's
    // trial position at u, a fixed slot's at its sorted place.  con: normal and coefficient.
    // rec, in node order: a slot's constraint (int bits) and weight; slot, by slot: where its
    // position is (int bits) and its weight.
    float4 *X, *G, *X1, *pos, *con;
    float2 *rec, *slot;
    float *lambda, *c;
};

// The solve of any size: thread t owns the nodes and constraints t, t + OB, ...  What it reads per
// evaluation is gathered once into short FP32 records; the constraint values and the objective of an
// accepted line-search point are those of the next evaluation and are not computed again.  Bound by
// the latency of slot -> position: positions and coefficients are in LDS while they fit (1,025 random
// impacts, 100 steps: 0.97 ms with them in memory, 0.64 in LDS; 2,000: 0.87; 2,023, in memory: 1.43).
template <class View, bool LDS>
__global__ void __launch_bounds__(OB) k_opt_solve(OptArgs<View> A, int* iterOut) {
    constexpr int K = View::K;
    extern __shared__ float4 mem[];
    __shared__ float2 part[OB / 64];
    const int nN = (int)*A.nNptr;
    if (nN == 0) return;
    const int m = K * A.nC, t = threadIdx.x;
    float4 *pos, *con;
    if constexpr (LDS) { pos = mem; con = mem + m; }
    else { pos = A.pos; con = A.con; }
    for (int k = t; k < m; k += OB) {
        const int slot = (int)A.sortedSlots[k], i = slot / K, j = slot % K, u = A.slotMap[slot];
        const float w = A.V.w(i, j);
        A.rec[k] = make_float2(__int_as_float(i), w);
        A.slot[slot] = make_float2(__int_as_float(u > -1 ? u : k), w);
        if (u < 0) pos[k] = A.x[A.V.node(i, j)];
    }
    float im = 0.0f, a = 0.0f;
    for (int u = t; u < nN; u += OB) {
        const int nd = A.nodes[u];
        const V3f x = ld3(A.x[nd]), x1 = ld3(A.x1[nd]);
        const float mass = nd < A.NC ? A.mass[nd] : A.obstacleMass;
        A.X[u] = pos[u] = st4(x);
        A.X1[u] = st4(x1, mass);
        im += 1.0f / mass;
        a += mass * norm2(x - x1);
    }
    const float2 ia = wg_sum2<OB>(im, a, part);
    const float invMass = ia.x / (float)nN;
    float obj = 0.5f * ia.y * invMass;
    const float mu = 1e3f;
    // c_i at the published positions
    auto constraint_at = [&](int i, V3f n) {
        float c = -A.thickness;
#pragma unroll
        for (int j = 0; j < K; j++) {
            const float2 q = A.slot[K * i + j];
            c += q.y * dot(n, ld3(pos[__float_as_int(q.x)]));
        }
        return c;
    };
    auto penalty = [&](float coef) { return coef != 0.0f ? 0.5f * mu * (coef * coef) : 0.0f; };
    for (int i = t; i < A.nC; i += OB) {
        const V3f n = A.V.n(i);
        con[i] = st4(n);
        A.lambda[i] = 0.0f;
        A.c[i] = constraint_at(i, n);
    }
    float s = 1e-3f * (float)nN;
    int iter = 0;
    for (; iter < 100; iter++) {
        // valueAndGradient (src/optimization/Optimization.cu:33-49)
        float pen = 0.0f;
        for (int i = t; i < A.nC; i += OB) {
            const float coef = tmin(A.c[i] + A.lambda[i] / mu, 0.0f);
            con[i].w = coef;
            pen += penalty(coef);
        }
        __syncthreads();
        float g2 = 0.0f;
        for (int u = t; u < nN; u += OB) {
            const float4 x1 = A.X1[u];
            V3f g = (invMass * x1.w) * (ld3(A.X[u]) - ld3(x1));
            const int last = A.end[u];
            float2 next = A.rec[A.start[u]];
            for (int k = A.start[u]; k < last; k++) {
                const float2 q = next;
                next = A.rec[tmin(k + 1, m - 1)];
                const float4 e = con[__float_as_int(q.x)];
                if (e.w != 0.0f) g += ((mu * e.w) * q.y) * ld3(e);
            }
            A.G[u] = st4(g);
            g2 += norm2(g);
        }
        const float2 pg = wg_sum2<OB>(pen, g2, part);
        const float f = obj + pg.x, norm2g = pg.y;
        s /= 0.7f;
        float ft, objt;
        do {
            s *= 0.7f;
            a = 0.0f;
            for (int u = t; u < nN; u += OB) {
                const V3f x = ld3(A.X[u]) - s * ld3(A.G[u]);
                const float4 x1 = A.X1[u];
                pos[u] = st4(x);
                a += x1.w * norm2(x - ld3(x1));
            }
            __syncthreads();
            pen = 0.0f;
            for (int i = t; i < A.nC; i += OB) {
                const float c = constraint_at(i, ld3(con[i]));
                A.c[i] = c;
                pen += penalty(tmin(c + A.lambda[i] / mu, 0.0f));
            }
            const float2 op = wg_sum2<OB>(a, pen, part);
            objt = 0.5f * op.x * invMass;
            ft = objt + op.y;
        } while (ft >= f - 0.5f * s * norm2g && s >= 1e-12f && tabs(f - ft) >= 1e-10f);
        if (s < 1e-12f || tabs(f - ft) < 1e-10f) break;
        for (int u = t; u < nN; u += OB) A.X[u] = pos[u];
        obj = objt;
        // updateMultiplier (src/optimization/Optimization.cu:51-57)
        for (int i = t; i < A.nC; i += OB) A.lambda[i] = tmin(A.lambda[i] + mu * A.c[i], 0.0f);
    }
    for (int u = t; u < nN; u += OB) A.x[A.nodes[u]] = A.X[u];
    if (t == 0 && iterOut) *iterOut = iter;
}

// ---- the solve in registers and LDS ----------------------------------------
// The solve is a serial chain of up to 100 gradient steps, each a few short sums over at most some
// thousand nodes and constraints, so latency bounds it.  Here a thread keeps its nodes (position,
// gradient, target, weight) and its constraint (normal, weights, multiplier) in registers;
// positions, coefficients and the slot lists are in LDS.  A cloth of 129x129 nodes draped on a
// sphere: 0.72 ms a call with every operand in memory and three barriers per sum, 0.19 ms here (100
// steps); 16 / 64 / 256 / 1024 random impacts, 100 steps: 0.11 / 0.14 / 0.23 / 0.42 ms.
constexpr int LDS_SLOTS = 4 * OB;
constexpr int LDS_SMALL = 256;  // one slot per thread of four wavefronts
constexpr size_t LDS_POS_BYTES = 158 * 1024;  // of 160 KiB

// LDS, in bytes per slot and constraint: 16 position, 8 (constraint, weight) in node order, 4 the
// slot's position; 16 normal and coefficient.
constexpr size_t lds_bytes(int K, int nC) { return (size_t)K * nC * 28 + (size_t)nC * 16; }

// T threads of NU nodes each: K * nC <= T * NU (a node has a slot), nC <= T.
template <class View, int T, int NU>
__global__ void __launch_bounds__(T) k_opt_solve_lds(OptArgs<View> A, int* iterOut) {
    constexpr int K = View::K;
    extern __shared__ float4 mem[];
    __shared__ float2 part[T / 64];
    const int nN = (int)*A.nNptr;
    if (nN == 0) return;
    const int m = K * A.nC, t = threadIdx.x;
    float4* pos = mem;                                  // [m]: node u at u, a fixed slot at its sorted place (>= nN)
    float4* con = pos + m;                              // [nC]: normal, coefficient
    float2* rec = reinterpret_cast<float2*>(con + A.nC);  // [m]: constraint (int bits), weight
    int* at = reinterpret_cast<int*>(rec + m);          // [m]: where the slot's position is

    for (int k = t; k < m; k += T) {
        const int slot = (int)A.sortedSlots[k], i = slot / K, j = slot % K, u = A.slotMap[slot];
        rec[k] = make_float2(__int_as_float(i), A.V.w(i, j));
        at[slot] = u > -1 ? u : k;
        if (u < 0) pos[k] = A.x[A.V.node(i, j)];
    }
    V3f X[NU], G[NU], X1[NU];
    float mass[NU];
    int first[NU], last[NU];
    float im = 0.0f, a = 0.0f;
#pragma unroll
    for (int r = 0; r < NU; r++) {
        const int u = t + r * T;
        X[r] = G[r] = X1[r] = mk(0.0f, 0.0f, 0.0f);
        mass[r] = 0.0f;
        first[r] = last[r] = 0;
        if (u < nN) {
            const int nd = A.nodes[u];
            X[r] = ld3(A.x[nd]);
            X1[r] = ld3(A.x1[nd]);
            mass[r] = nd < A.NC ? A.mass[nd] : A.obstacleMass;
            first[r] = A.start[u];
            last[r] = A.end[u];
            pos[u] = st4(X[r]);
            im += 1.0f / mass[r];
            a += mass[r] * norm2(X[r] - X1[r]);
        }
    }
    const float2 ia = wg_sum2<T>(im, a, part);
    const float invMass = ia.x / (float)nN;
    float obj = 0.5f * ia.y * invMass;
    V3f n = mk(0.0f, 0.0f, 0.0f);
    float w[K], lambda = 0.0f;
    int p[K];
    if (t < A.nC) {
        n = A.V.n(t);
#pragma unroll
        for (int j = 0; j < K; j++) {
            w[j] = A.V.w(t, j);
            p[j] = at[K * t + j];
        }
    }
    const float mu = 1e3f;
    // c_t at the published positions
    auto constraint_at = [&]() {
        float c = -A.thickness;
#pragma unroll
        for (int j = 0; j < K; j++) c += w[j] * dot(n, ld3(pos[p[j]]));
        return c;
    };
    auto penalty = [&](float coef) { return coef != 0.0f ? 0.5f * mu * (coef * coef) : 0.0f; };
    // the objective's terms at X - s G
    auto distance = [&](float s) {
        float a = 0.0f;
#pragma unroll
        for (int r = 0; r < NU; r++)
            if (t + r * T < nN) a += mass[r] * norm2((X[r] - s * G[r]) - X1[r]);
        return a;
    };
    float c = t < A.nC ? constraint_at() : 0.0f;
    float s = 1e-3f * (float)nN;
    int iter = 0;
    for (; iter < 100; iter++) {
        // valueAndGradient (src/optimization/Optimization.cu:33-49)
        float pen = 0.0f;
        if (t < A.nC) {
            const float coef = tmin(c + lambda / mu, 0.0f);
            con[t] = make_float4(n.x, n.y, n.z, coef);
            pen = penalty(coef);
        }
        __syncthreads();
        float g2 = 0.0f;
#pragma unroll
        for (int r = 0; r < NU; r++) {
            if (t + r * T >= nN) continue;
            V3f g = (invMass * mass[r]) * (X[r] - X1[r]);
            for (int k = first[r]; k < last[r]; k++) {
                const float2 q = rec[k];
                const float4 e = con[__float_as_int(q.x)];
                if (e.w != 0.0f) g += ((mu * e.w) * q.y) * mk(e.x, e.y, e.z);
            }
            G[r] = g;
            g2 += norm2(g);
        }
        const float2 pg = wg_sum2<T>(pen, g2, part);
        const float f = obj + pg.x, norm2g = pg.y;
        s /= 0.7f;
        float ft, objt;
        do {
            s *= 0.7f;
#pragma unroll
            for (int r = 0; r < NU; r++)
                if (t + r * T < nN) pos[t + r * T] = st4(X[r] - s * G[r]);
            __syncthreads();
            pen = 0.0f;
            if (t < A.nC) {
                c = constraint_at();
                pen = penalty(tmin(c + lambda / mu, 0.0f));
            }
            const float2 op = wg_sum2<T>(distance(s), pen, part);
            objt = 0.5f * op.x * invMass;
            ft = objt + op.y;
        } while (ft >= f - 0.5f * s * norm2g && s >= 1e-12f && tabs(f - ft) >= 1e-10f);
        if (s < 1e-12f || tabs(f - ft) < 1e-10f) break;
#pragma unroll
        for (int r = 0; r < NU; r++)
            if (t + r * T < nN) X[r] = X[r] - s * G[r];
        obj = objt;
        // updateMultiplier (src/optimization/Optimization.cu:51-57)
        if (t < A.nC) lambda = tmin(lambda + mu * c, 0.0f);
    }
#pragma unroll
    for (int r = 0; r < NU; r++)
        if (t + r * T < nN) A.x[A.nodes[t + r * T]] = st4(X[r]);
    if (t == 0 && iterOut) *iterOut = iter;
}

template <class View, int T, int NU>
void launch_lds(const OptArgs<View>& A, int* iterOut, hipStream_t s) {
    hipLaunchKernelGGL((k_opt_solve_lds<View, T, NU>), dim3(1), dim3(T), lds_bytes(View::K, A.nC), s, A, iterOut);
}

template <class View>
void opt_response(cs_ctx* C, View V, int nImp, int deform, const float* weight, float obstacleWeight) {
    if (nImp <= 0) return;
    hipStream_t s = C->stream;
    const int m = View::K * nImp;
    uint64_t* keys = C->optKeys.as<uint64_t>(m);
    uint64_t* ktmp = C->optKeysTmp.as<uint64_t>(m);
    uint32_t* vals = C->optVals.as<uint32_t>(m);
    uint32_t* vtmp = C->optValsTmp.as<uint32_t>(m);
    uint32_t* flag = C->optFlag.as<uint32_t>(m + 1);
    uint32_t* pos = C->optPos.as<uint32_t>(m + 1);
    int* nodes = C->optNodes.as<int>(m);
    int* start = C->optStart.as<int>(2 * (size_t)m);
    int* end = start + m;
    int* slotMap = C->optSlot.as<int>(m);
    hipLaunchKernelGGL(k_opt_collect<View>, dim3(cdiv(m, 256)), dim3(256), 0, s, m, V, deform, C->NC, C->N, keys,
                       vals);
    CS_LAUNCH_CHECK();
    int bits = 1;
    while ((1L << bits) <= C->N) bits++;
    radix_sort_pairs(keys, vals, ktmp, vtmp, m, 0, bits, C->ws, s);
    hipLaunchKernelGGL(k_opt_heads, dim3(cdiv(m, 256)), dim3(256), 0, s, m, C->N, keys, flag);
    CS_LAUNCH_CHECK();
    scan_exclusive(flag, pos, m, C->ws, s);
    fill_u32(reinterpret_cast<uint32_t*>(slotMap), 0xffffffffu, m, s);
    hipLaunchKernelGGL(k_opt_map, dim3(cdiv(m, 256)), dim3(256), 0, s, m, C->N, keys, vals, flag, pos, nodes, start,
                       end, slotMap);
    CS_LAUNCH_CHECK();
    OptArgs<View> A{};
    A.nC = nImp;
    A.nNptr = pos + m;
    A.V = V;
    A.nodes = nodes; A.start = start; A.end = end; A.slotMap = slotMap; A.sortedSlots = vals;
    A.x = C->x.ptr<float4>(); A.x1 = C->x1.ptr<float4>(); A.mass = weight;
    A.NC = C->NC;
    A.obstacleMass = obstacleWeight;
    A.thickness = C->P.collision_thickness;
    const size_t posBytes = sizeof(float4) * ((size_t)m + nImp);
    const bool ldsPos = posBytes <= LDS_POS_BYTES;
    if (m > LDS_SLOTS) {
        A.X = C->optX.as<float4>(2 * (size_t)m);
        A.X1 = A.X + m;
        if (!ldsPos) {
            A.pos = C->optNext.as<float4>(m);
            A.con = C->optCoef.as<float4>(nImp);
        }
        A.rec = reinterpret_cast<float2*>(C->optGrad.as<float4>(2 * (size_t)m));
        A.slot = A.rec + m;
        A.G = reinterpret_cast<float4*>(A.slot + m);
        A.lambda = C->optLambda.as<float>(2 * (size_t)nImp);
        A.c = A.lambda + nImp;
    }
    int* iterOut = C->optScal.as<int>(4);
    // A slot per thread while the slots fit a workgroup of four or sixteen wavefronts (fewer waves
    // make shorter barriers and sums), four up to LDS_SLOTS (LDS: 128 KiB then).
    if (m <= LDS_SMALL) launch_lds<View, LDS_SMALL, 1>(A, iterOut, s);
    else if (m <= OB) launch_lds<View, OB, 1>(A, iterOut, s);
    else if (m <= LDS_SLOTS) launch_lds<View, OB, 4>(A, iterOut, s);
    else if (ldsPos) hipLaunchKernelGGL((k_opt_solve<View, true>), dim3(1), dim3(OB), posBytes, s, A, iterOut);
    else hipLaunchKernelGGL((k_opt_solve<View, false>), dim3(1), dim3(OB), 0, s, A, iterOut);
    CS_LAUNCH_CHECK();
}

}  // namespace

void collision_response(cs_ctx* C, int nImp, int deform, float obstacleMass) {
    ImpView V;
    V.r = C->impAcc.ptr<cs_impact_rec>();
    opt_response(C, V, nImp, deform, C->mass.ptr<float>(), obstacleMass);
}

// SeparationOptimization (src/optimization/SeparationOptimization.cu:3-158): the same solve with
// per-node area weights (obstacle nodes: obstacleArea) and 6-node constraints.
void separation_response(cs_ctx* C, const SepRec* recs, int n, int deform, float obstacleArea) {
    SepView V;
    V.r = recs;
    opt_response(C, V, n, deform, C->area.ptr<float>(), obstacleArea);
}

}  // namespace cs
