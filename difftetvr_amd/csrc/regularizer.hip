// Tet-quality regulariser gradient on gfx950 (Data/Shaders/Optimizer/TetRegularizer.glsl:108-166,
// Renderer/TetRegularizerPass.cpp:91-95).
//
// Per tet: q = 6 sqrt(2) V / l_rms^3 (Parthasarathy et al. 1991) with V = -dot(cross(p1-p0, p2-p0), p3-p0) / 6
// and l_rms^2 = S / 6, S = sum of the 6 squared edge lengths; the loss term is the mirrored softplus
// (lambda / beta) log(1 + exp(-beta q)), whose derivative is dL/dq = -lambda / (1 + exp(beta q)).
// Written as q = -12 sqrt(3) D / S^{3/2} with the triple product D = dot(cross(p1-p0, p2-p0), p3-p0):
//   dq/dp = (12 sqrt(3) * dD/dp * S - 18 sqrt(3) * D * dS/dp) / S^{5/2} * (-1)
// and, as in the reference, S^{5/2} is clamped below at 1e-5 (this damps the gradient of small tets).
// Gradients are accumulated (+=) into grad_positions.
//
// What bounds it: the float atomics.  One per value (12 a tet), its wave's lanes at scattered addresses, go to the
// memory side at about 25 G/s: 742 us for 1.57M tets, against about 20 us for the mesh's bytes.  Neighbouring tets of a
// mesh file share most vertices, so a workgroup sums the tets of its range per vertex in LDS first (a hash table of
// vertex ids) and issues one atomic per value of each distinct vertex, consecutive lanes to consecutive addresses
// (about 180 G/s where every tet has its own vertices).  The sums are doubles: on gfx950 an LDS addition of doubles
// takes about half a cycle per lane, one of floats about four (146 us with float sums). 24 us for the 1.57M tets of a
// 64^3 grid; 272 -> 32 us for a Delaunay ball of 400K tets; with the grid's tets shuffled, 930 -> 773 us, and with
// vertices of their own, 714 -> 105 us.
#include "dtv_kernels.h"
#include "dtv_prims.h"
#include "vertex_table.h"

namespace dtv {

__device__ __forceinline__ void reg_tet(const int32_t* __restrict__ cells, const float* __restrict__ pos, int64_t t,
                                        float lambda, float beta, int32_t vid[4], float3_ g[4]) {
    const int4 idx = *reinterpret_cast<const int4*>(cells + 4 * t);
    vid[0] = idx.x;
    vid[1] = idx.y;
    vid[2] = idx.z;
    vid[3] = idx.w;
    float3_ p[4];
#pragma unroll
    for (int i = 0; i < 4; i++) p[i] = load_pos(pos, vid[i]);
    const float3_ a = sub(p[1], p[0]), b = sub(p[2], p[0]), c = sub(p[3], p[0]);
    const float D = dot(cross(a, b), c);
    float S = 0.f;
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = i + 1; j < 4; j++) {
            const float3_ e = sub(p[i], p[j]);
            S += dot(e, e);
        }
    const float k12 = 20.784609690826528f;   // 12 sqrt(3)
    const float q = -k12 * D / (S * sqrtf(S));
    const float dLdq = -lambda / (1.0f + expf(beta * q));
    const float S52 = fmaxf(S * S * sqrtf(S), 1e-5f);
    // dD/dp: p1 -> cross(b, c), p2 -> cross(c, a), p3 -> cross(a, b), p0 -> minus their sum
    float3_ dD[4];
    dD[1] = cross(b, c);
    dD[2] = cross(c, a);
    dD[3] = cross(a, b);
    dD[0] = scale(add(add(dD[1], dD[2]), dD[3]), -1.0f);
    float3_ sum = add(add(p[0], p[1]), add(p[2], p[3]));
#pragma unroll
    for (int i = 0; i < 4; i++) {
        // dS/dp_i = 2 (4 p_i - sum)
        const float3_ dS = scale(sub(scale(p[i], 4.0f), sum), 2.0f);
        g[i] = scale(sub(scale(dD[i], k12 * S), scale(dS, 1.5f * k12 * D)), -dLdq / S52);
    }
}

// One workgroup sums kThreads * kPer consecutive tets.  A thread takes consecutive ones, so that the lanes of a wave,
// kPer tets apart, seldom add to one vertex at once (LDS atomics on one address serialise).  A vertex that finds no
// entry (a mesh without locality fills the table) adds its values to the gradient directly.
template <int kThreads, int kPer>
__global__ __launch_bounds__(kThreads) void k_tet_regularizer(const int32_t* __restrict__ cells,
                                                              const float* __restrict__ pos, int64_t T, float lambda,
                                                              float beta, float* __restrict__ grad_pos) {
    constexpr int kTab = 4 * kThreads;
    __shared__ int32_t keys[kTab];
    __shared__ double sums[3 * kTab];
    for (int e = threadIdx.x; e < kTab; e += kThreads) {
        keys[e] = -1;
        sums[3 * e] = sums[3 * e + 1] = sums[3 * e + 2] = 0.0;
    }
    __syncthreads();
    const int64_t t0 = ((int64_t)blockIdx.x * kThreads + threadIdx.x) * kPer;
    for (int i = 0; i < kPer; i++) {
        if (t0 + i >= T) break;
        int32_t vid[4];
        float3_ g[4];
        reg_tet(cells, pos, t0 + i, lambda, beta, vid, g);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int e = grouped_entry<kTab, kRegProbes>(
                vid[k], [&](int at, int32_t v) { return atomicCAS(&keys[at], -1, v); });
            if (e >= 0) {
                lds_add_f64(&sums[3 * e + 0], g[k].x);
                lds_add_f64(&sums[3 * e + 1], g[k].y);
                lds_add_f64(&sums[3 * e + 2], g[k].z);
            } else {
                float* to = grad_pos + 3 * (int64_t)vid[k];
                atomic_add_f32(&to[0], g[k].x);
                atomic_add_f32(&to[1], g[k].y);
                atomic_add_f32(&to[2], g[k].z);
            }
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 3 * kTab; i += kThreads) {
        const int e = i / 3;
        const int32_t v = keys[e];
        const float sum = (float)sums[i];
        if (v >= 0 && sum != 0.f) atomic_add_f32(&grad_pos[3 * (int64_t)v + (i - 3 * e)], sum);
    }
}

template <int kThreads, int kPer>
static void launch_range(const int32_t* cells, const float* pos, int64_t T, float lambda, float beta, float* grad_pos,
                         hipStream_t s) {
    constexpr int64_t kRange = (int64_t)kThreads * kPer;
    hipLaunchKernelGGL((k_tet_regularizer<kThreads, kPer>), dim3((unsigned)((T + kRange - 1) / kRange)), dim3(kThreads),
                       0, s, cells, pos, T, lambda, beta, grad_pos);
}

void launch_tet_regularizer(const int32_t* cells, const float* pos, int64_t T, int64_t V, float lambda, float beta,
                            float* grad_pos, hipStream_t s) {
    if (T <= 0) return;
    switch (regularizer_range(T, V).per) {
        case 1: return launch_range<128, 1>(cells, pos, T, lambda, beta, grad_pos, s);
        case 2: return launch_range<256, 2>(cells, pos, T, lambda, beta, grad_pos, s);
        default: return launch_range<512, 4>(cells, pos, T, lambda, beta, grad_pos, s);
    }
}

}  // namespace dtv
