// flow_field.hip -- flow-field velocity at tracer points from segment and blob
// sources, for gfx950.
//
// Two modes:
//   Stokeslet + rotlet  -- the reference evaluator flow_velocities
//                          (src/flow_field/flow_field_evaluator.cu:13-228):
//                          Stokeslet of every segment force, rotlet of every
//                          segment torque, Stokeslet of every blob force, the
//                          Blakelet image system when there are no blobs
//                          (:83-116), optional removal of each body's net-force
//                          Stokeslet placed at the body centre (:125-143,
//                          :191-209), scaled by 1/(8 pi mu) (:549).
//   RPY                 -- the point-tracer limit (target radius 0) of the RPY
//                          pair tensor, <3,6> from segments and <3,3> from blobs.
//
// Sources are streamed through LDS in batches of BLOCK.  Two forms (flow_plan
// picks one from the point count): each lane holds two targets of its own, or
// (SHARED) the BLOCK/64 waves of a workgroup hold the same 64 targets and
// divide every batch between them, adding their sums in LDS in wave order.
// Either form may also divide the sources between gridDim.y workgroups, which
// write FP64 partial sums that flow_finish_kernel adds in chunk order, so a
// result does not change from run to run.  FP32 evaluation uses double-float
// positions and flushes FP32 partial sums into FP64 accumulators after every
// batch.
//
// Bound by VALU issue: at 4.2M points (FP32) the kernel's time equals the sum
// of its instructions' issue times (about 97 cycles per segment source and 64
// targets, 68 per blob).  What the divided forms give (MI355X): 10,007 points
// x 2,320 sources in FP64, where 20 workgroups were left for 256 CUs, and 1M
// points x 34,600 sources in FP32, where 1,954 workgroups made 7.6 per CU;
// times at flow_plan.
#include <algorithm>

#include "rpy_pair.h"
#include "tfs_internal.h"

namespace tfs {
namespace {

template <typename T>
constexpr int flow_rec() {
    // FP64: x y z f0..f5 (+pad).  FP32: xh yh zh xl yl zl f0..f5.  (Staging the
    // negated torque too, so that the rotlet terms become accumulates, measured
    // slower: the extra 16 B per source outweighs the saved issue slots.)
    return sizeof(T) == 8 ? 10 : 12;
}

// Image system of a Stokeslet above the no-slip wall z = 0 (Blake 1971):
// subtracts the image Stokeslet and adds the Stokeslet doublet and source
// dipole terms of flow_field_evaluator.cu:83-116.  acc += image velocity.
__device__ __forceinline__ void blakelet(double* acc, double zi, double zj, double ddx, double ddy, double fx,
                                         double fy, double fz) {
    const double Rz = zi + zj;
    const double R2 = ddx * ddx + ddy * ddy + Rz * Rz;
    const double Rm1 = __builtin_sqrt(1.0 / R2);
    const double kk = (ddx * fx + ddy * fy + Rz * fz) * Rm1 * Rm1;
    acc[0] -= Rm1 * (fx + ddx * kk);
    acc[1] -= Rm1 * (fy + ddy * kk);
    acc[2] -= Rm1 * (fz + Rz * kk);
    const double Dxx = (3.0 * ddx * ddx - R2) * zi;
    const double Dxy = 3.0 * ddx * ddy * zi;
    const double Dxz = (R2 - 3.0 * Rz * zi) * ddx;
    const double Dyy = (3.0 * ddy * ddy - R2) * zi;
    const double Dyz = (R2 - 3.0 * Rz * zi) * ddy;
    const double Dzx = (3.0 * Rz * zi + R2) * ddx;
    const double Dzy = (3.0 * Rz * zi + R2) * ddy;
    const double Dzz = (R2 - 3.0 * Rz * Rz) * zi;
    const double g = 2.0 * zj * Rm1 * Rm1 * Rm1 * Rm1 * Rm1;
    acc[0] += g * (Dxx * fx + Dxy * fy + Dxz * fz);
    acc[1] += g * (Dxy * fx + Dyy * fy + Dyz * fz);
    acc[2] += g * (Dzx * fx + Dzy * fy + Dzz * fz);
}

// The sources [s_lo, s_hi) of one class added into acc.  SHARED: wave w takes
// the w-th part of every batch.
template <typename T, int MODE, bool BLAKE, int FS, int BLOCK, int R, bool SHARED>
__device__ __forceinline__ void flow_sources(const FlowArgs& a, CView xsrc, CView fsrc, int s_lo, int s_hi, double aj,
                                             const double (&xi)[R][3], const T (&xh)[R][3],
                                             const T (&xl)[R][3], double (&acc)[R][3], T* lds) {
    constexpr int REC = flow_rec<T>();
    constexpr bool F32 = sizeof(T) == 4;
    const int tid = threadIdx.x;
    const T s3 = T(aj * aj / 3.0);
    const T m3s3 = T(-3) * s3;
    const T aj2 = T(aj * aj);
    T part[R][3];
    // FP32: the rotlet's negative cross-product halves, summed apart and
    // subtracted at the flush (every operation an accumulate).  FP64: the
    // terms in 1/r^3 (times 8), apart from the A f ones (times 2).
    T negp[R][3];
    for (int s0 = s_lo; s0 < s_hi; s0 += BLOCK) {
        const int n = (s_hi - s0) < BLOCK ? (s_hi - s0) : BLOCK;
        int j0 = 0, j1 = n;
        if constexpr (SHARED) {  // uniform over the wave
            const int per = (n + BLOCK / 64 - 1) / (BLOCK / 64);
            j0 = __builtin_amdgcn_readfirstlane(tid >> 6) * per;
            j1 = j0 + per < n ? j0 + per : n;
        }
        __syncthreads();
        if (tid < n) {
            const int64_t s = s0 + tid;
            T* rec = lds + tid * REC;
            const double p0 = xsrc.p[s * xsrc.ld_p], p1 = xsrc.p[s * xsrc.ld_p + xsrc.ld_c],
                         p2 = xsrc.p[s * xsrc.ld_p + 2 * xsrc.ld_c];
            if constexpr (F32) {
                const float h0 = float(p0), h1 = float(p1), h2 = float(p2);
                rec[0] = h0; rec[1] = h1; rec[2] = h2;
                rec[3] = float(p0 - double(h0)); rec[4] = float(p1 - double(h1)); rec[5] = float(p2 - double(h2));
#pragma unroll
                for (int k = 0; k < FS; ++k) rec[6 + k] = float(fsrc.p[s * fsrc.ld_p + k * fsrc.ld_c]);

            } else {
                rec[0] = p0; rec[1] = p1; rec[2] = p2;
#pragma unroll
                for (int k = 0; k < FS; ++k) rec[3 + k] = fsrc.p[s * fsrc.ld_p + k * fsrc.ld_c];
            }
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < R; ++r) {
            part[r][0] = part[r][1] = part[r][2] = T(0);
            negp[r][0] = negp[r][1] = negp[r][2] = T(0);
        }
        for (int j = j0; j < j1; ++j) {
            const T* rec = lds + j * REC;
            constexpr int F0 = F32 ? 6 : 3;
            T f[FS];
#pragma unroll
            for (int k = 0; k < FS; ++k) f[k] = rec[F0 + k];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                T dx, dy, dz;
                if constexpr (F32) {
                    dx = (xh[r][0] - rec[0]) + (xl[r][0] - rec[3]);
                    dy = (xh[r][1] - rec[1]) + (xl[r][1] - rec[4]);
                    dz = (xh[r][2] - rec[2]) + (xl[r][2] - rec[5]);
                } else {
                    dx = T(xi[r][0]) - rec[0];
                    dy = T(xi[r][1]) - rec[1];
                    dz = T(xi[r][2]) - rec[2];
                }
                const T r2 = fma_t(dz, dz, fma_t(dy, dy, dx * dx));
                // Stokeslet (+ rotlet): flow_field_evaluator.cu:66-78, 119-124; RPY point
                // tracer: the pair tensor with ai = 0.  Both are A f + Q (d.f) d / r^3 +
                // (tau x d) / r^3, with A = 1/r, Q = 1 or A = 1/r + s3/r^3, Q = 1 - 3 s3/r^2.
                // A tracer within the source's radius gets nothing here (its w = 0) and the
                // inner form below.
                bool inside = false;
                if constexpr (MODE == 1) inside = !(r2 > aj2);
                if constexpr (F32) {
                    // accumulates only
                    T rm1 = rsqrt_refined(r2);
                    if constexpr (MODE == 1) rm1 = inside ? T(0) : rm1;
                    const T rm2 = rm1 * rm1;
                    const T rm3 = rm1 * rm2;
                    const T A = MODE == 1 ? fma_t(s3, rm3, rm1) : rm1;
                    T sd;
                    T ex, ey, ez;
                    if constexpr (FS == 6) {
                        ex = rm3 * dx, ey = rm3 * dy, ez = rm3 * dz;
                        sd = fma_t(ez, f[2], fma_t(ey, f[1], ex * f[0]));
                    } else {
                        sd = rm3 * fma_t(dz, f[2], fma_t(dy, f[1], dx * f[0]));
                    }
                    if constexpr (MODE == 1) sd = fma_t(m3s3 * rm2, sd, sd);
                    part[r][0] = fma_t(sd, dx, fma_t(A, f[0], part[r][0]));
                    part[r][1] = fma_t(sd, dy, fma_t(A, f[1], part[r][1]));
                    part[r][2] = fma_t(sd, dz, fma_t(A, f[2], part[r][2]));
                    if constexpr (FS == 6) {
                        // (tau x d) / r^3 as + and - halves
                        part[r][0] = fma_t(f[4], ez, part[r][0]);
                        negp[r][0] = fma_t(f[5], ey, negp[r][0]);
                        part[r][1] = fma_t(f[5], ex, part[r][1]);
                        negp[r][1] = fma_t(f[3], ez, negp[r][1]);
                        part[r][2] = fma_t(f[3], ey, part[r][2]);
                        negp[r][2] = fma_t(f[4], ex, negp[r][2]);
                    }
                } else {
                    // w = 2/r: part = 2 A f, negp = 8 [Q (d.f) d + tau x d] / r^3
                    T w = rsqrt_twice(r2);
                    if constexpr (MODE == 1) w = inside ? T(0) : w;
                    const T w2 = w * w;
                    const T w3 = w * w2;
                    const T A = MODE == 1 ? fma_t(T(0.25) * s3, w3, w) : w;
                    part[r][0] = fma_t(A, f[0], part[r][0]);
                    part[r][1] = fma_t(A, f[1], part[r][1]);
                    part[r][2] = fma_t(A, f[2], part[r][2]);
                    T sd;
                    T ex, ey, ez;
                    if constexpr (FS == 6) {
                        ex = w3 * dx, ey = w3 * dy, ez = w3 * dz;
                        sd = fma_t(ez, f[2], fma_t(ey, f[1], ex * f[0]));
                    } else {
                        sd = w3 * fma_t(dz, f[2], fma_t(dy, f[1], dx * f[0]));
                    }
                    if constexpr (MODE == 1) sd = fma_t(T(0.25) * m3s3 * w2, sd, sd);
                    negp[r][0] = fma_t(sd, dx, negp[r][0]);
                    negp[r][1] = fma_t(sd, dy, negp[r][1]);
                    negp[r][2] = fma_t(sd, dz, negp[r][2]);
                    if constexpr (FS == 6) {
                        negp[r][0] = fma_t(f[4], ez, fma_t(-f[5], ey, negp[r][0]));
                        negp[r][1] = fma_t(f[5], ex, fma_t(-f[3], ez, negp[r][1]));
                        negp[r][2] = fma_t(f[3], ey, fma_t(-f[4], ex, negp[r][2]));
                    }
                }
                if constexpr (BLAKE) {
                    // Blakelet image system, flow_field_evaluator.cu:83-116, evaluated in
                    // double (the image distance of a wall-adjacent pair is small).
                    const double zi = xi[r][2];
                    double zj;
                    if constexpr (F32) zj = double(rec[2]) + double(rec[5]);
                    else zj = rec[2];
                    blakelet(acc[r], zi, zj, double(dx), double(dy), double(f[0]), double(f[1]), double(f[2]));
                }
                if constexpr (MODE == 1) {
                    if (inside) {
                        // rare: the rigid-body limit f / (6 pi mu aj) + tau x d / (8 pi mu aj^3)
                        // (cuda_functions.cu:207-354 with ai = 0), before the common factor
                        double ddx, ddy, ddz;
                        if constexpr (F32) {
                            ddx = xi[r][0] - (double(rec[0]) + double(rec[3]));
                            ddy = xi[r][1] - (double(rec[1]) + double(rec[4]));
                            ddz = xi[r][2] - (double(rec[2]) + double(rec[5]));
                        } else {
                            ddx = dx; ddy = dy; ddz = dz;
                        }
                        const double ca = 4.0 / (3.0 * aj), cc = 1.0 / (aj * aj * aj);
                        double u[3] = {ca * double(f[0]), ca * double(f[1]), ca * double(f[2])};
                        if constexpr (FS == 6) {
                            u[0] += cc * (double(f[4]) * ddz - double(f[5]) * ddy);
                            u[1] += cc * (double(f[5]) * ddx - double(f[3]) * ddz);
                            u[2] += cc * (double(f[3]) * ddy - double(f[4]) * ddx);
                        }
#pragma unroll
                        for (int k = 0; k < 3; ++k) acc[r][k] += u[k];
                    }
                }
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                if constexpr (!F32) acc[r][k] += 0.5 * part[r][k] + 0.125 * negp[r][k];
                else acc[r][k] += double(part[r][k]) - double(negp[r][k]);
            }
    }
}

// Each body's total force as one Stokeslet at its centre, taken out of acc
// (the per-source sums of flow_field_evaluator.cu:125-143, 191-209).
__device__ __forceinline__ void take_out_net_force(const FlowArgs& a, const double* __restrict__ net,
                                                   const double (&x)[3], double (&acc)[3]) {
    for (int b = 0; b < a.num_bodies; ++b) {
        const double dx = x[0] - a.x_bodies[3 * b], dy = x[1] - a.x_bodies[3 * b + 1],
                     dz = x[2] - a.x_bodies[3 * b + 2];
        const double fx = net[3 * b], fy = net[3 * b + 1], fz = net[3 * b + 2];
        const double rm2 = 1.0 / (dx * dx + dy * dy + dz * dz);
        const double rm1 = __builtin_sqrt(rm2);
        const double k = rm2 * (dx * fx + dy * fy + dz * fz);
        acc[0] -= rm1 * (fx + dx * k);
        acc[1] -= rm1 * (fy + dy * k);
        acc[2] -= rm1 * (fz + dz * k);
    }
}

// The common factor of every term.
__device__ __forceinline__ double flow_prefactor(double mu) { return 1.0 / (8.0 * 3.14159265358979323846 * mu); }

// Finish stamp of a workgroup: the largest of them is the evaluation's end.
__device__ __forceinline__ void stamp_end(unsigned long long* stamps) {
    if (threadIdx.x == 0) atomicMax(stamps + 1, (unsigned long long)wall_clock64());
}

// blockIdx.x: a tile of targets (BLOCK x R, or 64 x R shared by the waves);
// blockIdx.y: a chunk of a.chunk sources of the segments followed by the blobs.
// With a.part the sums go to part[(blockIdx.y * 3 + k) * nt + t], otherwise
// (one chunk) straight to the velocities.
template <typename T, int MODE, bool BLAKE, int BLOCK, int R, bool SHARED>
__global__ __launch_bounds__(BLOCK) void flow_kernel(FlowArgs a, const double* __restrict__ net) {
    constexpr int LANES = SHARED ? 64 : BLOCK;
    constexpr int SUMS = SHARED ? (BLOCK / 64 - 1) * 64 * R * 3 * (int)(sizeof(double) / sizeof(T)) : 0;
    constexpr int BATCH = BLOCK * flow_rec<T>();
    __shared__ __align__(16) T lds[BATCH > SUMS ? BATCH : SUMS];
    constexpr bool F32 = sizeof(T) == 4;
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) a.stamps[0] = (unsigned long long)wall_clock64();
    const int lane = (int)threadIdx.x & (LANES - 1);
    const int64_t t0 = (int64_t)blockIdx.x * (LANES * R) + lane;
    double xi[R][3];
    T xh[R][3], xl[R][3];
    double acc[R][3];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        int64_t t = t0 + (int64_t)r * LANES;
        t = t < a.nt ? t : a.nt - 1;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            xi[r][k] = a.xt.p[t * a.xt.ld_p + k * a.xt.ld_c];
            if constexpr (F32) {
                xh[r][k] = T(xi[r][k]);
                xl[r][k] = T(xi[r][k] - double(xh[r][k]));
            } else {
                xh[r][k] = xl[r][k] = T(0);
            }
            acc[r][k] = 0.0;
        }
    }
    const int64_t total = (int64_t)a.ns_total + a.nb_total;
    const int64_t c0 = (int64_t)blockIdx.y * a.chunk, c1 = c0 + a.chunk < total ? c0 + a.chunk : total;
    if (c0 < a.ns_total)
        flow_sources<T, MODE, BLAKE, 6, BLOCK, R, SHARED>(a, a.xs, a.fs, (int)c0,
                                                          (int)(c1 < a.ns_total ? c1 : a.ns_total), a.a_seg, xi, xh,
                                                          xl, acc, lds);
    if (c1 > a.ns_total)
        flow_sources<T, MODE, false, 3, BLOCK, R, SHARED>(a, a.xb, a.fb, (int)(c0 > a.ns_total ? c0 - a.ns_total : 0),
                                                          (int)(c1 - a.ns_total), a.a_blob, xi, xh, xl, acc, lds);
    bool writes = true;
    if constexpr (SHARED && BLOCK > 64) {
        double* buf = reinterpret_cast<double*>(lds);
        const int w = (int)threadIdx.x >> 6;
        __syncthreads();  // every wave is done with the last batch's records
        if (w > 0) {
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int k = 0; k < 3; ++k) buf[(((w - 1) * R + r) * 3 + k) * 64 + lane] = acc[r][k];
        }
        __syncthreads();
        writes = w == 0;
        if (writes) {
            for (int v = 0; v < BLOCK / 64 - 1; ++v)
#pragma unroll
                for (int r = 0; r < R; ++r)
#pragma unroll
                    for (int k = 0; k < 3; ++k) acc[r][k] += buf[((v * R + r) * 3 + k) * 64 + lane];
        }
    }
    const double prefac = flow_prefactor(a.mu);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int64_t t = t0 + (int64_t)r * LANES;
        if (!writes || t >= a.nt) continue;
        if (a.part) {
#pragma unroll
            for (int k = 0; k < 3; ++k) a.part[((int64_t)blockIdx.y * 3 + k) * a.nt + t] = acc[r][k];
            continue;
        }
        if (MODE == 0 && a.remove_net_force) take_out_net_force(a, net, xi[r], acc[r]);
#pragma unroll
        for (int k = 0; k < 3; ++k) a.vt.p[t * a.vt.ld_p + k * a.vt.ld_c] = prefac * acc[r][k];
    }
    if (!a.part) stamp_end(a.stamps);
}

// Adds the chunks' partial sums of each target in chunk order.
template <int MODE>
__global__ __launch_bounds__(256) void flow_finish_kernel(FlowArgs a, int nchunk, const double* __restrict__ net) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t < a.nt) {
        double acc[3] = {0.0, 0.0, 0.0};
#pragma unroll 4
        for (int c = 0; c < nchunk; ++c)
#pragma unroll
            for (int k = 0; k < 3; ++k) acc[k] += a.part[((int64_t)c * 3 + k) * a.nt + t];
        if (MODE == 0 && a.remove_net_force) {
            const double x[3] = {a.xt.p[t * a.xt.ld_p], a.xt.p[t * a.xt.ld_p + a.xt.ld_c],
                                 a.xt.p[t * a.xt.ld_p + 2 * a.xt.ld_c]};
            take_out_net_force(a, net, x, acc);
        }
        const double prefac = flow_prefactor(a.mu);
#pragma unroll
        for (int k = 0; k < 3; ++k) a.vt.p[t * a.vt.ld_p + k * a.vt.ld_c] = prefac * acc[k];
    }
    stamp_end(a.stamps);
}

// Per-body total force (segments + blobs), one thread per body.
__global__ void net_force_kernel(FlowArgs a, double* __restrict__ net, int nbod) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nbod) return;
    double f[3] = {0, 0, 0};
    for (int64_t s = (int64_t)b * a.ns_per_body; s < (int64_t)(b + 1) * a.ns_per_body; ++s)
        for (int k = 0; k < 3; ++k) f[k] += a.fs.p[s * a.fs.ld_p + k * a.fs.ld_c];
    for (int64_t s = (int64_t)b * a.nb_per_body; s < (int64_t)(b + 1) * a.nb_per_body; ++s)
        for (int k = 0; k < 3; ++k) f[k] += a.fb.p[s * a.fb.ld_p + k * a.fb.ld_c];
    for (int k = 0; k < 3; ++k) net[3 * b + k] = f[k];
}

template <typename T, int MODE, bool BLAKE, int BLOCK>
void launch_block(const FlowArgs& a, const double* net, const FlowPlan& p, hipStream_t s) {
    const int64_t tile = p.shared ? 64 : 2 * BLOCK;
    const dim3 grid((unsigned)((a.nt + tile - 1) / tile), (unsigned)p.chunks);
    if (p.shared) hipLaunchKernelGGL((flow_kernel<T, MODE, BLAKE, BLOCK, 1, true>), grid, dim3(BLOCK), 0, s, a, net);
    else hipLaunchKernelGGL((flow_kernel<T, MODE, BLAKE, BLOCK, 2, false>), grid, dim3(BLOCK), 0, s, a, net);
}

template <typename T, int MODE, bool BLAKE>
hipError_t launch_typed(const FlowArgs& a, const double* net, const FlowPlan& p, hipStream_t s) {
    switch (p.block) {
        case 64: launch_block<T, MODE, BLAKE, 64>(a, net, p, s); break;
        case 128: launch_block<T, MODE, BLAKE, 128>(a, net, p, s); break;
        case 256: launch_block<T, MODE, BLAKE, 256>(a, net, p, s); break;
        default: return hipErrorInvalidValue;
    }
    if (a.part)
        hipLaunchKernelGGL(flow_finish_kernel<MODE>, dim3((unsigned)((a.nt + 255) / 256)), dim3(256), 0, s, a, p.chunks,
                           net);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_flow_net(const FlowArgs& a, double* net, int nbod, hipStream_t s) {
    if (nbod <= 0) return hipSuccess;
    hipLaunchKernelGGL(net_force_kernel, dim3((nbod + 63) / 64), dim3(64), 0, s, a, net, nbod);
    return hipGetLastError();
}

// The launch form for nt points and nsrc sources on num_cus CUs.
//
// Each lane two targets of its own (every LDS read of a source serves both)
// where that form, with chunks of at least four batches, gives every CU 16
// workgroups, or undivided four; below, one target per lane, shared by the
// workgroup's waves.  Then the sources are divided until every CU has ~32
// (own targets) or ~12 (shared) workgroups of four waves, chunks at least
// four batches (own: the partial sums then cost under 1%) or half a batch
// (shared), partial sums within 256 MB.  Measured (MI355X, call of 320
// segments + 2,000 blobs at 10,007 points, FP64): 334 us undivided, own
// targets; 32 us shared and divided.  13,000 sources at 300,000 points, FP32:
// 3,240 and 2,140 us (own targets both).  34,600 sources at 1M points, FP32:
// 22.2 and 19.6 ms.
FlowPlan flow_plan(int64_t nt, int64_t nsrc, int block, int num_cus, bool may_divide) {
    FlowPlan p;
    p.block = block;
    const int64_t own = (nt + 2 * block - 1) / (2 * block);
    const int64_t least_own = 4LL * block;
    p.shared = own < 4LL * num_cus && own * (nsrc / least_own) < 16LL * num_cus;
    const int64_t tiles = p.shared ? (nt + 63) / 64 : own;
    const int64_t unit = p.shared ? 64 : block;                       // chunks are multiples of this
    const int64_t least = p.shared ? std::max(64, block / 2) : least_own;
    const int64_t waves = block / 64;
    const int64_t want = (p.shared ? 48LL : 128LL) * num_cus / waves;  // workgroups
    int64_t n = may_divide && tiles > 0 ? (want + tiles - 1) / tiles : 1;
    n = std::min<int64_t>(n, std::max<int64_t>(nsrc / least, 1));
    n = std::min<int64_t>(n, std::max<int64_t>((256LL << 20) / (24 * std::max<int64_t>(nt, 1)), 1));
    n = std::max<int64_t>(std::min<int64_t>(n, 65535), 1);
    int64_t chunk = (nsrc + n - 1) / n;
    if (n > 1) chunk = (chunk + unit - 1) / unit * unit;
    p.chunk = (int)std::max<int64_t>(std::min<int64_t>(chunk, INT32_MAX), 1);
    p.chunks = (int)std::max<int64_t>((nsrc + p.chunk - 1) / p.chunk, 1);
    return p;
}

hipError_t launch_flow_eval(int precision, const FlowArgs& a, const double* net, const FlowPlan& plan, hipStream_t s) {
    if (a.nt <= 0) return hipSuccess;
    const bool blake = a.mode == 0 && a.nb_per_body == 0 && a.ns_total > 0;
    if (precision == 0) {
        if (a.mode == 1) return launch_typed<double, 1, false>(a, net, plan, s);
        return blake ? launch_typed<double, 0, true>(a, net, plan, s) : launch_typed<double, 0, false>(a, net, plan, s);
    }
    if (a.mode == 1) return launch_typed<float, 1, false>(a, net, plan, s);
    return blake ? launch_typed<float, 0, true>(a, net, plan, s) : launch_typed<float, 0, false>(a, net, plan, s);
}

}  // namespace tfs
