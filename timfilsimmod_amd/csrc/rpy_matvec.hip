// rpy_matvec.hip -- fused, tiled RPY mobility matvec for gfx950.
//
// Replaces the four reference kernels Mss_mult / Msb_mult / Mbb_mult /
// Mbs_mult (src/cilia/cuda_functions.cu:362-757) with one launch over a work
// list.  A work item pairs a tile of targets (segments or blobs of one body)
// with a chunk of sources (segments or blobs of the same body).  A workgroup
// stages its chunk through LDS in batches of BLOCK sources (one coalesced
// load per lane, converted to the evaluation type as it is stored); every
// lane then walks the batch with broadcast LDS reads and accumulates
// PER_THREAD targets in registers.  Each item writes its partial sums to its
// own slot; a second kernel adds the slots of a tile in a fixed order and
// applies the reference's write rule (= or +=), so results are deterministic
// run to run, unlike atomics.
//
// The pair loop is branch-free: it evaluates the far-field RPY forms for
// every pair, with r^2 clamped below at (ai+aj)^2 (the self pair included).
// The pairs that clamp touches -- r^2 <= (ai+aj)^2, a handful per particle --
// are listed once per geometry by build_near_list (a hashed uniform grid),
// using the pair loop's own arithmetic for r^2, and the reduce kernel takes out their clamped far-field
// value and adds the reference's overlap and inner-branch formulas in FP64.
// Every pair is counted exactly once.
//
// Splitting the source range into chunks is what fills the chip: 21,800
// targets are only 341 wave64s, far fewer than the 1,024 SIMDs of an MI355X.
// The default shape also splits each item's sources between the waves of its
// workgroup (the waves share one tile of 64 x per_thread targets and add
// their sums in LDS before the item's one store): 12,800 segments + 9,000
// blobs in FP32 tiles are ~10k items of 64 targets x 768 sources, each
// writing 64 x 3 FP32 sums, a quarter of what four waves with their own
// targets would write.
//
// Two evaluation types:
//   double : the FP64 path (parity with the FP64 oracle at <= 1e-12).
//   float  : pair tensors in FP32 from fixed-point positions (per body,
//            X = rint(2^k (x - centre)) with |X| < 2^30): the separation is an
//            exact integer difference rounded once to FP32, so near pairs --
//            the ones that dominate -- lose nothing to cancellation, in two
//            full-rate instructions per component; per-batch FP32 partial sums
//            are flushed into FP64 accumulators after every LDS batch.
#include <algorithm>
#include <type_traits>

#include "rpy_pair.h"
#include "tfs_internal.h"

namespace tfs {
namespace {

constexpr int kMaxDof = 6;
constexpr int kXcds = 8;  // accelerator complex dies of an MI355X

// LDS record length (in T) of one staged source with FS strength components
// for targets with VT velocity components.  FP64: x y z f0..f(FS-1) [pad].
// FP32: X Y Z (fixed-point integers, stored as their bits) f0..f(FS-1), then
// the negated torque (FS = 6) and the negated force (VT = 6), padded to 16 B:
// with the negations staged, every cross-product term of the pair loop is an
// accumulate (the double-rate VOP2 form on gfx950) instead of a negated fma.
template <typename T, int FS, int VT = 3>
constexpr int rec_len() {
    if constexpr (sizeof(T) == 8) {
        return FS == 6 ? 10 : 6;
    } else {
        return (3 + FS + (FS == 6 ? 3 : 0) + (VT == 6 ? 3 : 0) + 3) / 4 * 4;
    }
}

// Largest record over the class combinations a kernel can stage.
template <typename T>
constexpr int rec_len_max() {
    return rec_len<T, 6, 6>();
}

// Separation and squared distance exactly as the pair loop evaluates them;
// build_near_list calls the same functions so the two agree bit for bit.
// FP64: d = x_i - x_j.  FP32: d = lambda (x_i - x_j) from the fixed-point
// coordinates -- an exact integer difference (|X| < 2^30) rounded once to
// FP32, two full-rate instructions per component.
__device__ __forceinline__ double separation(const double* xi, const double* rec, double& dx, double& dy,
                                             double& dz) {
    dx = xi[0] - rec[0];
    dy = xi[1] - rec[1];
    dz = xi[2] - rec[2];
    return __builtin_fma(dz, dz, __builtin_fma(dy, dy, dx * dx));
}
__device__ __forceinline__ float separation(const int32_t* Xi, const float* rec, float& dx, float& dy, float& dz) {
    dx = float(Xi[0] - __float_as_int(rec[0]));
    dy = float(Xi[1] - __float_as_int(rec[1]));
    dz = float(Xi[2] - __float_as_int(rec[2]));
    return __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
}

// Target coordinates in the evaluation type's form.
__device__ __forceinline__ void load_target(const MatvecArgs& a, int cls, int t, double* xi) {
    const CView x = cls == 0 ? a.xs : a.xb;
#pragma unroll
    for (int k = 0; k < 3; ++k) xi[k] = x.p[(int64_t)t * x.ld_p + k * x.ld_c];
}
__device__ __forceinline__ void load_target(const MatvecArgs& a, int cls, int t, int32_t* Xi) {
    const int4 q = a.xfx[(cls == 0 ? 0 : a.ns) + t];
    Xi[0] = q.x;
    Xi[1] = q.y;
    Xi[2] = q.z;
}

// One source of class src_cls into its LDS record: its position and, if
// with_force, its strengths -- forces multiplied by fscale, torques by
// tscale.
template <typename T, int FS, int VT = 3>
__device__ __forceinline__ void stage_source(T* rec, const MatvecArgs& a, int src_cls, int s, bool with_force,
                                             double fscale = 1.0, double tscale = 1.0) {
    constexpr int F0 = 3;
    if constexpr (sizeof(T) == 4) {
        const int4 q = a.xfx[(src_cls == 0 ? 0 : a.ns) + s];
        rec[0] = __int_as_float(q.x);
        rec[1] = __int_as_float(q.y);
        rec[2] = __int_as_float(q.z);
    } else {
        const CView x = src_cls == 0 ? a.xs : a.xb;
#pragma unroll
        for (int k = 0; k < 3; ++k) rec[k] = x.p[(int64_t)s * x.ld_p + k * x.ld_c];
    }
    if (with_force) {
        const CView f = src_cls == 0 ? a.fs : a.fb;
#pragma unroll
        for (int k = 0; k < FS; ++k) rec[F0 + k] = T((k < 3 ? fscale : tscale) * f.p[(int64_t)s * f.ld_p + k * f.ld_c]);
        if constexpr (sizeof(T) == 4) {
            int o = F0 + FS;
            if constexpr (FS == 6) {
#pragma unroll
                for (int k = 0; k < 3; ++k) rec[o + k] = -rec[F0 + 3 + k];
                o += 3;
            }
            if constexpr (VT == 6) {
#pragma unroll
                for (int k = 0; k < 3; ++k) rec[o + k] = -rec[F0 + k];
            }
        }
    }
}

// Target coordinates of a tile for the lanes of this thread (clamped into
// the tile; surplus lanes compute a duplicate and their slot entries are
// never read).  A tile has LANES x R targets: LANES = the workgroup size, or
// 64 when the waves split the sources (every wave then holds the same
// targets).
template <typename T>
using TargetT = typename std::conditional<sizeof(T) == 4, int32_t, double>::type;

template <typename T, int LANES, int R>
__device__ __forceinline__ void load_targets(const MatvecTile& tl, const MatvecArgs& a, TargetT<T> (&xi)[R][3]) {
    const int lane = (int)threadIdx.x & (LANES - 1);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        int t = tl.t_begin + lane + r * LANES;
        t = t < tl.t_end ? t : tl.t_end - 1;
        load_target(a, tl.cls, t, xi[r]);
    }
}

// The pairs of one work item added into acc (the first VT entries of each
// target's AV).  FP32 tiles work in the fixed-point frame d' = lambda d
// (lambda = 2^k, exact): with forces staged as lambda c8 F and torques as
// lambda^2 c8 tau, the translational sums come out in physical units and the
// rotational ones divided by lambda, which store_slot multiplies back.  FP32
// sums one LDS batch in `part` and flushes it into the FP64 accumulators.
// With SPLIT, wave w evaluates records [64 w, 64 w + 64) of every batch.
template <int VT, int FS, typename T, int BLOCK, int R, int AV, bool SPLIT = false>
__device__ __forceinline__ void accumulate_item(const MatvecItem it, const MatvecTile tl, const MatvecArgs& a,
                                                const TargetT<T> (&xi)[R][3], double (&acc)[R][AV],
                                                T* __restrict__ lds) {
    constexpr int REC = rec_len<T, FS, VT>();
    constexpr int F0 = 3;
    constexpr bool F32 = sizeof(T) == 4;
    const int tid = threadIdx.x;

    const double ai = tl.cls == 0 ? a.a_seg : a.a_blob;
    const double aj = it.src_cls == 0 ? a.a_seg : a.a_blob;
    const double PI = 3.14159265358979323846;
    const double lam = F32 ? *a.lam : 1.0;
    const T sum_a2 = T(lam * lam * ((ai + aj) * (ai + aj)));
    const T s3 = T(lam * lam * ((ai * ai + aj * aj) / 3.0));
    // -3 s3 as its own value (a negated operand would force the VOP3 form of the fma)
    const T m3s3 = T(-3) * s3;
    const double c8 = 1.0 / (8.0 * PI * a.mu);  // folded into the staged strengths

    T part[R][F32 ? VT : 1];
    // this wave's records of a batch start at j0 (uniform over the wave)
    const int j0 = SPLIT ? __builtin_amdgcn_readfirstlane(tid >> 6) * 64 : 0;
    for (int s0 = it.s_begin; s0 < it.s_end; s0 += BLOCK) {
        const int n = (it.s_end - s0) < BLOCK ? (it.s_end - s0) : BLOCK;
        const int j1 = SPLIT ? (n < j0 + 64 ? n : j0 + 64) : n;
        __syncthreads();  // the previous batch has been consumed
        if (tid < n) stage_source<T, FS, VT>(lds + tid * REC, a, it.src_cls, s0 + tid, true, lam * c8, lam * lam * c8);
        __syncthreads();
        if constexpr (F32) {
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int k = 0; k < VT; ++k) part[r][k] = T(0);
        }

#pragma unroll 2
        for (int j = j0; j < j1; ++j) {
            const T* rec = lds + j * REC;
            T f[FS];
#pragma unroll
            for (int k = 0; k < FS; ++k) f[k] = rec[F0 + k];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                T dx, dy, dz;
                const T r2 = separation(xi[r], rec, dx, dy, dz);
                // Overlapping pairs (and the self pair) are evaluated here with r
                // clamped to ai + aj -- one max instead of a compare and select --
                // and the reduce kernel swaps that value for the exact one.
                const T rm1 = rsqrt_refined(fmax_t(r2, sum_a2));
                if constexpr (F32) pair_far_scaled<T, VT, FS>(part[r], dx, dy, dz, rm1, f, rec + F0 + FS, s3, m3s3);
                else pair_far_scaled<T, VT, FS>(acc[r], dx, dy, dz, rm1, f, nullptr, s3, m3s3);
            }
        }
        if constexpr (F32) {
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int k = 0; k < VT; ++k) acc[r][k] += double(part[r][k]);
        }
    }
}

// A tile's sums (VT per target) into its partial slot (LANES x R targets).
// FP32 tiles store them in FP32: the reduce kernel reads half the bytes.
template <int VT, typename T, int LANES, int R, int AV>
__device__ __forceinline__ void store_slot(T* __restrict__ slot, const double (&acc)[R][AV], double lam) {
    constexpr int TILE = LANES * R;
    const int lane = (int)threadIdx.x & (LANES - 1);
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int k = 0; k < VT; ++k)
            slot[k * TILE + lane + r * LANES] = T(k < 3 ? acc[r][k] : lam * acc[r][k]);
}

// Source split: waves 1 .. S-1 hand their sums to wave 0 through LDS, which
// adds them in wave order (a fixed order: results are reproducible).
template <int VT, int BLOCK, int R, int AV>
__device__ __forceinline__ void combine_waves(double (&acc)[R][AV], double* __restrict__ buf) {
    const int w = (int)threadIdx.x >> 6, lane = (int)threadIdx.x & 63;
    __syncthreads();  // every wave is done with the last batch's records
    if (w > 0) {
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int k = 0; k < VT; ++k) buf[(((w - 1) * R + r) * VT + k) * 64 + lane] = acc[r][k];
    }
    __syncthreads();
    if (w == 0) {
        for (int v = 1; v < BLOCK / 64; ++v)
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int k = 0; k < VT; ++k) acc[r][k] += buf[(((v - 1) * R + r) * VT + k) * 64 + lane];
    }
}

// LDS of the one-workgroup-per-item kernel, in T: a batch of the largest
// records, or (source split) the sums of BLOCK/64 - 1 waves, if larger.
template <typename T, int BLOCK, int R, bool SPLIT>
constexpr int item_lds_len() {
    constexpr int batch = BLOCK * rec_len_max<T>();
    constexpr int sums = SPLIT ? (BLOCK / 64 - 1) * 64 * R * kMaxDof * (int)(sizeof(double) / sizeof(T)) : 0;
    return batch > sums ? batch : sums;
}

// The pairs of one work item into its own slot.
template <int VT, int FS, typename T, int BLOCK, int R, bool SPLIT>
__device__ __forceinline__ void run_item(const MatvecItem it, const MatvecTile tl, const MatvecArgs& a,
                                         T* __restrict__ slot, T* __restrict__ lds) {
    constexpr int LANES = SPLIT ? 64 : BLOCK;
    TargetT<T> xi[R][3];
    load_targets<T, LANES, R>(tl, a, xi);
    double acc[R][VT];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int k = 0; k < VT; ++k) acc[r][k] = 0.0;
    accumulate_item<VT, FS, T, BLOCK, R, VT, SPLIT>(it, tl, a, xi, acc, lds);
    if constexpr (SPLIT) {
        combine_waves<VT, BLOCK, R, VT>(acc, reinterpret_cast<double*>(lds));
        if (threadIdx.x >= 64) return;
    }
    store_slot<VT, T, LANES, R, VT>(slot, acc, sizeof(T) == 4 ? *a.lam : 1.0);
}

// One workgroup per item.  With `stamps`, thread 0 stores the item's start
// and finish (wall_clock64 ticks; equal for an item of a skipped body).
// SPLIT: the BLOCK/64 waves share the tile's 64 x R targets and split every
// batch of sources (BLOCK/64 times fewer partial bytes per item).
template <typename T, int SEGDOF, int BLOCK, int R, bool SPLIT>
__global__ __launch_bounds__(BLOCK) void rpy_pairs_kernel(const MatvecItem* __restrict__ items,
                                                          const MatvecTile* __restrict__ tiles,
                                                          MatvecArgs a, T* __restrict__ partial,
                                                          int64_t* __restrict__ stamps) {
    constexpr int TILE = (SPLIT ? 64 : BLOCK) * R;
    __shared__ __align__(16) T lds[item_lds_len<T, BLOCK, R, SPLIT>()];
    if (a.skip && *a.skip) return;
    const int64_t t_start = stamps ? (int64_t)wall_clock64() : 0;
    const MatvecItem it = items[blockIdx.x];
    const MatvecTile tl = tiles[it.tile];
    if (!(a.body_skip && a.body_skip[tl.body])) {
        T* slot = partial + (size_t)blockIdx.x * (kMaxDof * TILE);
        if (tl.cls == 0) {
            if (it.src_cls == 0) run_item<SEGDOF, SEGDOF, T, BLOCK, R, SPLIT>(it, tl, a, slot, lds);
            else run_item<SEGDOF, 3, T, BLOCK, R, SPLIT>(it, tl, a, slot, lds);
        } else {
            if (it.src_cls == 0) run_item<3, SEGDOF, T, BLOCK, R, SPLIT>(it, tl, a, slot, lds);
            else run_item<3, 3, T, BLOCK, R, SPLIT>(it, tl, a, slot, lds);
        }
    }
    if (stamps && threadIdx.x == 0) {
        const int64_t t_end = (a.body_skip && a.body_skip[tl.body]) ? t_start : (int64_t)wall_clock64();
        stamps[2 * (int64_t)blockIdx.x] = t_start;
        stamps[2 * (int64_t)blockIdx.x + 1] = t_end;
    }
}

// ---- symmetric form ------------------------------------------------------------
//
// The mobility of a pair is symmetric (M_ji = M_ij^T): the translational and
// rotational tensors are the same seen from either particle, the couplings
// change sign with the separation.  One evaluation of 1/r and its powers so
// serves both particles.  Tiles hold 64 particles of one class of one body; a
// panel is kSymWaves x R tiles.  An item pairs a panel with a run of tiles from
// the panel's first on: wave w owns the panel's tiles w, w + kSymWaves, ... (R
// particles per lane) and meets each tile of the run from LDS, lane l pairing
// its particles with source (l + k) mod 64 at step k: the lane's own sums get
// the source's term and the source's sums get the lane's terms.  The source
// sums live in one register per component that moves one lane per step (a DPP
// wave rotation ahead of the accumulates; the R particles of a lane share it),
// so after step k lane l holds the sum of source (l + k) mod 64.  The waves'
// sums of a source tile meet in LDS and are added in wave order.  Tile pairs
// a < b are evaluated once, a == b one-sided (the self pair and the overlapping
// pairs take the clamped far field, which the reduce kernel swaps for the exact
// value), and a > b not at all.  Within a body the segment tiles come first, so
// a blob target never meets a segment source.
//
// Partial slots: tile t of panel P has one slot per panel A < P its body
// overlaps (its sums as a source of panel A), then one per run of P from the
// one that holds t up to its body's last (its own sums; in its own run the sums
// it received as a source from its panel added), each written once per launch,
// so the reduce kernel sums them in slot order.
//
// Bound by VALU issue.  Cycles per wave instruction measured on MI355X (nominal
// 2.4 GHz): FP32 add, subtract, multiply 2.3-2.5, multiply-accumulate 2.7-3.1;
// maximum, int-to-float, DPP move, three-operand fma 4.3; rsq 8.2; FP64 4.4-5.6,
// its rsq 16.2 (FP32 and FP64 MFMA occupy the same pipes: their time adds to the
// VALU's, so moving sums there gains nothing).  Per launch at 12,800 segments +
// 9,000 blobs: 3 components FP32 195 us, FP64 320 (one particle per lane, items
// of 4 x 4 tiles: 212 and 354); 6 components FP32 325, FP64 540 (every ordered
// pair with the source split: 384 and 690).  Two particles per lane halve the
// rotations and the LDS reads; the three-operation Newton step saves one FP64
// operation; runs that shorten towards the end keep the CUs evenly loaded
// (FP32, 6 components: 355 us with two tiles per item throughout).
constexpr int kSymRot = 0x134;  // DPP wave_rol:1 -- lane l reads lane l + 1 (mod 64)
__device__ __forceinline__ float rotate_lanes(float x) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), kSymRot, 0xF, 0xF, false));
}
__device__ __forceinline__ double rotate_lanes(double x) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), kSymRot, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), kSymRot, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}

// LDS records of one source tile, split into arrays of 16 (or 8) bytes per
// record so that consecutive lanes, reading consecutive records, share no banks
// within a read phase.  FP32 positions are fixed-point integers as their bits.
// 3 components: held twice over (index j and j + 64 hold particle j), so that
// lane l reads record l + k without a wrap (the two index instructions per
// step cost more than the LDS).  6 components: held once, the index masked (of
// ~100 instructions per step two more matter less than a workgroup per CU),
// every array 16 bytes wide so that one address serves all.
template <typename T, int DOF>
struct SymTileLds;
template <>
struct SymTileLds<float, 3> {
    static constexpr bool kTwice = true;
    float4 xf[128];
    float2 yz[128];
    __device__ __forceinline__ void get(int j, float (&X)[3], float (&f)[3]) const {
        const float4 a = xf[j];
        const float2 b = yz[j];
        X[0] = a.x, X[1] = a.y, X[2] = a.z;
        f[0] = a.w, f[1] = b.x, f[2] = b.y;
    }
    __device__ __forceinline__ void put(int j, const int32_t (&X)[3], const float (&f)[3]) {
        xf[j] = make_float4(__int_as_float(X[0]), __int_as_float(X[1]), __int_as_float(X[2]), f[0]);
        yz[j] = make_float2(f[1], f[2]);
    }
};
template <>
struct SymTileLds<double, 3> {
    static constexpr bool kTwice = true;
    double2 xy[128];
    double2 zf[128];
    double2 gh[128];
    __device__ __forceinline__ void get(int j, double (&X)[3], double (&f)[3]) const {
        const double2 a = xy[j], b = zf[j], c = gh[j];
        X[0] = a.x, X[1] = a.y, X[2] = b.x;
        f[0] = b.y, f[1] = c.x, f[2] = c.y;
    }
    __device__ __forceinline__ void put(int j, const double (&X)[3], const double (&f)[3]) {
        xy[j] = make_double2(X[0], X[1]);
        zf[j] = make_double2(X[2], f[0]);
        gh[j] = make_double2(f[1], f[2]);
    }
};
template <>
struct SymTileLds<float, 6> {
    static constexpr bool kTwice = false;
    float4 a[64], b[64], c[64];
    template <int N>
    __device__ __forceinline__ void get(int j, float (&X)[3], float (&f)[N]) const {
        const float4 p = a[j], q = b[j];
        X[0] = p.x, X[1] = p.y, X[2] = p.z;
        f[0] = p.w, f[1] = q.x, f[2] = q.y;
        if constexpr (N == 6) f[3] = q.z, f[4] = q.w, f[5] = c[j].x;
    }
    __device__ __forceinline__ void put(int j, const int32_t (&X)[3], const float (&f)[6]) {
        a[j] = make_float4(__int_as_float(X[0]), __int_as_float(X[1]), __int_as_float(X[2]), f[0]);
        b[j] = make_float4(f[1], f[2], f[3], f[4]);
        c[j].x = f[5];
    }
};
template <>
struct SymTileLds<double, 6> {
    static constexpr bool kTwice = false;
    double2 a[64], b[64], c[64], d[64], e[64];
    template <int N>
    __device__ __forceinline__ void get(int j, double (&X)[3], double (&f)[N]) const {
        const double2 p = a[j], q = b[j], r = c[j];
        X[0] = p.x, X[1] = p.y, X[2] = q.x;
        f[0] = q.y, f[1] = r.x, f[2] = r.y;
        if constexpr (N == 6) {
            const double2 s = d[j];
            f[3] = s.x, f[4] = s.y, f[5] = e[j].x;
        }
    }
    __device__ __forceinline__ void put(int j, const double (&X)[3], const double (&f)[6]) {
        a[j] = make_double2(X[0], X[1]);
        b[j] = make_double2(X[2], f[0]);
        c[j] = make_double2(f[1], f[2]);
        d[j] = make_double2(f[3], f[4]);
        e[j].x = f[5];
    }
};

// Pair constants of one class pair.  FP32 tiles work in the fixed-point frame
// (separation from integer coordinates, s3 and (ai+aj)^2 scaled by lambda^2)
// with 1/r from the rsq instruction; FP64 with w = 2/r (one Newton-Raphson
// step without its factor 1/2, three operations), the powers of two folded
// into these constants and the staged strengths (sym_scale).
template <typename T>
struct SymConsts {
    T sum_a2;  // (ai + aj)^2
    T s3;      // s3, or s3/4
    T m3s3;    // -3 s3, or -3 s3/16
};
template <typename T>
__device__ __forceinline__ SymConsts<T> sym_consts(double ai, double aj, double lam) {
    const double s3 = lam * lam * ((ai * ai + aj * aj) / 3.0);
    SymConsts<T> c;
    c.sum_a2 = T(lam * lam * ((ai + aj) * (ai + aj)));
    c.s3 = sizeof(T) == 4 ? T(s3) : T(0.25 * s3);
    c.m3s3 = sizeof(T) == 4 ? T(-3) * T(s3) : T(-3.0 / 16.0 * s3);
    return c;
}

// Factors of the staged forces and torques, and of the rotational sums as they
// are stored.  FP32: forces lambda c8, torques lambda^2 c8 (c8 = 1/(8 pi mu)):
// rotational sums come out divided by lambda.  FP64: forces c8/2, torques
// c8/8: rotational sums come out times 4.
template <typename T>
__device__ __forceinline__ void sym_scale(const MatvecArgs& a, double& force, double& torque, double& rot) {
    const double c8 = 1.0 / (8.0 * 3.14159265358979323846 * a.mu);
    if constexpr (sizeof(T) == 4) {
        const double lam = *a.lam;
        force = lam * c8;
        torque = lam * lam * c8;
        rot = lam;
    } else {
        force = 0.5 * c8;
        torque = 0.125 * c8;
        rot = 0.25;
    }
}

// The pair term at separation d: pi += (i's velocity from fj), and with BOTH
// pj += (j's velocity from fi).  IT, JT: components of the target and source
// (6: force and torque in, velocity and angular velocity out).  `neg` is -1,
// opaque to the compiler in FP32 so that negated products stay two-operand
// accumulates (half the issue time of the three-operand form).
template <bool BOTH, typename T, int IT, int JT>
__device__ __forceinline__ void sym_pair(T dx, T dy, T dz, T r2, const SymConsts<T>& c, T neg, const T (&fi)[IT],
                                         const T (&fj)[JT], T (&pi)[IT], T (&pj)[JT]) {
    constexpr bool F32 = sizeof(T) == 4;
    r2 = fmax_t(r2, c.sum_a2);
    T w;
    if constexpr (F32) {
        w = rsqrt_refined(r2);
    } else {
        w = rsqrt_twice(r2);
    }
    const T w2 = w * w;
    const T w3 = w * w2;
    const T A = fma_t(c.s3, w3, w);
    // (1 - 3 s3 / r^2) as a factor: FP32 1 + u, FP64 u = a quarter of it
    const T u = F32 ? c.m3s3 * w2 : fma_t(c.m3s3, w2, T(0.25));
    if constexpr (IT == 3 && JT == 3) {
        const T B = F32 ? fma_t(u, w3, w3) : u * w3;
        const T Bd = B * fma_t(dz, fj[2], fma_t(dy, fj[1], dx * fj[0]));
        pi[0] = fma_t(Bd, dx, fma_t(A, fj[0], pi[0]));
        pi[1] = fma_t(Bd, dy, fma_t(A, fj[1], pi[1]));
        pi[2] = fma_t(Bd, dz, fma_t(A, fj[2], pi[2]));
        if constexpr (BOTH) {
            const T Be = B * fma_t(dz, fi[2], fma_t(dy, fi[1], dx * fi[0]));
            pj[0] = fma_t(Be, dx, fma_t(A, fi[0], pj[0]));
            pj[1] = fma_t(Be, dy, fma_t(A, fi[1], pj[1]));
            pj[2] = fma_t(Be, dz, fma_t(A, fi[2], pj[2]));
        }
    } else {
        const T ex = w3 * dx, ey = w3 * dy, ez = w3 * dz;
        const T nw3 = neg * w3;
        const T nx = nw3 * dx, ny = nw3 * dy, nz = nw3 * dz;
        T s = fma_t(ez, fj[2], fma_t(ey, fj[1], ex * fj[0]));
        s = F32 ? fma_t(u, s, s) : u * s;
        pi[0] = fma_t(s, dx, fma_t(A, fj[0], pi[0]));
        pi[1] = fma_t(s, dy, fma_t(A, fj[1], pi[1]));
        pi[2] = fma_t(s, dz, fma_t(A, fj[2], pi[2]));
        if constexpr (BOTH) {
            T t = fma_t(ez, fi[2], fma_t(ey, fi[1], ex * fi[0]));
            t = F32 ? fma_t(u, t, t) : u * t;
            pj[0] = fma_t(t, dx, fma_t(A, fi[0], pj[0]));
            pj[1] = fma_t(t, dy, fma_t(A, fi[1], pj[1]));
            pj[2] = fma_t(t, dz, fma_t(A, fi[2], pj[2]));
        }
        if constexpr (JT == 6) {
            // v_i += tau_j x d / r^3
            pi[0] = fma_t(fj[5], ny, fma_t(fj[4], ez, pi[0]));
            pi[1] = fma_t(fj[3], nz, fma_t(fj[5], ex, pi[1]));
            pi[2] = fma_t(fj[4], nx, fma_t(fj[3], ey, pi[2]));
            if constexpr (BOTH) {
                // omega_j -= F_i x d / r^3
                pj[3] = fma_t(fi[2], ey, fma_t(fi[1], nz, pj[3]));
                pj[4] = fma_t(fi[0], ez, fma_t(fi[2], nx, pj[4]));
                pj[5] = fma_t(fi[1], ex, fma_t(fi[0], ny, pj[5]));
            }
        }
        if constexpr (IT == 6) {
            // omega_i += F_j x d / r^3
            pi[3] = fma_t(fj[2], ny, fma_t(fj[1], ez, pi[3]));
            pi[4] = fma_t(fj[0], nz, fma_t(fj[2], ex, pi[4]));
            pi[5] = fma_t(fj[1], nx, fma_t(fj[0], ey, pi[5]));
            if constexpr (BOTH) {
                // v_j -= tau_i x d / r^3
                pj[0] = fma_t(fi[5], ey, fma_t(fi[4], nz, pj[0]));
                pj[1] = fma_t(fi[3], ez, fma_t(fi[5], nx, pj[1]));
                pj[2] = fma_t(fi[4], ex, fma_t(fi[3], ny, pj[2]));
            }
        }
        if constexpr (IT == 6 && JT == 6) {
            // omega_i += -tau_j / (2 r^3) + 3 (tau_j . d) d / (2 r^5), and with i and j swapped
            const T Ar = (F32 ? T(-0.5) : T(-2)) * w3;
            const T h = T(1.5) * w2;
            const T q = h * fma_t(ez, fj[5], fma_t(ey, fj[4], ex * fj[3]));
            pi[3] = fma_t(q, dx, fma_t(Ar, fj[3], pi[3]));
            pi[4] = fma_t(q, dy, fma_t(Ar, fj[4], pi[4]));
            pi[5] = fma_t(q, dz, fma_t(Ar, fj[5], pi[5]));
            if constexpr (BOTH) {
                const T p = h * fma_t(ez, fi[5], fma_t(ey, fi[4], ex * fi[3]));
                pj[3] = fma_t(p, dx, fma_t(Ar, fi[3], pj[3]));
                pj[4] = fma_t(p, dy, fma_t(Ar, fi[4], pj[4]));
                pj[5] = fma_t(p, dz, fma_t(Ar, fi[5], pj[5]));
            }
        }
    }
}

// Steps [k0, k1) of one stage: R target particles of the lane (IT of their DOF
// components) against the tile's sources (JT components).  BOTH: the sources'
// sums pj rotate and gather the lanes' terms (an off-diagonal tile pair);
// otherwise only the lane's own sums (the tile against itself).
template <bool BOTH, int IT, int JT, int R, typename T, int DOF>
__device__ __forceinline__ void sym_stage(const SymTileLds<T, DOF>& recs, int lane, int k0, int k1,
                                          const TargetT<T> (&Xi)[R][3], const T (&fi)[R][IT], const SymConsts<T>& c,
                                          T neg, T (&pi)[R][IT], T (&pj)[JT]) {
    // Not unrolled: more waves hide the LDS and dependency latency better than
    // a longer body (3 components, R = 1, FP32: 0.212 ms per launch of the
    // production body, 0.219 unrolled twice, 0.239 eight times).
#pragma unroll 1
    for (int k = k0; k < k1; ++k) {
        T X[3], fj[JT];
        recs.get(SymTileLds<T, DOF>::kTwice ? lane + k : (lane + k) & 63, X, fj);
        if constexpr (BOTH) {
#pragma unroll
            for (int q = 0; q < JT; ++q) pj[q] = rotate_lanes(pj[q]);
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            T dx, dy, dz;
            const T r2 = separation(Xi[r], X, dx, dy, dz);
            sym_pair<BOTH, T, IT, JT>(dx, dy, dz, r2, c, neg, fi[r], fj, pi[r], pj);
        }
    }
}

// One particle of a tile: its position (FP32 tiles: fixed-point) and strengths
// scaled by fsc and tsc (zero, with the tile's first position, for lanes past
// the tile's end; no torque for blobs).
template <typename T, int DOF>
__device__ __forceinline__ void sym_particle(const MatvecTile& tl, const MatvecArgs& a, int lane, double fsc,
                                             double tsc, TargetT<T> (&X)[3], T (&f)[DOF]) {
    const int s = tl.t_begin + lane;
    const bool ok = s < tl.t_end;
    const int sc = ok ? s : tl.t_begin;
    load_target(a, tl.cls, sc, X);
    const CView fv = tl.cls == 0 ? a.fs : a.fb;
#pragma unroll
    for (int k = 0; k < 3; ++k) f[k] = ok ? T(fsc * fv.p[(int64_t)sc * fv.ld_p + k * fv.ld_c]) : T(0);
    if constexpr (DOF == 6) {
        const bool tq = ok && tl.cls == 0;
#pragma unroll
        for (int k = 3; k < 6; ++k) f[k] = tq ? T(tsc * fv.p[(int64_t)sc * fv.ld_p + k * fv.ld_c]) : T(0);
    }
}

// Parts of a stage.  After each, a lane's own sums go to FP64 and the sources'
// sums to an LDS set of their own, in the evaluation type; the sets of all waves
// and parts are added in FP64.  An FP32 chain so has at most 64 particles' terms
// (a lane's own 32 where there are two parts: two particles per lane, and always
// with rotations, whose terms add four times to a component and not twice); in
// panels whose two tiles differ the second one's chain is added to the first
// one's, 32 terms each.  The length of these chains sets the FP32 error: 12,800
// segments + 9,000 blobs with rotations, 2.1e-7 with one part, 1.2e-7 with four
// (5% slower).
template <typename T, int DOF, int R>
constexpr int sym_parts() {
    return sizeof(T) == 4 ? (DOF == 6 ? 2 : R) : 1;
}

// R tiles of the lane against one source tile: own sums into acc, the sources'
// sums (BOTH) of every part to the wave's LDS sets js[part] (added to what they
// hold with `add`).
template <bool BOTH, int IT, int JT, int R, int PARTS, typename T, int DOF>
__device__ __forceinline__ void sym_tiles(const SymTileLds<T, DOF>& recs, int lane, const TargetT<T> (&Xi)[R][3],
                                          const T (&fi)[R][DOF], const SymConsts<T>& c, T neg, double (&acc)[R][DOF],
                                          T (*js)[DOF][64], bool add) {
    constexpr bool F32 = sizeof(T) == 4;
    T fv[R][IT];
    double sum[R][IT];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int k = 0; k < IT; ++k) {
            fv[r][k] = fi[r][k];
            sum[r][k] = acc[r][k];
        }
#pragma unroll 1
    for (int p = 0; p < PARTS; ++p) {
        T pi[R][IT], pj[JT];
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int k = 0; k < IT; ++k) {
                if constexpr (F32) pi[r][k] = T(0);
                else pi[r][k] = sum[r][k];
            }
#pragma unroll
        for (int k = 0; k < JT; ++k) pj[k] = T(0);
        const int k0 = p * (64 / PARTS), k1 = k0 + 64 / PARTS;
        sym_stage<BOTH, IT, JT, R, T, DOF>(recs, lane, k0, k1, Xi, fv, c, neg, pi, pj);
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int k = 0; k < IT; ++k) {
                if constexpr (F32) sum[r][k] += double(pi[r][k]);
                else sum[r][k] = pi[r][k];
            }
        if constexpr (BOTH) {
            const int j = (lane + k1 - 1) & 63;  // the source whose sums the lane holds now
#pragma unroll
            for (int k = 0; k < JT; ++k) js[p][k][j] = add ? js[p][k][j] + pj[k] : pj[k];
        }
    }
    // every component is written, also the ones that this class pair leaves as
    // they are: the instances then end in the same stores and the array stays
    // in registers
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int k = 0; k < DOF; ++k) acc[r][k] = k < IT ? sum[r][k < IT ? k : 0] : acc[r][k] + 0.0;
}

// The class pair's instance of sym_tiles.
template <bool BOTH, int R, int PARTS, typename T, int DOF>
__device__ __forceinline__ void sym_classes(int cls_a, int cls_b, const SymTileLds<T, DOF>& recs, int lane,
                                            const TargetT<T> (&Xi)[R][3], const T (&fi)[R][DOF],
                                            const SymConsts<T>& c, T neg, double (&acc)[R][DOF], T (*js)[DOF][64],
                                            bool add) {
    if constexpr (DOF == 3) {
        sym_tiles<BOTH, 3, 3, R, PARTS, T, DOF>(recs, lane, Xi, fi, c, neg, acc, js, add);
    } else if (cls_a == 1) {
        sym_tiles<BOTH, 3, 3, R, PARTS, T, DOF>(recs, lane, Xi, fi, c, neg, acc, js, add);
    } else if (cls_b == 0) {
        sym_tiles<BOTH, 6, 6, R, PARTS, T, DOF>(recs, lane, Xi, fi, c, neg, acc, js, add);
    } else {
        // a segment tile against a blob tile: never the tile itself
        if constexpr (BOTH) sym_tiles<true, 6, 3, R, PARTS, T, DOF>(recs, lane, Xi, fi, c, neg, acc, js, add);
    }
}

template <typename T, int DOF, int R>
constexpr int sym_min_waves() {
    if (R == 1) return DOF == 3 ? (sizeof(T) == 4 ? 8 : 6) : (sizeof(T) == 4 ? 6 : 4);
    return DOF == 3 ? (sizeof(T) == 4 ? 6 : 4) : (sizeof(T) == 4 ? 4 : 3);
}

// One workgroup of kSymWaves waves per item (tile = panel, source tiles
// [src_cls, s_begin), s_end = the run's number within the panel).
// `bb`: blob-blob pairs are evaluated (off when an overwriting BS block
// replaces BB).  Tile pairs of different bodies are skipped, and so is an item
// whose bodies all have their stop flag set; with `stamps`, thread 0 stores
// the item's start and finish (wall_clock64 ticks).
template <typename T, int DOF, int R>
__global__ __launch_bounds__(64 * kSymWaves, (sym_min_waves<T, DOF, R>())) void rpy_pairs_sym_kernel(
    const MatvecItem* __restrict__ items, const MatvecTile* __restrict__ tiles, int n_tiles, int bb, MatvecArgs a,
    T* __restrict__ partial, int64_t* __restrict__ stamps) {
    constexpr bool F32 = sizeof(T) == 4;
    constexpr int NW = kSymWaves, PANEL = NW * R, PARTS = sym_parts<T, DOF, R>();
    __shared__ SymTileLds<T, DOF> recs;
    __shared__ T jsum[NW * PARTS][DOF][64];
    if (a.skip && *a.skip) return;
    const int64_t t_start = stamps ? (int64_t)wall_clock64() : 0;
    const int w = (int)threadIdx.x >> 6, lane = (int)threadIdx.x & 63;
    const MatvecItem it = items[blockIdx.x];
    const int pa = it.tile, q0 = it.src_cls, q1 = it.s_begin;
    if (a.body_skip) {
        // the bodies of the item's tiles are a contiguous range
        const int b0 = tiles[PANEL * pa].body, b1 = tiles[q1 - 1].body;
        bool any = false;
        for (int b = b0; b <= b1 && !any; ++b) any = a.body_skip[b] == 0;
        if (!any) {
            if (stamps && threadIdx.x == 0) {
                stamps[2 * (int64_t)blockIdx.x] = t_start;
                stamps[2 * (int64_t)blockIdx.x + 1] = t_start;
            }
            return;
        }
    }
    const double lam = F32 ? *a.lam : 1.0;
    double fsc, tsc, rot;
    sym_scale<T>(a, fsc, tsc, rot);
    T neg = T(-1);
    if constexpr (F32 && DOF == 6) asm volatile("" : "+v"(neg));
    TargetT<T> Xi[R][3];
    T fi[R][DOF];
    double acc[R][DOF];
    int cls[R], body[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int ta = PANEL * pa + NW * r + w;
        cls[r] = 0;
        body[r] = -1;  // nothing to evaluate
#pragma unroll
        for (int k = 0; k < 3; ++k) Xi[r][k] = 0;
#pragma unroll
        for (int k = 0; k < DOF; ++k) {
            fi[r][k] = T(0);
            acc[r][k] = 0.0;
        }
        if (ta < n_tiles) {
            const MatvecTile tl = tiles[ta];
            cls[r] = tl.cls;
            if (!(a.body_skip && a.body_skip[tl.body])) body[r] = tl.body;
            sym_particle<T, DOF>(tl, a, lane, fsc, tsc, Xi[r], fi[r]);
        }
    }
    for (int tb = q0; tb < q1; ++tb) {
        const MatvecTile tlb = tiles[tb];
        if (w == (tb & (NW - 1))) {
            TargetT<T> X[3];
            T f[DOF];
            sym_particle<T, DOF>(tlb, a, lane, fsc, tsc, X, f);
            recs.put(lane, X, f);
            if constexpr (SymTileLds<T, DOF>::kTwice) recs.put(lane + 64, X, f);
        }
        __syncthreads();  // the records are in, the sums of the tile before are taken
        int mode[R];      // 0 nothing, 1 one-sided, 2 both particles
        bool all2 = true;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int ta = PANEL * pa + NW * r + w;
            mode[r] = ta < tb ? 2 : (ta == tb ? 1 : 0);
            if (body[r] != tlb.body || (cls[r] == 1 && tlb.cls == 1 && !bb)) mode[r] = 0;
            all2 = all2 && mode[r] == 2 && cls[r] == cls[0];
        }
        const double aj = tlb.cls == 0 ? a.a_seg : a.a_blob;
        T(*js)[DOF][64] = jsum + w * PARTS;  // this wave's sets
        if (!all2) {
#pragma unroll
            for (int p = 0; p < PARTS; ++p)
#pragma unroll
                for (int k = 0; k < DOF; ++k) js[p][k][lane] = T(0);
        }
        if (all2) {
            const SymConsts<T> c = sym_consts<T>(cls[0] == 0 ? a.a_seg : a.a_blob, aj, lam);
            sym_classes<true, R, PARTS, T, DOF>(cls[0], tlb.cls, recs, lane, Xi, fi, c, neg, acc, js, false);
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if (mode[r] == 0) continue;
                const SymConsts<T> c = sym_consts<T>(cls[r] == 0 ? a.a_seg : a.a_blob, aj, lam);
                TargetT<T> X1[1][3];
                T f1[1][DOF];
                double a1[1][DOF];
#pragma unroll
                for (int k = 0; k < 3; ++k) X1[0][k] = Xi[r][k];
#pragma unroll
                for (int k = 0; k < DOF; ++k) {
                    f1[0][k] = fi[r][k];
                    a1[0][k] = acc[r][k];
                }
                if (R > 1 && mode[r] == 2)  // R = 1: all2
                    sym_classes<true, 1, PARTS, T, DOF>(cls[r], tlb.cls, recs, lane, X1, f1, c, neg, a1, js, true);
                else
                    sym_classes<false, 1, PARTS, T, DOF>(cls[r], tlb.cls, recs, lane, X1, f1, c, neg, a1, js, true);
#pragma unroll
                for (int k = 0; k < DOF; ++k) acc[r][k] = a1[0][k];
            }
        }
        __syncthreads();  // every wave's sums are in
        auto source_sum = [&](int k) {
            double v = 0.0;
#pragma unroll
            for (int h = 0; h < NW * PARTS; ++h) v += double(jsum[h][k][lane]);
            return v;
        };
        if (tb < PANEL * pa + PANEL) {
            // one of the panel's own tiles: into its owner's sums
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (tb == PANEL * pa + NW * r + w) {
#pragma unroll
                    for (int k = 0; k < DOF; ++k)
                        if (k < 3 || tlb.cls == 0) acc[r][k] += source_sum(k);
                }
        } else {
            T* s = partial + (size_t)(tlb.first_item + pa - tlb.panel0) * (DOF * 64);
            const int ncomp = tlb.cls == 0 ? DOF : 3;
            for (int k = w; k < ncomp; k += NW) s[k * 64 + lane] = T(k < 3 ? source_sum(k) : rot * source_sum(k));
        }
    }
    // own sums: the slot of this run, if one of the tile's own to its body's last
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int ta = PANEL * pa + NW * r + w;
        if (ta >= n_tiles) continue;
        const MatvecTile tl = tiles[ta];
        const int slot = (pa - tl.panel0) + it.s_end - tl.run0;  // after the panels before the tile's
        if (it.s_end < tl.run0 || slot >= tl.n_items) continue;
        T* s = partial + (size_t)(tl.first_item + slot) * (DOF * 64);
#pragma unroll
        for (int k = 0; k < DOF; ++k)
            if (k < 3 || tl.cls == 0) s[k * 64 + lane] = T(k < 3 ? acc[r][k] : rot * acc[r][k]);
    }
    if (stamps && threadIdx.x == 0) {
        stamps[2 * (int64_t)blockIdx.x] = t_start;
        stamps[2 * (int64_t)blockIdx.x + 1] = (int64_t)wall_clock64();
    }
}

// Half-space domain (no-slip wall at z = 0): every pair of an item through
// pair_wall; the self pair (same global index) takes the wall self-mobility.
// Four waves share a tile of 64 targets, one per lane, and divide each batch
// of up to 256 sources; their sums are added in wave order.  FP64 tiles stage
// positions as they are.  FP32 tiles take separations from the fixed-point
// positions (exact integer differences, scaled by 1/lambda) and heights as
// floats of the FP64 positions, sum a wave's share of one batch in FP32 and
// flush it into FP64 accumulators.  Partial slots as run_item, in the
// evaluation type.
//
// Bound by the FP64 operations of pair_wall and by how evenly the waves fill
// the device.  5,120 segments with rotations, FP64, the whole call: 155 us,
// 251 with a target per lane of 256 x 256 items (400 workgroups) and the
// formulas as printed; 630 segments: 16 us, 145 before.
constexpr int kWallBatch = kWallBlock;  // sources staged at a time
template <int VT, int FS, typename T>
__device__ void run_item_wall(const MatvecItem it, const MatvecTile tl, const MatvecArgs& a,
                              T* __restrict__ slot, T* __restrict__ lds, double (*sums)[6][64]) {
    constexpr bool F32 = sizeof(T) == 4;
    constexpr int F0 = F32 ? 4 : 3;          // FP32 records: X bits (3), height, strengths
    constexpr int REC = F0 + FS;
    const double k6 = 1.0 / (6.0 * 3.14159265358979323846);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int t = tl.t_begin + lane;
    t = t < tl.t_end ? t : tl.t_end - 1;
    const CView xt = tl.cls == 0 ? a.xs : a.xb;
    const double zi_d = xt.p[(int64_t)t * xt.ld_p + 2 * xt.ld_c];
    double xi[3];
    int32_t Xi[3];
    if constexpr (F32) load_target(a, tl.cls, t, Xi);
    else load_target(a, tl.cls, t, xi);
    const T zi = T(zi_d);
    const T inv_lam = T(F32 ? 1.0 / *a.lam : 1.0);
    const int tg = (tl.cls == 0 ? 0 : a.ns) + t;
    const int src_base = it.src_cls == 0 ? 0 : a.ns;
    const CView xsrc = it.src_cls == 0 ? a.xs : a.xb;
    const CView fsrc = it.src_cls == 0 ? a.fs : a.fb;
    double acc[VT];
    T part[VT];
#pragma unroll
    for (int k = 0; k < VT; ++k) acc[k] = 0.0;
    for (int s0 = it.s_begin; s0 < it.s_end; s0 += kWallBatch) {
        const int n = (it.s_end - s0) < kWallBatch ? (it.s_end - s0) : kWallBatch;
        __syncthreads();
        if (tid < n) {
            T* rec = lds + tid * REC;
            const int s = s0 + tid;
            if constexpr (F32) {
                const int4 q = a.xfx[src_base + s];
                rec[0] = __int_as_float(q.x);
                rec[1] = __int_as_float(q.y);
                rec[2] = __int_as_float(q.z);
                rec[3] = float(xsrc.p[(int64_t)s * xsrc.ld_p + 2 * xsrc.ld_c]);
            } else {
#pragma unroll
                for (int k = 0; k < 3; ++k) rec[k] = xsrc.p[(int64_t)s * xsrc.ld_p + k * xsrc.ld_c];
            }
#pragma unroll
            for (int k = 0; k < FS; ++k) rec[F0 + k] = T(k6 * fsrc.p[(int64_t)s * fsrc.ld_p + k * fsrc.ld_c]);
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < VT; ++k) part[k] = T(0);
        const int share = (n + 3) / 4, j0 = wave * share, j1 = j0 + share < n ? j0 + share : n;
        for (int j = j0; j < j1; ++j) {
            const T* rec = lds + j * REC;
            T dx, dy, dz, zj;
            if constexpr (F32) {
                dx = float(Xi[0] - __float_as_int(rec[0])) * inv_lam;
                dy = float(Xi[1] - __float_as_int(rec[1])) * inv_lam;
                dz = float(Xi[2] - __float_as_int(rec[2])) * inv_lam;
                zj = rec[3];
            } else {
                dx = xi[0] - rec[0];
                dy = xi[1] - rec[1];
                dz = xi[2] - rec[2];
                zj = rec[2];
            }
            pair_wall<T, VT, FS>(part, src_base + s0 + j == tg, dx, dy, dz, zi, zj, rec + F0);
        }
#pragma unroll
        for (int k = 0; k < VT; ++k) acc[k] += double(part[k]);
    }
    if (wave > 0) {
#pragma unroll
        for (int k = 0; k < VT; ++k) sums[wave - 1][k][lane] = acc[k];
    }
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int w = 0; w < 3; ++w)
#pragma unroll
        for (int k = 0; k < VT; ++k) acc[k] += sums[w][k][lane];
#pragma unroll
    for (int k = 0; k < VT; ++k) slot[k * kWallTile + lane] = T(acc[k]);
}

template <int SEGDOF, typename T>
__global__ __launch_bounds__(kWallBlock) void rpy_pairs_wall_kernel(const MatvecItem* __restrict__ items,
                                                                    const MatvecTile* __restrict__ tiles,
                                                                    MatvecArgs a, T* __restrict__ partial) {
    __shared__ __align__(16) T lds[kWallBatch * (4 + 6)];
    __shared__ double sums[3][6][64];
    if (a.skip && *a.skip) return;
    const MatvecItem it = items[blockIdx.x];
    const MatvecTile tl = tiles[it.tile];
    if (a.body_skip && a.body_skip[tl.body]) return;
    T* slot = partial + (size_t)blockIdx.x * (kMaxDof * kWallTile);
    if (tl.cls == 0) {
        if (it.src_cls == 0) run_item_wall<SEGDOF, SEGDOF, T>(it, tl, a, slot, lds, sums);
        else run_item_wall<SEGDOF, 3, T>(it, tl, a, slot, lds, sums);
    } else {
        if (it.src_cls == 0) run_item_wall<3, SEGDOF, T>(it, tl, a, slot, lds, sums);
        else run_item_wall<3, 3, T>(it, tl, a, slot, lds, sums);
    }
}

// Persistent form: workgroup w takes the contiguous items [w k, (w+1) k) of
// the work list (items of one tile are contiguous, of similar size) and keeps
// one tile's sums in registers across its items, storing them once per tile
// segment, into the slot of the segment's first item: the reduce kernel reads
// only those slots (segment starts are the tiles' first items and the
// multiples of k), about k times fewer partial bytes than one slot per item.
// Loop counts and exits are uniform over the workgroup.  With timing on,
// every lane of a workgroup stores the same per-item start/finish stamps
// (wall_clock64 ticks; equal for an item of a skipped body).
template <typename T, int SEGDOF, int BLOCK, int R>
__global__ __launch_bounds__(BLOCK) void rpy_pairs_persistent_kernel(const MatvecItem* __restrict__ items,
                                                                     const MatvecTile* __restrict__ tiles,
                                                                     MatvecArgs a, T* __restrict__ partial,
                                                                     int n_items, int k, PersistState ps) {
    constexpr int REC = rec_len_max<T>();
    __shared__ __align__(16) T lds[BLOCK * REC];
    if (a.skip && *a.skip) return;
    const int i0 = blockIdx.x * k;
    const int i1 = i0 + k < n_items ? i0 + k : n_items;
    const double lam = sizeof(T) == 4 ? *a.lam : 1.0;
    TargetT<T> xi[R][3];
    double acc[R][SEGDOF];
    int cur = -1, cur_cls = 0, seg = 0;
    auto flush = [&]() {
        T* slot = partial + (size_t)seg * (kMaxDof * BLOCK * R);
        if (cur_cls == 0) store_slot<SEGDOF, T, BLOCK, R, SEGDOF>(slot, acc, lam);
        else store_slot<3, T, BLOCK, R, SEGDOF>(slot, acc, lam);
    };
    for (int item = i0; item < i1; ++item) {
        if (ps.item_stamps) ps.item_stamps[2 * item] = (int64_t)wall_clock64();
        const MatvecItem it = items[item];
        const MatvecTile tl = tiles[it.tile];
        if (a.body_skip && a.body_skip[tl.body]) {  // uniform over the workgroup
            if (ps.item_stamps) ps.item_stamps[2 * item + 1] = ps.item_stamps[2 * item];
            continue;
        }
        if (it.tile != cur) {
            if (cur >= 0) flush();
            cur = it.tile;
            cur_cls = tl.cls;
            seg = item;
            load_targets<T, BLOCK, R>(tl, a, xi);
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int c = 0; c < SEGDOF; ++c) acc[r][c] = 0.0;
        }
        if (tl.cls == 0) {
            if (it.src_cls == 0) accumulate_item<SEGDOF, SEGDOF, T, BLOCK, R, SEGDOF>(it, tl, a, xi, acc, lds);
            else accumulate_item<SEGDOF, 3, T, BLOCK, R, SEGDOF>(it, tl, a, xi, acc, lds);
        } else {
            if (it.src_cls == 0) accumulate_item<3, SEGDOF, T, BLOCK, R, SEGDOF>(it, tl, a, xi, acc, lds);
            else accumulate_item<3, 3, T, BLOCK, R, SEGDOF>(it, tl, a, xi, acc, lds);
        }
        if (ps.item_stamps) ps.item_stamps[2 * item + 1] = (int64_t)wall_clock64();
    }
    if (cur >= 0) flush();
}

// ---------------------------------------------------------------------------
// New positions: the fixed-point frame of FP32 tiles and the near-pair lists.
//
// Bound by the launches and the round trips to the host between them, not by
// the particles: three launches (clear + bounding boxes, place, list) and one
// read-back that the caller takes while the pair kernel runs.  What new
// positions add to an FP32 evaluation, two uploads included: 30 us for one body
// of 12,800 + 9,000 particles and 74 us for twelve of 1,000-29,000 (164 and 620
// with one workgroup per body for the boxes and the conversion, the frame
// computed on the host, and a counting sort with a one-workgroup scan for the
// cells).  Small FP64 problems test every pair instead (near_small_kernel).
//
// Cells have side h >= (1 + 1e-5) max(ai + aj), so every pair that either
// arithmetic (FP64, or FP32 fixed point, whose r^2 errs by well under 1e-5
// relative) could classify as overlapping lies in neighbouring cells; each
// candidate is then classified with the pair kernel's own staging and
// separation functions for the requested precision, so the lists and the pair
// loop's clamp agree bit for bit.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void particle_pos(const MatvecArgs& a, int p, double* x) {
    const CView v = p < a.ns ? a.xs : a.xb;
    const int i = p < a.ns ? p : p - a.ns;
#pragma unroll
    for (int k = 0; k < 3; ++k) x[k] = v.p[(int64_t)i * v.ld_p + k * v.ld_c];
}

__device__ __forceinline__ int cell_coord(double x, double inv_h) {
    const double c = __builtin_floor(x * inv_h);
    return (int)(c < -1073741824.0 ? -1073741824.0 : (c > 1073741824.0 ? 1073741824.0 : c));
}

__device__ __forceinline__ uint32_t cell_hash(int cx, int cy, int cz, uint32_t mask) {
    return ((uint32_t)cx * 73856093u ^ (uint32_t)cy * 19349663u ^ (uint32_t)cz * 83492791u) & mask;
}

__global__ __launch_bounds__(256) void grid_count_kernel(MatvecArgs a, int n, double inv_h, uint32_t mask,
                                                        int32_t* __restrict__ bucket_of,
                                                        int32_t* __restrict__ fill) {
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p >= n) return;
    double x[3];
    particle_pos(a, p, x);
    const uint32_t b = cell_hash(cell_coord(x[0], inv_h), cell_coord(x[1], inv_h), cell_coord(x[2], inv_h), mask);
    bucket_of[p] = (int32_t)b;
    atomicAdd(&fill[b], 1);
}

// start = exclusive prefix sum of fill (table entries, a power of two >= 1024),
// start[table] = total; fill is cleared for the scatter.  One workgroup, in
// chunks of up to 16384 entries (1024 x per).  The chunk is loaded and stored
// coalesced, every load (and store) of a thread issued together, and staged in
// LDS with one pad word per 16 entries, so that each thread's `per`
// consecutive entries (a stride of 17 words across the lanes) share no bank.
// Every thread sums its entries, the sums are scanned across each wave by
// shuffles and across the sixteen waves from their totals, and a running
// carry joins the chunks.
__global__ __launch_bounds__(1024) void grid_scan_kernel(int32_t* __restrict__ fill, int32_t* __restrict__ start,
                                                        int table) {
    constexpr int kChunk = 16384, kMaxPer = kChunk / 1024, kWaves = 1024 / 64;
    __shared__ int32_t buf[kChunk + kChunk / 16];
    __shared__ int32_t wsum[kWaves];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const auto pad = [](int i) { return i + (i >> 4); };
    int32_t carry = 0;
    for (int c0 = 0; c0 < table; c0 += kChunk) {
        const int len = table - c0 < kChunk ? table - c0 : kChunk;
        const int per = len / 1024;
        int32_t v[kMaxPer];
#pragma unroll
        for (int k = 0; k < kMaxPer; ++k) v[k] = k < per ? fill[c0 + k * 1024 + tid] : 0;
#pragma unroll
        for (int k = 0; k < kMaxPer; ++k)
            if (k < per) buf[pad(k * 1024 + tid)] = v[k];
        __syncthreads();
        const int b = tid * per;  // this thread's first entry of the chunk
        int32_t sum = 0;
#pragma unroll
        for (int i = 0; i < kMaxPer; ++i)
            if (i < per) sum += buf[pad(b + i)];
        int32_t inc = sum;  // inclusive scan of the threads' sums across the wave
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int32_t t = __shfl_up(inc, off, 64);
            if (lane >= off) inc += t;
        }
        if (lane == 63) wsum[wid] = inc;
        __syncthreads();
        int32_t before = 0, total = 0;
#pragma unroll
        for (int k = 0; k < kWaves; ++k) {
            const int32_t t = wsum[k];
            before += k < wid ? t : 0;
            total += t;
        }
        int32_t run = carry + before + inc - sum;  // exclusive prefix of this thread's entries
#pragma unroll
        for (int i = 0; i < kMaxPer; ++i)
            if (i < per) {
                const int32_t cnt = buf[pad(b + i)];
                buf[pad(b + i)] = run;
                run += cnt;
            }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kMaxPer; ++k) v[k] = k < per ? buf[pad(k * 1024 + tid)] : 0;
#pragma unroll
        for (int k = 0; k < kMaxPer; ++k)
            if (k < per) {
                start[c0 + k * 1024 + tid] = v[k];
                fill[c0 + k * 1024 + tid] = 0;
            }
        carry += total;
        __syncthreads();  // buf and wsum are written again by the next chunk
    }
    if (tid == 0) start[table] = carry;
}

__global__ __launch_bounds__(256) void grid_scatter_kernel(int n, const int32_t* __restrict__ bucket_of,
                                                          const int32_t* __restrict__ start,
                                                          int32_t* __restrict__ fill, int32_t* __restrict__ order) {
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p >= n) return;
    const int32_t b = bucket_of[p];
    order[start[b] + atomicAdd(&fill[b], 1)] = p;
}

// Puts each bucket's particles in increasing index order (the scatter's
// atomics leave them in arrival order), so that sums over a cell's particles
// are reproducible.  Insertion sort per bucket; buckets hold a few particles
// (cells of side ~2a hold at most a handful), larger ones are left as they are.
__global__ __launch_bounds__(256) void grid_sort_buckets_kernel(int table, const int32_t* __restrict__ start,
                                                               int32_t* __restrict__ order) {
    const int b = blockIdx.x * 256 + threadIdx.x;
    if (b >= table) return;
    const int lo = start[b], hi = start[b + 1];
    if (hi - lo < 2 || hi - lo > 256) return;
    for (int i = lo + 1; i < hi; ++i) {
        const int32_t v = order[i];
        int k = i - 1;
        while (k >= lo && order[k] > v) {
            order[k + 1] = order[k];
            --k;
        }
        order[k + 1] = v;
    }
}

// Particle t of body range r (its segments, then its blobs).
__device__ __forceinline__ int body_particle(const int4& r, int ns, int t) {
    const int segs = r.y - r.x;
    return t < segs ? r.x + t : ns + r.z + (t - segs);
}

// Bucket of a cell of one body: bodies that overlap in space (independent
// bodies solved together) keep to buckets of their own.
__device__ __forceinline__ uint32_t body_cell_hash(int cx, int cy, int cz, int body, uint32_t mask) {
    return cell_hash((int)((uint32_t)cx + (uint32_t)body * 2654435761u), cy, cz, mask);
}

// Empties the grid (head, table entries, may be null), clears *max_cnt and,
// with BOX, writes box[blockIdx.x gridDim.y + blockIdx.y]: the bounds (min
// xyz, max xyz) of the workgroup's share of body blockIdx.x, NaN if any of its
// coordinates is not finite.  Workgroups of 256.  (Bodies are counted in x here
// and below: a grid's y ends at 65,535.)
template <bool BOX>
__global__ __launch_bounds__(256) void geometry_clear_kernel(MatvecArgs a, const int4* __restrict__ ranges,
                                                            double* __restrict__ box, int32_t* __restrict__ head,
                                                            int table, int32_t* __restrict__ max_cnt) {
    const int tid = (int)threadIdx.x;
    const int block = (int)(blockIdx.y * gridDim.x + blockIdx.x);
    if (head)
        for (int64_t i = ((int64_t)block * 256 + tid) * 4; i < table; i += (int64_t)(gridDim.x * gridDim.y) * 1024)
            *reinterpret_cast<int4*>(head + i) = make_int4(-1, -1, -1, -1);
    if (block == 0 && tid == 0) *max_cnt = 0;
    if constexpr (BOX) {
        __shared__ double red[4][6];
        const int4 r = ranges[blockIdx.x];
        const int m = (r.y - r.x) + (r.w - r.z);
        double lo[3] = {__builtin_inf(), __builtin_inf(), __builtin_inf()};
        double hi[3] = {-__builtin_inf(), -__builtin_inf(), -__builtin_inf()};
        bool bad = false;
        for (int t = (int)blockIdx.y * 256 + tid; t < m; t += (int)gridDim.y * 256) {
            double x[3];
            particle_pos(a, body_particle(r, a.ns, t), x);
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                bad |= !__builtin_isfinite(x[k]);
                lo[k] = __builtin_fmin(lo[k], x[k]);
                hi[k] = __builtin_fmax(hi[k], x[k]);
            }
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1)
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                lo[k] = __builtin_fmin(lo[k], __shfl_xor(lo[k], off, 64));
                hi[k] = __builtin_fmax(hi[k], __shfl_xor(hi[k], off, 64));
            }
        if ((tid & 63) == 0)
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                red[tid >> 6][k] = lo[k];
                red[tid >> 6][3 + k] = hi[k];
            }
        const bool any_bad = __syncthreads_or(bad);
        if (tid < 6) {
            double v = red[0][tid];
            for (int w = 1; w < 4; ++w) v = tid < 3 ? __builtin_fmin(v, red[w][tid]) : __builtin_fmax(v, red[w][tid]);
            box[6 * ((int64_t)blockIdx.x * gridDim.y + blockIdx.y) + tid] = any_bad ? __builtin_nan("") : v;
        }
    }
}

// The fixed-point frame of the bodies' boxes (`shares` per body): each body is
// centred on its bounding box; lambda = 2^k is the largest power of two with
// lambda * (largest half-extent) <= 2^30 - 2, so every coordinate and every
// difference of two fits an int32, and lambda amin < 2^40, so that the third
// power of 1/r at the clamp r = ai + aj is no denormal float (a particle on
// its own, bodies of coincident particles), and lambda <= 2^60, so that the
// lambda^2 of a staged torque stays far inside a float.  Returns lambda, 0
// with *status set where the positions are not finite or the step 1/lambda is
// not below 2^-19 amin, and the centre of body `own`.  Every workgroup of
// geometry_place_kernel works it out for itself from up to kFrameBodies boxes;
// more bodies have geometry_frame_kernel do it once.
constexpr int kFrameBodies = 1024;  // at least kBoxShares: more have one box each
template <int THREADS>
__device__ double fixed_frame(const double* __restrict__ box, int nbody, int shares, int own, double amin,
                              double* centre, int* status) {
    __shared__ double wave_ext[THREADS / 64], own_centre[3];
    const int tid = (int)threadIdx.x;
    int width = 1;  // lanes per body
    while (width < shares && width < 64) width <<= 1;
    double ext = 0.0;
    bool bad = false;
    for (int b = tid / width; b < nbody; b += THREADS / width) {
        double lo[3] = {__builtin_inf(), __builtin_inf(), __builtin_inf()};
        double hi[3] = {-__builtin_inf(), -__builtin_inf(), -__builtin_inf()};
        for (int g = tid % width; g < shares; g += width) {
            const double* q = box + 6 * ((int64_t)b * shares + g);
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                bad |= q[k] != q[k];
                lo[k] = __builtin_fmin(lo[k], q[k]);
                hi[k] = __builtin_fmax(hi[k], q[3 + k]);
            }
        }
        for (int off = width >> 1; off > 0; off >>= 1)
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                lo[k] = __builtin_fmin(lo[k], __shfl_xor(lo[k], off, width));
                hi[k] = __builtin_fmax(hi[k], __shfl_xor(hi[k], off, width));
            }
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const bool some = lo[k] <= hi[k];  // a body without particles has no box
            const double c = some ? 0.5 * (lo[k] + hi[k]) : 0.0;
            ext = some ? __builtin_fmax(ext, __builtin_fmax(hi[k] - c, c - lo[k])) : ext;
            if (b == own && tid % width == 0) own_centre[k] = c;
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) ext = __builtin_fmax(ext, __shfl_xor(ext, off, 64));
    if ((tid & 63) == 0) wave_ext[tid >> 6] = ext;
    const bool any_bad = __syncthreads_or(bad);
    for (int w = 0; w < THREADS / 64; ++w) ext = __builtin_fmax(ext, wave_ext[w]);
    for (int k = 0; k < 3; ++k) centre[k] = own_centre[k];
    *status = any_bad ? kFrameNonFinite : ext < 1e300 ? 0 : kFrameTooLarge;
    if (*status) return 0.0;
    int k = 1000;
    if (ext > 0.0) {
        int e;
        const double m = frexp(ext, &e);  // ext = m 2^e, 1/2 <= m < 1
        k = m <= 1073741822.0 / 1073741824.0 ? 30 - e : 29 - e;
    }
    int ea;
    (void)frexp(amin, &ea);
    k = k < 40 - ea ? k : 40 - ea;
    k = k < 60 ? k : 60;
    if (ldexp(1.0, -k) > ldexp(amin, -19)) {
        *status = kFrameTooLarge;
        return 0.0;
    }
    return ldexp(1.0, k);
}

// One box per body.
__global__ __launch_bounds__(1024) void geometry_frame_kernel(const double* __restrict__ box, int nbody, double amin,
                                                             GeomFrame* __restrict__ frame) {
    double centre[3];
    int status;
    const double lam = fixed_frame<1024>(box, nbody, 1, -1, amin, centre, &status);
    if (threadIdx.x == 0) {
        frame->lam = lam;
        frame->status = status;
    }
}

// FIXED: X = rint(lambda (x - c_body)) of every particle, and the frame (shares
// = 0: it is there already, and each body has one box).
// head not null: every particle into the grid, each bucket a list linked
// through nodes[p] = (cell, next particle or -1), newest first (the order
// varies between runs; near_grid_kernel sorts what it finds).  body_of (may be
// null) gets each particle's body.  Grid (bodies, workgroups per body).
template <bool FIXED>
__global__ __launch_bounds__(256) void geometry_place_kernel(MatvecArgs a, const int4* __restrict__ ranges,
                                                            const double* __restrict__ box, int shares, double amin,
                                                            int4* __restrict__ fixed, GeomFrame* __restrict__ frame,
                                                            double inv_h, uint32_t mask, int32_t* __restrict__ head,
                                                            int4* __restrict__ nodes, int32_t* __restrict__ body_of) {
    const int body = (int)blockIdx.x;
    const int4 r = ranges[body];
    const int m = (r.y - r.x) + (r.w - r.z);
    double centre[3] = {0.0, 0.0, 0.0}, lam = 0.0;
    if constexpr (FIXED) {
        int status;
        if (shares == 0) {
            lam = frame->lam;
            status = frame->status;
            const double* q = box + 6 * (int64_t)body;
#pragma unroll
            for (int k = 0; k < 3; ++k) centre[k] = q[k] <= q[3 + k] ? 0.5 * (q[k] + q[3 + k]) : 0.0;
        } else {
            lam = fixed_frame<256>(box, (int)gridDim.x, shares, body, amin, centre, &status);
            if (blockIdx.y == 0 && body == 0 && threadIdx.x == 0) {
                frame->lam = lam;
                frame->status = status;
            }
        }
        if (status) return;  // the same in every workgroup
    }
    for (int t = (int)(blockIdx.y * 256 + threadIdx.x); t < m; t += (int)gridDim.y * 256) {
        const int p = body_particle(r, a.ns, t);
        double x[3];
        particle_pos(a, p, x);
        if constexpr (FIXED)
            fixed[p] = make_int4((int)__builtin_rint((x[0] - centre[0]) * lam),
                                 (int)__builtin_rint((x[1] - centre[1]) * lam),
                                 (int)__builtin_rint((x[2] - centre[2]) * lam), 0);
        if (body_of) body_of[p] = body;
        if (head) {
            const int cx = cell_coord(x[0], inv_h), cy = cell_coord(x[1], inv_h), cz = cell_coord(x[2], inv_h);
            const int32_t next = atomicExch(head + body_cell_hash(cx, cy, cz, body, mask), p);
            nodes[p] = make_int4(cx, cy, cz, next);
        }
    }
}

// 32 lanes per target, lane l < 27 visiting neighbour cell l; the near sources
// are appended in any order and then put into increasing order by rank (the
// entries are distinct), from LDS for up to 64 of them, so the lists are the
// same on every run.  cnt is the full count, entries past cap are dropped and
// *max_cnt gets any count above cap.
//
// Crowded places (a bucket longer than `walk` particles, or a list of more than
// 256): the target's lanes test all of its body's particles
// in order instead, 32 at a time, so that no cell and no list, whatever the
// positions (coincident, not finite), takes more than a walk of those lengths
// and one pass over the body: a launch costs at most about what the pair kernel
// does.  Sorting such a list by itself would take a lane as many dependent moves
// as its length squared.
constexpr int kNearLds = 64, kRankPer = 8;
template <typename T>
__global__ __launch_bounds__(256) void near_grid_kernel(MatvecArgs a, int n, double inv_h, uint32_t mask,
                                                       const int4* __restrict__ ranges, int walk,
                                                       const int32_t* __restrict__ head,
                                                       const int4* __restrict__ nodes,
                                                       const int32_t* __restrict__ body_of, int32_t* __restrict__ cnt,
                                                       int32_t* idx, int cap, int32_t* __restrict__ max_cnt) {
    constexpr bool F32 = sizeof(T) == 4;
    constexpr int REC = rec_len<T, 3>();
    __shared__ int32_t found[8], crowded[8];
    __shared__ int32_t list[8][kNearLds + 1];
    const int s = (int)(threadIdx.x >> 5);
    const int tg = (int)blockIdx.x * 8 + s;
    const int lane = (int)(threadIdx.x & 31);
    const double lam = F32 ? *a.lam : 1.0;
    if (!(lam > 0.0)) return;  // no frame: uniform over the launch
    if (threadIdx.x < 8) found[threadIdx.x] = crowded[threadIdx.x] = 0;
    __syncthreads();
    int32_t* e = idx + (int64_t)tg * cap;
    const bool in = tg < n;
    // (past the end: the last target's, so that the loads go out together)
    const int tc = in ? tg : n - 1;
    const int cls = tc < a.ns ? 0 : 1;
    const int4 own = nodes[tc];
    using XT = typename std::conditional<F32, int32_t, double>::type;
    XT xi[3];
    load_target(a, cls, cls == 0 ? tc : tc - a.ns, xi);
    const int body = body_of ? body_of[tc] : 0;
    const double ai = cls == 0 ? a.a_seg : a.a_blob;
    const T sum_seg = T(lam * lam * ((ai + a.a_seg) * (ai + a.a_seg)));
    const T sum_blob = T(lam * lam * ((ai + a.a_blob) * (ai + a.a_blob)));
    auto is_near = [&](int j) {
        const int jcls = j < a.ns ? 0 : 1;
        T rec[REC];
        stage_source<T, 3>(rec, a, jcls, jcls == 0 ? j : j - a.ns, false);
        T ddx, ddy, ddz;
        const T r2 = separation(xi, rec, ddx, ddy, ddz);
        return !(r2 > (jcls == 0 ? sum_seg : sum_blob));
    };
    if (in && lane < 27) {
        const int nx = own.x + lane % 3 - 1, ny = own.y + (lane / 3) % 3 - 1, nz = own.z + lane / 9 - 1;
        int j = head[body_cell_hash(nx, ny, nz, body, mask)];
        for (int left = walk; j >= 0 && left > 0; --left) {
            const int4 nd = nodes[j];
            // the bucket may also hold other cells (and bodies): visit j from its own only
            if (nd.x == nx && nd.y == ny && nd.z == nz && (!body_of || body_of[j] == body) && is_near(j)) {
                const int k = atomicAdd(&found[s], 1);
                if (k < kNearLds) list[s][k] = j;
                if (k < cap) e[k] = j;
            }
            j = nd.w;
        }
        if (j >= 0) crowded[s] = 1;
    }
    __syncthreads();
    int total = in ? found[s] : 0;
    const bool scan = in && (crowded[s] || total > 32 * kRankPer);
    if (scan) {
        const int shift = (int)(threadIdx.x & 32);  // the target's half of the wave
        const int4 r = ranges[body];
        const int m = (r.y - r.x) + (r.w - r.z);
        total = 0;
        for (int t0 = 0; t0 < m; t0 += 32) {
            const int t = t0 + lane;
            const int j = body_particle(r, a.ns, t < m ? t : m - 1);
            const bool near = t < m && is_near(j);
            const uint32_t hits = (uint32_t)(__ballot(near) >> shift);
            const int k = total + __popc(hits & ((1u << lane) - 1u));
            if (near && k < cap) e[k] = j;
            total += __popc(hits);
        }
    }
    if (in && lane == 0) {
        cnt[tg] = total;
        if (total > cap) atomicMax(max_cnt, total);
    }
    if (!scan && total <= kNearLds) {
        for (int i = lane; i < total; i += 32) {
            const int32_t v = list[s][i];
            int q = 0;
            for (int j = 0; j < total; ++j) q += list[s][j] < v ? 1 : 0;
            if (q < cap) e[q] = v;
        }
    }
    const bool by_rank = !scan && total > kNearLds;
    if (!__syncthreads_or(by_rank)) return;
    // longer lists: ranked against what the barrier above made readable
    const int c = total < cap ? total : cap;
    int32_t val[kRankPer];
    int rank[kRankPer];
#pragma unroll
    for (int q = 0; q < kRankPer; ++q) {
        const int i = lane + 32 * q;
        val[q] = 0;
        rank[q] = -1;
        if (by_rank && i < c) {
            const int32_t v = e[i];
            int below = 0;
            for (int j = 0; j < c; ++j) below += e[j] < v ? 1 : 0;
            val[q] = v;
            rank[q] = below;
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kRankPer; ++q)
        if (rank[q] >= 0) e[rank[q]] = val[q];
}

// The FP64 lists of small problems by testing every pair of a body in one launch:
// four targets per wave, whose lanes take 64 sources at a time (four batches'
// loads in flight); a ballot places the near ones, so the lists come out in
// increasing order.  Grid (bodies, 16 targets each).  *max_cnt is zero before
// (geometry_clear_kernel's job otherwise).
__global__ __launch_bounds__(256) void near_small_kernel(MatvecArgs a, const int4* __restrict__ ranges,
                                                        int32_t* __restrict__ cnt, int32_t* __restrict__ idx, int cap,
                                                        int32_t* __restrict__ max_cnt) {
    constexpr int REC = rec_len<double, 3>(), U = 4, Q = 4;
    const int4 r = ranges[blockIdx.x];
    const int m = (r.y - r.x) + (r.w - r.z);
    const int lane = (int)threadIdx.x & 63;
    const int t0 = ((int)blockIdx.y * 4 + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6)) * U;
    if (t0 >= m) return;
    double xi[U][3], sum_seg[U], sum_blob[U];
    int32_t* e[U];
    int n[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int p = body_particle(r, a.ns, t0 + u < m ? t0 + u : m - 1);
        const int cls = p < a.ns ? 0 : 1;
        load_target(a, cls, cls == 0 ? p : p - a.ns, xi[u]);
        const double ai = cls == 0 ? a.a_seg : a.a_blob;
        sum_seg[u] = (ai + a.a_seg) * (ai + a.a_seg);
        sum_blob[u] = (ai + a.a_blob) * (ai + a.a_blob);
        e[u] = idx + (int64_t)p * cap;
        n[u] = 0;
    }
    for (int s0 = 0; s0 < m; s0 += 64 * Q) {
        double rec[Q][REC];
        int src[Q];
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int t = s0 + 64 * q + lane;
            src[q] = body_particle(r, a.ns, t < m ? t : m - 1);
            const int cls = src[q] < a.ns ? 0 : 1;
            stage_source<double, 3>(rec[q], a, cls, cls == 0 ? src[q] : src[q] - a.ns, false);
        }
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const bool in = s0 + 64 * q + lane < m;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                double ddx, ddy, ddz;
                const double r2 = separation(xi[u], rec[q], ddx, ddy, ddz);
                const bool near = in && !(r2 > (src[q] < a.ns ? sum_seg[u] : sum_blob[u]));
                const uint64_t hits = __ballot(near);
                const int k = n[u] + __popcll(hits & ((uint64_t(1) << lane) - 1));
                if (near && k < cap && t0 + u < m) e[u][k] = src[q];
                n[u] += __popcll(hits);
            }
        }
    }
    if (lane != 0) return;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        if (t0 + u >= m) continue;
        cnt[body_particle(r, a.ns, t0 + u)] = n[u];
        if (n[u] > cap) atomicMax(max_cnt, n[u]);
    }
}

__global__ void fill_int_kernel(int32_t* p, int32_t v, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// Barrier (short-range repulsion) forces of the elastic model
// (cuda_functions.cu:1240-1436).  Per particle p, over every other particle j
// within 1.1 (ai + aj) -- except, for segments, j itself and its neighbours
// on the same filament --
//   f_p += S fac^4 (x_p - x_j)/|x_p - x_j|,  fac = min(1, 1 - 10 (r - ai - aj)/(ai + aj)),
// and for segments below z = DL/2 with the plane wall a normal force
// S min(1, 1 - (z - a)/(DL/2 - a))^4 first.  Segment forces are added to
// slots 0-2 of fs (stride 6); blob forces overwrite fb (stride 3, may be
// null).  Candidates come from the 27 neighbouring cells of side
// >= 1.1 * 2 max(a), in a fixed order (cells, then indices within a bucket),
// so results are reproducible; each is visited from its own cell only.
__global__ __launch_bounds__(256) void barrier_kernel(MatvecArgs a, int n, double inv_h, uint32_t mask,
                                                     const int32_t* __restrict__ start,
                                                     const int32_t* __restrict__ order, BarrierParams bp,
                                                     double* __restrict__ fs, double* __restrict__ fb) {
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p >= n) return;
    double xi[3];
    particle_pos(a, p, xi);
    const bool seg = p < a.ns;
    const double ai = seg ? a.a_seg : a.a_blob;
    const int fili = seg ? p / bp.nseg : -1;
    double f[3] = {0.0, 0.0, 0.0};
    if (seg && bp.wall && xi[2] < 0.5 * bp.dl) {
        double fz = fmin(1.0, 1.0 - (xi[2] - a.a_seg) / (0.5 * bp.dl - a.a_seg));
        fz *= bp.strength * fz * fz * fz;
        f[2] = fz;
    }
    const int cx = cell_coord(xi[0], inv_h), cy = cell_coord(xi[1], inv_h), cz = cell_coord(xi[2], inv_h);
    for (int dz = -1; dz <= 1; ++dz)
        for (int dy = -1; dy <= 1; ++dy)
            for (int dx = -1; dx <= 1; ++dx) {
                const int nx = cx + dx, ny = cy + dy, nz = cz + dz;
                const uint32_t b = cell_hash(nx, ny, nz, mask);
                for (int q = start[b]; q < start[b + 1]; ++q) {
                    const int j = order[q];
                    if (j == p) continue;
                    const bool jseg = j < a.ns;
                    if (seg && jseg && j / bp.nseg == fili && (j - p <= 1 && p - j <= 1)) continue;
                    double xj[3];
                    particle_pos(a, j, xj);
                    if (cell_coord(xj[0], inv_h) != nx || cell_coord(xj[1], inv_h) != ny ||
                        cell_coord(xj[2], inv_h) != nz)
                        continue;
                    const double asum = ai + (jseg ? a.a_seg : a.a_blob);
                    const double ddx = xi[0] - xj[0], ddy = xi[1] - xj[1], ddz = xi[2] - xj[2];
                    const double dist = sqrt(ddx * ddx + ddy * ddy + ddz * ddz);
                    if (dist < 1.1 * asum) {
                        double fac = fmin(1.0, 1.0 - (10.0 / asum) * (dist - asum));
                        fac *= bp.strength * fac * fac * fac;
                        const double dm1 = 1.0 / dist;
                        f[0] += fac * ddx * dm1;
                        f[1] += fac * ddy * dm1;
                        f[2] += fac * ddz * dm1;
                    }
                }
            }
    if (seg) {
#pragma unroll
        for (int k = 0; k < 3; ++k) fs[(int64_t)p * 6 + k] += f[k];
    } else if (fb) {
#pragma unroll
        for (int k = 0; k < 3; ++k) fb[(int64_t)(p - a.ns) * 3 + k] = f[k];
    }
}

template <int VT>
__device__ void add_near(double* acc, int src, const double* xi, double ai, const MatvecArgs& a, int seg_dof,
                         uint32_t cls_mask) {
    const bool seg = src < a.ns;
    if (!(cls_mask & (seg ? 1u : 2u))) return;  // that block is not active
    const int s = seg ? src : src - a.ns;
    const CView xv = seg ? a.xs : a.xb;
    const CView fv = seg ? a.fs : a.fb;
    const double d0 = xi[0] - xv.p[(int64_t)s * xv.ld_p];
    const double d1 = xi[1] - xv.p[(int64_t)s * xv.ld_p + xv.ld_c];
    const double d2 = xi[2] - xv.p[(int64_t)s * xv.ld_p + 2 * xv.ld_c];
    double f[6];
    const int fs = seg ? seg_dof : 3;
    for (int k = 0; k < 6; ++k) f[k] = k < fs ? fv.p[(int64_t)s * fv.ld_p + k * fv.ld_c] : 0.0;
    const double aj = seg ? a.a_seg : a.a_blob;
    // Take out what the pair loop added for this pair -- the far-field form at
    // r clamped to ai + aj, with the strengths scaled by 1/(8 pi mu) -- then add
    // the reference's overlap / inner-branch value.
    const double PI = 3.14159265358979323846;
    const double c8 = 1.0 / (8.0 * PI * a.mu);
    const double s3 = (ai * ai + aj * aj) / 3.0;
    double fsc[6], clamp[6] = {0, 0, 0, 0, 0, 0};
    for (int k = 0; k < 6; ++k) fsc[k] = c8 * f[k];
    const double rm1c = rsqrt_refined((ai + aj) * (ai + aj));
    if (fs == 6) pair_far_scaled<double, VT, 6>(clamp, d0, d1, d2, rm1c, fsc, nullptr, s3, -3.0 * s3);
    else pair_far_scaled<double, VT, 3>(clamp, d0, d1, d2, rm1c, fsc, nullptr, s3, -3.0 * s3);
    for (int k = 0; k < VT; ++k) acc[k] -= clamp[k];
    if (fs == 6) pair_near<VT, 6>(acc, d0, d1, d2, f, ai, aj, a.mu);
    else pair_near<VT, 3>(acc, d0, d1, d2, f, ai, aj, a.mu);
}

// Filament rows of the saddle-point operator: -K_phi^T lambda and
// -K_theta^T lambda over the filament's 3*nseg entries, by one wave.
__device__ void saddle_filament_rows(const SaddleEpilogue& e, int m, int lane) {
    const int len = 3 * e.nseg;
    const int64_t seg0 = (int64_t)m * len;
    double sp = 0.0, st = 0.0;
    for (int k = lane; k < len; k += 64) {
        const double lam = e.in[seg0 + k];
        sp += lam * e.kphi[seg0 + k];
        st += lam * e.kth[seg0 + k];
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        sp += __shfl_down(sp, off, 64);
        st += __shfl_down(st, off, 64);
    }
    if (lane == 0) {
        if (e.dyn_phase) e.out[e.off_phase + m] = -sp;
        if (e.dyn_angle) e.out[e.off_angle + m] = -st;
    }
}

// Adds the partial slots of each tile and the overlapping pairs, and applies
// the write rule.  A slot holds slot_dof x tile_targets values (component k
// of target l at k * tile_targets + l).  A workgroup covers 64 targets of one
// tile with GR groups of 64 threads: group g sums the items g, g+GR, g+2 GR,
// ... (loads of four items issued together) and then the near-list entries g,
// g+GR, ... of its target (the lists are sorted when built); the group sums
// are added in group order, so the result is the same on every run.
// Workgroups past `tile_blocks` write the filament rows of the saddle-point
// operator.
//
// Bound by latency and the slots' bytes: few tiles with many slots each want
// many loads in flight (reduce_groups: 12,800 segments + 9,000 blobs, 6
// components FP32, 28 MB of slots: 36 us with the component count a condition
// on every load, 13 without).
template <int SEGDOF, typename P, int GR>
__global__ __launch_bounds__(64 * GR) void rpy_reduce_kernel(const MatvecTile* __restrict__ tiles,
                                                             const P* __restrict__ partial, int tile_targets,
                                                             int tile_blocks, int merge_k, int slot_dof, OutArgs o,
                                                             MatvecArgs a, NearList near) {
    __shared__ double grp_acc[GR - 1][6][64];
    if (a.skip && *a.skip) return;
    const int grp = threadIdx.x >> 6;
    if ((int)blockIdx.x >= tile_blocks) {
        const int m = ((int)blockIdx.x - tile_blocks) * GR + grp;
        if (m < o.sad.nfil && !(a.body_skip && o.sad.fil_body && a.body_skip[o.sad.fil_body[m]]))
            saddle_filament_rows(o.sad, m, threadIdx.x & 63);
        return;
    }
    const int per_tile = (tile_targets + 63) / 64;
    const MatvecTile tl = tiles[blockIdx.x / per_tile];
    if (a.body_skip && a.body_skip[tl.body]) return;  // the whole workgroup has this tile
    const int l = (blockIdx.x % per_tile) * 64 + (threadIdx.x & 63);
    const int t = tl.t_begin + l;
    const bool active = l < tile_targets && t < tl.t_end;
    const bool seg_t = tl.cls == 0;
    const int vt = seg_t ? SEGDOF : 3;
    const size_t slot_len = (size_t)slot_dof * tile_targets;
    const int lc = l < tile_targets ? l : tile_targets - 1;
    const P* p = partial + (size_t)tl.first_item * slot_len + lc;
    // Filled slots: every item's, or (persistent form, merge_k items per
    // workgroup) the tile's first item and the multiples of merge_k after it.
    const int q0 = merge_k > 0 ? tl.first_item / merge_k : 0;
    const int nslots = merge_k > 0 && tl.n_items > 0 ? (tl.first_item + tl.n_items - 1) / merge_k - q0 + 1
                                                     : tl.n_items;
    auto slot_of = [&](int q) { return merge_k > 0 ? (q == 0 ? 0 : (q0 + q) * merge_k - tl.first_item) : q; };
    double acc[6] = {0, 0, 0, 0, 0, 0};
    // one instance per component count: with the count a condition on each load
    // the loads of an iteration would wait for one another
    auto sum_slots = [&](auto comps) {
        constexpr int VT = decltype(comps)::value;
        for (int m0 = grp; m0 < nslots; m0 += 4 * GR) {
            double v[4][VT];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int m = m0 + GR * u;
                const P* q = p + (size_t)slot_of(m < nslots ? m : grp) * slot_len;
#pragma unroll
                for (int k = 0; k < VT; ++k) v[u][k] = double(q[(size_t)k * tile_targets]);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const bool in = m0 + GR * u < nslots;
#pragma unroll
                for (int k = 0; k < VT; ++k) acc[k] += in ? v[u][k] : 0.0;
            }
        }
    };
    if (SEGDOF == 6 && seg_t) sum_slots(std::integral_constant<int, 6>{});
    else sum_slots(std::integral_constant<int, 3>{});
    // Active source classes for this target class: bit 0 segments, bit 1 blobs.
    const uint32_t cls_mask = seg_t ? ((o.blocks & 1u) ? 1u : 0u) | ((o.blocks & 2u) ? 2u : 0u)
                                    : ((o.blocks & 8u) ? 1u : 0u) | ((o.blocks & 4u) ? 2u : 0u);
    if (near.cnt && cls_mask && active) {
        const int tg = (seg_t ? 0 : a.ns) + t;
        const int c = near.cnt[tg] < near.cap ? near.cnt[tg] : near.cap;
        const int32_t* e = near.idx + (int64_t)tg * near.cap;
        const CView xv = seg_t ? a.xs : a.xb;
        const double xi[3] = {xv.p[(int64_t)t * xv.ld_p], xv.p[(int64_t)t * xv.ld_p + xv.ld_c],
                              xv.p[(int64_t)t * xv.ld_p + 2 * xv.ld_c]};
        const double ai = seg_t ? a.a_seg : a.a_blob;
        for (int q = grp; q < c; q += GR) {
            if (seg_t && SEGDOF == 6) add_near<6>(acc, e[q], xi, ai, a, SEGDOF, cls_mask);
            else add_near<3>(acc, e[q], xi, ai, a, SEGDOF, cls_mask);
        }
    }
    if (grp > 0) {
#pragma unroll
        for (int k = 0; k < 6; ++k) grp_acc[grp - 1][k][threadIdx.x & 63] = acc[k];
    }
    __syncthreads();
    if (grp > 0 || !active) return;
#pragma unroll
    for (int g = 0; g < GR - 1; ++g)
#pragma unroll
        for (int k = 0; k < 6; ++k) acc[k] += grp_acc[g][k][threadIdx.x];
    if (seg_t && o.sad.in && (o.sad.dyn_phase || o.sad.dyn_angle)) {
        const int m = t / o.sad.nseg;
        const double pd = o.sad.dyn_phase ? o.sad.in[o.sad.off_phase + m] : 0.0;
        const double td = o.sad.dyn_angle ? o.sad.in[o.sad.off_angle + m] : 0.0;
        for (int k = 0; k < 3; ++k) acc[k] -= pd * o.sad.kphi[3 * (int64_t)t + k] + td * o.sad.kth[3 * (int64_t)t + k];
    }
    if (o.sad.free_body) {
        // -(V + Omega x r) of the target's swimmer (mobility_solver.cpp:1856-1870, 1885-1894)
        const int sw = seg_t ? t / o.sad.segs_per_swim : t / o.sad.blobs_per_swim;
        const double* V = o.sad.in + o.sad.off_body + 6 * (int64_t)sw;
        const CView xv = seg_t ? a.xs : a.xb;
        const double r0 = xv.p[(int64_t)t * xv.ld_p] - o.sad.x_bodies[3 * sw];
        const double r1 = xv.p[(int64_t)t * xv.ld_p + xv.ld_c] - o.sad.x_bodies[3 * sw + 1];
        const double r2 = xv.p[(int64_t)t * xv.ld_p + 2 * xv.ld_c] - o.sad.x_bodies[3 * sw + 2];
        acc[0] -= V[0] + (V[4] * r2 - V[5] * r1);
        acc[1] -= V[1] + (V[5] * r0 - V[3] * r2);
        acc[2] -= V[2] + (V[3] * r1 - V[4] * r0);
    }
    const int slots = seg_t ? o.seg_out_slots : 3;
    const View out = seg_t ? o.vs : o.vb;
    for (int k = 0; k < slots; ++k) {
        double* dst = out.p + (int64_t)t * out.ld_p + k * out.ld_c;
        if (tl.write_mode == 0) *dst = k < vt ? acc[k] : 0.0;
        else if (k < vt) *dst += acc[k];
    }
}

// Items per workgroup of the persistent form: the work list over
// persistent x CUs workgroups, as contiguous ranges.
int persistent_items(const TileShape& sh, int n_items, int num_cus) {
    const long g = (long)sh.persistent * (num_cus > 0 ? num_cus : 256);
    return (int)std::max<long>(1, (n_items + g - 1) / g);
}

template <typename T, int SEGDOF, int BLOCK, int R, bool SPLIT>
hipError_t launch_pairs(const TileShape& sh, const MatvecArgs& a, const MatvecItem* d_items, int n_items,
                        const MatvecTile* d_tiles, double* partial, const PersistState& ps, hipStream_t stream) {
    if (SPLIT && sh.persistent > 0) return hipErrorInvalidValue;  // no persistent form of the split
    if (!SPLIT && sh.persistent > 0) {
        const int k = persistent_items(sh, n_items, ps.num_cus);
        hipLaunchKernelGGL((rpy_pairs_persistent_kernel<T, SEGDOF, BLOCK, R>), dim3((unsigned)((n_items + k - 1) / k)),
                           dim3(BLOCK), 0, stream, d_items, d_tiles, a, reinterpret_cast<T*>(partial), n_items, k,
                           ps);
    } else {
        hipLaunchKernelGGL((rpy_pairs_kernel<T, SEGDOF, BLOCK, R, SPLIT>), dim3(n_items), dim3(BLOCK), 0, stream,
                           d_items, d_tiles, a, reinterpret_cast<T*>(partial), ps.item_stamps);
    }
    return hipGetLastError();
}

template <typename T, int SEGDOF>
hipError_t dispatch_shape(const TileShape& sh, const MatvecArgs& a, const MatvecItem* d_items, int n_items,
                          const MatvecTile* d_tiles, double* partial, const PersistState& ps,
                          hipStream_t stream) {
#define TFS_SHAPE(B, R, S)                                                                    \
    if (sh.block == B && sh.per_thread == R && sh.split == S)                                \
        return launch_pairs<T, SEGDOF, B, R, S>(sh, a, d_items, n_items, d_tiles, partial, ps, stream);
    TFS_SHAPE(64, 1, 0) TFS_SHAPE(64, 2, 0) TFS_SHAPE(128, 1, 0) TFS_SHAPE(128, 2, 0) TFS_SHAPE(256, 1, 0)
    TFS_SHAPE(256, 2, 0) TFS_SHAPE(256, 1, 1) TFS_SHAPE(256, 2, 1) TFS_SHAPE(512, 1, 1) TFS_SHAPE(512, 2, 1)
#undef TFS_SHAPE
    return hipErrorInvalidValue;
}

template <typename T, int DOF>
hipError_t launch_sym(int kind, const MatvecArgs& a, const MatvecItem* d_items, int n_items, const MatvecTile* d_tiles,
                      int n_tiles, int bb, double* partial, const PersistState& ps, hipStream_t stream) {
    T* part = reinterpret_cast<T*>(partial);
    const dim3 grid((unsigned)n_items), block(64 * kSymWaves);
    if (kind == kSymWide)
        hipLaunchKernelGGL((rpy_pairs_sym_kernel<T, DOF, 2>), grid, block, 0, stream, d_items, d_tiles, n_tiles, bb, a,
                           part, ps.item_stamps);
    else
        hipLaunchKernelGGL((rpy_pairs_sym_kernel<T, DOF, 1>), grid, block, 0, stream, d_items, d_tiles, n_tiles, bb, a,
                           part, ps.item_stamps);
    return hipGetLastError();
}

}  // namespace

void build_worklist(const std::vector<BodyRange>& bodies, int tile_targets, int chunk, bool ss, bool sb,
                    bool bb, bool bs, int seg_write, int blob_write, std::vector<MatvecTile>& tiles,
                    std::vector<MatvecItem>& items) {
    tiles.clear();
    items.clear();
    // Target tiles of every body; with several bodies the tiles are then
    // interleaved in proportion to each body's tile count (tile k of T_b at
    // position (k + 1/2) / T_b), so that every body's work is spread over the
    // whole launch and the bodies finish together.
    struct Pending {
        MatvecTile tl;
        double pos;
    };
    std::vector<Pending> pend;
    for (const BodyRange& body : bodies) {
        const size_t first = pend.size();
        auto add_tiles = [&](int cls, int t_lo, int t_hi, int write) {
            if (write < 0) return;
            for (int t0 = t_lo; t0 < t_hi; t0 += tile_targets) {
                MatvecTile tl{};
                tl.cls = cls;
                tl.t_begin = t0;
                tl.t_end = std::min(t0 + tile_targets, t_hi);
                tl.write_mode = write;
                tl.body = (int32_t)(&body - bodies.data());
                pend.push_back({tl, 0.0});
            }
        };
        add_tiles(0, body.seg_begin, body.seg_end, seg_write);
        add_tiles(1, body.blob_begin, body.blob_end, blob_write);
        const size_t nt = pend.size() - first;
        for (size_t k = 0; k < nt; ++k) pend[first + k].pos = (double(k) + 0.5) / double(nt);
    }
    if (bodies.size() > 1)
        std::stable_sort(pend.begin(), pend.end(), [](const Pending& x, const Pending& y) { return x.pos < y.pos; });
    for (Pending& pt : pend) {
        MatvecTile tl = pt.tl;
        const BodyRange& body = bodies[tl.body];
        const bool from_segs = tl.cls == 0 ? ss : bs, from_blobs = tl.cls == 0 ? sb : bb;
        tl.first_item = (int)items.size();
        const int tile_id = (int)tiles.size();
        std::vector<MatvecItem> chunks;  // the tile's items in source order
        auto add_src = [&](int src_cls, int lo, int hi) {
            for (int s0 = lo; s0 < hi; s0 += chunk) chunks.push_back({tile_id, src_cls, s0, std::min(s0 + chunk, hi)});
        };
        if (from_segs) add_src(0, body.seg_begin, body.seg_end);
        if (from_blobs) add_src(1, body.blob_begin, body.blob_end);
        // Workgroup i of a launch runs on XCD i mod 8.  Chunk c of every tile
        // goes to a position p with p = c (mod 8) where one is free, so each
        // XCD's L2 holds about an eighth of the sources instead of all of them.
        const int n = (int)chunks.size();
        std::vector<int> next(kXcds, 0), order(n, -1);
        std::vector<char> used(n, 0);
        for (int i = 0; i < n; ++i) {
            const int want = (tl.first_item + i) % kXcds;
            int& c = next[want];
            while (c * kXcds + want < n && used[c * kXcds + want]) ++c;
            if (c * kXcds + want < n) {
                order[i] = c * kXcds + want;
                used[order[i]] = 1;
            }
        }
        for (int i = 0, c = 0; i < n; ++i) {
            if (order[i] >= 0) continue;
            while (used[c]) ++c;
            order[i] = c;
            used[c] = 1;
        }
        for (int i = 0; i < n; ++i) items.push_back(chunks[order[i]]);
        tl.n_items = n;
        tiles.push_back(tl);
    }
}

size_t build_sym_worklist(const std::vector<BodyRange>& bodies, int kind, int seg_dof, int num_cus, int seg_write,
                          int blob_write, std::vector<MatvecTile>& tiles, std::vector<MatvecItem>& items) {
    tiles.clear();
    items.clear();
    for (size_t b = 0; b < bodies.size(); ++b) {
        auto add_tiles = [&](int cls, int lo, int hi, int write) {
            for (int t0 = lo; t0 < hi; t0 += 64) {
                MatvecTile tl{};
                tl.cls = cls;
                tl.t_begin = t0;
                tl.t_end = std::min(t0 + 64, hi);
                tl.write_mode = write;
                tl.body = (int32_t)b;
                tiles.push_back(tl);
            }
        };
        add_tiles(0, bodies[b].seg_begin, bodies[b].seg_end, seg_write);
        add_tiles(1, bodies[b].blob_begin, bodies[b].blob_end, blob_write);
    }
    const int n_tiles = (int)tiles.size();
    const int panel = sym_panel(kind), n_panels = (n_tiles + panel - 1) / panel;
    std::vector<int> first(bodies.size(), 0), last(bodies.size(), -1);  // each body's tiles
    for (int t = n_tiles - 1; t >= 0; --t) {
        first[tiles[t].body] = t;
        if (last[tiles[t].body] < 0) last[tiles[t].body] = t;
    }
    // Source tiles of panel A: its own, then the rest of its last body's.
    auto end_of = [&](int A) { return last[tiles[std::min(panel * A + panel, n_tiles) - 1].body] + 1; };
    // Cost of a panel's tiles against one source tile, in 3-component tile pairs;
    // beyond the panel it depends on the source's class only.
    auto pair_cost = [&](int ta, int tb) {
        if (ta > tb || tiles[ta].body != tiles[tb].body) return 0.0;
        const bool sa = tiles[ta].cls == 0, sb = tiles[tb].cls == 0;
        return (seg_dof == 6 ? (sa && sb ? 2.2 : sa || sb ? 1.4 : 1.0) : 1.0) * (ta == tb ? 0.6 : 1.0);
    };
    auto cost_of = [&](int A, int tb) {
        double c = 0.0;
        for (int ta = panel * A; ta < std::min(panel * A + panel, n_tiles); ++ta) c += pair_cost(ta, tb);
        return c;
    };
    std::vector<double> cost(n_tiles);  // of the current panel's source tiles
    auto panel_costs = [&](int A) {
        const int own_end = std::min(panel * A + panel, n_tiles), end = end_of(A);
        double sum = 0.0;
        for (int q = panel * A; q < end; ++q) {
            const bool as_before = q > own_end && tiles[q].cls == tiles[q - 1].cls;
            cost[q] = as_before ? cost[q - 1] : cost_of(A, q);
            sum += cost[q];
        }
        return sum;
    };
    double left = 0.0;
    for (int A = 0; A < n_panels; ++A) left += panel_costs(A);
    // Runs: about half of what is left shared by the workgroups that fit the
    // device, so that the last ones are single tiles and the launch ends evenly
    // without every tile costing its panel a slot.
    const double resident = 5.0 * (num_cus > 0 ? num_cus : 256);
    std::vector<int> run_of;                       // of the panel's source tiles
    for (int A = 0; A < n_panels; ++A) {
        const int q_lo = panel * A, q_hi = end_of(A);
        run_of.assign(q_hi - q_lo, 0);
        panel_costs(A);
        int run = 0;
        for (int q = q_lo; q < q_hi;) {
            const double want = std::max(left / (2.0 * resident), 1.0);
            int e = q;
            double c = 0.0;
            while (e < q_hi && e - q < kSymMaxRun && (e == q || c + 0.5 * cost[e] <= want)) {
                c += cost[e];
                run_of[e - q_lo] = run;
                ++e;
            }
            items.push_back({A, q, e, run});
            left -= c;
            q = e;
            ++run;
        }
        for (int t = q_lo; t < std::min(q_lo + panel, n_tiles); ++t) {
            MatvecTile& tl = tiles[t];
            tl.panel0 = first[tl.body] / panel;
            tl.run0 = run_of[t - q_lo];
            tl.n_items = (A - tl.panel0) + (run_of[last[tl.body] - q_lo] - tl.run0 + 1);
        }
    }
    size_t slots = 0;
    for (MatvecTile& tl : tiles) {
        tl.first_item = (int32_t)slots;
        slots += (size_t)tl.n_items;
    }
    return slots;
}

void free_grid(NearGrid& g) {
    for (int32_t* p : {g.start, g.fill, g.bucket_of, g.order, g.body_of})
        if (p) (void)hipFree(p);
    if (g.nodes) (void)hipFree(g.nodes);
    g = NearGrid{};
}

// The grid's size for n particles; arrays made for another go.
static void size_grid(NearGrid& grid, int n) {
    int table = 1024;
    while (table < 2 * n) table <<= 1;
    if (grid.n == n && grid.table == table) return;
    free_grid(grid);
    grid.n = n;
    grid.table = table;
}

// Sorts the n particles (segments, then blobs) into the grid's buckets for
// cells of side 1 / inv_h: start (exclusive bucket offsets) and order.
static hipError_t sort_into_grid(const MatvecArgs& a, NearGrid& grid, int n, double inv_h, hipStream_t stream) {
    size_grid(grid, n);
    const int table = grid.table;
    if (!grid.fill) TFS_HIP_CHECK(hipMalloc(&grid.fill, sizeof(int32_t) * table));
    if (!grid.order) {
        if (!grid.start) TFS_HIP_CHECK(hipMalloc(&grid.start, sizeof(int32_t) * (table + 1)));
        if (!grid.bucket_of) TFS_HIP_CHECK(hipMalloc(&grid.bucket_of, sizeof(int32_t) * n));
        TFS_HIP_CHECK(hipMalloc(&grid.order, sizeof(int32_t) * n));
    }
    const uint32_t mask = (uint32_t)table - 1;
    const unsigned gn = (unsigned)((n + 255) / 256);
    hipLaunchKernelGGL(fill_int_kernel, dim3((unsigned)((table + 255) / 256)), dim3(256), 0, stream, grid.fill, 0,
                       (int64_t)table);
    hipLaunchKernelGGL(grid_count_kernel, dim3(gn), dim3(256), 0, stream, a, n, inv_h, mask, grid.bucket_of, grid.fill);
    hipLaunchKernelGGL(grid_scan_kernel, dim3(1), dim3(1024), 0, stream, grid.fill, grid.start, table);
    hipLaunchKernelGGL(grid_scatter_kernel, dim3(gn), dim3(256), 0, stream, n, grid.bucket_of, grid.start, grid.fill,
                       grid.order);
    hipLaunchKernelGGL(grid_sort_buckets_kernel, dim3((unsigned)((table + 255) / 256)), dim3(256), 0, stream, table,
                       grid.start, grid.order);
    return hipGetLastError();
}

int box_shares(int nbody, int largest) {
    const int fit = nbody < kBoxShares ? kBoxShares / nbody : 1;
    return std::max(1, std::min(fit, (largest + 255) / 256));
}

// Clears (and with `fixed` the bounding boxes), then places: the fixed-point
// positions and, with nodes, the grid.
static void launch_geometry(const MatvecArgs& a, const GeometryArgs& g, bool fixed, NearGrid* grid, double inv_h,
                            int32_t* max_cnt, hipStream_t stream) {
    const int4* ranges = reinterpret_cast<const int4*>(g.ranges);
    int32_t* head = grid ? grid->fill : nullptr;
    const int table = grid ? grid->table : 0;
    const double amin = std::min(a.a_seg, a.a_blob);
    int shares = box_shares(g.nbody, g.largest);
    if (fixed)
        hipLaunchKernelGGL(geometry_clear_kernel<true>, dim3((unsigned)g.nbody, (unsigned)shares), dim3(256), 0, stream,
                           a, ranges, g.box, head, table, max_cnt);
    else
        hipLaunchKernelGGL(geometry_clear_kernel<false>, dim3((unsigned)std::max(1, table / 4096)), dim3(256), 0,
                           stream, a, ranges, g.box, head, table, max_cnt);
    const int per_body = std::max(1, std::min((g.largest + 255) / 256, std::max(1, 4096 / g.nbody)));
    const dim3 place((unsigned)g.nbody, (unsigned)per_body);
    if (fixed && g.nbody > kFrameBodies) {
        // (every box in every workgroup is the square of the bodies: an evaluation
        // of 20,000 bodies of 40 at new positions took 1,835 us, 980 so; the
        // launch takes 1.6 us more where there are 300)
        hipLaunchKernelGGL(geometry_frame_kernel, dim3(1), dim3(1024), 0, stream, (const double*)g.box, g.nbody, amin,
                           g.frame);
        shares = 0;
    }
    const uint32_t mask = (uint32_t)table - 1;
    int4* nodes = grid ? grid->nodes : nullptr;
    int32_t* body_of = grid && g.nbody > 1 ? grid->body_of : nullptr;
    if (fixed)
        hipLaunchKernelGGL(geometry_place_kernel<true>, place, dim3(256), 0, stream, a, ranges, (const double*)g.box,
                           shares, amin, g.fixed, g.frame, inv_h, mask, head, nodes, body_of);
    else
        hipLaunchKernelGGL(geometry_place_kernel<false>, place, dim3(256), 0, stream, a, ranges, (const double*)g.box,
                           shares, 0.0, g.fixed, g.frame, inv_h, mask, head, nodes, body_of);
}

hipError_t launch_fixed(const MatvecArgs& a, const GeometryArgs& g, hipStream_t stream) {
    launch_geometry(a, g, true, nullptr, 0.0, &g.frame->max_cnt[1], stream);
    return hipGetLastError();
}

hipError_t build_near_list(int precision, const MatvecArgs& a, const GeometryArgs& g, bool fixed, NearGrid& grid,
                           const NearList& near, hipStream_t stream) {
    const int n = a.ns + a.nb;
    if (n <= 0) return hipSuccess;
    if (precision == 0 && n <= kNearSmallMax) {
        hipLaunchKernelGGL(near_small_kernel, dim3((unsigned)g.nbody, (unsigned)((g.largest + 15) / 16)), dim3(256), 0,
                           stream, a, reinterpret_cast<const int4*>(g.ranges), near.cnt, near.idx, near.cap,
                           near.max_cnt);
        return hipGetLastError();
    }
    size_grid(grid, n);
    if (!grid.fill) TFS_HIP_CHECK(hipMalloc(&grid.fill, sizeof(int32_t) * grid.table));
    if (!grid.nodes) TFS_HIP_CHECK(hipMalloc(&grid.nodes, sizeof(int4) * n));
    if (g.nbody > 1 && !grid.body_of) TFS_HIP_CHECK(hipMalloc(&grid.body_of, sizeof(int32_t) * n));
    const double h = 2.0 * std::max(a.a_seg, a.a_blob) * (1.0 + 1e-5);
    const double inv_h = 1.0 / h;
    launch_geometry(a, g, fixed, &grid, inv_h, near.max_cnt, stream);
    const uint32_t mask = (uint32_t)grid.table - 1;
    const unsigned gl = (unsigned)((n + 7) / 8);   // 8 targets of 32 lanes per workgroup
    const int32_t* body_of = g.nbody > 1 ? grid.body_of : nullptr;
    // a step of the walk waits for the one before, a pass takes 32 particles at once
    const int walk = std::max(256, g.largest / 32);
    if (precision == 0)
        hipLaunchKernelGGL(near_grid_kernel<double>, dim3(gl), dim3(256), 0, stream, a, n, inv_h, mask,
                           reinterpret_cast<const int4*>(g.ranges), walk, grid.fill, grid.nodes, body_of, near.cnt, near.idx, near.cap, near.max_cnt);
    else
        hipLaunchKernelGGL(near_grid_kernel<float>, dim3(gl), dim3(256), 0, stream, a, n, inv_h, mask,
                           reinterpret_cast<const int4*>(g.ranges), walk, grid.fill, grid.nodes, body_of, near.cnt, near.idx, near.cap, near.max_cnt);
    return hipGetLastError();
}

hipError_t launch_barrier(const MatvecArgs& a, NearGrid& grid, const BarrierParams& bp, double* fs, double* fb,
                          hipStream_t stream) {
    const int n = a.ns + a.nb;
    if (n <= 0) return hipSuccess;
    const double h = 2.2 * std::max(a.a_seg, a.a_blob) * (1.0 + 1e-6);
    const double inv_h = 1.0 / h;
    TFS_HIP_CHECK(sort_into_grid(a, grid, n, inv_h, stream));
    hipLaunchKernelGGL(barrier_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, a, n, inv_h,
                       (uint32_t)grid.table - 1, grid.start, grid.order, bp, fs, fb);
    return hipGetLastError();
}

// Groups of a reduce workgroup: sixteen (eight with rotations, whose near-pair
// terms take too many registers for sixteen) where the tiles are few and have
// many slots each, else four.
template <int SEGDOF>
static int reduce_groups(int tile_blocks, int n_tiles, int n_slots) {
    return tile_blocks <= 1024 && n_slots >= 24 * n_tiles ? (SEGDOF == 6 ? 8 : 16) : 4;
}

template <int SEGDOF, typename P>
static void launch_reduce_typed(const MatvecArgs& a, const OutArgs& o, const MatvecTile* d_tiles, int n_tiles, int n_slots,
                                int tile_targets, int merge_k, int slot_dof, const P* partial, const NearList& near,
                                hipStream_t stream) {
    const int tile_blocks = n_tiles * ((tile_targets + 63) / 64);
    const int gr = reduce_groups<SEGDOF>(tile_blocks, n_tiles, n_slots);
    const int fil_blocks = o.sad.in ? (o.sad.nfil + gr - 1) / gr : 0;
    const dim3 grid((unsigned)(tile_blocks + fil_blocks));
    constexpr int MANY = SEGDOF == 6 ? 8 : 16;
    if (gr == MANY)
        hipLaunchKernelGGL((rpy_reduce_kernel<SEGDOF, P, MANY>), grid, dim3(64 * MANY), 0, stream, d_tiles, partial,
                           tile_targets, tile_blocks, merge_k, slot_dof, o, a, near);
    else
        hipLaunchKernelGGL((rpy_reduce_kernel<SEGDOF, P, 4>), grid, dim3(256), 0, stream, d_tiles, partial,
                           tile_targets, tile_blocks, merge_k, slot_dof, o, a, near);
}

// The reduce kernel over n_slots partial slots of the evaluation type.
static hipError_t launch_reduce(int precision, int seg_dof, const MatvecArgs& a, const OutArgs& o,
                                const MatvecTile* d_tiles, int n_tiles, int n_slots, int tile_targets, int merge_k,
                                int slot_dof, const double* partial, const NearList& near, hipStream_t stream) {
    const float* pf = reinterpret_cast<const float*>(partial);
    if (precision == 0) {
        if (seg_dof == 6)
            launch_reduce_typed<6>(a, o, d_tiles, n_tiles, n_slots, tile_targets, merge_k, slot_dof, partial, near, stream);
        else
            launch_reduce_typed<3>(a, o, d_tiles, n_tiles, n_slots, tile_targets, merge_k, slot_dof, partial, near, stream);
    } else {
        if (seg_dof == 6)
            launch_reduce_typed<6>(a, o, d_tiles, n_tiles, n_slots, tile_targets, merge_k, slot_dof, pf, near, stream);
        else
            launch_reduce_typed<3>(a, o, d_tiles, n_tiles, n_slots, tile_targets, merge_k, slot_dof, pf, near, stream);
    }
    return hipGetLastError();
}

hipError_t launch_wall_pairs(int precision, int seg_dof, const MatvecArgs& a, const MatvecTile* d_tiles, int n_tiles,
                             const MatvecItem* d_items, int n_items, double* partial, hipStream_t stream,
                             hipEvent_t ev_begin, hipEvent_t ev_end) {
    if (n_tiles > 0 && n_items > 0) {
        float* pf = reinterpret_cast<float*>(partial);
        if (ev_begin) TFS_HIP_CHECK(hipEventRecord(ev_begin, stream));
        const dim3 grid((unsigned)n_items), block(kWallBlock);
        if (precision == 0) {
            if (seg_dof == 6)
                hipLaunchKernelGGL((rpy_pairs_wall_kernel<6, double>), grid, block, 0, stream, d_items, d_tiles, a,
                                   partial);
            else
                hipLaunchKernelGGL((rpy_pairs_wall_kernel<3, double>), grid, block, 0, stream, d_items, d_tiles, a,
                                   partial);
        } else {
            if (seg_dof == 6)
                hipLaunchKernelGGL((rpy_pairs_wall_kernel<6, float>), grid, block, 0, stream, d_items, d_tiles, a, pf);
            else
                hipLaunchKernelGGL((rpy_pairs_wall_kernel<3, float>), grid, block, 0, stream, d_items, d_tiles, a, pf);
        }
        TFS_HIP_CHECK(hipGetLastError());
        if (ev_end) TFS_HIP_CHECK(hipEventRecord(ev_end, stream));
    }
    return hipSuccess;
}

hipError_t launch_wall_reduce(int precision, int seg_dof, const MatvecArgs& a, const OutArgs& o,
                              const MatvecTile* d_tiles, int n_tiles, int n_items, const double* partial,
                              hipStream_t stream) {
    if (n_tiles == 0) return hipSuccess;
    return launch_reduce(precision, seg_dof, a, o, d_tiles, n_tiles, n_items, kWallTile, 0, kMaxDof, partial, NearList{},
                         stream);
}

hipError_t launch_matvec_pairs(int precision, int seg_dof, const TileShape& shape, const MatvecArgs& a,
                               uint32_t blocks, const MatvecTile* d_tiles, int n_tiles, const MatvecItem* d_items,
                               int n_items, double* partial, const PersistState& ps, hipStream_t stream,
                               hipEvent_t ev_begin, hipEvent_t ev_end) {
    if (precision == 1 && (!a.xfx || !a.lam)) return hipErrorInvalidValue;
    if (n_tiles > 0 && n_items > 0) {
        hipError_t e;
        if (ev_begin) TFS_HIP_CHECK(hipEventRecord(ev_begin, stream));
        if (shape.symmetric) {
            const int bb = (blocks & 4u) ? 1 : 0;
            if (precision == 0)
                e = seg_dof == 6 ? launch_sym<double, 6>(shape.symmetric, a, d_items, n_items, d_tiles, n_tiles, bb, partial, ps, stream)
                                 : launch_sym<double, 3>(shape.symmetric, a, d_items, n_items, d_tiles, n_tiles, bb, partial, ps, stream);
            else
                e = seg_dof == 6 ? launch_sym<float, 6>(shape.symmetric, a, d_items, n_items, d_tiles, n_tiles, bb, partial, ps, stream)
                                 : launch_sym<float, 3>(shape.symmetric, a, d_items, n_items, d_tiles, n_tiles, bb, partial, ps, stream);
        } else if (precision == 0) {
            e = seg_dof == 6 ? dispatch_shape<double, 6>(shape, a, d_items, n_items, d_tiles, partial, ps, stream)
                             : dispatch_shape<double, 3>(shape, a, d_items, n_items, d_tiles, partial, ps, stream);
        } else {
            e = seg_dof == 6 ? dispatch_shape<float, 6>(shape, a, d_items, n_items, d_tiles, partial, ps, stream)
                             : dispatch_shape<float, 3>(shape, a, d_items, n_items, d_tiles, partial, ps, stream);
        }
        if (e != hipSuccess) return e;
        if (ev_end) TFS_HIP_CHECK(hipEventRecord(ev_end, stream));
    }
    return hipSuccess;
}

hipError_t launch_matvec_reduce(int precision, int seg_dof, const TileShape& shape, const MatvecArgs& a,
                                const OutArgs& o, const MatvecTile* d_tiles, int n_tiles, int n_items, int n_slots,
                                const double* partial, const NearList& near, const PersistState& ps,
                                hipStream_t stream) {
    if (n_tiles == 0) return hipSuccess;
    // The partial slots hold the evaluation type (FP32 sums for FP32 tiles);
    // the persistent form fills only its tile segments' first slots.
    const int merge_k = shape.persistent > 0 && n_items > 0 ? persistent_items(shape, n_items, ps.num_cus) : 0;
    const int slots = shape.symmetric ? n_slots : n_items;
    return launch_reduce(precision, seg_dof, a, o, d_tiles, n_tiles, slots, tile_targets(shape), merge_k,
                         shape.symmetric ? seg_dof : kMaxDof, partial, near, stream);
}

}  // namespace tfs
