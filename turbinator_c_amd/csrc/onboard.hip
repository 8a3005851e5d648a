// gfx950 kernel of the onboard tactical (24) and physics-prior (15) features.
//
// Semantics follow the reference device code
// src/network/onboard_features.cuh:6-519 (tb_onboard_tactical,
// tb_onboard_prior, tb_onboard_tactical_prior), which the reference runs as
// one thread per environment inside its actor input kernel
// (src/network/network_gpu.cu:274-304).  Here the two halves of the work get
// the execution shape that suits them:
//
//   * the LiDAR scan (two passes over 1,536 rays: closest return, corridor
//     minimum, cluster membership and y sum) runs one wave per environment,
//     24 rays per lane, so each load instruction reads 256 contiguous LiDAR
//     bytes and no workgroup barrier is needed.  The wave lists its
//     in-window rays in ray order (ballot + lane prefix) and runs both
//     passes over the list; above kListCap in-window rays it sweeps every
//     slot, branch-free, with the two heads' rays at the same azimuth and
//     elevation sharing the first two products of each rotated component.
//     The closest return is a 32-bit wave minimum of the range bits followed
//     by a lane-mask search for its first slot and lane (the first minimum
//     in the reference scan order); the corridor minimum is a DPP / permlane
//     fminf reduction, with a +0 / -0 tie settled as the reference's strict
//     < settles it (the first in ray order); the cluster count comes from
//     lane masks, and the cluster's y centres are added in float in ray
//     order, as the reference does, because the sign of that sum picks the
//     slalom lane.  The controller uses the closest return for dodge
//     missions only and the corridor and cluster for slalom missions only
//     (onboard_features.cuh:208-244), so unless the caller asks for the
//     scan's diagnostics each environment gets only the part its mission
//     uses, and the next environment's ranges are requested only as far as
//     it needs them.  The environments whose mission uses the scan are shared
//     out over a workgroup's waves from a pool in LDS, so the waves that
//     would have drawn several slalom missions do not set the kernel's time;
//     the actor entry's scan for large batches, which also writes the LiDAR
//     channels of every environment, keeps a static share;
//   * the tactical features and the controller (mission decode, targets,
//     landing / standard / inversion / BWB laws, cannon) run on one quad of
//     lanes per environment (lane a evaluates arm a and a quarter of the
//     independent transcendental calls), in the same workgroup as their
//     scan: a launch of their own cost its start, a second staging of the
//     inputs and the scan results' round trip.  Small batches give the
//     flight controller, the rest of the controller and the scan their own
//     waves, so that the chain that sets the time, the flight controller's,
//     runs beside the scan up to the point that needs it.  The angles that
//     reach its angle wraps use a correctly rounded atan2: exact angles
//     (from equal or zero components) reach a wrap's discontinuity, where
//     one ulp flips the wrapped error's sign.
//
// Ray directions come from a table generated at build time with the host
// libm (gen_ray_table.c), and the scan arithmetic is evaluated without FMA
// contraction in the reference's operation order, so the per-ray world
// vectors, and with them the closest return, its ray index, the corridor
// minimum, the cluster count and the cluster y sum, are reproducible
// bit-for-bit against the unfused C restatement.

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <atomic>
#include <mutex>

#include "turbinator/training/hip_features.h"
#include "onboard_math.h"
#include "recip_range.h"
#include "xcd_order.h"

#include "onboard_rays.inc"

namespace {

constexpr int kBlockThreads = 256;
constexpr int kWavesPerBlock = kBlockThreads / 64;
constexpr int kControlWaves = 4;  // control workgroup: waves 0..3 controller, 4..7 tactical
constexpr int kControlThreads = 2 * kControlWaves * 64;
constexpr int kScanRays = 1536 / 64;  // rays per lane: one wave scans one environment
// In-window rays a wave lists for the compact pass; with more, every slot is
// swept instead.
constexpr int kListCap = 512;
constexpr int kListRounds = kListCap / 64;
constexpr unsigned kMaxBlocks = 1u << 20;
constexpr int kStreamThreads = 1024;  // actor plane kernel: one workgroup per environment
constexpr unsigned kScanBlocks = 256 * 4;   // persistent scan grid: 4 per CU
// Widest row of the control kernel's grid; larger batches take more rows (a
// launch's x extent is limited to 2^32 threads).
constexpr unsigned kControlGridX = 1u << 20;
constexpr size_t kMaxBatch = 0x7fffffffu;
constexpr float kPi = 3.14159265358979323846f;

struct ScanResult {
    float min_r, min_r_dx, min_r_dy, min_dx_c, cluster_y_sum;
    int min_ray, cluster_count, pad;
};

// x / c for a constant float c, as one double product.  For each constant
// this file divides by (10, 20, 30, 45, pi/6, pi/4 and the thrust span) the
// result equals the IEEE quotient for every finite float x
// (tests/csrc/check_div_by_constant.c, run over all 4.28e9 finite floats);
// the IEEE division is a ten-instruction dependent sequence.
__device__ __forceinline__ float div_const(float x, float c) {
    return (float)((double)x * (1.0 / (double)c));
}

// onboard_features.cuh:6-22.  The tests are formed before the selects, so
// they stay selects: as nested conditionals each became two branches.
// TAME (onboard_math.h): no value is infinite or NaN.
template <bool TAME = false>
__device__ __forceinline__ float ob_clamp(float x, float lo, float hi) {
    const float y = fminf(hi, fmaxf(lo, x));
    if constexpr (TAME) return y;
    const bool nan = __builtin_isnan(x);
    return nan ? x : y;
}
__device__ __forceinline__ float finite_as(float x, float limit) {
    const bool nan = __builtin_isnan(x), inf = __builtin_isinf(x);
    const float y = inf ? copysignf(limit, x) : x;
    return nan ? 0.0f : y;
}
__device__ __forceinline__ float ob_obs(float x) { return finite_as(x, 1000.0f); }
__device__ __forceinline__ float ob_mission(float x) { return finite_as(x, 1.0f); }
// atan2 and the angle wrap.  ob_wrap is discontinuous where its two angles
// differ by pi, and that is reached exactly by angles such as -3pi/4 and pi/4
// (from equal or zero components), or pi and a yaw of +-0: there one ulp of
// either angle flips the wrapped error between about -pi and +pi and the
// controller's torques with it.  The single-precision atan2f can be an ulp
// from the correctly rounded value on such arguments; the host libm's
// atan2f, which the oracle calls, is correctly rounded on them (equal,
// opposite and zero components, results near +-pi: tests/csrc/
// check_atan2.hip), and so is atan2_float (check_onboard_math.hip).
// Elsewhere either may be an ulp off, which moves the angles continuously.
template <bool TAME>
__device__ __forceinline__ float ob_atan2(float y, float x) {
    return onboard_math::atan2_float<TAME>(y, x);
}
template <bool TAME>
__device__ __forceinline__ float ob_wrap(float target, float current) {
    return onboard_math::wrap_angle<TAME>(target - current);
}
template <bool TAME>
__device__ __forceinline__ float ob_norm3(float x, float y, float z) {
    return onboard_math::square_root<TAME>(x * x + y * y + z * z);
}
template <bool TAME>
__device__ __forceinline__ float ob_hypot(float x, float y) {
    return onboard_math::hypotenuse<TAME>(x, y);
}

// Normalised, sign-fixed attitude quaternion (onboard_features.cuh:105-109)
// and its rotation matrix rows (:137-145).
struct Attitude {
    float qw, qx, qy, qz;
    float r[9];
};

__device__ __forceinline__ Attitude attitude_of(float o6, float o7, float o8, float o9) {
    Attitude a;
    float qnorm = fmaxf(sqrtf(o6 * o6 + o7 * o7 + o8 * o8), 0.0f);
    qnorm = fmaxf(sqrtf(qnorm * qnorm + o9 * o9), 1.0e-8f);
    const float sign = o6 < 0.0f ? -1.0f : 1.0f;
    const onboard_math::Divisor over(qnorm);  // the IEEE quotients
    a.qw = over(sign * o6);
    a.qx = over(sign * o7);
    a.qy = over(sign * o8);
    a.qz = over(sign * o9);
    const float qw = a.qw, qx = a.qx, qy = a.qy, qz = a.qz;
    a.r[0] = 1.0f - 2.0f * (qy * qy + qz * qz);
    a.r[1] = 2.0f * (qx * qy - qw * qz);
    a.r[2] = 2.0f * (qx * qz + qw * qy);
    a.r[3] = 2.0f * (qx * qy + qw * qz);
    a.r[4] = 1.0f - 2.0f * (qx * qx + qz * qz);
    a.r[5] = 2.0f * (qy * qz - qw * qx);
    a.r[6] = 2.0f * (qx * qz - qw * qy);
    a.r[7] = 2.0f * (qy * qz + qw * qx);
    a.r[8] = 1.0f - 2.0f * (qx * qx + qy * qy);
    return a;
}

// Wave-wide reductions without the LDS crossbar: DPP exchanges inside each
// row of 16 lanes (quad_perm [1,0,3,2], [2,3,0,1], row_half_mirror,
// row_mirror) and the gfx950 permlane swaps across rows (partner l^16, then
// l^32).  Each step hands every lane the pair {own value, partner value};
// the combining operations below are symmetric, so every lane ends with the
// whole-wave result.
template <int CTRL>
__device__ __forceinline__ int dpp_partner(int v) {
    return __builtin_amdgcn_mov_dpp(v, CTRL, 0xF, 0xF, false);
}

template <bool SWAP32>
__device__ __forceinline__ int swap_pair(int v, int &other) {
    const auto s = SWAP32 ? __builtin_amdgcn_permlane32_swap(v, v, false, false)
                          : __builtin_amdgcn_permlane16_swap(v, v, false, false);
    other = s[1];
    return s[0];
}

__device__ __forceinline__ float wave_min(float v) {
    v = fminf(v, __int_as_float(dpp_partner<0xB1>(__float_as_int(v))));
    v = fminf(v, __int_as_float(dpp_partner<0x4E>(__float_as_int(v))));
    v = fminf(v, __int_as_float(dpp_partner<0x141>(__float_as_int(v))));
    v = fminf(v, __int_as_float(dpp_partner<0x140>(__float_as_int(v))));
    int o;
    float a = __int_as_float(swap_pair<false>(__float_as_int(v), o));
    v = fminf(a, __int_as_float(o));
    a = __int_as_float(swap_pair<true>(__float_as_int(v), o));
    return fminf(a, __int_as_float(o));
}

// Ray directions as three planes (x, y, z) of 1,536 floats in LDS.
struct RayPlanes {
    float d[3][1536];
};

__device__ __forceinline__ unsigned wave_min_u32(unsigned v) {
    v = min(v, (unsigned)dpp_partner<0xB1>((int)v));
    v = min(v, (unsigned)dpp_partner<0x4E>((int)v));
    v = min(v, (unsigned)dpp_partner<0x141>((int)v));
    v = min(v, (unsigned)dpp_partner<0x140>((int)v));
    int o;
    v = min((unsigned)swap_pair<false>((int)v, o), (unsigned)o);
    return min((unsigned)swap_pair<true>((int)v, o), (unsigned)o);
}

// Buffer resources (gfx9 word 3): loads read zero past num_records instead
// of faulting, so a resource of 0 bytes turns a prefetch into zeros (ranges
// outside the scan window) without a branch.  A branch-free prefetch also
// keeps the load counter exact: a load issued on one path only would make
// the compiler wait for every load at the join.
constexpr int kBufferWord3 = 0x00020000;
constexpr unsigned kObsRowBytes = 4148 * sizeof(float);
constexpr int kNontemporal = 2;  // cache policy bit 1 (nt)

__device__ __forceinline__ __amdgpu_buffer_rsrc_t obs_rsrc(const float *obs, bool valid) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(obs), (short)0,
                                             valid ? (int)kObsRowBytes : 0, kBufferWord3);
}

// The 24 ranges lane l of an environment's wave owns: slot u = 2 row + half
// is ray 128 row + 64 half + l (row = 6 head + el), so slots run in ray
// order and each load instruction reads 256 contiguous LiDAR bytes.
// Elevation rows 4..5 are read through `upper`, which a caller that needs
// only the closest return (rows 0..3) gives 0 bytes: they then read zeros,
// outside the scan window.
__device__ __forceinline__ void load_ranges(__amdgpu_buffer_rsrc_t obs,
                                            __amdgpu_buffer_rsrc_t upper, int lane,
                                            float (&rg)[kScanRays]) {
#pragma unroll
    for (int u = 0; u < kScanRays; ++u) {
        const int row = u / 2, head = row / 6, el = row % 6;
        // A head's rows lie within the instruction's 12-bit offset, the heads
        // 8,192 bytes apart: one scalar offset instead of one for each load.
        rg[u] = __builtin_bit_cast(
            float, __builtin_amdgcn_raw_buffer_load_b32(el < 4 ? obs : upper,
                                                        4 * (48 + lane) + 4 * (el * 128 + 64 * (u % 2)),
                                                        8192 * head, kNontemporal));
    }
}

// onboard_features.cuh:105-109,137-145 (attitude rows) and :183 (py) of one
// environment: the frame of its scan.
struct ScanFrame {
    float r[9], py;
};

struct FrameObs {
    float o1, o6, o7, o8, o9, m4, m5;  // and the two mission values scan_need reads
};

__device__ __forceinline__ FrameObs load_frame_obs(const float *obs, const float *mission) {
    return FrameObs{obs[1], obs[6], obs[7], obs[8], obs[9], mission[4], mission[5]};
}

__device__ __forceinline__ ScanFrame scan_frame(FrameObs &v) {
    // An empty asm that takes the seven values waits for their loads once,
    // here, instead of letting each load sink to its use inside the branchy
    // non-finite mapping (one memory round trip each).
    asm volatile("" : "+v"(v.o1), "+v"(v.o6), "+v"(v.o7), "+v"(v.o8), "+v"(v.o9), "+v"(v.m4),
                 "+v"(v.m5));
    const Attitude att = attitude_of(ob_obs(v.o6), ob_obs(v.o7), ob_obs(v.o8), ob_obs(v.o9));
    ScanFrame f;
#pragma unroll
    for (int k = 0; k < 9; ++k) f.r[k] = att.r[k];
    f.py = ob_obs(v.o1);
    return f;
}

// One listed in-window ray: its range (bits) and ray index.
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ bool in_window(float range) {
    return (int)(range > 0.35f) & (int)(range < 11.5f);
}

// in_window as one unsigned compare of the bits: 0x3eb33334 is the least
// float above 0.35f and 0x41380000 is 11.5f; negative values, zeros, NaN
// and infinities all fall outside [0x3eb33334, 0x41380000).  The listed
// pass stores the difference `bits - kWindowLo` itself: it orders in-window
// ranges like the ranges, and kWindowSpan marks "none".
constexpr unsigned kWindowLo = 0x3eb33334u;             // least float above 0.35f
constexpr unsigned kWindowSpan = 0x41380000u - kWindowLo;  // 11.5f - kWindowLo
__device__ __forceinline__ unsigned window_offset(float range) {
    return __float_as_uint(range) - kWindowLo;
}

// The 618M actor's three LiDAR channels of one range (network_gpu.cu:
// 467-479): inverse range, range / 30 and validity.  Both the plane kernel
// and the scan kernel of the actor entry form them here.  The divisor of the
// inverse range lies in [0.2, 30] for every input (non-finite ranges clamp
// to 0.05 or 30), where recip_range is the IEEE quotient; it is formed on
// every lane and selected, without a branch.
__device__ __forceinline__ float lidar_channel(float range, int kind) {
    const bool valid = range > 0.0f && __builtin_isfinite(range);
    const float clamped = fmaxf(0.05f, fminf(30.0f, range));
    if (kind == 0) return valid ? recip_range(fmaxf(0.2f, clamped)) : 0.0f;
    if (kind == 1) return valid ? div_const(clamped, 30.0f) : 1.0f;
    return valid ? 1.0f : 0.0f;
}

// Buffer cache-policy bits of the actor entry's plane stores: nt (1) and
// sc1 (4).
constexpr int kStorePolicy = 2 | 16;

// onboard_features.cuh:199-207 for one ray with rotated direction rw:
// returns the corridor centre x (+inf when the ray is outside the window or
// the corridor) and sets y_center.  Bitwise, so the compares stay one
// straight-line block.
__device__ __forceinline__ float corridor_centre(float rwx, float rwy, float rwz, float range,
                                                 float py, float &y_center) {
    const float wx = rwx * range, wy = rwy * range, wz = rwz * range;
    const float x_center = wx + rwx * 1.10f;
    y_center = py + wy + rwy * 1.10f;
    const bool corridor = (int)in_window(range) & (int)(fabsf(wz) <= 2.1f) &
                          (int)(x_center >= -0.35f) & (int)(x_center <= 10.5f) &
                          (int)(fabsf(y_center) <= 3.5f);
    return corridor ? x_center : __builtin_huge_valf();
}

// sum + v[l0] + v[l1] + ... in float, one rounding per term, over the lanes
// of `members` in ascending order (onboard_features.cuh:231-234 adds each
// cluster ray's y_center in scan order; the sign of the sum decides the
// slalom lane at :238, so the reference's rounding sequence is kept).  The
// loop runs on the scalar unit, one v_readlane and one add per member.
__device__ __forceinline__ float add_in_lane_order(float sum, float v, uint64_t members) {
    while (members) {
        const int l = (int)__builtin_ctzll(members);
        sum += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
        members &= members - 1;
    }
    return sum;
}

// The 618M actor's three LiDAR channel planes of the wave's 1,536 rays,
// written into `planes`, the environment's [6][16][128] channel block: these
// rays are in the wave's registers already, so the actor entry reads them
// from HBM once, and its plane kernel writes only the other elevation rows.
// Slot u holds row 6 head + el, azimuths 64 (u % 2) + lane: channel kind k
// of head h is plane h + 2k, so each store writes 256 consecutive bytes of
// one plane row.
__device__ __forceinline__ void write_channel_planes(const float (&rg)[kScanRays],
                                                     __amdgpu_buffer_rsrc_t planes, int lane) {
#pragma unroll
    for (int u = 0; u < kScanRays; ++u) {
        const int row = u / 2, head = row / 6, el = row % 6;
#pragma unroll
        for (int kind = 0; kind < 3; ++kind)
            __builtin_amdgcn_raw_buffer_store_b32(
                __builtin_bit_cast(unsigned, lidar_channel(rg[u], kind)), planes, 4 * lane,
                4 * ((head + 2 * kind) * 2048 + el * 128 + 64 * (u % 2)), kStorePolicy);
    }
}

// What the controller uses of an environment's scan (onboard_features.cuh:
// 107-109 for the mission flags, :208-244 for the uses): a dodge mission
// uses the closest return (min_r and its world offset), a slalom mission the
// corridor minimum and the cluster, and every other mission none of it.
// The two flags exclude each other (dodge needs m5 > 0.75, slalom m5 <= 0.25).
constexpr int kNeedNone = 0, kNeedClosest = 1, kNeedCorridor = 2, kNeedAll = 3;

__device__ __forceinline__ int scan_need(float raw_m4, float raw_m5) {
    const float m4 = ob_mission(raw_m4), m5 = ob_mission(raw_m5);
    const bool lateral = m4 > 0.75f && m5 > 0.25f;
    const bool slalom = m4 > 0.75f && !lateral;
    const bool dodge = m5 > 0.75f;
    return slalom ? kNeedCorridor : (dodge ? kNeedClosest : kNeedNone);
}

// Lane 0's closest-return fields of `out` from the winning ray and range
// bits (onboard_features.cuh:202, the world offset in the reference's
// operation order).
__device__ __forceinline__ void closest_fields(int ray, unsigned min_bits, const RayPlanes &rays,
                                               const ScanFrame &f, ScanResult &out) {
    const float range = ray >= 0 ? __uint_as_float(min_bits) : 30.0f;
    out.min_r = range;
    out.min_r_dx = 0.0f;
    out.min_r_dy = 0.0f;
    out.min_ray = -1;
    if (ray >= 0) {
        const float dx = rays.d[0][ray], dy = rays.d[1][ray], dz = rays.d[2][ray];
        const float rwx = f.r[0] * dx + f.r[1] * dy + f.r[2] * dz;
        const float rwy = f.r[3] * dx + f.r[4] * dy + f.r[5] * dz;
        out.min_r_dx = rwx * range;
        out.min_r_dy = rwy * range;
        out.min_ray = ray;
    }
}

// onboard_features.cuh:184-234 for one environment, on one wave (24 rays per
// lane, no workgroup barrier).  In a batch that fills the chip the scans are
// three quarters of its instructions, and their number bounds the kernel: the
// closest return takes about 150 and the corridor and cluster about 450 in an
// open scene (250 and 500 before the offsets became the key of the closest
// return, its slot search an early exit and the loads' offsets immediate:
// 25.9 -> 24.9 us at 32,768 environments, 16.1 -> 15.0 at 16,384).
//   * The reference maps non-finite ranges to 0 / +-1000 first; both fail
//     the 0.35 < r < 11.5 window, as NaN does, so the raw value is tested.
//     The reference skips rays outside the window (:193, :218), and so does
//     the common path here: the in-window rays are listed in the wave's
//     `list` (ballot + lane prefix count) and passes 1 and 2 run over the
//     list, 64 rays per instruction.  When more than kListCap rays are in
//     the window, every slot is swept instead (the same per-ray arithmetic).
//   * The closest return over elevation rows 0..3 is found straight from
//     the ranges, before any list, in two steps: the wave's minimum
//     in-window range (as bits: positive floats order like their bit
//     patterns), then the first slot in ray order and the first lane holding
//     exactly that range, from lane masks on the scalar unit.  That is the
//     reference's first minimum in scan order.  Lane 0 computes the winner's
//     world offset with the reference's expression.
//   * Pass 1 keeps each ray's corridor centre (x = +inf outside the window or
//     the corridor), so pass 2 is a compare-and-add.  The reference's
//     strict-< update over corridor rays is the minimum of their centres,
//     except that of a +0 and a -0 it keeps the first in ray order, which a
//     search over the zero centres restores when the minimum is zero.
//   * Once the ranges are consumed (listed, or swept by pass 1), the
//     registers take the next environment's (`next`, a 0-byte resource when
//     there is none): they have the rest of this environment to arrive.
//   * `f` and `need` are wave-uniform.  Only the corridor and cluster use
//     the list: with kNeedClosest only (a dodge mission) nothing is listed
//     and the corridor work is skipped; with kNeedCorridor only (slalom) the
//     closest-return search is skipped; with kNeedNone nothing is done.  The
//     fields skipped keep their empty values.
__device__ __forceinline__ void scan_env(float (&rg)[kScanRays], const RayPlanes &rays,
                                         const ScanFrame &f, __amdgpu_buffer_rsrc_t next,
                                         __amdgpu_buffer_rsrc_t next_upper, int lane,
                                         u32x2 *list, ScanResult &out, int need) {
    // Closest return, straight from the ranges: each lane's minimum over its
    // 16 slots of elevation rows 0..3 as window offsets (they order like the
    // ranges; everything outside the window is at or above kWindowSpan, so
    // it never wins), the wave's minimum, then the first slot (slots are in
    // ray order) and its first lane holding exactly that range: the
    // reference's first minimum in scan order.
    unsigned min_bits = kWindowSpan + kWindowLo;
    int min_ray = -1;
    if (need & kNeedClosest) {
        unsigned lane_min = kWindowSpan;
#pragma unroll
        for (int u = 0; u < kScanRays; ++u)
            if ((u / 2) % 6 < 4) lane_min = min(lane_min, window_offset(rg[u]));
        const unsigned wave_low = wave_min_u32(lane_min);
        if (wave_low != kWindowSpan) {
            min_bits = wave_low + kWindowLo;
#pragma unroll
            for (int u = 0; u < kScanRays; ++u) {
                if ((u / 2) % 6 >= 4) continue;
                const uint64_t hit =
                    __builtin_amdgcn_ballot_w64(__float_as_uint(rg[u]) == min_bits);
                if (hit) {
                    min_ray = 64 * u + (int)__builtin_ctzll(hit);
                    break;
                }
            }
        }
    }

    // List the in-window rays in slot order while counting them: entry =
    // (range bits - kWindowLo, ray).  The slot's first entry address is
    // uniform (scalar), so each lane's address is one shift-add of its lane
    // prefix.  Once a slot's rays would overflow the list, counting stops:
    // n then exceeds kListCap and the list is not used.
    int n = 0;
#pragma unroll
    for (int u = 0; u < kScanRays; ++u) {
        // Only the corridor and cluster use the list.
        if (!(need & kNeedCorridor)) break;
        // A slot adds at most 64 entries, so the list can be full only from
        // slot kListCap / 64 + 1 on.
        if (64 * u > kListCap && n > kListCap) break;
        const unsigned off = window_offset(rg[u]);
        const bool in = off < kWindowSpan;
        const uint64_t m = __builtin_amdgcn_ballot_w64(in);
        // The lane's list position: the running count plus the in-window
        // lanes below it (mbcnt adds its second operand).  With n <= kListCap
        // every position is below kListCap + 64, inside the list and its
        // spare entries; a slot that takes the count past kListCap abandons
        // the list, so what it wrote there is never read.  Lanes outside the
        // window write to their own spare entry, so the store needs no
        // branch.
        unsigned pos = __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                                 __builtin_amdgcn_mbcnt_lo((unsigned)m, (unsigned)n));
        asm volatile("" : "+v"(pos));  // formed on every lane, then selected
        *(list + (in ? pos : (unsigned)(kListCap + lane))) = u32x2{off, (unsigned)(64 * u + lane)};
        n += (int)__builtin_popcountll(m);
    }

    float min_dx_c = 30.0f;
    int count = 0;
    float y_sum = 0.0f;
    if (n <= kListCap) {
        // The list is written and read by this wave only.
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        load_ranges(next, next_upper, lane, rg);
        // Round r's values exist only when 64 r < n, and every later loop
        // stops at the same bound (initialising the unused rounds cost
        // about 35 moves per environment).
        float xl[kListRounds], yl[kListRounds];
#pragma unroll
        for (int r = 0; r < kListRounds; ++r) {
            if (64 * r < n) {
                const int e = 64 * r + lane;
                const u32x2 entry = list[e];
                const bool valid = e < n;
                // Entries past n are left from earlier environments: they
                // read as 11.5 (kWindowSpan + kWindowLo), outside the window.
                const unsigned off = valid ? entry.x : kWindowSpan;
                const float range = __uint_as_float(off + kWindowLo);
                const int ray = valid ? (int)entry.y : 0;
                const float dx = rays.d[0][ray], dy = rays.d[1][ray], dz = rays.d[2][ray];
                const float rwx = f.r[0] * dx + f.r[1] * dy + f.r[2] * dz;
                const float rwy = f.r[3] * dx + f.r[4] * dy + f.r[5] * dz;
                const float rwz = f.r[6] * dx + f.r[7] * dy + f.r[8] * dz;
                xl[r] = corridor_centre(rwx, rwy, rwz, range, f.py, yl[r]);
                min_dx_c = fminf(min_dx_c, xl[r]);
            }
        }
        if (need & kNeedCorridor) {
            min_dx_c = wave_min(min_dx_c);
            if (min_dx_c == 0.0f) {
                // +0 and -0 tie; the reference keeps the first in ray order.
#pragma unroll
                for (int r = 0; r < kListRounds; ++r) {
                    if (64 * r >= n) break;
                    const uint64_t zero = __builtin_amdgcn_ballot_w64(xl[r] == 0.0f);
                    if (zero) {
                        min_dx_c = __int_as_float(__builtin_amdgcn_readlane(
                            __float_as_int(xl[r]), (int)__builtin_ctzll(zero)));
                        break;
                    }
                }
            }
            const float limit = min_dx_c + 1.4f;
#pragma unroll
            for (int r = 0; r < kListRounds; ++r) {
                if (64 * r >= n) break;
                const uint64_t members = __builtin_amdgcn_ballot_w64(xl[r] <= limit);
                count += __builtin_popcountll(members);
                y_sum = add_in_lane_order(y_sum, yl[r], members);
            }
        }
    } else {
        // Every slot.  The rays of rows el and el + 6 (heads 0 and 1) at the
        // same azimuth have the same table x, y and the negated z, bit for
        // bit.  With the reference's order (R0 d.x + R1 d.y) + R2 d.z the
        // head-1 sum is therefore P - Q where the head-0 sum is P + Q,
        // exactly (a + (-b) and a - b are the same IEEE operation), so each
        // pair reads one direction and forms P and Q once.
        float xc[kScanRays], yc[kScanRays];
        int min_slot = kScanRays;
#pragma unroll
        for (int el = 0; el < 6; ++el) {
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const int ray = 128 * el + 64 * half + lane;
                const float dx = rays.d[0][ray], dy = rays.d[1][ray], dz = rays.d[2][ray];
                const float p0 = f.r[0] * dx + f.r[1] * dy, q0 = f.r[2] * dz;
                const float p1 = f.r[3] * dx + f.r[4] * dy, q1 = f.r[5] * dz;
                const float p2 = f.r[6] * dx + f.r[7] * dy, q2 = f.r[8] * dz;
#pragma unroll
                for (int head = 0; head < 2; ++head) {
                    const int u = 2 * (6 * head + el) + half;
                    xc[u] = corridor_centre(head ? p0 - q0 : p0 + q0, head ? p1 - q1 : p1 + q1,
                                            head ? p2 - q2 : p2 + q2, rg[u], f.py, yc[u]);
                    // The reference's strict < in ray order: the lane keeps
                    // its minimum at the lowest slot (slots are visited head
                    // innermost, not in ray order; equal values differ only
                    // as +0 / -0, which is settled across lanes below).
                    const bool lower = (int)(xc[u] < min_dx_c) |
                                       ((int)(xc[u] == min_dx_c) & (int)(u < min_slot));
                    min_dx_c = lower ? xc[u] : min_dx_c;
                    min_slot = lower ? u : min_slot;
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        load_ranges(next, next_upper, lane, rg);
        {
            // +0 and -0 tie; the reference keeps the first in ray order
            // (slot u holds rays 64 u .. 64 u + 63): the lowest ray among the
            // lanes' first zeros.  Formed on every environment and selected:
            // a branch here cost the kernel 50 VGPRs.
            const float lane_min = min_dx_c;
            min_dx_c = wave_min(lane_min);
            const unsigned key =
                lane_min == 0.0f ? 64u * (unsigned)min_slot + (unsigned)lane : ~0u;
            const float first_zero = __int_as_float(__builtin_amdgcn_readlane(
                __float_as_int(lane_min), (int)(wave_min_u32(key) & 63u)));
            min_dx_c = min_dx_c == 0.0f ? first_zero : min_dx_c;
        }
        // Pass 2: the cluster is counted from the lane masks (scalar unit)
        // and its y values summed in ray order (slot outer, lane inner).
        // All 24 masks are formed before the first sum: interleaving the
        // mask compares with the member loops took the kernel from 119 to
        // 182 VGPRs (2 waves per SIMD instead of 4).
        const float limit = min_dx_c + 1.4f;
        uint64_t members[kScanRays];
#pragma unroll
        for (int u = 0; u < kScanRays; ++u) {
            members[u] = __builtin_amdgcn_ballot_w64(xc[u] <= limit);
            count += __builtin_popcountll(members[u]);
        }
#pragma unroll
        for (int u = 0; u < kScanRays; ++u) y_sum = add_in_lane_order(y_sum, yc[u], members[u]);
    }
    if (lane == 0) {
        closest_fields(min_ray, min_bits, rays, f, out);
        out.min_dx_c = min_dx_c;
        out.cluster_count = count;
        out.cluster_y_sum = y_sum;
    }
}

// Lane k of every group of four (a quad) reads quad lane K's value.
template <int K>
__device__ __forceinline__ float quad_lane(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), K * 0x55, 0xF, 0xF, false));
}

// The four lanes' values of v, in every lane of the quad.
struct Quad4 {
    float v[4];
};
__device__ __forceinline__ Quad4 quad_all(float v) {
    return Quad4{{quad_lane<0>(v), quad_lane<1>(v), quad_lane<2>(v), quad_lane<3>(v)}};
}

// Quad lane a's choice among four values: three plain selects (as a nested
// conditional it became branches with the values' computation inside).
__device__ __forceinline__ float quad_pick(int a, float v0, float v1, float v2, float v3) {
    const bool odd = (a & 1) != 0, high = (a & 2) != 0;
    const float lo = odd ? v1 : v0;
    const float hi = odd ? v3 : v2;
    return high ? hi : lo;
}

// How the chains are spread over lanes.  QUAD: an environment's four lanes
// hold one arm each and repeat the shared part, except that independent calls
// of one function are spread over them and broadcast: the shortest chain, for
// batches that leave the chip waiting for it.  Otherwise one lane holds the
// environment and its four arms: 4,100 instead of 10,800 instructions for 64
// environments, for batches that fill the chip.  Both form every value by the
// same operations.
template <bool QUAD>
constexpr int kArms = QUAD ? 1 : 4;  // arms per lane

// Every arm's value from the lane's own.
template <bool QUAD>
__device__ __forceinline__ Quad4 every_arm(const float (&v)[kArms<QUAD>]) {
    if constexpr (QUAD) return quad_all(v[0]);
    else return Quad4{{v[0], v[1], v[2], v[3]}};
}
// Of four values the one of the lane's arm k.
template <bool QUAD>
__device__ __forceinline__ float arm_pick(int a, int k, float v0, float v1, float v2, float v3) {
    if constexpr (QUAD) return quad_pick(a, v0, v1, v2, v3);
    else return k == 0 ? v0 : (k == 1 ? v1 : (k == 2 ? v2 : v3));  // k is a constant
}
// f of four arguments, or pairs.
template <bool QUAD, class F>
__device__ __forceinline__ Quad4 spread(int a, F f, float x0, float x1, float x2, float x3) {
    if constexpr (QUAD) return quad_all(f(quad_pick(a, x0, x1, x2, x3)));
    else return Quad4{{f(x0), f(x1), f(x2), f(x3)}};
}
template <bool QUAD, class F>
__device__ __forceinline__ Quad4 spread2(int a, F f, float y0, float y1, float y2, float y3,
                                         float x0, float x1, float x2, float x3) {
    if constexpr (QUAD) return quad_all(f(quad_pick(a, y0, y1, y2, y3), quad_pick(a, x0, x1, x2, x3)));
    else return Quad4{{f(y0, x0), f(y1, x1), f(y2, x2), f(y3, x3)}};
}

// The staged inputs that a lane of the control kernel's chains reads,
// taken from LDS all at once: an empty asm on each value keeps the compiler
// from sinking its read to the first use, where every read would cost the
// chain its own LDS round trip.  `head` is obs[0..12], `arm` the four values
// obs[16 + 4 k + arm] of the lane's arms, `tail` obs[40], obs[41], obs[44..47].
template <bool QUAD>
struct ChainInputs {
    float head[13], arm[4][kArms<QUAD>], tail[6], m[10];
};

template <bool QUAD>
__device__ __forceinline__ ChainInputs<QUAD> chain_inputs(const float *obs, const float *mission,
                                                          int a) {
    constexpr int K = kArms<QUAD>;
    ChainInputs<QUAD> in;
#pragma unroll
    for (int i = 0; i < 13; ++i) in.head[i] = obs[i];
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int i = 0; i < K; ++i) in.arm[k][i] = obs[16 + 4 * k + (QUAD ? a : i)];
#pragma unroll
    for (int k = 0; k < 6; ++k) in.tail[k] = obs[k < 2 ? 40 + k : 42 + k];
#pragma unroll
    for (int i = 0; i < 10; ++i) in.m[i] = mission[i];
#pragma unroll
    for (int i = 0; i < 13; ++i) asm volatile("" : "+v"(in.head[i]));
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int i = 0; i < K; ++i) asm volatile("" : "+v"(in.arm[k][i]));
#pragma unroll
    for (int k = 0; k < 6; ++k) asm volatile("" : "+v"(in.tail[k]));
#pragma unroll
    for (int i = 0; i < 10; ++i) asm volatile("" : "+v"(in.m[i]));
    return in;
}

// Whether an input of the environment is infinite, NaN or not below
// onboard_math::kTameMax: unless for every arm the sum of its inputs' and the
// shared inputs' squares is below its square.  The same flag in a quad's lanes
// and in one lane per environment: ob_direction's results depend on it.
template <bool QUAD>
__device__ __forceinline__ bool wild_inputs(const ChainInputs<QUAD> &in) {
    float shared = 0.0f;
#pragma unroll
    for (int i = 0; i < 13; ++i) shared = __builtin_fmaf(in.head[i], in.head[i], shared);
#pragma unroll
    for (int k = 0; k < 6; ++k) shared = __builtin_fmaf(in.tail[k], in.tail[k], shared);
#pragma unroll
    for (int i = 0; i < 10; ++i) shared = __builtin_fmaf(in.m[i], in.m[i], shared);
    int wild = 0;
#pragma unroll
    for (int i = 0; i < kArms<QUAD>; ++i) {
        float s = shared;
#pragma unroll
        for (int k = 0; k < 4; ++k) s = __builtin_fmaf(in.arm[k][i], in.arm[k][i], s);
        wild |= !(s < onboard_math::kTameMax * onboard_math::kTameMax);
    }
    if constexpr (QUAD) {
        wild |= dpp_partner<0xB1>(wild);
        wild |= dpp_partner<0x4E>(wild);
    }
    return wild != 0;
}

// Sine and cosine of atan2(y, x) from the components; a wild environment's are
// those of the rounded angle, as the reference forms them: what they multiply may
// be infinite or near the largest float, and then it matters that the sine of
// a float near pi is about 1e-7 and not the exact value.
template <bool TAME>
__device__ __forceinline__ onboard_math::Direction ob_direction(float y, float x, bool wild) {
    onboard_math::Direction d = onboard_math::direction(y, x);
    if constexpr (!TAME) {
        if (__builtin_amdgcn_ballot_w64(wild)) {
            float s, c;
            sincosf(ob_atan2<false>(y, x), &s, &c);
            d.s = wild ? s : d.s;
            d.c = wild ? c : d.c;
        }
    }
    return d;
}

// The inputs as the controller reads them (onboard_features.cuh:12-22, 95-99).
template <bool QUAD>
__device__ __forceinline__ void controller_inputs(ChainInputs<QUAD> &in) {
#pragma unroll
    for (int i = 0; i < 13; ++i) in.head[i] = ob_obs(in.head[i]);
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int i = 0; i < kArms<QUAD>; ++i) in.arm[k][i] = ob_obs(in.arm[k][i]);
#pragma unroll
    for (int k = 0; k < 6; ++k) in.tail[k] = ob_obs(in.tail[k]);
#pragma unroll
    for (int i = 0; i < 10; ++i) in.m[i] = ob_mission(in.m[i]);
}

struct Direction2 {
    float s0, c0, s1, c1;
};
// Two directions; on a quad lane 0 forms the first and the others the second.
template <bool TAME, bool QUAD>
__device__ __forceinline__ Direction2 directions(int a, float y0, float x0, float y1, float x1,
                                                 bool wild) {
    if constexpr (QUAD) {
        const onboard_math::Direction d =
            ob_direction<TAME>(a == 0 ? y0 : y1, a == 0 ? x0 : x1, wild);
        return Direction2{quad_lane<0>(d.s), quad_lane<0>(d.c), quad_lane<1>(d.s),
                          quad_lane<1>(d.c)};
    } else {
        const onboard_math::Direction d = ob_direction<TAME>(y0, x0, wild),
                                      e = ob_direction<TAME>(y1, x1, wild);
        return Direction2{d.s, d.c, e.s, e.c};
    }
}

// onboard_features.cuh:25-86.  Every call takes the arguments the reference's
// code gives it, and the arm sums are formed in its order.  v[0..23] are the
// features before the reference's last mapping.
template <bool TAME, bool QUAD>
__device__ __forceinline__ void tactical_values(const ChainInputs<QUAD> &in, bool wild, int a,
                                                float (&v)[24]) {
    constexpr int K = kArms<QUAD>;
    const float pi = kPi;
    const float *o = in.head, *m = in.m;
    const float o44 = in.tail[2], o45 = in.tail[3], o46 = in.tail[4], o47 = in.tail[5];
    float spool_a[K], fz_a[K], tz_a[K];
#pragma unroll
    for (int i = 0; i < K; ++i) {
        spool_a[i] = ob_clamp<TAME>(in.arm[0][i], 0.0f, 1.0f);
        const float thrust_a = 0.036f + 0.964f * spool_a[i];
        const float ci_a = onboard_math::cos_float<TAME>(in.arm[3][i]);
        fz_a[i] = thrust_a * in.arm[2][i] * ci_a;
        tz_a[i] = thrust_a * in.arm[1][i] * ci_a;
    }
    const Quad4 spool = every_arm<QUAD>(spool_a), fz = every_arm<QUAD>(fz_a),
                tz = every_arm<QUAD>(tz_a);
    float tau_z = 0.0f, spool_mean = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        tau_z += tz.v[i];
        spool_mean += spool.v[i];
    }
    spool_mean *= 0.25f;
    v[0] = fz.v[1] - fz.v[3];
    v[1] = fz.v[2] - fz.v[0];
    v[2] = 0.5f * tau_z;
    v[3] = 0.25f * (fz.v[0] + fz.v[1] + fz.v[2] + fz.v[3]) - 0.5f;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[4 + i] = 2.0f * (spool.v[i] - spool_mean);
    const float qw = o[6], qx = o[7], qy = o[8], qz = o[9];
    const float bz_x = 2.0f * (qx * qz + qw * qy);
    const float bz_y = 2.0f * (qy * qz - qw * qx);
    const float ct = ob_clamp<TAME>(1.0f - 2.0f * (qx * qx + qy * qy), -1.0f, 1.0f);
    const float bx_x = 1.0f - 2.0f * (qy * qy + qz * qz);
    const float bx_y = 2.0f * (qx * qy + qw * qz);
    const Quad4 offsets = spread<QUAD>(
        a, [](float x) { return onboard_math::atanh_float(ob_clamp<TAME>(x, -0.995f, 0.995f)); },
        m[7], m[8], m[9], m[9]);
    const float rx = offsets.v[0] * 20.0f, ry = offsets.v[1] * 20.0f, rz = offsets.v[2] * 20.0f;
    // Sine and cosine of yaw = atan2(bx_y, bx_x) and of the target bearing
    // atan2(ry, rx), from their components; the angles themselves are used
    // nowhere else.
    const Direction2 dir = directions<TAME, QUAD>(a, bx_y, bx_x, ry, rx, wild);
    const float cy = dir.c0, sy = dir.s0, cb = dir.c1, sb = dir.s1;
    v[8] = cy * bz_y - sy * bz_x;
    v[9] = -sy * bz_y - cy * bz_x;
    v[10] = ct;
    v[11] = ct < 0.20f ? 1.0f : 0.0f;
    const float dist = fmaxf(ob_norm3<TAME>(rx, ry, rz), 1.0f);
    const float flight = div_const(dist, 20.0f);
    const float wx = rx - o[3] * 0.5f * flight;
    const float wy = ry - o[4] * 0.5f * flight;
    const float wz = rz - o[5] * 0.5f * flight + 0.5f * 9.80665f * flight * flight;
    const float ux = -qx, uy = -qy, uz = -qz;
    const float cx = uy * wz - uz * wy + qw * wx;
    const float cyq = uz * wx - ux * wz + qw * wy;
    const float cz = ux * wy - uy * wx + qw * wz;
    const float bx = wx + 2.0f * (uy * cz - uz * cyq);
    const float by = wy + 2.0f * (uz * cx - ux * cz);
    const float bz = wz + 2.0f * (ux * cyq - uy * cx);
    const Quad4 hyp = spread2<QUAD>(a, [](float x, float y) { return ob_hypot<TAME>(x, y); }, rx, bx,
                                    bx, bx, ry, by, by, by);
    const float h_rxy = hyp.v[0], h_bxy = fmaxf(hyp.v[1], 0.2f);
    const Quad4 aim = spread2<QUAD>(a, [](float y, float x) { return atan2f(y, x); }, by, bz, bz, bz,
                                    bx, h_bxy, h_bxy, h_bxy);
    const float az = ob_clamp<TAME>(aim.v[0], pi / 12.0f, pi * 5.0f / 12.0f);
    const float el = ob_clamp<TAME>(aim.v[1], -pi / 6.0f, pi / 6.0f);
    const float err = ob_hypot<TAME>(az - o44, el - o45);
    const Quad4 th1 = spread<QUAD>(a, [](float x) { return tanhf(x); }, (cy * rx + sy * ry) * 0.08f,
                                   (-sy * rx + cy * ry) * 0.08f, rz * 0.12f, h_rxy * 0.05f);
    const Quad4 th2 = spread<QUAD>(a, [](float x) { return tanhf(x); }, (cy * o[3] + sy * o[4]) * 0.15f,
                                   (-sy * o[3] + cy * o[4]) * 0.15f, err * 2.0f, 0.0f);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[12 + i] = th1.v[i];
    v[16] = th2.v[0];
    v[17] = th2.v[1];
    v[21] = th2.v[2];
    v[18] = expf(-fmaxf(o[2] - 0.62f, 0.0f));
    v[19] = div_const(az - pi * 0.25f, pi / 6.0f);
    v[20] = div_const(el, pi / 6.0f);
    const bool ready = (int)(o46 <= 0.02f) & (int)(o47 > 0.01f) & (int)(err < 0.26f) &
                       (int)(dist < 34.0f);
    v[22] = ready ? 1.0f : -1.0f;
    // sin(bearing - pi/4 - yaw) by the addition theorem.
    v[23] = ((sb * cy - cb * sy) - (cb * cy + sb * sy)) * 0x1.6a09e6p-1f;  // 1 / sqrt 2
}

// The reference's last mapping (NaN -> 0, +-inf -> +-1).
__device__ __forceinline__ float tactical_out(float x) { return finite_as(x, 1.0f); }

// The mission's flags (onboard_features.cuh:107-109, 126-136, 433-437).
struct MissionFlags {
    bool landing, cargo, inversion, turbine_out, lateral, slalom, dodge, arena;
    bool bwb_arena, bwb_endurance, bwb;
};

__device__ __forceinline__ MissionFlags mission_flags(const float (&m)[10]) {
    MissionFlags f;
    f.landing = m[1] > 0.75f;
    f.cargo = m[2] > 0.75f;
    f.inversion = (int)(m[3] > 0.75f) & (int)(m[0] < -0.25f);
    f.turbine_out = (int)(m[3] > 0.75f) & (int)(m[2] < -0.25f);
    f.lateral = (int)(m[4] > 0.75f) & (int)(m[5] > 0.25f);
    f.slalom = (int)(m[4] > 0.75f) & (int)!f.lateral;
    f.dodge = m[5] > 0.75f;
    f.arena = m[6] > 0.75f;
    f.bwb_arena = (int)f.arena & (int)(m[4] < -0.25f);
    const bool cruise = (int)(m[4] > 0.75f) & (int)(m[2] > 0.25f);
    f.bwb_endurance = (int)cruise & (int)(m[0] > 0.25f);
    f.bwb = (int)f.bwb_arena | (int)cruise | ((int)f.arena & (int)(m[5] > 0.60f));
    return f;
}

// The goal's position (onboard_features.cuh:157-172, before the arena's
// stand-off) from the mission offsets.
struct Goal {
    float x, y, z;
};

__device__ __forceinline__ Goal goal_of(const MissionFlags &f, float px, float py, float pz,
                                        float relx, float rely, float relz) {
    const bool chase = (int)f.arena | (int)f.lateral;
    Goal g;
    g.x = chase ? px + relx : 0.0f;
    g.x = f.cargo ? 15.0f : g.x;
    g.x = f.slalom ? 36.0f : g.x;
    g.y = chase ? py + rely : 0.0f;
    g.z = f.landing ? 0.60f : 8.0f;
    g.z = f.inversion ? 14.0f : g.z;
    g.z = (int)f.cargo | (int)f.arena ? pz + relz : g.z;
    return g;
}

// One lane's share of the flight controls: its arms' throttle, outer and
// inner commands.
template <bool QUAD>
struct ArmOutputs {
    float throttle[kArms<QUAD>], outer[kArms<QUAD>], inner[kArms<QUAD>];
};

// The flight controller: onboard_features.cuh:88-432 without the cannon, with
// the LiDAR passes replaced by the scan's result (the two per-arm loops are
// :114-125 and :376-391).  The arm sums and the running maximum are formed in
// the reference's order, so every value is the one its code forms.  The
// cannon and the BWB law share nothing with this chain but its inputs: other
// waves form them (gunnery_values).
// `fetch` returns the scan result; everything that does not depend on it is
// formed before it is called.
template <bool TAME, bool QUAD, class Fetch>
__device__ __forceinline__ ArmOutputs<QUAD> flight_values(const ChainInputs<QUAD> &in, bool wild,
                                                          const MissionFlags &f, int a,
                                                          Fetch fetch) {
    constexpr int K = kArms<QUAD>;
    using onboard_math::quotient;
    const float pi = kPi;
    const float max_installed = 294.2f * 0.85f;
    const float idle_frac = 0.08f;
    const float min_thrust = max_installed * idle_frac;
    const float gravity = 9.80665f;
    const float outer_limit = 2.0f;
    const float inner_limit = pi / 4.0f;
    const float cannon_az_ctr = pi / 4.0f;
    const float *o = in.head, *m = in.m;
    const float px = o[0], py = o[1], pz = o[2], vx = o[3], vy = o[4], vz = o[5];
    const Attitude att = attitude_of(o[6], o[7], o[8], o[9]);
    const float qw = att.qw, qx = att.qx, qy = att.qy, qz = att.qz;
    const float ux = -qx, uy = -qy, uz = -qz;
    const float r00 = att.r[0], r10 = att.r[3], r22 = att.r[8];
    const float ox = o[10], oy = o[11], oz = o[12];
    const float omega_norm = ob_norm3<TAME>(ox, oy, oz);

    // This lane's arms; then every arm's forces.
    float spool[K], thrust[K], outer[K], fz_a[K], ft_a[K];
#pragma unroll
    for (int i = 0; i < K; ++i) {
        spool[i] = ob_clamp<TAME>(in.arm[0][i], 0.0f, 1.0f);
        thrust[i] = max_installed * (idle_frac + (1.0f - idle_frac) * spool[i]);
        outer[i] = ob_atan2<TAME>(in.arm[1][i], in.arm[2][i]);
        const onboard_math::Direction o_sc = ob_direction<TAME>(in.arm[1][i], in.arm[2][i], wild);
        const float c_inner = onboard_math::cos_float<TAME>(in.arm[3][i]);
        fz_a[i] = thrust[i] * o_sc.c * c_inner;
        ft_a[i] = thrust[i] * o_sc.s * c_inner;
    }
    const Quad4 fz = every_arm<QUAD>(fz_a), ft = every_arm<QUAD>(ft_a);
    float total_fz = 0.0f, jammed_yaw_ft = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        total_fz += fz.v[i];
        jammed_yaw_ft += ft.v[i];
    }
    const float fuel = ob_clamp<TAME>(in.tail[0], 0.0f, 1.0f) * 9.0f;
    const float ammo_mass = ob_clamp<TAME>(in.tail[5], 0.0f, 4.0f) * 6.0f;
    const bool payload = in.tail[1] > 0.5f;
    const float mass = (f.arena ? 40.0f : 43.0f) + fuel + ammo_mass + (payload ? 30.0f : 0.0f);
    const float weight = mass * gravity;
    const float body_z_x = 2.0f * (qx * qz + qw * qy);
    const float body_z_y = 2.0f * (qy * qz - qw * qx);
    const float ct = ob_clamp<TAME>(r22, -1.0f, 1.0f);
    const float tau_x_actual = fz.v[1] - fz.v[3];
    const float tau_y_actual = fz.v[2] - fz.v[0];
    const float az_actual = quotient<TAME>(total_fz * ct - weight, mass);
    const bool heavy_cargo = (int)f.cargo & (int)payload;
    const bool landing_like = (int)f.landing | (int)heavy_cargo;

    const Quad4 offsets = spread<QUAD>(
        a, [](float x) { return onboard_math::atanh_float(ob_clamp<TAME>(x, -0.9995f, 0.9995f)); },
        m[7], m[8], m[9], m[9]);
    const float relx = offsets.v[0] * 20.0f;
    const float rely = offsets.v[1] * 20.0f;
    const float relz = offsets.v[2] * 20.0f;
    const Goal goal = goal_of(f, px, py, pz, relx, rely, relz);
    const float tx = goal.x, ty = goal.y, tz = goal.z;
    const float dx_opp = tx - px, dy_opp = ty - py;
    const Quad4 angles = spread2<QUAD>(a, [](float y, float x) { return ob_atan2<TAME>(y, x); },
                                       r10, m[1], dy_opp, dy_opp, r00, m[2], dx_opp, dx_opp);
    const float yaw = angles.v[0], opp_bearing = angles.v[1], raw_bearing = angles.v[2];

    float ex = tx, ey = ty, ez = tz;
    const float dxy = ob_hypot<TAME>(dx_opp, dy_opp);
    const bool valid_d = dxy > 1.0e-3f;
    const onboard_math::Divisor over_d(valid_d ? dxy : 1.0f);
    const bool intercept = (int)f.arena & (int)(m[0] > 0.75f) & (int)(m[5] < -0.25f);
    const float desired_range = intercept ? 8.5f : 12.5f;
    const float stand_x = tx - over_d(dx_opp) * desired_range;
    const float stand_y = ty - over_d(dy_opp) * desired_range;
    float ax = valid_d ? stand_x : tx;
    float ay = valid_d ? stand_y : ty;
    const float scale =
        fminf(quotient<TAME>(16.0f, fmaxf(ob_hypot<TAME>(ax, ay), 1.0e-3f)), 1.0f);
    ax *= scale;
    ay *= scale;
    const float pull =
        ob_clamp<TAME>(div_const(ob_hypot<TAME>(px, py) - 21.0f, 10.0f), 0.0f, 1.0f);
    ax *= 1.0f - pull;
    ay *= 1.0f - pull;
    const bool low_or_sinking = (int)(pz < 8.0f) | (int)(vz < -1.0f);
    const float tz_held = ob_clamp<TAME>(tz, 8.5f, 12.2f);
    const float az_t = low_or_sinking ? 12.2f : tz_held;
    ex = f.arena ? ax : ex;
    ey = f.arena ? ay : ey;
    ez = f.arena ? az_t : ez;
    const float errx = ex - px, erry = ey - py;
    const float horiz_dist = ob_hypot<TAME>(errx, erry);

    const float tilt = acosf(ct);
    const bool need_headroom = (int)f.inversion | (int)f.arena | (int)(ct < 0.88f);
    const bool urgent_climb = (int)f.arena & ((int)(pz < 8.5f) | (int)(vz < -1.2f)) &
                              (int)(ct > 0.58f);
    const float room = ob_clamp<TAME>(3.95f - 0.90f * omega_norm - 1.30f * tilt, 2.55f, 3.95f);
    const float calm_coll = need_headroom ? room : 3.95f;
    const float max_coll = urgent_climb ? 3.95f : calm_coll;
    const float tilt_scale_h =
        ob_clamp<TAME>(1.0f - 1.5f * fmaxf(tilt - 0.15f, 0.0f), 0.0f, 1.0f);
    const float calm_scale = need_headroom ? tilt_scale_h : 1.0f;
    const float horiz_scale = urgent_climb ? 0.0f : calm_scale;
    const float cw_x = body_z_y, cw_y = -body_z_x;
    const float tt_x = 2.0f * (-uz * cw_y), tt_y = 2.0f * (uz * cw_x);
    const float tt_z = 2.0f * (ux * cw_y - uy * cw_x);
    const float te_x = cw_x + qw * tt_x + (uy * tt_z - uz * tt_y);
    const float te_y = cw_y + qw * tt_y + (uz * tt_x - ux * tt_z);
    const float te_z = qw * tt_z + (ux * tt_y - uy * tt_x);
    const float te_norm = ob_norm3<TAME>(te_x, te_y, te_z);
    const float per_te = quotient<TAME>(tilt, fmaxf(te_norm, 1.0e-5f));
    const float tilt_scale = te_norm > 1.0e-5f ? per_te : 0.0f;
    const float e_rx = te_x * tilt_scale, e_ry = te_y * tilt_scale;

    const bool inv_hold_yaw = ((int)f.inversion | (int)f.arena) &
                              ((int)(pz < 6.0f) | (int)(vz < -0.5f) | (int)(ct < 0.88f));
    const bool opp_bearing_valid = (int)f.arena & (int)(fabsf(m[1]) + fabsf(m[2]) > 0.1f);
    const float target_bearing = opp_bearing_valid ? opp_bearing : raw_bearing;
    const bool face = (int)f.arena & (int)(horiz_dist > 1.0f) & (int)!inv_hold_yaw;
    const float held_yaw = inv_hold_yaw ? yaw : 0.0f;
    const float facing_yaw = target_bearing - cannon_az_ctr;
    const float desired_yaw = face ? facing_yaw : held_yaw;
    const float yaw_err = ob_wrap<TAME>(desired_yaw, yaw);

    const float horiz_speed = ob_hypot<TAME>(vx, vy);
    const float hill = ob_clamp<TAME>(div_const(px - 6.0f, 30.0f), 0.0f, 1.0f);
    const float hill_sin = onboard_math::sin_half_turn(hill);

    const ScanResult scan = fetch();

    // Sine and cosine of yaw and of the closest return's bearing from their
    // components (a rotation's rows; a range inside the window).
    const Direction2 dir =
        directions<TAME, QUAD>(a, r10, r00, scan.min_r_dy, scan.min_r_dx, wild);
    const float cyaw = dir.c0, syaw = dir.s0;

    const bool avoid = (int)f.dodge & (int)(scan.min_r < 7.5f);
    const float away_x = -dir.s1 * 2.2f, away_y = dir.c1 * 2.2f;
    const float avoid_x = avoid ? away_x : 0.0f, avoid_y = avoid ? away_y : 0.0f;
    const float min_dx_c = scan.min_dx_c;
    const int cluster_count = scan.cluster_count;
    // Its sign alone is used, and the divisor is positive.
    const float cluster_y = scan.cluster_y_sum;
    const bool has_slalom_obs = (int)f.slalom & (int)(horiz_dist > 2.5f) & (int)(min_dx_c < 10.2f) &
                                (int)(cluster_count > 0);
    const float nearest_dx = has_slalom_obs ? min_dx_c : 30.0f;
    const float side_y = cluster_y >= 0.0f ? -1.85f : 1.85f;
    ey = has_slalom_obs ? side_y : ey;
    const float lane_err = fabsf(py - ey);
    float speed_limit = lane_err > 0.55f ? 2.75f : 4.10f;
    speed_limit = lane_err > 1.05f ? 1.55f : speed_limit;
    const bool open_road = (int)(min_dx_c >= 6.6f) & (int)(px > 4.0f);
    speed_limit = open_road ? 3.10f : speed_limit;
    const float slalom_speed = has_slalom_obs ? speed_limit : 3.8f;
    const bool over_hill = (int)f.slalom & (int)(horiz_dist > 3.5f);
    const float hill_z = 2.5f * hill_sin + 8.0f;
    ez = over_hill ? hill_z : ez;
    const float upx = ex - px, upy = ey - py, upz = ez - pz;
    const float up_horiz = ob_hypot<TAME>(upx, upy);
    const bool active_slalom =
        (int)f.slalom & (int)(nearest_dx < 10.2f) & (int)(horiz_dist > 3.0f);

    const float pad_z = fmaxf(ez, 0.60f), above_pad = pz - pad_z;
    const float transit_cap = heavy_cargo ? 2.65f : 3.4f;
    const float near_cap = heavy_cargo ? 1.25f : 1.6f;
    const float low_cap = above_pad < 1.2f ? 0.55f : near_cap;
    const float max_vxy_land = up_horiz > 1.8f ? transit_cap : low_cap;
    const float kp_land = heavy_cargo ? 0.75f : 1.05f;
    const float des_vx_land = ob_clamp<TAME>(kp_land * upx, -max_vxy_land, max_vxy_land);
    const float des_vy_land = ob_clamp<TAME>(kp_land * upy, -max_vxy_land, max_vxy_land);
    const float vz_land_touch = pz > 0.635f ? -0.16f : 0.0f;
    const float vz_land_cargo = ob_clamp<TAME>(1.6f * (0.64f - pz), -0.30f, 0.18f);
    const float vz_land_low = f.cargo ? vz_land_cargo : vz_land_touch;
    const float max_desc = f.cargo ? -0.82f : -1.4f;
    const float vz_land_mid = ob_clamp<TAME>(-0.70f * above_pad, max_desc, -0.25f);
    const float vz_land_align = ob_clamp<TAME>(1.2f * (pad_z + 0.90f - pz), -0.30f, 0.60f);
    const float heavy_transit = fmaxf(1.2f + 0.28f * up_horiz, 2.0f);
    const float transit_z = heavy_cargo ? heavy_transit : 2.0f;
    const float max_desc_trans = heavy_cargo ? -1.05f : -1.6f;
    const float vz_land_trans = ob_clamp<TAME>(1.3f * (transit_z - pz), max_desc_trans, 1.4f);
    float des_vz_land = above_pad > 1.05f ? vz_land_mid : vz_land_low;
    const bool align = ((int)(up_horiz > 0.85f) | (int)(horiz_speed > 0.65f)) &
                       (int)(above_pad < 0.95f);
    des_vz_land = align ? vz_land_align : des_vz_land;
    des_vz_land = up_horiz > 1.8f ? vz_land_trans : des_vz_land;
    const float max_axy_land = heavy_cargo ? 2.2f : 2.6f;
    const float des_ax_land = ob_clamp<TAME>(2.4f * (des_vx_land - vx), -max_axy_land, max_axy_land);
    const float des_ay_land = ob_clamp<TAME>(2.4f * (des_vy_land - vy), -max_axy_land, max_axy_land);
    const float kp_az_land = heavy_cargo ? 5.0f : 4.5f;
    const float kd_az_land = heavy_cargo ? 1.0f : 0.80f;
    const float min_az_land = heavy_cargo ? -1.8f : -2.8f;
    const float des_az_land = ob_clamp<TAME>(
        kp_az_land * (des_vz_land - vz) - kd_az_land * az_actual, min_az_land, 5.5f);

    const bool dash = (int)(up_horiz > 9.0f) & (int)(fabsf(upz) < 2.5f) & (int)(ct > 0.90f);
    const float inv_max_v = dash ? 6.2f : 4.2f;
    const float lat_vx = fabsf(upy) > 1.35f ? 1.45f : 3.8f;
    float max_vx = f.arena ? 3.2f : 3.0f;
    max_vx = f.inversion ? inv_max_v : max_vx;
    float max_vy = f.lateral ? 3.4f : max_vx;
    max_vx = f.lateral ? lat_vx : max_vx;
    max_vx = f.slalom ? 3.5f : max_vx;
    max_vx = active_slalom ? slalom_speed : max_vx;
    max_vy = active_slalom ? 3.2f : max_vy;
    const bool climb_fast = (int)(vz < -2.0f) | (int)f.inversion;
    const float max_vz = climb_fast ? 6.5f : 2.6f;
    const float kp_side = f.lateral ? 0.95f : 0.90f;
    const float kp_xy = f.inversion ? 0.85f : kp_side;
    const float kp_vx = active_slalom ? 1.25f : kp_xy;
    const float kp_vy_calm = f.lateral ? 1.05f : kp_xy;
    const float kp_vy = active_slalom ? 1.45f : kp_vy_calm;
    const float des_vx = ob_clamp<TAME>(kp_vx * upx + avoid_x, -max_vx, max_vx);
    const float des_vy = ob_clamp<TAME>(kp_vy * upy + avoid_y, -max_vy, max_vy);
    float des_vz = ob_clamp<TAME>(1.25f * upz, -2.6f, max_vz);
    const bool recover = ((int)f.inversion | (int)f.arena) & (int)(vz < -1.0f);
    const float des_vz_up = fmaxf(des_vz, 0.8f);
    des_vz = recover ? des_vz_up : des_vz;
    const float kp_ax = active_slalom ? 3.0f : 2.4f;
    const float kp_ay = active_slalom ? 3.0f : 2.6f;
    const float des_ax_std = ob_clamp<TAME>(kp_ax * (des_vx - vx), -3.8f, 3.8f);
    const float des_ay_std = ob_clamp<TAME>(kp_ay * (des_vy - vy), -3.8f, 3.8f);
    const bool pull_up = (int)(vz < -1.8f) | (int)f.inversion;
    const float max_az = pull_up ? 14.0f : 6.5f;
    const float des_az_std =
        ob_clamp<TAME>(3.8f * (des_vz - vz) - 0.80f * az_actual, -4.0f, max_az);
    const float des_ax = landing_like ? des_ax_land : des_ax_std;
    const float des_ay = landing_like ? des_ay_land : des_ay_std;
    const float des_az = landing_like ? des_az_land : des_az_std;

    const float fz_des = ob_clamp<TAME>(quotient<TAME>(weight + mass * des_az, fmaxf(ct, 0.45f)),
                                        0.10f * weight, max_coll * max_installed);
    const float tilt_comp = f.turbine_out ? 0.65f : 0.0f;
    const float damp_v = active_slalom ? 0.8f : 0.4f;
    const float fx_world =
        (mass * des_ax + damp_v * vx - tilt_comp * total_fz * body_z_x) * horiz_scale;
    const float fy_world =
        (mass * des_ay + damp_v * vy - tilt_comp * total_fz * body_z_y) * horiz_scale;
    const float std_fh = heavy_cargo ? 52.0f : 80.0f;
    const float lat_fh = f.lateral ? 125.0f : std_fh;
    const float max_fh = active_slalom ? 105.0f : lat_fh;
    const float fx_body = ob_clamp<TAME>(cyaw * fx_world + syaw * fy_world, -max_fh, max_fh);
    const float fy_body = ob_clamp<TAME>(-syaw * fx_world + cyaw * fy_world, -max_fh, max_fh);

    const float parasite_scale = f.turbine_out ? 0.35f : 1.0f;
    const float tau_x_par = -0.1625f * fy_body * parasite_scale;
    const float tau_y_par = 0.1625f * fx_body * parasite_scale;
    const float tau_x_net = tau_x_actual + tau_x_par;
    const float tau_y_net = tau_y_actual + tau_y_par;
    const float max_txy = heavy_cargo ? 120.0f : 260.0f;
    const float tau_x_cmd = ob_clamp<TAME>(
        95.0f * e_rx - 64.0f * ox - 0.90f * tau_x_net - tau_x_par, -max_txy, max_txy);
    const float tau_y_cmd = ob_clamp<TAME>(
        95.0f * e_ry - 64.0f * oy - 0.90f * tau_y_net - tau_y_par, -max_txy, max_txy);
    const float tau_z_cmd = ob_clamp<TAME>(22.0f * yaw_err - 18.0f * oz, -70.0f, 70.0f);
    const float half_tx = tau_x_cmd * 0.5f, half_ty = tau_y_cmd * 0.5f;
    const float yaw_ft = (tau_z_cmd - 0.40f * jammed_yaw_ft) * 0.25f;
    const float fx_outer = ft.v[3] - ft.v[1];
    const float fy_outer = ft.v[0] - ft.v[2];
    const float fx_rem = fx_body - fx_outer, fy_rem = fy_body - fy_outer;
    const float std_sin = heavy_cargo ? 0.22f : 0.32f;
    const float road_sin = active_slalom ? 0.42f : std_sin;
    const float max_sin_inner = f.lateral ? 0.44f : road_sin;
    const float std_gain = heavy_cargo ? 4.5f : 2.4f;
    const float spool_gain = f.turbine_out ? 10.5f : std_gain;
    const bool land_idle = (int)f.landing & (int)(pz <= 0.638f) & (int)(up_horiz < 0.85f) &
                           (int)(fabsf(vz) < 0.20f);
    const float idle_thrust = 0.15f * weight * 0.25f;
    float outer_cmd[K], inner_cmd[K], u_raw[K];
#pragma unroll
    for (int i = 0; i < K; ++i) {
        // {q - ty, q + tx, q + ty, q - tx}[arm]; q - t and q + (-t) are the
        // same IEEE operation.
        const float fz_cmd =
            0.25f * fz_des + arm_pick<QUAD>(a, i, -half_ty, half_tx, half_ty, -half_tx);
        const float sin_alpha =
            ob_clamp<TAME>(quotient<TAME>(yaw_ft, fmaxf(thrust[i], 30.0f)), -0.35f, 0.35f);
        const float yaw_alpha = asinf(sin_alpha);
        outer_cmd[i] =
            ob_clamp<TAME>(6.5f * ob_wrap<TAME>(yaw_alpha, outer[i]), -outer_limit, outer_limit);
        const float urx = arm_pick<QUAD>(a, i, 1.0f, 0.0f, -1.0f, 0.0f);
        const float ury = arm_pick<QUAD>(a, i, 0.0f, 1.0f, 0.0f, -1.0f);
        const float fr_req = 0.5f * (fx_rem * urx + fy_rem * ury);
        const float sin_in = ob_clamp<TAME>(quotient<TAME>(fr_req, fmaxf(thrust[i], 40.0f)),
                                            -max_sin_inner, max_sin_inner);
        inner_cmd[i] = ob_clamp<TAME>(asinf(sin_in), -inner_limit * 0.90f, inner_limit * 0.90f);
        // cos(yaw_alpha) cos(inner_cmd), both arcsines (|sin_in| <= 0.44, so
        // the limit on inner_cmd is never met).
        const float nominal_cos = fmaxf(onboard_math::cosine_product(sin_alpha, sin_in), 0.70f);
        const float lift_thrust = quotient<TAME>(fmaxf(fz_cmd, 0.0f), nominal_cos);
        const float target_thrust = land_idle ? idle_thrust : lift_thrust;
        const float u_des = ob_clamp<TAME>(
            div_const(target_thrust - min_thrust, max_installed - min_thrust), 0.0f, 1.0f);
        u_raw[i] = u_des + spool_gain * (u_des - spool[i]);
    }
    // The reference's running maximum over arms 0..3, from -inf.
    const Quad4 u_all = every_arm<QUAD>(u_raw);
    float max_raw = -__builtin_huge_valf();
#pragma unroll
    for (int i = 0; i < 4; ++i) max_raw = fmaxf(max_raw, u_all.v[i]);
    const float excess = ob_clamp<TAME>(max_raw - 1.0f, 0.0f, urgent_climb ? 0.10f : 0.45f);
    const float shed = need_headroom ? excess : 0.0f;
    const bool inv_mode = ct < 0.20f;
    const float inv_rx = te_norm > 1.0e-5f ? e_rx : tilt;
    const float tx_inv = 130.0f * inv_rx - 52.0f * ox;
    const float ty_inv = 130.0f * e_ry - 52.0f * oy;
    ArmOutputs<QUAD> out;
#pragma unroll
    for (int i = 0; i < K; ++i) {
        float throttle = ob_clamp<TAME>(u_raw[i] - shed, 0.0f, 1.0f);
        const float arm_mom = arm_pick<QUAD>(a, i, -ty_inv, tx_inv, ty_inv, -tx_inv);
        const float inv_throttle = arm_mom > 12.0f ? 0.58f : 0.0f;
        const float inv_outer = ob_clamp<TAME>(-outer[i] * 6.0f, -outer_limit, outer_limit);
        throttle = inv_mode ? inv_throttle : throttle;
        const float outer_out = inv_mode ? inv_outer : outer_cmd[i];
        const float inner_out = inv_mode ? 0.0f : inner_cmd[i];
        out.throttle[i] = ob_clamp<TAME>(throttle * 2.0f - 1.0f, -1.0f, 1.0f);
        out.outer[i] = ob_clamp<TAME>(outer_out * (1.0f / outer_limit), -1.0f, 1.0f);
        out.inner[i] = ob_clamp<TAME>(div_const(inner_out, inner_limit), -1.0f, 1.0f);
    }
    return out;
}

// The cannon (onboard_features.cuh:393-430) and, for BWB missions, the BWB
// law, which replaces every prior value (:433-510): the cannon's azimuth,
// elevation and fire (identical in a quad's lanes) and, for a BWB mission,
// the lane's arm commands.
template <bool QUAD>
struct GunOutputs {
    float az, el, fire;
    ArmOutputs<QUAD> arm;  // BWB missions only
};

template <bool TAME, bool QUAD>
__device__ __forceinline__ GunOutputs<QUAD> gunnery_values(const ChainInputs<QUAD> &in, bool wild,
                                                           const MissionFlags &f, int a) {
    constexpr int K = kArms<QUAD>;
    using onboard_math::quotient;
    const float pi = kPi;
    const float gravity = 9.80665f;
    const float inner_limit = pi / 4.0f;
    const float cannon_az_ctr = pi / 4.0f;
    const float cannon_az_half = pi / 6.0f;
    const float cannon_el_lim = pi / 6.0f;
    const float *o = in.head, *m = in.m;
    const float o44 = in.tail[2], o45 = in.tail[3], o46 = in.tail[4], o47 = in.tail[5];
    const float px = o[0], py = o[1], pz = o[2], vx = o[3], vy = o[4], vz = o[5];
    const Attitude att = attitude_of(o[6], o[7], o[8], o[9]);
    const float qw = att.qw, qx = att.qx, qy = att.qy, qz = att.qz;
    const float ux = -qx, uy = -qy, uz = -qz;
    const float r00 = att.r[0], r01 = att.r[1], r02 = att.r[2];
    const float r10 = att.r[3], r11 = att.r[4], r12 = att.r[5];
    const float r20 = att.r[6], r21 = att.r[7], r22 = att.r[8];
    const float ct = ob_clamp<TAME>(r22, -1.0f, 1.0f);
    const bool inv_mode = ct < 0.20f;

    const Quad4 offsets = spread<QUAD>(
        a, [](float x) { return onboard_math::atanh_float(ob_clamp<TAME>(x, -0.9995f, 0.9995f)); },
        m[7], m[8], m[9], m[9]);
    const Goal goal = goal_of(f, px, py, pz, offsets.v[0] * 20.0f, offsets.v[1] * 20.0f,
                              offsets.v[2] * 20.0f);
    // The aim point in the body frame.
    const float to_x = goal.x - px, to_y = goal.y - py, to_z = goal.z - pz;
    const float dist = fmaxf(ob_norm3<TAME>(to_x, to_y, to_z), 1.0f);
    const float flight = div_const(dist, 20.0f);
    const float aim_x = to_x - vx * (0.65f * flight);
    const float aim_y = to_y - vy * (0.65f * flight);
    const float aim_z = to_z - vz * (0.65f * flight) + 0.53f * gravity * flight * flight;
    const float cx = uy * aim_z - uz * aim_y + qw * aim_x;
    const float cyq = uz * aim_x - ux * aim_z + qw * aim_y;
    const float cz = ux * aim_y - uy * aim_x + qw * aim_z;
    const float aim_bx = aim_x + 2.0f * (uy * cz - uz * cyq);
    const float aim_by = aim_y + 2.0f * (uz * cx - ux * cz);
    const float aim_bz = aim_z + 2.0f * (ux * cyq - uy * cx);
    // The aim's azimuth and elevation, and for the BWB law roll and course
    // (the ground track above 2.5 m/s, else yaw).
    const float gs = ob_hypot<TAME>(vx, vy);
    const float course_y = gs > 2.5f ? vy : r10, course_x = gs > 2.5f ? vx : r00;
    const auto atan2_of = [](float y, float x) { return ob_atan2<TAME>(y, x); };
    const Quad4 angles = spread2<QUAD>(a, atan2_of, aim_by, aim_bz, r21, course_y, aim_bx,
                                       fmaxf(ob_hypot<TAME>(aim_bx, aim_by), 0.2f), r22, course_x);
    const float des_cannon_az =
        ob_clamp<TAME>(angles.v[0], cannon_az_ctr - cannon_az_half, cannon_az_ctr + cannon_az_half);
    const float des_cannon_el = ob_clamp<TAME>(angles.v[1], -cannon_el_lim, cannon_el_lim);
    const float roll_right = angles.v[2], course_yaw = angles.v[3];

    const float aim_err = ob_hypot<TAME>(ob_wrap<TAME>(des_cannon_az, o44), des_cannon_el - o45);
    const bool loaded = (int)f.arena & (int)(o46 <= 0.02f) & (int)(o47 > 0.01f);
    const bool fire =
        (int)loaded & (int)!inv_mode & (int)(aim_err < 0.28f) & (int)(dist < 34.0f);
    const bool cannon = (int)f.arena & (int)!inv_mode;
    const float aimed_az =
        ob_clamp<TAME>(div_const(des_cannon_az - cannon_az_ctr, cannon_az_half), -1.0f, 1.0f);
    const float aimed_el = ob_clamp<TAME>(div_const(des_cannon_el, cannon_el_lim), -1.0f, 1.0f);
    GunOutputs<QUAD> out;
    out.az = cannon ? aimed_az : 0.0f;
    out.az = inv_mode ? -1.0f : out.az;
    out.el = cannon ? aimed_el : 0.0f;
    out.fire = fire ? 0.8f : -0.8f;
    out.arm = ArmOutputs<QUAD>{};
    if (!f.bwb) return out;

    const float vb_x = r00 * vx + r10 * vy + r20 * vz;
    const float vb_y = r01 * vx + r11 * vy + r21 * vz;
    const Quad4 b_offsets = spread<QUAD>(
        a, [](float x) { return onboard_math::atanh_float(ob_clamp<TAME>(x, -0.9999f, 0.9999f)); },
        m[7], m[8], m[9], m[9]);
    const float brx = b_offsets.v[0] * 20.0f;
    const float bry = b_offsets.v[1] * 20.0f;
    const float brz = b_offsets.v[2] * 20.0f;
    float btx = px + brx;
    float bty = py + bry;
    float btz = pz + brz;
    const float rxy = ob_hypot<TAME>(px, py);
    const float pull_b = ob_clamp<TAME>(div_const(rxy - 235.0f, 45.0f), 0.0f, 0.85f);
    const bool fenced = (int)f.arena & (int)(rxy > 235.0f);
    const float in_x = btx * (1.0f - pull_b), in_y = bty * (1.0f - pull_b);
    btx = fenced ? in_x : btx;
    bty = fenced ? in_y : bty;
    const float in_z = ob_clamp<TAME>(btz, 28.0f, 135.0f);
    btz = f.arena ? in_z : btz;
    const float gx = btx - px, gy = bty - py;
    const float gz = btz - pz;
    const float gdist = fmaxf(ob_norm3<TAME>(gx, gy, gz), 1.0f);
    const float climb_des = ob_clamp<TAME>(0.42f * gz, -5.0f, 5.0f);
    const float oppx = brx - vx * 0.10f, oppy = bry - vy * 0.10f, oppz = brz - vz * 0.10f;
    const float bdist = fmaxf(ob_norm3<TAME>(oppx, oppy, oppz), 1.0f);
    const bool head_on = (int)f.bwb_arena & (int)(btx * px + bty * py < -800.0f) &
                         (int)(bdist > 45.0f);
    const float head_closing = 75.0f + 2.0f * fmaxf(vb_x, 0.0f);
    const float closing = head_on ? head_closing : 75.0f;
    const float bflight = quotient<TAME>(bdist, closing);
    const float bax = oppx, bay = oppy;
    const float sink = -vz * (0.85f * bflight);
    const float baz = oppz + (head_on ? sink : 0.0f) + 0.50f * gravity * bflight * bflight;
    const float bbx = r00 * bax + r10 * bay + r20 * baz;
    const float bby = r01 * bax + r11 * bay + r21 * baz;
    const float bbz = r02 * bax + r12 * bay + r22 * baz;
    const Quad4 b_angles = spread2<QUAD>(a, atan2_of, gy, climb_des, bby, bbz, gx, fmaxf(gs, 14.0f),
                                         fmaxf(bbx, 0.2f), fmaxf(ob_hypot<TAME>(bbx, bby), 0.2f));
    const float desired_yaw_b = b_angles.v[0], gamma_des = b_angles.v[1];
    const float b_az = ob_clamp<TAME>(b_angles.v[2], -pi / 6.0f, pi / 6.0f);
    const float b_el = ob_clamp<TAME>(b_angles.v[3], -cannon_el_lim, cannon_el_lim);

    const float course_err = ob_wrap<TAME>(desired_yaw_b, course_yaw);
    const float arena_speed = gdist > 38.0f ? 26.0f : 24.0f;
    const float free_speed = f.arena ? arena_speed : 22.4f;
    const float desired_speed = f.bwb_endurance ? 18.5f : free_speed;
    const float speed_err = desired_speed - vb_x;
    const float u_coll = ob_clamp<TAME>((f.bwb_endurance ? 0.36f : 0.44f) + 0.065f * speed_err +
                                            0.018f * gz, 0.12f, 0.90f);
    const float desired_roll = ob_clamp<TAME>(-1.35f * course_err, -0.55f, 0.55f);
    const float diff_u = ob_clamp<TAME>(0.90f * (desired_roll - roll_right) - 0.34f * o[10],
                                        -0.45f, 0.45f);
    const float u0 = ob_clamp<TAME>(u_coll + diff_u, 0.05f, 1.0f);
    const float u1 = ob_clamp<TAME>(u_coll - diff_u, 0.05f, 1.0f);
    const float pitch_up = asinf(ob_clamp<TAME>(r20, -1.0f, 1.0f));
    const float climb_err = climb_des - vz;
    const onboard_math::Direction bank = ob_direction<TAME>(r21, r22, wild);
    const float cos_bank = bank.c, sin_bank = bank.s;
    float desired_pitch = ob_clamp<TAME>(0.062831853f + 0.75f * gamma_des + 0.035f * climb_err +
                                             0.09f * (1.0f - fmaxf(cos_bank, 0.5f)),
                                         -0.15f, 0.25f);
    const float slow_pitch = fminf(desired_pitch, 0.02f);
    desired_pitch = vb_x < 15.5f ? slow_pitch : desired_pitch;
    const float theta_dot = 2.20f * (desired_pitch - pitch_up);
    const float psi_dot = quotient<TAME>(gravity, fmaxf(vb_x, 12.0f)) *
                              onboard_math::tan_float(ob_clamp<TAME>(-roll_right, -0.75f, 0.75f)) +
                          0.35f * course_err;
    const float q_up = cos_bank * theta_dot - sin_bank * psi_dot;
    const float r_left = sin_bank * theta_dot + cos_bank * psi_dot;
    const float gimbal = pi / 6.0f;
    const float inner0 = ob_clamp<TAME>(0.85f * (q_up + o[11]) + 0.03f, -gimbal, gimbal);
    const float inner1 = ob_clamp<TAME>(-0.65f * (r_left - o[12]) - 0.025f * vb_y, -gimbal, gimbal);
    const float b_err = ob_hypot<TAME>(ob_wrap<TAME>(b_az, o44), b_el - o45);
    const bool b_fire = (int)loaded & (int)(b_err < 0.045f) & (int)(bdist < 165.0f) &
                        (int)(bbx > 0.0f);
    const float b_norm_az = ob_clamp<TAME>(div_const(b_az, pi / 6.0f), -1.0f, 1.0f);
    const float b_norm_el = ob_clamp<TAME>(div_const(b_el, cannon_el_lim), -1.0f, 1.0f);
    out.az = f.arena ? b_norm_az : 0.0f;
    out.el = f.arena ? b_norm_el : 0.0f;
    out.fire = b_fire ? 0.8f : -0.8f;
#pragma unroll
    for (int i = 0; i < K; ++i) {
        const float throttle = arm_pick<QUAD>(a, i, u0, u1, u0, u1);
        const float inner_cmd = arm_pick<QUAD>(a, i, inner0, inner1, 0.0f, 0.0f);
        out.arm.throttle[i] = ob_clamp<TAME>(throttle * 2.0f - 1.0f, -1.0f, 1.0f);
        out.arm.outer[i] = 0.0f;
        out.arm.inner[i] = ob_clamp<TAME>(div_const(inner_cmd, inner_limit), -1.0f, 1.0f);
    }
    return out;
}

struct OnboardRows {
    const unsigned char *obs;
    size_t obs_stride;
    const unsigned char *mission;
    size_t mission_stride;
    float *tactical;
    float *prior;
    float *diag;
    float *proprio;      // optional [batch, 91]: tactical -> 52..75, prior -> 76..90
    float *mission_vec;  // optional [batch, 49]: tactical -> 10..33, prior -> 34..48
    float *lidar;        // optional [batch, 6, 16, 128]: channels of the scan rays
    size_t batch;
};

// log1p(x) for x >= 0 (any magnitude): 1 + x = u + c exactly (Fast2Sum),
// log1p(x) = log2(u)*ln2 + c/u with ln2 as a hi+lo pair.
__device__ __forceinline__ float log1p_pos(float x) {
    const float a = fmaxf(x, 1.0f), b = fminf(x, 1.0f);
    const float u = a + b;
    const float c = b - (u - a);
    const float l2 = __builtin_amdgcn_logf(u);
    const float t = c * __builtin_amdgcn_rcpf(u);
    const float r = __builtin_fmaf(l2, 0x1.62e43p-1f, __builtin_fmaf(l2, -0x1.05c61p-29f, t));
    return x == 0.0f ? x : r;
}

__device__ __forceinline__ float actor_scale(int i) {  // network_gpu.cu:287-293
    if (i < 3) return 0.05f;
    if (i < 6) return 0.10f;
    if (i >= 10 && i < 13) return 0.20f;
    if (i >= 13 && i < 16) return 0.10f;
    if (i >= 28 && i < 32) return 0.50f;
    if (i >= 32 && i < 36) return 0.20f;
    return 1.0f;
}

// network_gpu.cu:285-297 (scalar_inputs): lanes 0..51 of a wave write the
// environment's 52 symlog scalars, lanes 52..61 its 10 finite mission values.
// The input of lane l is obs[l] (l < 48), obs[4144 + l - 48] (l < 52) or
// mission[l - 52] (l < 62).  Branch-free: every lane forms both values, and
// buffer stores (discarded past num_records) write lanes 0..51 into proprio
// and 52..61 into mission_vec; an environment that is not `valid` writes
// nothing.
constexpr int kPastRecords = 0x40000000;  // past every resource
// RN_double(1 / sqrtf(1.0001f)): (float)((double)x * this) equals the IEEE
// quotient x / sqrtf(1.0001f) for every float |x| <= 8 (checked
// exhaustively by tests/csrc/check_div_by_constant.c), and |symlog| < 7.
constexpr double kInvSqrt10001 = 0x1.fff974156e01ep-1;

__device__ __forceinline__ void actor_scalars(float raw, int lane, float *proprio,
                                              float *mission_vec, bool valid) {
    const bool finite = __builtin_isfinite(raw);
    const float clamped = finite ? fmaxf(-1000.0f, fminf(1000.0f, raw)) : 0.0f;
    const float symlog = copysignf(log1p_pos(fabsf(clamped * actor_scale(lane))), clamped);
    const float scaled = fmaxf(-8.0f, fminf(8.0f, (float)((double)symlog * kInvSqrt10001)));
    __builtin_amdgcn_raw_buffer_store_b32(
        __builtin_bit_cast(unsigned, scaled),
        __builtin_amdgcn_make_buffer_rsrc(proprio, (short)0, valid ? 52 * 4 : 0, kBufferWord3),
        lane < 52 ? 4 * lane : kPastRecords, 0, 0);
    __builtin_amdgcn_raw_buffer_store_b32(
        __builtin_bit_cast(unsigned, finite ? raw : 0.0f),
        __builtin_amdgcn_make_buffer_rsrc(mission_vec, (short)0, valid ? 10 * 4 : 0,
                                          kBufferWord3),
        lane >= 52 && lane < 62 ? 4 * (lane - 52) : kPastRecords, 0, 0);
}

// A scan result parked in its environment's prior row (7 of its 15 words)
// until the control kernel has read it.
__device__ __forceinline__ void park_scan(float *park, const ScanResult &s) {
    park[0] = s.min_r;
    park[1] = s.min_r_dx;
    park[2] = s.min_r_dy;
    park[3] = s.min_dx_c;
    park[4] = s.cluster_y_sum;
    park[5] = __int_as_float(s.min_ray);
    park[6] = __int_as_float(s.cluster_count);
}

// Phase 1 of the actor entry's two-stream form.  Each wave scans one
// environment at a time;
// workgroups are persistent (the ray table is loaded into LDS once per
// workgroup, the only barrier).  Wave g of the grid takes environments g,
// g + W, g + 2W, ... (W waves in the grid).  Their scan frames (attitude
// rows, py) and scan needs (scan_need) are formed up front, lane j for the
// wave's j-th environment, and each environment's frame and need are then
// read from its lane into scalar registers.  Each environment's ranges are
// requested while the previous one finishes; every range is read, for the
// LiDAR channels of the scan rays.  The 32-byte result is parked in the
// environment's own prior row (60 bytes), which phase 2 reads before it
// writes the 15 prior values there: no scratch memory is needed.
__global__ __launch_bounds__(kBlockThreads) __attribute__((amdgpu_waves_per_eu(4)))
void actor_scan_kernel(OnboardRows rows) {
    __shared__ RayPlanes rays;
    __shared__ u32x2 lists[kWavesPerBlock][kListCap + 64];  // + a spare entry per lane
    const int tid = threadIdx.x, lane = tid & 63;
    for (int i = tid; i < 1536; i += kBlockThreads) {
        rays.d[0][i] = kRayDir[i * 3 + 0];
        rays.d[1][i] = kRayDir[i * 3 + 1];
        rays.d[2][i] = kRayDir[i * 3 + 2];
    }
    __syncthreads();
    const size_t waves = (size_t)gridDim.x * kWavesPerBlock;
    size_t env = (size_t)blockIdx.x * kWavesPerBlock + __builtin_amdgcn_readfirstlane(tid >> 6);
    if (env >= rows.batch) return;
    auto obs_of = [&](size_t e) {
        return reinterpret_cast<const float *>(rows.obs + e * rows.obs_stride);
    };
    // Lane j forms the frame of the wave's j-th environment from here (a
    // lane past the batch repeats the current one, whose row exists), and
    // what its mission uses of the scan.
    auto frame_obs = [&](size_t first) {
        const size_t e0 = first + (size_t)lane * waves, e = e0 < rows.batch ? e0 : first;
        return load_frame_obs(obs_of(e), reinterpret_cast<const float *>(
                                             rows.mission + e * rows.mission_stride));
    };
    auto frame_need = [&](const FrameObs &v) { return scan_need(v.m4, v.m5); };
    FrameObs first_obs = frame_obs(env);
    float rg[kScanRays];
    load_ranges(obs_rsrc(obs_of(env), true), obs_rsrc(obs_of(env), true), lane, rg);
    ScanFrame mine = scan_frame(first_obs);
    int need_mine = frame_need(first_obs);
    for (int k = 0;;) {
        ScanFrame f;
#pragma unroll
        for (int i = 0; i < 9; ++i)
            f.r[i] = __builtin_bit_cast(
                float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, mine.r[i]), k));
        f.py = __builtin_bit_cast(float,
                                  __builtin_amdgcn_readlane(__builtin_bit_cast(int, mine.py), k));
        const size_t next_env = env + waves;
        const bool has_next = next_env < rows.batch;
        const int need = __builtin_amdgcn_readlane(need_mine, k);
        const __amdgpu_buffer_rsrc_t next =
            obs_rsrc(has_next ? obs_of(next_env) : nullptr, has_next);
        write_channel_planes(
            rg, __builtin_amdgcn_make_buffer_rsrc(rows.lidar + env * 12288, (short)0,
                                                  12288 * 4, kBufferWord3),
            lane);
        ScanResult s;
        scan_env(rg, rays, f, next, next, lane, lists[__builtin_amdgcn_readfirstlane(tid >> 6)],
                 s, need);
        if (lane == 0) park_scan(rows.prior + env * 15, s);
        if (!has_next) break;
        env = next_env;
        if (++k == 64) {  // the next 64 environments of this wave
            k = 0;
            FrameObs v = frame_obs(env);
            mine = scan_frame(v);
            need_mine = frame_need(v);
        }
    }
}

// The onboard entry's workgroups take equal shares of the batch, at least
// kMinShare environments: one workgroup for each CU up to 4,096 environments,
// two above, as many as are resident at once.  A share of up to 16 runs as one
// group, up to 32 as two, above that as four (whose flight chains take one
// lane per environment), and batches above 32,768 take further rounds.  Fewer
// environments are shorter chains and fewer scans for a workgroup's waves,
// more share the ray table and the launch.  What the scans cost depends on the
// scene and the missions: where every environment is scanned through a
// cluttered corridor they are nine tenths of the time, and shares of 16 left
// most CUs idle (64 environments on four).  Measured on one box, us, scenes as
// the generator makes them / cluttered with every mission a slalom (two
// launches, a scan and a control kernel; 16, 32 or 64 environments per
// workgroup; these shares):
//       64  15.5 / 22.0   7.9 / 26.6   7.9 / 21.2
//    1,000  15.8 / 23.2   8.8 / 28.0   8.5 / 22.4
//    2,560  17.7 / 28.6   9.0 / 28.4   8.7 / 23.6
//    4,096  17.9 / 28.8   9.1 / 28.6   (the same)
//    6,000  19.0 / 35.6  10.4 / 33.1  10.1 / 29.1
//    9,000  20.2 / 42.5  13.4 / 56.0  12.7 / 40.5
//   12,000  20.9 / 74.0  14.4 / 57.1  13.5 / 49.0
//   16,384  21.0 / 74.4  14.9 / 57.7  (the same)
//   17,000  34.1 / 69.9  (already equal shares)  16.7 / 54.7
//   32,768  44.8 / 106   22.9 / 87.0  (the same)
// Shares below 8 gain for the smallest batches when all are scanned (4 each:
// 64 8.1 / 14.6) and lose from 2,048 (9.6 / 18.0; 3,000 15.1 / 29.9).  Of the
// groups, one / two / four: 8,192 environments 10.6 / 12.9 / 14.6, 16,384 20.2
// / 14.9 / 16.4, 17,000 -- / 22.5 / 16.7.
constexpr unsigned kMinShare = 8;
constexpr size_t kCus = 256, kRoundBlocks = 512;  // workgroups resident at once: two per CU

// Above one round of 64 environments in every workgroup the last round holds
// the rest.  A rest of up to one workgroup of 32 for each CU is shared out by
// 32: in shares of 64 a few CUs kept the others waiting, which in scenes full
// of scans took longer than two launches.  Smaller shares gain more there and
// lose in open scenes, whose last workgroups start when the first of the
// round before end; above 8,192 the same holds for shares of 32.  us, scenes
// as generated / with a quarter of the returns within 12 m / cluttered, every
// mission a slalom (two launches; shares of 64; the rest by 32; over all CUs):
//   34,000  51.4 / 55.3 / 118.9  31.4 / 35.7 / 133.8  29.7 / 33.6 / 110.2  30.0 / 33.6 / 90.3
//   39,999  54.8 / 58.3 / 133.0  32.7 / 37.0 / 135.3  32.2 / 36.4 / 112.0  33.3 / 37.8 / 110.8
//   45,000  57.8 / 61.3 / 144.0  35.4 / 39.5 / 135.9  37.5 / 41.4 / 131.7  36.3 / 41.5 / 126.6
//   70,000  89.8 / 93.4 / 220.6  50.0 / 55.7 / 207.1  49.6 / 55.0 / 185.3  50.9 / 56.0 / 176.8
// (Equal shares over both rounds lose: 39,999 at 40 each cluttered 45.2 us for
// 40.7, since a CU's last workgroup alone runs faster than two.)
constexpr unsigned kRestShare = 32;
constexpr size_t kRoundRows = 64 * kRoundBlocks, kRestRows = kRestShare * kCus;
constexpr int kPoolWaves = kControlThreads / 64;

// The inputs of N environments in LDS: obs[0..47], mission[0..9], the scan
// result, and for the actor obs[4144..4147].  Odd row pitches put the rows a
// wave reads (64 lanes, or 16 quads) on different LDS banks.
constexpr int kStageObs = 48, kStageObsPitch = 49, kStageMissionPitch = 11, kStageScanPitch = 9;
template <int N>
struct Stage {
    float obs[N][kStageObsPitch];
    float mission[N][kStageMissionPitch];
    float scan[N][kStageScanPitch];
    float tail[N][5];
};

// Stages environments base .. base + N - 1, every load issued at once and
// coalesced over the rows' first 192 bytes, so that the chains read LDS: read
// from global memory at their points of use, the values came in a dozen
// dependent round trips.  PARKED: also the scan results parked in the prior
// rows.  Rows past the batch end re-read the last row; nothing uses them.
template <int N, bool TAIL, bool PARKED>
__device__ __forceinline__ void stage_inputs(const OnboardRows &rows, size_t base, Stage<N> &stage,
                                             int tid) {
    constexpr int kThreads = kControlThreads;
    auto row_of = [&](int e) {
        const size_t env = base + (size_t)e;
        return env < rows.batch ? env : rows.batch - 1;
    };
    constexpr int kObsLoads = (N * kStageObs + kThreads - 1) / kThreads;
    constexpr int kMissionLoads = (N * 10 + kThreads - 1) / kThreads;
    constexpr int kScanLoads = (N * 7 + kThreads - 1) / kThreads;
    // Every thread issues all its loads unconditionally (an index past the
    // stage re-reads the stage's last value), so they leave at once.
    float vo[kObsLoads], vm[kMissionLoads], vs[kScanLoads], vt = 0.0f;
#pragma unroll
    for (int k = 0; k < kObsLoads; ++k) {
        const int idx = min(tid + kThreads * k, N * kStageObs - 1);
        const int e = idx / kStageObs, i = idx - kStageObs * e;
        vo[k] = reinterpret_cast<const float *>(rows.obs + row_of(e) * rows.obs_stride)[i];
    }
#pragma unroll
    for (int k = 0; k < kMissionLoads; ++k) {
        const int idx = min(tid + kThreads * k, N * 10 - 1);
        const int e = idx / 10, i = idx - 10 * e;
        vm[k] = reinterpret_cast<const float *>(rows.mission + row_of(e) * rows.mission_stride)[i];
    }
    if (PARKED) {
#pragma unroll
        for (int k = 0; k < kScanLoads; ++k) {
            const int idx = min(tid + kThreads * k, N * 7 - 1);
            const int e = idx / 7, i = idx - 7 * e;
            vs[k] = rows.prior[row_of(e) * 15 + i];
        }
    }
    if (TAIL) {
        const int idx = min(tid, N * 4 - 1);
        const int e = idx / 4;
        vt = reinterpret_cast<const float *>(rows.obs +
                                             row_of(e) * rows.obs_stride)[4144 + idx - 4 * e];
    }
#pragma unroll
    for (int k = 0; k < kObsLoads; ++k) {
        const int idx = tid + kThreads * k;
        const int e = idx / kStageObs;
        if (idx < N * kStageObs) stage.obs[e][idx - kStageObs * e] = vo[k];
    }
#pragma unroll
    for (int k = 0; k < kMissionLoads; ++k) {
        const int idx = tid + kThreads * k;
        const int e = idx / 10;
        if (idx < N * 10) stage.mission[e][idx - 10 * e] = vm[k];
    }
    if (PARKED) {
#pragma unroll
        for (int k = 0; k < kScanLoads; ++k) {
            const int idx = tid + kThreads * k;
            const int e = idx / 7;
            if (idx < N * 7) stage.scan[e][idx - 7 * e] = vs[k];
        }
    }
    if (TAIL && tid < N * 4) stage.tail[tid / 4][tid % 4] = vt;
}

template <int N>
__device__ __forceinline__ void stage_result(Stage<N> &stage, int e, const ScanResult &r) {
    float *sc = stage.scan[e];
    sc[0] = r.min_r;
    sc[1] = r.min_r_dx;
    sc[2] = r.min_r_dy;
    sc[3] = r.min_dx_c;
    sc[4] = r.cluster_y_sum;
    sc[5] = __int_as_float(r.min_ray);
    sc[6] = __int_as_float(r.cluster_count);
}

template <int N>
__device__ __forceinline__ ScanResult staged_result(const Stage<N> &stage, int e) {
    const float *sc = stage.scan[e];
    ScanResult s;
    s.min_r = sc[0];
    s.min_r_dx = sc[1];
    s.min_r_dy = sc[2];
    s.min_dx_c = sc[3];
    s.cluster_y_sum = sc[4];
    s.min_ray = __float_as_int(sc[5]);
    s.cluster_count = __float_as_int(sc[6]);
    // Read from LDS at once, like the other inputs.
    asm volatile("" : "+v"(s.min_r), "+v"(s.min_r_dx), "+v"(s.min_r_dy), "+v"(s.min_dx_c),
                 "+v"(s.cluster_y_sum), "+v"(s.min_ray), "+v"(s.cluster_count));
    return s;
}

__device__ __forceinline__ void store_scan_diag(float *d, const ScanResult &s) {
    d[0] = s.min_r;
    d[1] = (float)s.min_ray;
    d[2] = s.min_dx_c;
    d[3] = (float)s.cluster_count;
    d[4] = s.cluster_y_sum;
}

// Where an environment's tactical and prior values go: their rows, and for
// the actor their copies in proprio and mission_vec.
struct OutputRows {
    float *tactical, *prior, *proprio, *mission_vec;
    __device__ __forceinline__ OutputRows(const OnboardRows &rows, size_t env)
        : tactical(rows.tactical + env * 24), prior(rows.prior + env * 15),
          proprio(rows.proprio ? rows.proprio + env * 91 + 52 : nullptr),
          mission_vec(rows.proprio ? rows.mission_vec + env * 49 + 10 : nullptr) {}
    __device__ __forceinline__ void arm(int a, const ArmOutputs<true> &n) const {
        prior[a] = n.throttle[0];
        prior[4 + a] = n.outer[0];
        prior[8 + a] = n.inner[0];
        if (proprio) {
            proprio[24 + a] = n.throttle[0];
            proprio[28 + a] = n.outer[0];
            proprio[32 + a] = n.inner[0];
            mission_vec[24 + a] = n.throttle[0];
            mission_vec[28 + a] = n.outer[0];
            mission_vec[32 + a] = n.inner[0];
        }
    }
};

// One wave: the tactical features, the cannon and the BWB law of the 16
// environments from `first` of the stage on, a quad of lanes each.
template <int N>
__device__ __forceinline__ void support_wave(const OnboardRows &rows, size_t base,
                                             const Stage<N> &stage, int first, int lane) {
    const int a = lane & 3, slot = first + (lane >> 2);
    const size_t env = base + (size_t)slot;
    if (env >= rows.batch) return;
    ChainInputs<true> in = chain_inputs<true>(stage.obs[slot], stage.mission[slot], a);
    const bool wild = wild_inputs(in), tame = __builtin_amdgcn_ballot_w64(wild) == 0;
    const OutputRows out(rows, env);
    // Lane a of the quad writes features 6a .. 6a + 5.
    float t[6];
    {
        float v[24];
        if (tame) tactical_values<true, true>(in, wild, a, v);
        else tactical_values<false, true>(in, wild, a, v);
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            t[k] = tactical_out(quad_pick(a, v[k], v[6 + k], v[12 + k], v[18 + k]));
        }
    }
#pragma unroll
    for (int i = 0; i < 6; ++i) out.tactical[6 * a + i] = t[i];
    if (out.proprio) {
#pragma unroll
        for (int i = 0; i < 6; ++i) {
            out.proprio[6 * a + i] = t[i];
            out.mission_vec[6 * a + i] = t[i];
        }
    }
    if (!tame) controller_inputs(in);
    const MissionFlags f = mission_flags(in.m);
    const GunOutputs<true> g = tame ? gunnery_values<true, true>(in, wild, f, a)
                                    : gunnery_values<false, true>(in, wild, f, a);
    if (f.bwb) out.arm(a, g.arm);
    if (a == 0) {
        out.prior[12] = g.az;
        out.prior[13] = g.el;
        out.prior[14] = g.fire;
        if (out.proprio) {
            out.proprio[36] = g.az;
            out.proprio[37] = g.el;
            out.proprio[38] = g.fire;
            out.mission_vec[36] = g.az;
            out.mission_vec[37] = g.el;
            out.mission_vec[38] = g.fire;
        }
    }
}

// One wave: the flight controller of the 16 environments from `first` on.
// `wait` returns when their scan results are in the stage.
template <int N, class Wait>
__device__ __forceinline__ void flight_wave(const OnboardRows &rows, size_t base,
                                            const Stage<N> &stage, int first, int lane, Wait wait) {
    const int a = lane & 3, slot = first + (lane >> 2);
    const size_t env = base + (size_t)slot;
    if (env >= rows.batch) return;
    ChainInputs<true> in = chain_inputs<true>(stage.obs[slot], stage.mission[slot], a);
    const bool wild = wild_inputs(in), tame = __builtin_amdgcn_ballot_w64(wild) == 0;
    if (!tame) controller_inputs(in);
    const MissionFlags f = mission_flags(in.m);
    ScanResult s;
    auto fetch = [&]() {
        wait();
        s = staged_result(stage, slot);
        return s;
    };
    const ArmOutputs<true> n = tame ? flight_values<true, true>(in, wild, f, a, fetch)
                                    : flight_values<false, true>(in, wild, f, a, fetch);
    if (!f.bwb) OutputRows(rows, env).arm(a, n);  // a BWB mission's are the support wave's
    if (rows.diag && a == 0) store_scan_diag(rows.diag + env * 5, s);
}

// The same for 64 staged environments, one lane each: three waves of a
// workgroup, one for each part, write the rows in LDS, from where the
// workgroup stores them coalesced.
struct LaneRows {
    float tactical[64][25];
    float prior[64][15];
    __device__ __forceinline__ void arms(int lane, const ArmOutputs<false> &n) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            prior[lane][i] = n.throttle[i];
            prior[lane][4 + i] = n.outer[i];
            prior[lane][8 + i] = n.inner[i];
        }
    }
};

__device__ __forceinline__ void tactical_lanes(const Stage<64> &stage, int lane, LaneRows &out) {
    const ChainInputs<false> in = chain_inputs<false>(stage.obs[lane], stage.mission[lane], 0);
    const bool wild = wild_inputs(in);
    float v[24];
    if (__builtin_amdgcn_ballot_w64(wild) == 0) tactical_values<true, false>(in, wild, 0, v);
    else tactical_values<false, false>(in, wild, 0, v);
#pragma unroll
    for (int k = 0; k < 24; ++k) out.tactical[lane][k] = tactical_out(v[k]);
}

__device__ __forceinline__ void gunnery_lanes(const Stage<64> &stage, int lane, LaneRows &out) {
    ChainInputs<false> in = chain_inputs<false>(stage.obs[lane], stage.mission[lane], 0);
    const bool wild = wild_inputs(in), tame = __builtin_amdgcn_ballot_w64(wild) == 0;
    if (!tame) controller_inputs(in);
    const MissionFlags f = mission_flags(in.m);
    const GunOutputs<false> g = tame ? gunnery_values<true, false>(in, wild, f, 0)
                                     : gunnery_values<false, false>(in, wild, f, 0);
    out.prior[lane][12] = g.az;
    out.prior[lane][13] = g.el;
    out.prior[lane][14] = g.fire;
    if (f.bwb) out.arms(lane, g.arm);
}

__device__ __forceinline__ void flight_lanes(const Stage<64> &stage, int lane, LaneRows &out,
                                             float *diag) {
    ChainInputs<false> in = chain_inputs<false>(stage.obs[lane], stage.mission[lane], 0);
    const bool wild = wild_inputs(in), tame = __builtin_amdgcn_ballot_w64(wild) == 0;
    if (!tame) controller_inputs(in);
    const MissionFlags f = mission_flags(in.m);
    auto fetch = [&] { return staged_result(stage, lane); };
    const ArmOutputs<false> n = tame ? flight_values<true, false>(in, wild, f, 0, fetch)
                                     : flight_values<false, false>(in, wild, f, 0, fetch);
    if (!f.bwb) out.arms(lane, n);
    if (diag) store_scan_diag(diag, staged_result(stage, lane));
}

// One wave: the actor's symlog scalars and mission values of `Count`
// environments first, first + step, ... of the stage.  Lane l's input:
// obs[l] (l < 48), obs[4144 + l - 48] (l < 52), mission[l - 52] (l < 62).
template <int Count, int N>
__device__ __forceinline__ void scalars_wave(const OnboardRows &rows, size_t base,
                                             const Stage<N> &stage, int first, int step,
                                             int lane) {
    const int lo = min(lane, kStageObs - 1), lt = min(max(lane - 48, 0), 3),
              lm = min(max(lane - 52, 0), 9);
    // All inputs are read first, so the chains are independent; rows past
    // the stage or the batch end (staged as copies of the last row) store
    // nothing.
    float raw[Count];
#pragma unroll
    for (int j = 0; j < Count; ++j) {
        const int e = min(first + step * j, N - 1);
        raw[j] = lane < 48 ? stage.obs[e][lo]
                           : (lane < 52 ? stage.tail[e][lt] : stage.mission[e][lm]);
    }
#pragma unroll
    for (int j = 0; j < Count; ++j) {
        const int e = first + step * j;
        const size_t env = base + (size_t)e;
        const bool valid = e < N && env < rows.batch;
        const size_t row = valid ? env : base;
        actor_scalars(raw[j], lane, rows.proprio + row * 91, rows.mission_vec + row * 49, valid);
    }
}

// Phase 2 of the actor entry's two-stream form: the tactical features, the
// controller and the actor's scalars from the parked scan results.  A
// workgroup covers 64 environments: waves 0..3 run the flight controller,
// waves 4..7 the tactical features, the cannon and the BWB law, each on one
// quad of lanes per environment (16 per wave), so every SIMD holds one wave
// of each; the latter then write the symlog scalars and mission values, one
// row per store (on the scan waves they cost the scan kernel 6 µs and the
// plane kernel of the next call 6 µs more).
//
// The time of the chains is their instruction count (onboard_math.h), so they
// are written without branches (conditions are formed first and values
// selected; as nested conditionals they became 130 branches, with the
// computation inside and five instructions of mask handling each), take short
// forms of the functions, and have a form for tame inputs without the
// reference's checks for infinities and NaN.  Cycles of a workgroup's chains
// at 1,000 environments, before these and after: 16,800 in the flight wave
// that held BWB missions (13,700 in the others) and 4,800 in the tactical
// waves -> 7,000 and 11,600.
//   * One pass per workgroup, without a grid-stride loop: in a loop the
//     compiler kept 64-bit coefficients and literals in registers across it,
//     256 of them; without it the chains fit in 128.
__global__ __launch_bounds__(kControlThreads) __attribute__((amdgpu_waves_per_eu(4)))
void actor_control_kernel(OnboardRows rows) {
    __shared__ Stage<64> stage;
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const size_t base = ((size_t)blockIdx.y * gridDim.x + blockIdx.x) * 64;
    if (base >= rows.batch) return;
    stage_inputs<64, true, true>(rows, base, stage, tid);
    __syncthreads();
    if (w < kControlWaves) {
        flight_wave(rows, base, stage, 16 * w, lane, [] {});
    } else {
        support_wave(rows, base, stage, 16 * (w - kControlWaves), lane);
        scalars_wave<16>(rows, base, stage, 16 * (w - kControlWaves), 1, lane);
    }
}

// The onboard entry, and the actor entry's small batches: the scan, the
// tactical features and the controller of G groups of 16 environments in one
// workgroup of eight waves.
//   * G = 1, 2: waves 0 .. G-1 run the flight controllers, waves G .. 2G-1
//     the tactical features, cannon and BWB law, which need no scan; the
//     others scan, and the support waves join them when they are done.
//   * G = 4: all waves scan, then three run the flight controllers, the
//     tactical features and the cannon and BWB law, one lane per environment,
//     and all store the rows.  Two workgroups fit a CU and fill its issue
//     slots, so instructions count and not the chain's length: one lane per
//     environment takes 4,100 for 64 environments where quads take 10,800
//     (27.3 -> 25.9 us at 32,768 environments, 54.4 -> 52.1 at 65,536
//     cluttered; below 16,384 the quads' shorter chains win).
//   * Wave 7 forms each environment's frame and need (lane e), stages the
//     empty result of those whose mission uses no scan result and enters the
//     others in a pool in LDS, corridor scans (the longest) first.  The
//     scanning waves take entries one at a time, the next one taken before
//     the current one is scanned so that its ranges are requested as far as
//     its need goes.  Which wave scans which environment varies from call to
//     call; each result depends only on its environment.
//   * The flight waves form what does not depend on the scan and then wait
//     until their group's results are staged: wave 7 publishes each group's
//     count, every scanner takes its result off it.  The waves of a workgroup
//     are resident together and no scanner waits for a flight wave, so the
//     wait ends.
struct alignas(16) PoolEntry {
    float r[9], py;
    unsigned env;
    int need;
};

template <int G>
struct OnboardLds {
    RayPlanes rays;
    u32x2 lists[kPoolWaves][kListCap + 64];  // + a spare entry per lane
    PoolEntry pool[16 * G];
    Stage<16 * G> stage;
    int count, next, ready;
    int left[G];  // results the group still lacks, once ready
};

template <int G, bool SCALARS>
__device__ __forceinline__ void onboard_block(const OnboardRows &rows, size_t base,
                                              OnboardLds<G> &s) {
    constexpr int N = 16 * G, kThreads = kControlThreads;
    constexpr bool kRoles = 2 * G < kPoolWaves;
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    stage_inputs<N, SCALARS, false>(rows, base, s.stage, tid);
    for (int i = tid; i < 1536; i += kThreads) {
        s.rays.d[0][i] = kRayDir[i * 3 + 0];
        s.rays.d[1][i] = kRayDir[i * 3 + 1];
        s.rays.d[2][i] = kRayDir[i * 3 + 2];
    }
    if (tid == 0) {
        s.next = 0;
        s.ready = 0;
    }
    __syncthreads();
    auto spin = [](int *word, int until) {
        while (__hip_atomic_load(word, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) != until)
            __builtin_amdgcn_s_sleep(1);
    };
    if (kRoles && w < G) {
        flight_wave(rows, base, s.stage, 16 * w, lane, [&] {
            spin(&s.ready, 1);
            spin(&s.left[w], 0);
        });
        return;
    }
    auto obs_of = [&](int e) {
        return reinterpret_cast<const float *>(rows.obs + (base + (size_t)e) * rows.obs_stride);
    };
    if (w == kPoolWaves - 1) {
        const int e = lane & (N - 1);
        const bool valid = (N == 64 || lane < N) && base + (size_t)e < rows.batch;
        FrameObs v{s.stage.obs[e][1], s.stage.obs[e][6], s.stage.obs[e][7], s.stage.obs[e][8],
                   s.stage.obs[e][9], s.stage.mission[e][4], s.stage.mission[e][5]};
        const ScanFrame f = scan_frame(v);
        const int need = rows.diag ? kNeedAll : scan_need(v.m4, v.m5);
        const bool entered = valid && need != kNeedNone;
        if (valid && !entered)
            stage_result(s.stage, e, ScanResult{30.0f, 0.0f, 0.0f, 30.0f, 0.0f, -1, 0, 0});
        const bool front = (need & kNeedCorridor) != 0;
        const uint64_t mf = __builtin_amdgcn_ballot_w64(entered && front);
        const uint64_t mb = __builtin_amdgcn_ballot_w64(entered && !front);
        if (entered) {
            const uint64_t mine = front ? mf : mb;
            const unsigned rank = __builtin_amdgcn_mbcnt_hi(
                (unsigned)(mine >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mine, 0u));
            PoolEntry &p = s.pool[(front ? 0u : (unsigned)__builtin_popcountll(mf)) + rank];
            p.env = (unsigned)e;
            p.need = need;
#pragma unroll
            for (int k = 0; k < 9; ++k) p.r[k] = f.r[k];
            p.py = f.py;
        }
        if (lane == 0) {
            s.count = (int)__builtin_popcountll(mf | mb);
#pragma unroll
            for (int g = 0; g < G; ++g)
                s.left[g] = __builtin_popcount((unsigned)((mf | mb) >> (16 * g)) & 0xffffu);
        }
        // The wave's LDS writes are in order; the release waits for them.
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        if (lane == 0)
            __hip_atomic_store(&s.ready, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    if (kRoles && w < 2 * G) support_wave(rows, base, s.stage, 16 * (w - G), lane);
    spin(&s.ready, 1);
    const int count = __builtin_amdgcn_readfirstlane(s.count);
    auto take = [&]() {
        int t = 0;
        if (lane == 0)
            t = __hip_atomic_fetch_add(&s.next, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        return __builtin_amdgcn_readfirstlane(t);
    };
    auto entry = [&](int t, int &slot, int &need) {
        slot = __builtin_amdgcn_readfirstlane((int)s.pool[t].env);
        need = __builtin_amdgcn_readfirstlane(s.pool[t].need);
    };
    int t = take();
    if (t < count) {
        int slot, need;
        entry(t, slot, need);
        float rg[kScanRays];
        load_ranges(obs_rsrc(obs_of(slot), true), obs_rsrc(obs_of(slot), (need & kNeedCorridor) != 0),
                    lane, rg);
        for (;;) {
            ScanFrame f;
#pragma unroll
            for (int i = 0; i < 9; ++i) f.r[i] = s.pool[t].r[i];
            f.py = s.pool[t].py;
            const int t_next = take();
            const bool has_next = t_next < count;
            int next_slot = slot, next_need = kNeedNone;
            if (has_next) entry(t_next, next_slot, next_need);
            const float *next_obs = obs_of(next_slot);
            ScanResult r;
            scan_env(rg, s.rays, f, obs_rsrc(next_obs, has_next),
                     obs_rsrc(next_obs, has_next && (next_need & kNeedCorridor)), lane, s.lists[w],
                     r, need);
            if (lane == 0) {
                stage_result(s.stage, slot, r);
                __hip_atomic_fetch_sub(&s.left[slot / 16], 1, __ATOMIC_RELEASE,
                                       __HIP_MEMORY_SCOPE_WORKGROUP);
            }
            if (!has_next) break;
            t = t_next;
            slot = next_slot;
            need = next_need;
        }
    }
    if constexpr (!kRoles) {
        // Rows past the batch end (copies of the last one, staged without a
        // scan result) are computed and not stored.
        static_assert(G == 4 && !SCALARS && sizeof(LaneRows) <= sizeof(s.lists));
        LaneRows &out = *reinterpret_cast<LaneRows *>(&s.lists[0][0]);
        __syncthreads();
        const size_t rows_here = rows.batch - base < 64 ? rows.batch - base : 64;
        if (w == 0) {
            flight_lanes(s.stage, lane, out,
                         rows.diag && (size_t)lane < rows_here ? rows.diag + (base + lane) * 5
                                                               : nullptr);
        } else if (w == 1) {
            tactical_lanes(s.stage, lane, out);
        } else if (w == 2) {
            gunnery_lanes(s.stage, lane, out);
        }
        __syncthreads();
        for (int i = tid; i < (int)rows_here * 24; i += kThreads)
            rows.tactical[base * 24 + i] = out.tactical[i / 24][i % 24];
        for (int i = tid; i < (int)rows_here * 15; i += kThreads)
            rows.prior[base * 15 + i] = out.prior[i / 15][i % 15];
    }
    if (SCALARS) {
        constexpr int kWaves = kPoolWaves - G, kEach = (N + kWaves - 1) / kWaves;
        scalars_wave<kEach>(rows, base, s.stage, w - G, kWaves, lane);
    }
}

// `share` environments per workgroup, at most 16 G; with REST (G = 4) 64 in the
// batch's whole rounds and kRestShare after them.
template <int G, bool REST = false>
__global__ __launch_bounds__(kControlThreads) __attribute__((amdgpu_waves_per_eu(4)))
void onboard_kernel(OnboardRows rows, unsigned share) {
    __shared__ OnboardLds<G> lds;
    const size_t block = (size_t)blockIdx.y * gridDim.x + blockIdx.x;
    size_t base = block * share;
    if constexpr (REST) {
        const size_t whole = rows.batch / kRoundRows * kRoundBlocks;
        share = block < whole ? 64 : kRestShare;
        base = 64 * block - (block < whole ? 0 : (64 - kRestShare) * (block - whole));
    }
    if (base >= rows.batch) return;
    if (rows.batch - base > share) rows.batch = base + share;  // this workgroup's end
    onboard_block<G, false>(rows, base, lds);
}

// Environments per workgroup of a batch that one round of workgroups takes.
size_t share_of(size_t batch) {
    const size_t blocks = batch <= 16 * kCus ? kCus : kRoundBlocks;
    const size_t share = (batch + blocks - 1) / blocks;
    return share < kMinShare ? kMinShare : share;
}

// A grid of `want` workgroups.
dim3 wide_grid(size_t want) {
    return dim3((unsigned)(want < kControlGridX ? want : kControlGridX),
                (unsigned)((want + kControlGridX - 1) / kControlGridX));
}

}  // namespace

extern "C" int tb_hip_onboard_tactical_prior_device(const float *obs, const float *mission,
                                                    float *tactical, float *prior, float *diag,
                                                    size_t batch_size, void *stream) {
    if (!obs || !mission || !tactical || !prior || batch_size == 0 || batch_size > kMaxBatch)
        return 0;
    OnboardRows rows;
    rows.obs = reinterpret_cast<const unsigned char *>(obs);
    rows.obs_stride = 4148 * sizeof(float);
    rows.mission = reinterpret_cast<const unsigned char *>(mission);
    rows.mission_stride = 10 * sizeof(float);
    rows.tactical = tactical;
    rows.prior = prior;
    rows.diag = diag;
    rows.proprio = nullptr;
    rows.mission_vec = nullptr;
    rows.lidar = nullptr;
    rows.batch = batch_size;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    (void)hipGetLastError();
    const size_t rest = batch_size % kRoundRows;
    if (batch_size > kRoundRows && rest != 0 && rest <= kRestRows) {
        const size_t blocks = (batch_size - rest) / 64 + (rest + kRestShare - 1) / kRestShare;
        onboard_kernel<4, true><<<wide_grid(blocks), kControlThreads, 0, s>>>(rows, kRestShare);
        return hipGetLastError() == hipSuccess;
    }
    const size_t want = share_of(batch_size), share = want < 64 ? want : 64;
    const dim3 grid = wide_grid((batch_size + share - 1) / share);
    if (share <= 16)
        onboard_kernel<1><<<grid, kControlThreads, 0, s>>>(rows, (unsigned)share);
    else if (share <= 32)
        onboard_kernel<2><<<grid, kControlThreads, 0, s>>>(rows, (unsigned)share);
    else
        onboard_kernel<4><<<grid, kControlThreads, 0, s>>>(rows, (unsigned)share);
    return hipGetLastError() == hipSuccess;
}

// ---------------------------------------------------------------------------
// The 618M actor's sensor preparation, fused (reference
// src/network/network_gpu.cu:274-304 scalar_inputs, :467-479 lidar_channels,
// :480-483 camera_luma, launched back to back at :1446-1451).  One workgroup
// per environment streams the LiDAR block once into the six channel planes
// and the cameras once into luma: LiDAR in 16-byte loads, camera bytes in
// 4-byte loads so that each lane's 4 luma values are one float4 and every
// store instruction writes 1 KiB of consecutive output.  In the two-stream
// form the scan kernel writes the channels of the rays it reads (elevation
// rows 0..5) and the plane kernel only those of rows 6..15, so each LiDAR
// range is read from HBM once.  The onboard workgroups also write each
// environment's 52 symlog scalars and mission values, and the copies of
// tactical / prior.  In large batches, fusing the scan into the streaming
// workgroups was measured
// slower: next to saturated HBM traffic the scan's dependent loads stall.  Luma is
// the reference's `(float)b * (1.0f / 255.0f) - 0.5f` as its CUDA build
// evaluates it: nvcc contracts the product and difference into one fused
// multiply-add by default, so it is one explicit fma here (this file is built
// without automatic contraction, like every restatement of the reference's
// arithmetic here).

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// Threads of a head whose LiDAR float4 lies in the scan's elevation rows
// 0..5 (6 rows of 32 float4).
constexpr int kScanRowThreads = 6 * 128 / 4;

struct ActorRows {
    const float *obs;
    const unsigned char *cameras;
    float *lidar, *luma;
    size_t batch;
};

__device__ __forceinline__ f32x4 lidar_channel4(f32x4 r, int kind) {
    f32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = lidar_channel(r[e], kind);
    return o;
}

// Four camera bytes as luma.
__device__ __forceinline__ f32x4 luma4(unsigned w) {
    f32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e)
        o[e] = __builtin_fmaf((float)((w >> (8 * e)) & 0xffu), 1.0f / 255.0f, -0.5f);
    return o;
}

// One 1,024-thread workgroup per environment: thread t loads LiDAR float4 t
// and camera words t + 1024 k, and every store instruction of the
// workgroup writes 16 KB of consecutive output (the two heads' planes of a
// channel kind are adjacent, as are consecutive luma float4).  With the
// XCD-contiguous environment order a pure fill of this pattern reaches
// 6.3 TB/s on MI355X, against 5.5 TB/s for 256-thread workgroups in
// dispatch order.
// One 16-byte store into an environment's output block (`bytes` long) with
// cache policy nt + sc1.  Entry at 16,384 environments on MI355X, one
// workgroup per CU, identical outputs: default policy 461.5 us, nt 450.7,
// sc0 + nt 449.9, sc1 442.4, sc0 + sc1 442.4, nt + sc1 434.1, sc0 + nt +
// sc1 434.3 (with two workgroups per CU: default 440.3 us for the plane
// kernel, sc1 416.7).
__device__ __forceinline__ void store_plane(float *block, unsigned bytes, unsigned index, f32x4 v) {
    __builtin_amdgcn_raw_buffer_store_b128(
        __builtin_bit_cast(u32x4, v),
        __builtin_amdgcn_make_buffer_rsrc(block, (short)0, (int)bytes, 0x00020000), index * 16u,
        0, kStorePolicy);
}

__global__ __launch_bounds__(kStreamThreads) void actor_stream_kernel(ActorRows rows) {
    const int t = threadIdx.x;
    for (size_t env = xcd_contiguous(blockIdx.x, gridDim.x); env < rows.batch;
         env += gridDim.x) {
        // float4 t is bins 4(t%512).. of head t/512, elevation row
        // (t%512)/32.  The scan kernel writes rows 0..5
        // (threads with t%512 < 192, whole waves) and this kernel the other
        // ten.
        const bool lidar = rows.lidar && (t & 511) >= kScanRowThreads;
        f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
        if (lidar)
            v = __builtin_nontemporal_load(
                reinterpret_cast<const f32x4 *>(rows.obs + env * 4148 + 48) + t);
        unsigned px[4];
        if (rows.luma) {
            const unsigned *cam = reinterpret_cast<const unsigned *>(rows.cameras + env * 16384);
#pragma unroll
            for (int k = 0; k < 4; ++k) px[k] = __builtin_nontemporal_load(cam + t + 1024 * k);
        }
        if (lidar) {
            // Head h feeds channels h, h+2, h+4.
            float *dst = rows.lidar + env * 12288;
            const int head = t >> 9, q = t & 511;
#pragma unroll
            for (int kind = 0; kind < 3; ++kind)
                store_plane(dst, 12288 * 4, (head + 2 * kind) * 512 + q, lidar_channel4(v, kind));
        }
        if (rows.luma) {
            float *dst = rows.luma + env * 16384;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                store_plane(dst, 16384 * 4, t + 1024 * k, luma4(px[k]));
            }
        }
    }
}

// The same planes by half a workgroup: 512 threads, each both heads' float4 t
// and camera words t + 512 k.
__device__ __forceinline__ void actor_planes_block(const ActorRows &rows, size_t env) {
    const int t = threadIdx.x;
    f32x4 v[2];
    if (rows.lidar) {
        const f32x4 *src = reinterpret_cast<const f32x4 *>(rows.obs + env * 4148 + 48);
#pragma unroll
        for (int head = 0; head < 2; ++head) v[head] = __builtin_nontemporal_load(src + 512 * head + t);
    }
    unsigned px[8];
    if (rows.luma) {
        const unsigned *cam = reinterpret_cast<const unsigned *>(rows.cameras + env * 16384);
#pragma unroll
        for (int k = 0; k < 8; ++k) px[k] = __builtin_nontemporal_load(cam + t + 512 * k);
    }
    if (rows.lidar) {
        float *dst = rows.lidar + env * 12288;
#pragma unroll
        for (int kind = 0; kind < 3; ++kind)
#pragma unroll
            for (int head = 0; head < 2; ++head)
                store_plane(dst, 12288 * 4, (head + 2 * kind) * 512 + t,
                            lidar_channel4(v[head], kind));
    }
    if (rows.luma) {
        float *dst = rows.luma + env * 16384;
#pragma unroll
        for (int k = 0; k < 8; ++k) store_plane(dst, 16384 * 4, t + 512 * k, luma4(px[k]));
    }
}

// The onboard features and scalars of one workgroup's environments: SPREAD a
// share below 16, else 16 (a constant: the end of a share held in registers
// cost the full workgroups 0.2 us and beside plane workgroups up to 4%).
template <bool SPREAD>
__device__ __forceinline__ void actor_share(OnboardRows &rows, size_t block, unsigned share,
                                            OnboardLds<1> &lds) {
    const size_t base = block * (SPREAD ? share : 16);
    if (base >= rows.batch) return;
    if (SPREAD && rows.batch - base > share) rows.batch = base + share;
    onboard_block<1, true>(rows, base, lds);
}

// The whole preparation of a small batch in one launch: the first
// `onboard_blocks` workgroups take a share of the environments' onboard
// features and scalars each (the longest chains start first), the others one
// environment's planes each.
template <bool SPREAD>
__global__ __launch_bounds__(kControlThreads) __attribute__((amdgpu_waves_per_eu(4)))
void actor_one_kernel(OnboardRows rows, ActorRows planes, unsigned onboard_blocks) {
    __shared__ OnboardLds<1> lds;
    if (blockIdx.x < onboard_blocks)
        actor_share<SPREAD>(rows, blockIdx.x, kMinShare, lds);
    else
        actor_planes_block(planes, blockIdx.x - onboard_blocks);
}

// The onboard features and scalars alone, for any batch.
template <bool SPREAD>
__global__ __launch_bounds__(kControlThreads) __attribute__((amdgpu_waves_per_eu(4)))
void actor_onboard_kernel(OnboardRows rows, unsigned share) {
    __shared__ OnboardLds<1> lds;
    actor_share<SPREAD>(rows, (size_t)blockIdx.y * gridDim.x + blockIdx.x, share, lds);
}

void launch_actor_onboard(const OnboardRows &rows, hipStream_t s) {
    const size_t share = share_of(rows.batch);
    if (share < 16)
        actor_onboard_kernel<true><<<wide_grid((rows.batch + share - 1) / share), kControlThreads,
                                     0, s>>>(rows, (unsigned)share);
    else
        actor_onboard_kernel<false><<<wide_grid((rows.batch + 15) / 16), kControlThreads, 0, s>>>(
            rows, 16);
}

// From kOverlapMinBatch environments the scan and control kernels run beside
// the plane kernel on a second stream of the device, forked from and joined
// back to the caller's stream.  The plane kernel is write-bound and keeps one
// workgroup per CU; the scan and control workgroups fit beside it, and their
// latency-bound chains overlap its streams.  It is the controller that gains
// most: the scan alone on the second stream, with the controller after the
// join, measured 437.9 against 433.0 us at 16,384 environments (before the
// split below).
//
// Split of the LiDAR channel planes: the scan kernel writes the channels of
// the 1,536 rays it reads (elevation rows 0..5 of each head) and the plane
// kernel only the other rows, so the entry reads every LiDAR range from HBM
// once instead of reading the scan rows twice (428.5 -> 412.5 us at 16,384).
// Without LiDAR channels the second stream runs the onboard kernel instead.
//
// Smaller batches take one launch (actor_one_kernel): the fork and join cost
// several microseconds, and the onboard workgroups are spread over CUs that
// also run plane workgroups.  Measured on one box, us (before: one stream and
// three launches up to 1,792 environments, two streams above; one launch; two
// streams with the split):
//       64   19.9    8.6    --       2,048   67.6   54.9   70.1
//      256   22.9   12.7    --       2,560   75.6   70.3   77.2
//    1,000   42.6   28.0   52.9      3,072   87.4   85.6   87.3
//    1,500   56.5   41.1   63.2      3,500   97.1   97.6   97.3
//                                    4,096  112.8  116.4  112.5
constexpr size_t kOverlapMinBatch = 3072;
// In that one launch the onboard workgroups take 8 environments each while the
// plane workgroups leave CUs idle, and 16 above, where they would hold more of
// the CUs' places (both planes, generated scenes / cluttered slaloms, us;
// three launches before, 16 and 8 each): 64 19.6 / 26.3, 8.0 / 26.9, 7.6 /
// 21.6; 512 28.4 / 35.5, 13.2 / 31.5, 12.6 / 25.6; 700 32.8 / 39.8, 15.8 /
// 33.5, 16.5 / 27.1; 3,071 86.8 / 86.8, 84.1 / 84.5, 87.3 / 89.2.
constexpr size_t kSpreadMax = 512;
constexpr int kMaxDevices = 64;

struct SideStream {
    std::mutex order;           // one fork ... join sequence at a time
    std::atomic<int> state{0};  // 0 not made, 1 ready, -1 creation failed
    hipStream_t stream = nullptr;
    hipEvent_t fork = nullptr, join = nullptr;
};
SideStream side_streams[kMaxDevices];

// The current device's side stream (default priority, non-blocking), made
// on first use.  nullptr when it cannot be made, and while `s` is being
// captured into a graph before it exists (a capture may use one made
// earlier: the fork and join events bring it into the capture).  A failed
// query or creation is cleared from the runtime's last error, so the call
// goes on with one stream and its own launch check stays meaningful.
SideStream *side_stream(hipStream_t s) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
        (void)hipGetLastError();
        return nullptr;
    }
    SideStream &ss = side_streams[dev];
    int state = ss.state.load(std::memory_order_acquire);
    if (state == 0) {
        hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(s, &capture) != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
        if (capture != hipStreamCaptureStatusNone) return nullptr;
        std::lock_guard<std::mutex> made(ss.order);
        state = ss.state.load(std::memory_order_acquire);
        if (state == 0) {
            const bool ok =
                hipStreamCreateWithFlags(&ss.stream, hipStreamNonBlocking) == hipSuccess &&
                hipEventCreateWithFlags(&ss.fork, hipEventDisableTiming) == hipSuccess &&
                hipEventCreateWithFlags(&ss.join, hipEventDisableTiming) == hipSuccess;
            state = ok ? 1 : -1;
            if (!ok) (void)hipGetLastError();
            ss.state.store(state, std::memory_order_release);
        }
    }
    return state == 1 ? &ss : nullptr;
}

}  // namespace

extern "C" int tb_hip_actor_inputs_device(const float *obs, const float *mission,
                                          const unsigned char *cameras, float *proprio,
                                          float *mission_vec, float *tactical, float *prior,
                                          float *lidar_channels, float *camera_luma,
                                          size_t batch_size, void *stream) {
    if (!obs || !mission || !proprio || !mission_vec || !tactical || !prior || batch_size == 0 ||
        batch_size > kMaxBatch || (camera_luma && !cameras))
        return 0;
    const uintptr_t align = reinterpret_cast<uintptr_t>(obs) |
                            reinterpret_cast<uintptr_t>(lidar_channels) |
                            reinterpret_cast<uintptr_t>(camera_luma) |
                            reinterpret_cast<uintptr_t>(cameras);
    if ((align & 15u) != 0) return 0;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    (void)hipGetLastError();
    const bool planes = lidar_channels || camera_luma;
    OnboardRows rows;
    rows.obs = reinterpret_cast<const unsigned char *>(obs);
    rows.obs_stride = 4148 * sizeof(float);
    rows.mission = reinterpret_cast<const unsigned char *>(mission);
    rows.mission_stride = 10 * sizeof(float);
    rows.tactical = tactical;
    rows.prior = prior;
    rows.diag = nullptr;
    rows.proprio = proprio;
    rows.mission_vec = mission_vec;
    rows.lidar = nullptr;
    rows.batch = batch_size;
    ActorRows ar;
    ar.obs = obs;
    ar.cameras = cameras;
    ar.lidar = lidar_channels;
    ar.luma = camera_luma;
    ar.batch = batch_size;
    if (!planes) {
        launch_actor_onboard(rows, s);
        return hipGetLastError() == hipSuccess;
    }
    if (batch_size < kOverlapMinBatch) {
        const bool spread = batch_size <= kSpreadMax;
        const unsigned n = (unsigned)batch_size, share = spread ? kMinShare : 16,
                       onboard_blocks = (n + share - 1) / share;
        if (spread)
            actor_one_kernel<true><<<onboard_blocks + n, kControlThreads, 0, s>>>(rows, ar,
                                                                                 onboard_blocks);
        else
            actor_one_kernel<false><<<onboard_blocks + n, kControlThreads, 0, s>>>(rows, ar,
                                                                                  onboard_blocks);
        return hipGetLastError() == hipSuccess;
    }
    SideStream *side = side_stream(s);
    std::unique_lock<std::mutex> order;
    if (side) {
        order = std::unique_lock<std::mutex>(side->order);
        if (hipEventRecord(side->fork, s) != hipSuccess ||
            hipStreamWaitEvent(side->stream, side->fork, 0) != hipSuccess)
            return 0;
    }
    // One workgroup per CU: the launch asks for more than half of the
    // CU's 160 KB of LDS, which the kernel does not use (by registers a
    // CU holds two; one measured 462.7 -> 445.0 us for the entry,
    // identical outputs: fewer requests in flight keep the write-bound
    // streams more efficient).
    constexpr unsigned kOneWorkgroupLds = (160 * 1024 / 2 + 1 + 1023) / 1024 * 1024;
    actor_stream_kernel<<<batch_size > kMaxBlocks ? kMaxBlocks : (unsigned)batch_size,
                          kStreamThreads, kOneWorkgroupLds, s>>>(ar);
    const hipStream_t beside = side ? side->stream : s;
    if (lidar_channels) {
        rows.lidar = lidar_channels;
        const size_t scan_want = (batch_size + kWavesPerBlock - 1) / kWavesPerBlock;
        actor_scan_kernel<<<scan_want > kScanBlocks ? kScanBlocks : (unsigned)scan_want,
                            kBlockThreads, 0, beside>>>(rows);
        actor_control_kernel<<<wide_grid((batch_size + 63) / 64), kControlThreads, 0, beside>>>(
            rows);
    } else {
        launch_actor_onboard(rows, beside);
    }
    const int ok = hipGetLastError() == hipSuccess;
    if (side && (hipEventRecord(side->join, side->stream) != hipSuccess ||
                 hipStreamWaitEvent(s, side->join, 0) != hipSuccess))
        return 0;
    return ok;
}
