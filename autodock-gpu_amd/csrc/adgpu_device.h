// adgpu_device.h -- gfx950 device code of the docking hot path (included by
// the kernel translation units k_*.hip; each instantiates its own kernels).
//
// Execution model (CDNA, 64-wide wavefronts):
//   * a "team" of TW lanes (TW = 16, 32 or 64) evaluates one individual, so a
//     wavefront carries 64/TW individuals; a workgroup stages the ligand
//     tables (pair records, torsion vectors) into LDS once and every team of
//     the workgroup shares them;
//   * team lane l owns atoms l, l+TW, ... (NC chunks) and walks each atom's
//     own torsion chain, so pose -> coordinates needs no barrier (the
//     reference's rotation list is a barrier per cycle, calcenergy.cl:232-275);
//   * team lane l owns genes l and l+TW (when TW = 32) for a whole local
//     search, so minimiser updates are register code; each gene lane also
//     evaluates the sine/cosine of its own angle once per evaluation;
//   * pairs are strided over the team; pair forces go to per-atom int32
//     fixed-point accumulators in LDS through ds_add (order independent);
//   * energies, forces and torques are summed with DPP row reductions and row
//     swaps or broadcasts, in one order whatever the lanes that need the sum;
//   * local searches run as persistent kernels: a team that finishes its
//     entity takes the next one from a global counter, so teams of one
//     wavefront never wait for each other and uneven searches balance out.
// The arithmetic of every device function follows the reference file:line
// given at its definition (ccsb-scripps/AutoDock-GPU v1.5, device/ = OpenCL).
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>

#include "adgpu_internal.h"

namespace adgpu {

#define DEV __device__ __forceinline__
// Workgroups of up to 1024 threads (choose_ls_shape).
// Waves per SIMD the register budget is sized for (4: at most 128 VGPRs).
#ifndef ADGPU_WAVES_PER_EU
#define ADGPU_WAVES_PER_EU 4
#endif
#define ADGPU_GROUP_KERNEL __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(ADGPU_WAVES_PER_EU)))

// common/calcenergy_basic.h
constexpr float kDegToRad = 0.0174533f;
constexpr float kPi = 3.14159265358979323846f;
constexpr float kTwoPi = 2.0f * kPi;
constexpr float kTermScale = 1024.0f;
constexpr float kOneOverTermScale = 1.0f / 1024.0f;
constexpr float kMaxTerm = 8192.0f;

// ---------------------------------------------------------------------------
// wavefront / team primitives
// ---------------------------------------------------------------------------
DEV int lane_id() { return (int)__lane_id(); }

// Orders LDS accesses of the lanes of one wavefront (no workgroup barrier).
DEV void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ZERO: lanes without a source read 0.
template <int CTRL, bool ZERO = false>
DEV float dpp(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, ZERO));
}
DEV float rdl(float v, int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l)); }
DEV int rdl_i(int v, int l) { return __builtin_amdgcn_readlane(v, l); }

template <int TW>
struct Team {
    static_assert(TW == 16 || TW == 32 || TW == 64, "team width");
    static constexpr int kPerWave = 64 / TW;
    static constexpr int kGPL = 64 / TW;          // genes per lane
    DEV static int lane() { return lane_id() & (TW - 1); }
    DEV static int slot() { return lane_id() / TW; }
    // Sum over the team; every lane of the team receives the same bits.
    // Rows of 16 lanes: xor 1, xor 2 (quad_perm), half-row mirror, row mirror;
    // then the row sums are combined with gfx950's row swaps: permlane16_swap
    // gives rows 2k and 2k+1 both (row 2k, row 2k+1), so both add
    // row 2k + row 2k+1 in that order; permlane32_swap does the same for the
    // two halves of the wavefront.
    // A 16-lane team is one row: the four DPP steps give its sum.
    DEV static float sum(float v) {
        v += dpp<0xB1>(v);
        v += dpp<0x4E>(v);
        v += dpp<0x141>(v);
        v += dpp<0x140>(v);
        if constexpr (TW == 16) return v;
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
        if constexpr (TW == 64) {
            const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
            v = __uint_as_float(h[0]) + __uint_as_float(h[1]);
        }
        return v;
    }
    // The same sum, the same bits, in the lanes of the team's last row only:
    // each row's last lane is broadcast to the next row, then the first half's
    // to the second, one instruction each where the row swaps take three.
    static constexpr int kTop = TW - 16;
    DEV static float sum_top(float v) {
        v += dpp<0xB1>(v);
        v += dpp<0x4E>(v);
        v += dpp<0x141>(v);
        v += dpp<0x140>(v);
        if constexpr (TW >= 32) v += dpp<0x142, true>(v);
        if constexpr (TW == 64) v += dpp<0x143, true>(v);
        return v;
    }
    // Value of team lane k (k uniform).
    DEV static float bcast(float v, int k) {
        if constexpr (TW == 16) {
            const float a = rdl(v, k), b = rdl(v, 16 + k), c = rdl(v, 32 + k), d = rdl(v, 48 + k);
            const int s = lane_id() >> 4;
            return s == 0 ? a : s == 1 ? b : s == 2 ? c : d;
        } else if constexpr (TW == 32) {
            return lane_id() < 32 ? rdl(v, k) : rdl(v, 32 + k);
        } else {
            return rdl(v, k);
        }
    }
    DEV static int bcast_i(int v, int k) {
        if constexpr (TW == 16) {
            const int a = rdl_i(v, k), b = rdl_i(v, 16 + k), c = rdl_i(v, 32 + k), d = rdl_i(v, 48 + k);
            const int s = lane_id() >> 4;
            return s == 0 ? a : s == 1 ? b : s == 2 ? c : d;
        } else if constexpr (TW == 32) {
            return lane_id() < 32 ? rdl_i(v, k) : rdl_i(v, 32 + k);
        } else {
            return rdl_i(v, k);
        }
    }
    // True when any lane of the wavefront has p set.
    DEV static bool any_in_wave(bool p) { return __ballot(p) != 0ull; }
};

// ---------------------------------------------------------------------------
// scalar helpers
// ---------------------------------------------------------------------------
DEV float fast_rcp(float x) { return __builtin_amdgcn_rcpf(x); }
DEV float fast_sqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
DEV float fast_rsq(float x) { return __builtin_amdgcn_rsqf(x); }

// max(x, lo) and min(x, hi) with a wave-uniform bound, as one instruction (the
// library forms first canonicalize both operands).  A NaN x gives the bound,
// as fmaxf and fminf do.
DEV float max_s(float x, float lo) {
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "s"(lo), "v"(x));
    return r;
}
DEV float min_s(float x, float hi) {
    float r;
    asm("v_min_f32 %0, %1, %2" : "=v"(r) : "s"(hi), "v"(x));
    return r;
}

// LDS atomic subtract without a returned value (ds_sub_u32; HIP's atomicSub
// would negate and add).
DEV void lds_sub(int* p, int v) {
    (void)__hip_atomic_fetch_sub(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// fmod_pi2, calcenergy.cl:86-91
DEV float fmod_pi2(float x) { return x - (float)((int)((1.0f / kTwoPi) * x)) * kTwoPi; }

// fast_acos, calcenergy.cl:93-108
DEV float fast_acos(float cosine) {
    const float a = 9.78056e-05f, b = -0.00104588f, c = 0.00418716f, d = -0.00314347f;
    const float e = 2.74084f, f = 0.370388f;
    const float o = -(a + b + c + d);
    float x = fabsf(cosine);
    float x2 = x * x, x3 = x2 * x, x4 = x3 * x;
    float ac = (((o * x4 + a) * x3 + b) * x2 + c) * x + d +
               e * fast_sqrt(2.0f - fast_sqrt(2.0f + 2.0f * x)) - f * fast_sqrt(2.0f - 2.0f * x);
    return copysignf(ac, cosine) + (cosine < 0.0f ? kPi : 0.0f);
}

// float2int_round of the clamped term, calcMergedEneGra.cl:30-35 (the half is
// moved toward zero before truncation, as the reference does).
// v - copysign(0.5, v) equals the reference's v + 0.5 * (v < 0 ? 1 : v > 0 ? -1 : 0)
// for every v, including +-0.
DEV int quant(float x) {
    const float v = fminf(kMaxTerm, fmaxf(-kMaxTerm, x));
    return (int)(v - copysignf(0.5f, v));
}

// quaternion_rotate, calcenergy.cl:119-127
DEV float3 qrot(float3 v, float4 q) {
    float zx = (q.y * v.z - q.z * v.y) * 2.0f;
    float zy = (q.z * v.x - q.x * v.z) * 2.0f;
    float zz = (q.x * v.y - q.y * v.x) * 2.0f;
    return make_float3(v.x + zx * q.w + (q.y * zz - q.z * zy),
                       v.y + zy * q.w + (q.z * zx - q.x * zz),
                       v.z + zz * q.w + (q.x * zy - q.y * zx));
}

// The same bits with q2 = (2 q.x, 2 q.y, 2 q.z, q.w): both cross products come
// out doubled, which is exact, the first as it is needed and the second halved
// by the addition that takes it -- three additions less.
DEV float3 qrot2(float3 v, float4 q2) {
#pragma clang fp contract(off)
    const float zx = fmaf(q2.y, v.z, -(q2.z * v.y));
    const float zy = fmaf(q2.z, v.x, -(q2.x * v.z));
    const float zz = fmaf(q2.x, v.y, -(q2.y * v.x));
    return make_float3(fmaf(0.5f, fmaf(q2.y, zz, -(q2.z * zy)), fmaf(zx, q2.w, v.x)),
                       fmaf(0.5f, fmaf(q2.z, zx, -(q2.x * zz)), fmaf(zy, q2.w, v.y)),
                       fmaf(0.5f, fmaf(q2.x, zy, -(q2.y * zx)), fmaf(zz, q2.w, v.z)));
}

// quaternion_multiply, calcenergy.cl:110-117
DEV float4 qmul(float4 a, float4 b) {
    return make_float4(a.w * b.x + a.x * b.w + a.y * b.z - a.z * b.y,
                       a.w * b.y - a.x * b.z + a.y * b.w + a.z * b.x,
                       a.w * b.z + a.x * b.y - a.y * b.x + a.z * b.w,
                       a.w * b.w - a.x * b.x - a.y * b.y - a.z * b.z);
}

// map_angle, auxiliary_genetic.cl:72-85.  Values the subtraction loop could
// not bring into range (|a| >= 1e6, where a - 360 may round back to a, and
// inf) are reduced with fmodf first; the reference loops forever on them.
DEV void map_angle(float& a) {
    if (!(fabsf(a) < 1.0e6f)) a = fmodf(a, 360.0f);
    if (!(a == a) || isinf(a)) return;
    while (a >= 360.0f) a -= 360.0f;
    while (a < 0.0f) a += 360.0f;
}

// LCG, auxiliary_genetic.cl:29-67
DEV float randf(uint32_t& s) {
    s = 1103515245u * s + 12345u;
    return ((float)s * (1.0f / 4294967296.0f)) * 0.999999f;
}

// ---------------------------------------------------------------------------
// map gathers: one grid point of one map = 4 values (packed-4 layout)
// ---------------------------------------------------------------------------
// Bytes of a point, as a shift.
template <int MF>
constexpr int kPointShift = MF == ADGPU_MAP_F32 ? 4 : 3;

template <int MF>
DEV float4 load_pt(const void* p);

template <>
DEV float4 load_pt<ADGPU_MAP_F32>(const void* p) {
    return *reinterpret_cast<const float4*>(p);
}
template <>
DEV float4 load_pt<ADGPU_MAP_F16>(const void* p) {
    uint2 r = *reinterpret_cast<const uint2*>(p);
    __half2 lo = *reinterpret_cast<__half2*>(&r.x), hi = *reinterpret_cast<__half2*>(&r.y);
    float2 a = __half22float2(lo), b = __half22float2(hi);
    return make_float4(a.x, a.y, b.x, b.y);
}
template <>
DEV float4 load_pt<ADGPU_MAP_BF16>(const void* p) {
    uint2 r = *reinterpret_cast<const uint2*>(p);
    return make_float4(__uint_as_float(r.x << 16), __uint_as_float(r.x & 0xffff0000u),
                       __uint_as_float(r.y << 16), __uint_as_float(r.y & 0xffff0000u));
}
template <int MF>
DEV float4 load_pt(const void* base, uint32_t idx) {
    return load_pt<MF>(reinterpret_cast<const char*>(base) + ((uint64_t)idx << kPointShift<MF>));
}

// ---------------------------------------------------------------------------
// LDS layout
// ---------------------------------------------------------------------------
// One rotatable bond in a team's LDS block: its rotation, then (once the
// coordinates are made) its axis; its moving vector; the bond's first atom.
struct TorRec {
    float4 q;
    float4 m;
    float4 r0;
};

// A pair's record as the energy takes it.
struct PairRec {
    uint32_t ij;
    float fn, ac, bd, reqm, cq, dsol, g;
};
DEV PairRec unpack(const PairA& a, const PairB& b) {
    return PairRec{a.ij, a.fn, a.ac, a.bd, b.reqm, b.cq, b.dsol, b.g};
}
DEV PairRec unpack(const PairC& c) {   // g: with the flags
    return PairRec{c.ij & ~kPairTen, (int)c.ij < 0 ? 10.0f : 6.0f, c.ac, c.bd, c.reqm, c.cq, c.dsol, 0.0f};
}

struct SharedView {           // staged once per workgroup
    const PairA* pa;          // LDS (or global when the pairs do not fit): record p of step k is
    const PairB* pb;          //   [k * pair_stride<TW, PL> + lane] of both
    const PairC* pc;          // in place of pa and pb (compact_pairs)
    const PairX* px;          // global (rarely read)
    const float4* tor_unit;
    const int2* tor_atoms;
};

// Element at byte offset `bytes` of an array.
template <class V>
DEV V* at(V* p, uint32_t bytes) { return reinterpret_cast<V*>(reinterpret_cast<char*>(p) + bytes); }

struct TeamView {             // private to one team
    float* cx;                // [coord_array] atom coordinates (grid units), one
    float* cy;                //   array per axis: lanes reading different
    float* cz;                //   atoms hit different banks
    int* fx;                  // [slot_array] int32 fixed-point pair forces
    int* fy;
    int* fz;
    TorRec* tor;              // [T]
    int* gi;                  // [T][4] torsion gene gradients (int fixed point), in four
                              //   parts: lanes add to the part of their index mod 4
    float* pg;                // [12] genes 0..5, sin/cos of phi, theta, rot/2; then the
                              //   gradients of genes 0..5 (int fixed point)
};

__host__ __device__ inline size_t align16(size_t x) { return (x + 15) & ~size_t(15); }

// Records from one step of the pair loop to the next.  In LDS the two halves
// of a step's TW records follow each other (TW PairA, then TW PairB), so that
// one address register reaches both, at a fixed offset.
template <int TW, bool PL>
constexpr int pair_stride = PL ? 2 * TW : TW;

__host__ __device__ inline size_t shared_bytes_for(int TW, int NC, int T, int P, bool pairs_in_lds, bool GRAD) {
    size_t s = pairs_in_lds ? (size_t)padded_pairs(P, TW) * (compact_pairs(TW * NC, GRAD) ? sizeof(PairC) : sizeof(PairA) + sizeof(PairB)) : 0;
    s += (size_t)T * (sizeof(float4) + sizeof(int2));
    return align16(s);
}

// Copies of the atoms' coordinates that the pair loop reads, and the words of
// one coordinate array.  Kernels that only take energies (GRAD false) add no
// forces: their staged records name first copies.
__host__ __device__ constexpr int coord_copies(int TW, int NC, bool PL, bool GRAD) {
    return PL && !GRAD ? 1 : slot_copies(TW, NC);
}
__host__ __device__ constexpr int coord_array(int TW, int NC, bool PL, bool GRAD) {
    return PL && !GRAD ? TW * NC + 4 : slot_array(TW, NC);
}
// Slot that lanes without an atom write, behind the atoms of every copy and
// named by no pair: in one copy's arrays the first spare word, in two copies'
// a slot between the first copy of a ligand of `atoms` atoms and its second.
__host__ __device__ constexpr int idle_slot(int TW, int NC, bool PL, bool GRAD, int atoms) {
    return coord_copies(TW, NC, PL, GRAD) == 2 ? slot_stride(atoms) - 16 : TW * NC;
}
// Whether its last copy lies inside the arrays for the shape's largest ligand.
__host__ __device__ constexpr bool idle_slot_fits(int TW, int NC, bool PL, bool GRAD) {
    return idle_slot(TW, NC, PL, GRAD, TW * NC) + (coord_copies(TW, NC, PL, GRAD) - 1) * slot_stride(TW * NC) <
           coord_array(TW, NC, PL, GRAD);
}

__host__ __device__ inline size_t team_bytes_for(int TW, int NC, int T, bool PL, bool GRAD) {
    const size_t coords = 3 * (size_t)coord_array(TW, NC, PL, GRAD) * 4 + (size_t)T * sizeof(TorRec) + 48;
    return GRAD ? coords + 3 * (size_t)slot_array(TW, NC) * 4 + (size_t)T * 16 : coords;
}

// LDS of one workgroup of `threads` threads (threads / TW teams).
__host__ __device__ inline size_t lds_bytes_for(int TW, int NC, int T, int P, bool PL, bool GRAD, int threads) {
    return shared_bytes_for(TW, NC, T, P, PL, GRAD) + (size_t)(threads / TW) * team_bytes_for(TW, NC, T, PL, GRAD);
}

// Stages the shared tables (all threads of the workgroup) and carves the
// team's region.  Contains the only workgroup barrier of every kernel.  GRAD:
// the kernel evaluates gradients.
template <int TW, int NC, bool PL, bool GRAD>
DEV void stage(const LigandDev* L, char* lds, SharedView& sv, TeamView& tv) {
    const char* gbase = reinterpret_cast<const char*>(L);
    const int T = L->num_rotbonds, P = L->num_pairs;
    char* p = lds;
    const PairA* gpa = reinterpret_cast<const PairA*>(gbase + L->off_pair_a[slot_copies(TW, NC) - 1]);
    const PairB* gpb = reinterpret_cast<const PairB*>(gbase + L->off_pair_b);
    sv.px = reinterpret_cast<const PairX*>(gbase + L->off_pair_x);
    constexpr bool kCompact = compact_pairs(TW * NC, GRAD);
    sv.pc = reinterpret_cast<const PairC*>(gbase + L->off_pair_c);
    if constexpr (PL && kCompact) {
        static_assert(slot_copies(TW, NC) == 1, "staged as it is stored");
        const int PP = padded_pairs(P, TW);
        PairC* lc = reinterpret_cast<PairC*>(p);
        for (int k = threadIdx.x; k < PP; k += blockDim.x) lc[k] = sv.pc[k];
        sv.pc = lc;
        p += (size_t)PP * sizeof(PairC);
    } else if (PL) {
        const int PP = padded_pairs(P, TW);
        PairA* la = reinterpret_cast<PairA*>(p);
        PairB* lb = reinterpret_cast<PairB*>(la + TW);
        for (int k = threadIdx.x; k < PP; k += blockDim.x) {
            const int at = k / TW * pair_stride<TW, true> + k % TW;
            PairA r = gpa[k];
            if (coord_copies(TW, NC, PL, GRAD) < slot_copies(TW, NC)) {
                const uint32_t second = 4u * (uint32_t)slot_stride(L->num_atoms);
                const uint32_t i = r.ij & 0xffffu, j = r.ij >> 16;
                r.ij = (i >= second ? i - second : i) | (j >= second ? j - second : j) << 16;
            }
            la[at] = r;
            lb[at] = gpb[k];
        }
        sv.pa = la;
        sv.pb = lb;
        p += (size_t)PP * (sizeof(PairA) + sizeof(PairB));
    } else {
        sv.pa = gpa;
        sv.pb = gpb;
    }
    float4* tu = reinterpret_cast<float4*>(p);
    int2* ta = reinterpret_cast<int2*>(tu + T);
    const float4* gtu = reinterpret_cast<const float4*>(gbase + L->off_tor_unit);
    const float4* gtm = reinterpret_cast<const float4*>(gbase + L->off_tor_move);
    const int2* gta = reinterpret_cast<const int2*>(gbase + L->off_tor_atoms);
    for (int k = threadIdx.x; k < T; k += blockDim.x) { tu[k] = gtu[k]; ta[k] = gta[k]; }
    sv.tor_unit = tu; sv.tor_atoms = ta;
    char* w = lds + shared_bytes_for(TW, NC, T, P, PL, GRAD) + (size_t)(threadIdx.x / TW) * team_bytes_for(TW, NC, T, PL, GRAD);
    constexpr int kCoords = coord_array(TW, NC, PL, GRAD), kForces = slot_array(TW, NC);
    tv.cx = reinterpret_cast<float*>(w);
    tv.cy = tv.cx + kCoords;
    tv.cz = tv.cy + kCoords;
    w += 3 * (size_t)kCoords * 4;
    if (GRAD) {
        tv.fx = reinterpret_cast<int*>(w);
        tv.fy = tv.fx + kForces;
        tv.fz = tv.fy + kForces;
        w += 3 * (size_t)kForces * 4;
        tv.gi = reinterpret_cast<int*>(w);
        w += (size_t)T * 16;
    }
    tv.tor = reinterpret_cast<TorRec*>(w);
    for (int t = Team<TW>::lane(); t < T; t += TW) tv.tor[t].m = gtm[t];
    w += (size_t)T * sizeof(TorRec);
    tv.pg = reinterpret_cast<float*>(w);
    __syncthreads();
}

// ---------------------------------------------------------------------------
// per-lane atom data, loaded once per kernel
// ---------------------------------------------------------------------------
template <int TW, int NC>
struct Atoms {
    float3 ref[NC];
    float q[NC];
    uint32_t mlo[NC];         // rotatable bonds 0..31 that move the atom
    uint32_t mapoff[NC];      // map index * g3
    uint32_t slot[NC];        // byte offset of the atom's first copy in the slot arrays
    uint32_t copy;            // bytes from there to its second copy
    bool valid[NC], ign[NC], lig[NC];

    // PL, GRAD: the kernel's layout, as stage is told.
    template <bool PL, bool GRAD>
    DEV void load(const LigandDev* L, const GridDev& G) {
        static_assert(idle_slot_fits(TW, NC, PL, GRAD), "lanes without an atom write inside their team's arrays");
        const char* gb = reinterpret_cast<const char*>(L);
        const float4* ar = reinterpret_cast<const float4*>(gb + L->off_atom_ref);
        const int4* ai = reinterpret_cast<const int4*>(gb + L->off_atom_info);
        const uint2* am = reinterpret_cast<const uint2*>(gb + L->off_atom_mask);
        const int tl = Team<TW>::lane();
        const int stride = slot_stride(L->num_atoms);
        copy = (uint32_t)stride * 4u;
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            int a = tl + TW * k;
            valid[k] = a < L->num_atoms;
            slot[k] = 4u * (uint32_t)(valid[k] ? a : idle_slot(TW, NC, PL, GRAD, L->num_atoms));
            int aa = valid[k] ? a : 0;
            float4 r = ar[aa];
            int4 inf = ai[aa];
            uint2 m = am[aa];
            ref[k] = make_float3(r.x, r.y, r.z);
            q[k] = r.w;
            mlo[k] = valid[k] ? m.x : 0u;
            mapoff[k] = valid[k] ? (uint32_t)inf.x * G.g3 : 0u;
            ign[k] = !valid[k] || inf.z != 0;
            lig[k] = valid[k] && a < L->true_ligand_atoms;
        }
    }
};

// Ligand scalars read once per kernel (kept in registers, not re-read from
// global memory inside the loops).
struct LigScalars {
    int T, P, NG;
    bool has_lig, any_general;
    float half_smooth, elec_min, inv_elec_min, coeff_desolv;
    DEV void load(const LigandDev* L) {
        T = L->num_rotbonds; P = L->num_pairs; NG = L->num_genes;
        has_lig = L->true_ligand_atoms != 0;
        any_general = L->any_general != 0;
        half_smooth = L->half_smooth; elec_min = L->elec_min_distance; coeff_desolv = L->coeff_desolv;
        inv_elec_min = L->inv_elec_min;
    }
};

template <int TW, int NC>
struct EvalCtx {
    const LigandDev* L;
    GridDev G;
    SharedView sv;
    TeamView tv;
    Atoms<TW, NC> A;
    LigScalars ls;
};

// Calls f(t, q, v) for the rotatable bonds t that move atom chunk k of the
// lane, in ascending order, with the bond's record members `second` (v) and q.
// 64-lane teams read the next bond's members while f runs, so that only the
// first read's latency shows; 32-lane ones have no registers for it (ADAM, 41
// atoms, 64 lanes 400 -> 452 M evals/s; ADADELTA, 30 atoms, 32 lanes 366 -> 371
// ms a docking, were it done there).  Bonds beyond the 32nd are rare: their bits are read from the
// ligand block instead of keeping a register.
template <int TW, int NC, class F>
DEV void for_bonds(const EvalCtx<TW, NC>& X, int k, float4 TorRec::*second, F&& f) {
    const int T = X.ls.T;
    // a 24-bit product: 64-bit address arithmetic takes four times as long
    auto rec = [&](int t) { return at(X.tv.tor, __umul24((uint32_t)t, (uint32_t)sizeof(TorRec))); };
    if (uint32_t m = X.A.mlo[k]) {
        int t = __builtin_ctz(m);
        float4 q = rec(t)->q, v = rec(t)->*second;
        for (;;) {
            m &= m - 1;
            if constexpr (TW == 64) {
                const int next = m ? __builtin_ctz(m) : t;
                const float4 nq = rec(next)->q, nv = rec(next)->*second;
                f(t, q, v);
                if (!m) break;
                t = next; q = nq; v = nv;
            } else {
                f(t, q, v);
                if (!m) break;
                t = __builtin_ctz(m);
                q = rec(t)->q; v = rec(t)->*second;
            }
        }
    }
    if (__builtin_expect(T > 32, 0)) {
        const LigandDev* L = X.L;
        const uint2* am = reinterpret_cast<const uint2*>(reinterpret_cast<const char*>(L) + L->off_atom_mask);
        uint32_t m = X.A.valid[k] ? am[Team<TW>::lane() + TW * k].y : 0u;
        for (; m; m &= m - 1) {
            const int t = 32 + __builtin_ctz(m);
            f(t, rec(t)->q, rec(t)->*second);
        }
    }
}

// ---------------------------------------------------------------------------
// Pose (calcenergy.cl:201-221): genes 0..5 and the sine/cosine of the
// orientation angles, which the gene lanes left in the team's LDS block.
// ---------------------------------------------------------------------------
struct Pose {
    float4 q;          // genrot quaternion
    float3 mv;         // translation (grid units)
    float phi, theta, rotangle, sin_theta, sin_half, is_theta_gt_pi;
};

// Every gene lane computes the trigonometry of its own angle gene once:
// orientation genes into pg, torsion genes into the torsion quaternions
// (calcenergy.cl:201-221, 248-260).  Followed by wave_sync by the caller.
template <int TW>
DEV void gene_trig(const LigScalars& ls, const SharedView& sv, const TeamView& tv, const float (&gene)[64 / TW]) {
    const int tl = Team<TW>::lane();
    const int NG = ls.NG;
#pragma unroll
    for (int j = 0; j < Team<TW>::kGPL; ++j) {
        const int g = tl + TW * j;
        if (j > 0 && NG <= TW) break;
        const float v = gene[j];
        if (g < 6) tv.pg[g] = v;
        if (g >= 3 && g < NG) {
            float ang = v * kDegToRad;
            if (g >= 5) ang = ang * 0.5f;
            float s, c;
            sincosf(ang, &s, &c);
            if (g < 6) {
                tv.pg[6 + 2 * (g - 3)] = s;
                tv.pg[7 + 2 * (g - 3)] = c;
            } else {
                float4 u = sv.tor_unit[g - 6];
                s += s;
                tv.tor[g - 6].q = make_float4(s * u.x, s * u.y, s * u.z, c);   // as qrot2 takes it
            }
        }
    }
}

DEV Pose read_pose(const TeamView& tv, bool has_ligand) {
    Pose P;
    const float4 p0 = *reinterpret_cast<const float4*>(tv.pg);       // g0 g1 g2 g3
    const float4 p1 = *reinterpret_cast<const float4*>(tv.pg + 4);   // g4 g5 sin(phi) cos(phi)
    const float4 p2 = *reinterpret_cast<const float4*>(tv.pg + 8);   // sin/cos theta, sin/cos rot/2
    P.phi = p0.w * kDegToRad;
    P.theta = p1.x * kDegToRad;
    P.rotangle = p1.y * kDegToRad;
    P.q = make_float4(0.f, 0.f, 0.f, 1.f);
    P.mv = make_float3(0.f, 0.f, 0.f);
    P.sin_theta = 0.f; P.sin_half = 0.f; P.is_theta_gt_pi = 1.f;
    if (has_ligand) {
        const float sp = p1.z, cp = p1.w, st = p2.x, ct = p2.y, sh = p2.z, ch = p2.w;
        P.mv = make_float3(p0.x, p0.y, p0.z);
        P.q = make_float4(sh * st * cp, sh * st * sp, sh * ct, ch);
        P.sin_theta = st;
        P.sin_half = sh;
        P.is_theta_gt_pi = 1.0f - 2.0f * (float)(st < 0.0f);
    }
    return P;
}

// Pose -> coordinates (calcenergy.cl:232-275).  Per atom: the rotatable bonds
// moving it in ascending index, then the general rotation (the per-atom order
// gen_rotlist encodes, host/src/calcenergy.cpp:387-488).
template <int TW, int NC, int COPIES>
DEV void compute_coords(const EvalCtx<TW, NC>& X, const Pose& P, float3 (&c)[NC]) {
    const TeamView& tv = X.tv;
    const Atoms<TW, NC>& A = X.A;
#pragma unroll
    for (int k = 0; k < NC; ++k) {
        float3 v = A.ref[k];
        for_bonds<TW, NC>(X, k, &TorRec::m, [&](int, const float4& q, const float4& m) {
            float3 r = qrot2(make_float3(v.x - m.x, v.y - m.y, v.z - m.z), q);
            v = make_float3(r.x + m.x, r.y + m.y, r.z + m.z);
        });
        if (A.lig[k]) {
            float3 r = qrot(v, P.q);
            v = make_float3(r.x + P.mv.x, r.y + P.mv.y, r.z + P.mv.z);
        }
        c[k] = v;
#pragma unroll
        for (int copy = 0; copy < COPIES; ++copy) {
            const uint32_t o = A.slot[k] + copy * A.copy;
            *at(tv.cx, o) = v.x; *at(tv.cy, o) = v.y; *at(tv.cz, o) = v.z;
        }
    }
}

// ---------------------------------------------------------------------------
// Intermolecular energy (+ map gradient) of one atom, calcenergy.cl:280-379,
// calcMergedEneGra.cl:222-443.  Split in two so the map loads of all atoms
// are in flight while the pair loop runs.
// ---------------------------------------------------------------------------
template <int MF>
struct Gather {
    float4 a0, a1, e0, e1, d0, d1;
    bool in;
};

template <int MF>
DEV void gather_issue(const GridDev& G, float3 c, uint32_t mapoff, Gather<MF>& g) {
    // out of the grid (calcenergy.cl:293-301); NaN coordinates count as out,
    // so no map index is ever formed from them
    g.in = (c.x >= 0.f) && (c.y >= 0.f) && (c.z >= 0.f) && (c.x < (float)(G.gx - 1)) &&
           (c.y < (float)(G.gy - 1)) && (c.z < (float)(G.gz - 1));
    // Cell of the low corner; coordinates in the grid are not negative, so the
    // conversion's truncation is their floor.  The e and d maps lie at uniform
    // addresses, one 32-bit offset apart from which the loads reach both
    // corners along x; only the type map's address is 64-bit arithmetic.
    const uint32_t cell = (uint32_t)c.x + __umul24((uint32_t)c.y, G.g1) + __umul24((uint32_t)c.z, G.g2);
    const uint32_t p = g.in ? cell : 0u;
    constexpr uint32_t kPt = 1u << kPointShift<MF>;
    const char* base = reinterpret_cast<const char*>(G.data);
    const char* em = base + ((uint64_t)((uint32_t)(G.nmaps - 2) * G.g3) << kPointShift<MF>);
    const char* dm = em + ((uint64_t)G.g3 << kPointShift<MF>);
    const char* am = base + ((uint64_t)(mapoff + p) << kPointShift<MF>);
    const uint32_t off = p << kPointShift<MF>;
    g.a0 = load_pt<MF>(am); g.a1 = load_pt<MF>(am + kPt);
    g.e0 = load_pt<MF>(em + off); g.e1 = load_pt<MF>(em + off + kPt);
    g.d0 = load_pt<MF>(dm + off); g.d1 = load_pt<MF>(dm + off + kPt);
}

// The three maps are combined per cube corner first (type + q e + |q| d),
// then interpolated once: the same sum as the reference's three separate
// interpolations (calcenergy.cl:338-379), with one interpolation's work.
template <int MF, bool GRAD>
DEV float gather_finish(const GridDev& G, float3 c, float q, const Gather<MF>& g, int3& fi) {
    if (!g.in) {
        if (GRAD) { fi.x += 16777216; fi.y += 16777216; fi.z += 16777216; }
        return 16777216.0f;
    }
    const float dx = __builtin_amdgcn_fractf(c.x), omdx = 1.0f - dx;
    const float dy = __builtin_amdgcn_fractf(c.y), omdy = 1.0f - dy;
    const float dz = __builtin_amdgcn_fractf(c.z), omdz = 1.0f - dz;
    const float aq = fabsf(q);
    // cube corner k: 0 000, 1 010, 2 001, 3 011 (low x: .x .y .z .w of a0/e0/d0), 4..7 the same at x+1
    const float4 l = make_float4(fmaf(aq, g.d0.x, fmaf(q, g.e0.x, g.a0.x)), fmaf(aq, g.d0.y, fmaf(q, g.e0.y, g.a0.y)),
                                 fmaf(aq, g.d0.z, fmaf(q, g.e0.z, g.a0.z)), fmaf(aq, g.d0.w, fmaf(q, g.e0.w, g.a0.w)));
    const float4 h = make_float4(fmaf(aq, g.d1.x, fmaf(q, g.e1.x, g.a1.x)), fmaf(aq, g.d1.y, fmaf(q, g.e1.y, g.a1.y)),
                                 fmaf(aq, g.d1.z, fmaf(q, g.e1.z, g.a1.z)), fmaf(aq, g.d1.w, fmaf(q, g.e1.w, g.a1.w)));
    // interpolate along x, then y, then z
    const float x00 = omdx * l.x + dx * h.x, x10 = omdx * l.y + dx * h.y;
    const float x01 = omdx * l.z + dx * h.z, x11 = omdx * l.w + dx * h.w;
    const float y0 = omdy * x00 + dy * x10, y1 = omdy * x01 + dy * x11;
    const float e = omdz * y0 + dz * y1;
    if (GRAD) {
        const float ig = kTermScale * G.inv_spacing;   // a power of two: the same rounded products
        const float gx = omdz * (omdy * (h.x - l.x) + dy * (h.y - l.y)) + dz * (omdy * (h.z - l.z) + dy * (h.w - l.w));
        const float gy = omdz * (x10 - x00) + dz * (x11 - x01);
        const float gz = y1 - y0;
        fi.x += quant(gx * ig);
        fi.y += quant(gy * ig);
        fi.z += quant(gz * ig);
    }
    return e;
}

// ---------------------------------------------------------------------------
// Intramolecular pair energy and dE/dr (calcenergy.cl:397-536,
// calcMergedEneGra.cl:455-583).
// ---------------------------------------------------------------------------
// The cutoff tests select terms instead of branching: over a team's pairs
// both ranges are almost always present, so branches would only add mask
// handling.  Adding the zero of an excluded term leaves the sum unchanged.
// dist = distance in grid units, rdist = 1 / dist, inv_sp = 1 / spacing: 1/r in
// A is rdist * inv_sp unless r is clamped at elec_min_distance.  Every fused
// multiply-add is written out, so all kernels round alike.
// flags(): the pair's PairX::flags.
template <bool GRAD, bool COMPACT, class F>
DEV float pair_energy(const LigScalars& ls, const PairRec& pr, F&& flags, float spacing, float dist,
                      float rdist, float inv_sp, float& dedr) {
#pragma clang fp contract(off)
    // vdW / H-bond with smoothing, r < 8 A: with qm = sd^-m and qn = sd^-n,
    // E = AC qm - BD qn and dE/dsd = -(m AC qm - n BD qn) / sd.  sd^-12 is one
    // reciprocal of sd^12 (a few ulp; the 12th power of 1/sd would carry up to
    // 12 ulp), and sd^-n = sd^-12 sd^(12-n)
    const float ad = dist * spacing;
    const float delta = fmaf(-spacing, dist, pr.reqm);
    const float sd = (fabsf(delta) >= ls.half_smooth) ? fmaf(spacing, dist, copysignf(ls.half_smooth, delta)) : pr.reqm;
    const float r2 = sd * sd, r4 = r2 * r2, r6 = r4 * r2;
    const float qm = fast_rcp(r6 * r6);               // m = 12
    const float qn = qm * (pr.fn == 6.0f ? r6 : r2);  // n = 6 or 10
    const float q = GRAD ? fast_rcp(sd) : 0.0f;
    const float am = pr.ac * qm, bn = pr.bd * qn;
    float evdw = fmaf(pr.ac, qm, -bn);
    float dvdw = GRAD ? fmaf(bn, pr.fn, -(12.0f * am)) * q : 0.0f;
    float g = pr.g;                                   // CG-G0 bond constant: 50 for a CG-G0 pair, else 0
    if (__builtin_expect(ls.any_general, 0)) {        // other exponents (modified pairs): rare,
        const uint32_t fl = flags();                  // kept off the common path
        if (COMPACT && (fl & kPairCgG0)) g = 50.0f;
        if (!(fl & kPairFast)) {
            const float fm = (float)(fl & 0xffu), fn = (float)((fl >> 8) & 0xffu);
            const float l2 = __builtin_amdgcn_logf(sd);
            const float gm = __builtin_amdgcn_exp2f(-fm * l2);
            const float ga = pr.ac * gm, gb = pr.bd * __builtin_amdgcn_exp2f(-fn * l2);
            evdw = fmaf(pr.ac, gm, -gb);
            if (GRAD) dvdw = fmaf(gb, fn, -(fm * ga)) * q;
        }
    }
    // electrostatics and desolvation, r < 20.48 A, r clamped at elec_min_distance:
    // 1/max(r, r_min) = min(1/r, 1/r_min)
    const float d = max_s(ad, ls.elec_min);
    const float d2 = d * d;
    const float num = fmaf(-0.1063f * d2, fmaf(-0.001947f, d2, 1.0f), 12.96f);
    const float den = fmaf(d2, fmaf(d2, fmaf(0.000112f, d2, 0.00357f), 0.4137f), 12.96f);
    const float desolv = pr.dsol * (ls.coeff_desolv * num * fast_rcp(den));
    const float rds = fast_rcp(d + 1.26366f);
    const float rds2 = rds * rds;
    const float diel = fmaf(1.10859f, rds2, 0.010358f);
    const float rd = min_s(rdist * inv_sp, ls.inv_elec_min);
    const float es = pr.cq * rd;
    const float eel = fmaf(es, diel, desolv);
    const bool in8 = ad < 8.0f, in20 = ad < 20.48f;
    const float e = fmaf(g, ad, in8 ? evdw : 0.0f) + (in20 ? eel : 0.0f);
    if (GRAD) {
        const float del = fmaf(-0.0771605f * d, desolv, fmaf(rds, es * -2.21718f * rds2, -(es * rd * diel)));
        dedr = g + (in8 ? dvdw : 0.0f) + (in20 ? del : 0.0f);
    } else {
        dedr = 0.f;
    }
    return e;
}

// ---------------------------------------------------------------------------
// One evaluation of one genotype by one team.
//   GRAD = false: gpu_calc_energy (calcenergy.cl:132-554)
//   GRAD = true : gpu_calc_energrad (calcMergedEneGra.cl:46-936); grad[j]
//                 receives d E / d gene (lane + TW j), 0 beyond the genes.
// All lanes of the wavefront must call it together (uniform control flow).
// ---------------------------------------------------------------------------
// GRAD_KERNEL: what stage was told.
template <int TW, int NC, int MF, bool PL, bool GRAD, bool GRAD_KERNEL = true>
DEV float evaluate(const EvalCtx<TW, NC>& X, const float (&gene)[64 / TW], float (&grad)[64 / TW]) {
    using TM = Team<TW>;
    const LigandDev* L = X.L;
    const GridDev& G = X.G;
    const TeamView& tv = X.tv;
    const SharedView& sv = X.sv;
    const int tl = TM::lane();
    const int T = X.ls.T, NG = X.ls.NG;
    const bool has_lig = X.ls.has_lig;
    (void)L;

    gene_trig<TW>(X.ls, sv, tv, gene);
    if (GRAD) {
#pragma unroll
        for (int k = 0; k < NC; ++k)
#pragma unroll
            for (int copy = 0; copy < slot_copies(TW, NC); ++copy) {
                const uint32_t o = X.A.slot[k] + copy * X.A.copy;
                *at(tv.fx, o) = 0; *at(tv.fy, o) = 0; *at(tv.fz, o) = 0;
            }
#pragma unroll
        for (int j = 0; j < TM::kGPL; ++j) {
            if (j > 0 && T <= TW) break;
            if (tl + TW * j < T) reinterpret_cast<int4*>(tv.gi)[tl + TW * j] = make_int4(0, 0, 0, 0);
        }
    }
    wave_sync();
    const Pose pose = read_pose(tv, has_lig);
    float3 c[NC];
    compute_coords<TW, NC, coord_copies(TW, NC, PL, GRAD_KERNEL)>(X, pose, c);

    // with one atom per lane the map loads go out before the pair loop and
    // land while it runs; with more, each chunk is gathered after it (the
    // loads of all chunks would not fit the register budget)
    Gather<MF> gth0;
    if constexpr (NC == 1) gather_issue<MF>(G, c[0], X.A.mapoff[0], gth0);
    wave_sync();

    const float spacing = G.spacing;
    float e = 0.f;
    constexpr bool kCompact = compact_pairs(TW * NC, GRAD_KERNEL);
    const PairA* ra = sv.pa + tl;
    const PairB* rb = sv.pb + tl;
    const PairC* rc = sv.pc + tl;
    // Every lane has a record in every step (padding), so the loop count is
    // uniform: no execution masks, and the counter is scalar.  With the atoms
    // kept as byte offsets, the exponent as a float, the two halves of a step
    // behind one address and the bounds taken by max_s / min_s, a step is 91
    // VALU and 8 SALU instructions (105 and 15 with counted lanes, packed
    // indices and library fmaxf / fminf): Solis-Wets nrun 20 on the 30-atom
    // ligand 95.6 -> 89.5 ms a docking, ADADELTA nrun 50 on 54 atoms 222.8 ->
    // 218.0 ms, ADADELTA nrun 100 on 30 atoms 389.2 -> 386.2 ms.
    const int steps = (X.ls.P + TW - 1) / TW;
    // Records that stay in memory are read a step ahead (the last step reads its
    // own again), so that L2's latency runs beside the arithmetic: 90 atoms in
    // 64-lane teams 27.5 -> 22.6 us an iteration of one search, 76 -> 89 M
    // evals/s with 7500 searches.  The same for records in LDS (the next
    // pair's atoms only) gave 6.1 -> 5.8 us for one search but 608 -> 590 M
    // evals/s with many, and is not done.
    PairA pa{};
    PairB pb{};
    PairC pc{};
    if (!PL && steps > 0) {
        if constexpr (kCompact) pc = *rc;
        else { pa = *ra; pb = *rb; }
    }
#pragma unroll 1
    for (int k = 0; k < steps; ++k) {
        PairA pa_next{};
        PairB pb_next{};
        PairC pc_next{};
        const int next = k + 1 < steps ? TW : 0;
        if constexpr (PL && kCompact) pc = *rc;
        else if constexpr (PL) { pa = *ra; pb = *rb; }
        else if constexpr (kCompact) pc_next = rc[next];
        else { pa_next = ra[next]; pb_next = rb[next]; }
        const PairRec pr = kCompact ? unpack(pc) : unpack(pa, pb);
        const uint32_t io = pr.ij & 0xffffu, jo = pr.ij >> 16;
        const float sx = *at(tv.cx, io) - *at(tv.cx, jo), sy = *at(tv.cy, io) - *at(tv.cy, jo),
                    sz = *at(tv.cz, io) - *at(tv.cz, jo);
        const float d2g = fmaf(sz, sz, fmaf(sx, sx, sy * sy));
        const float rdist = fast_rsq(d2g);            // one transcendental for r and 1/r
        const float dist = d2g * rdist;
        float dedr;
        auto flags = [&] {
            const uint32_t at = kCompact ? (uint32_t)(rc - sv.pc) : (uint32_t)(ra - sv.pa);
            return sv.px[PL && !kCompact ? (at + tl) >> 1 : at].flags;   // a step's records are TW PairA apart
        };
        e += pair_energy<GRAD, kCompact>(X.ls, pr, flags, spacing, dist, rdist, G.inv_spacing, dedr);
        if (GRAD) {
            // TERMSCALE * s * gdd with the power-of-two scale folded into gdd:
            // the same rounded product
            const float gdd = dedr * rdist * -kTermScale;
            const int ix = quant(sx * gdd), iy = quant(sy * gdd), iz = quant(sz * gdd);
            lds_sub(at(tv.fx, io), ix); lds_sub(at(tv.fy, io), iy); lds_sub(at(tv.fz, io), iz);
            atomicAdd(at(tv.fx, jo), ix); atomicAdd(at(tv.fy, jo), iy); atomicAdd(at(tv.fz, jo), iz);
        }
        if constexpr (!PL) { pa = pa_next; pb = pb_next; pc = pc_next; }
        ra += pair_stride<TW, PL>;
        rb += pair_stride<TW, PL>;
        rc += TW;
    }
    int3 fi[NC];
#pragma unroll
    for (int k = 0; k < NC; ++k) {
        fi[k] = make_int3(0, 0, 0);
        if constexpr (NC == 1) {
            const float ea = gather_finish<MF, GRAD>(G, c[k], X.A.q[k], gth0, fi[k]);
            if (!X.A.ign[k]) e += ea;
        } else {
            Gather<MF> gk;
            gather_issue<MF>(G, c[k], X.A.mapoff[k], gk);
            const float ea = gather_finish<MF, GRAD>(G, c[k], X.A.q[k], gk, fi[k]);
            if (!X.A.ign[k]) e += ea;
        }
    }
    const float energy = TM::sum(e);
    if (!GRAD) return energy;

    wave_sync();
    // total per-atom forces (kcal/mol/A), int fixed point -> float
    float3 F[NC];
    float sfx = 0.f, sfy = 0.f, sfz = 0.f, tx = 0.f, ty = 0.f, tz = 0.f;
#pragma unroll
    for (int k = 0; k < NC; ++k) {
        F[k] = make_float3(0.f, 0.f, 0.f);
        if (X.A.valid[k]) {
            int fx = 0, fy = 0, fz = 0;
#pragma unroll
            for (int copy = 0; copy < slot_copies(TW, NC); ++copy) {
                const uint32_t o = X.A.slot[k] + copy * X.A.copy;
                fx += *at(tv.fx, o); fy += *at(tv.fy, o); fz += *at(tv.fz, o);
            }
            if (!X.A.ign[k]) { fx += fi[k].x; fy += fi[k].y; fz += fi[k].z; }
            F[k] = make_float3(kOneOverTermScale * (float)fx, kOneOverTermScale * (float)fy,
                               kOneOverTermScale * (float)fz);
            sfx += F[k].x; sfy += F[k].y; sfz += F[k].z;
            if (X.A.lig[k]) {   // torque about the ligand centre, calcMergedEneGra.cl:712-745
                const float rx = (c[k].x - pose.mv.x) * spacing, ry = (c[k].y - pose.mv.y) * spacing,
                            rz = (c[k].z - pose.mv.z) * spacing;
                tx += ry * F[k].z - rz * F[k].y;
                ty += rz * F[k].x - rx * F[k].z;
                tz += rx * F[k].y - ry * F[k].x;
            }
        }
    }
    // Rigid-body genes in lanes 0..5 of the team's last row, which the sums
    // above reach: every lane runs one chain, its gene's operands selected, and
    // one rounding to the fixed point.
    sfx = TM::sum_top(sfx); sfy = TM::sum_top(sfy); sfz = TM::sum_top(sfz);
    tx = TM::sum_top(tx); ty = TM::sum_top(ty); tz = TM::sum_top(tz);
    const int r = tl - TM::kTop;
    int ig = 0;
    if (has_lig) {
#pragma clang fp contract(off)
        // translation genes, calcMergedEneGra.cl:679-697
        const float move = kTermScale * (r == 0 ? sfx : r == 1 ? sfy : sfz) * spacing;
        // rotation genes (3 phi, 4 theta, 5 angle), calcMergedEneGra.cl:756-861
        const bool is_phi = r == 3, is_theta = r == 4, is_rot = r == 5;
        const float tlen = fast_sqrt(fmaf(tz, tz, fmaf(tx, tx, ty * ty)));
        const float tlen2 = tlen * tlen;
        const bool small = tlen < 1e-3f;
        const float oscale = small ? 1.0f : tlen * (1.0f / 1e-3f);
        const float sc = small ? fmaf(tlen2, -1.0f / 48.0f, 0.5f) : 0.0005f * fast_rcp(tlen);
        const float4 qt = make_float4(tx * sc, ty * sc, tz * sc, small ? fmaf(tlen2, -0.125f, 1.0f) : 0.99999988f);
        const float4 tq = qmul(qt, pose.q);
        const float inv_sin = fast_rsq(fmaf(-tq.w, tq.w, 1.0f));
        const float ac = fast_acos(is_theta ? tq.z * inv_sin : tq.w);
        const float at = atan2f(pose.is_theta_gt_pi * tq.y, pose.is_theta_gt_pi * tq.x);
        const float target = is_phi ? fmod_pi2(at + kTwoPi) : is_theta ? fmaf(pose.is_theta_gt_pi, ac, kTwoPi) : 2.0f * ac;
        const float current = fmod_pi2(fmaf(tv.pg[tl & 7], kDegToRad, kTwoPi));
        const float turn = oscale * (fmod_pi2(target - current + kPi) - kPi);
        const float corr = 4.0f * pose.sin_half * pose.sin_half;
        const float s = is_phi ? pose.sin_theta : 1.0f;
        const float rot = kTermScale * turn * s * s * (is_rot ? 1.0f : corr) * kDegToRad;
        ig = quant(r < 3 ? move : rot);
    }
    if ((unsigned)r < 6u) reinterpret_cast<int*>(tv.pg)[r] = ig;   // every lane has read its pose
    // torsion genes, calcMergedEneGra.cl:866-915
    for (int t = tl; t < T; t += TW) {
        const int2 ab = sv.tor_atoms[t];
        const float4 r0 = make_float4(tv.cx[ab.x], tv.cy[ab.x], tv.cz[ab.x], 0.f);
        const float ax = tv.cx[ab.y] - r0.x, ay = tv.cy[ab.y] - r0.y, az = tv.cz[ab.y] - r0.z;
        const float inv = fast_rsq(ax * ax + ay * ay + az * az);
        tv.tor[t].q = make_float4(ax * inv, ay * inv, az * inv, 0.f);
        tv.tor[t].r0 = r0;
    }
    wave_sync();
#pragma unroll
    for (int k = 0; k < NC; ++k) {
        for_bonds<TW, NC>(X, k, &TorRec::r0, [&](int t, const float4& ax, const float4& r0) {
            const float rx = c[k].x - r0.x, ry = c[k].y - r0.y, rz = c[k].z - r0.z;
            const float qx = ry * F[k].z - rz * F[k].y, qy = rz * F[k].x - rx * F[k].z,
                        qz = rx * F[k].y - ry * F[k].x;
            const float toa = (ax.x * qx + ax.y * qy + ax.z * qz) * spacing;
            atomicAdd(&tv.gi[4 * t + (tl & 3)], quant(toa * (kTermScale * kDegToRad)));
        });
    }
    wave_sync();
    const float conv = spacing * spacing * 1.0f / (kDegToRad * kDegToRad);   // CONVERT_INTO_ANGSTROM_RADIAN
#pragma unroll
    for (int j = 0; j < TM::kGPL; ++j) {
        const int g = tl + TW * j;
        int iv = 0;
        if (g < 6) {
            iv = reinterpret_cast<const int*>(tv.pg)[g];
        } else if (g < NG) {
            const int4 part = reinterpret_cast<const int4*>(tv.gi)[g - 6];
            iv = part.x + part.y + part.z + part.w;
        }
        const float gv = (float)iv * (g >= 3 ? kOneOverTermScale * conv : kOneOverTermScale);
        grad[j] = g < NG ? gv : 0.f;
    }
    return energy;
}

// ---------------------------------------------------------------------------
// Float gradient with the exact Mehler-Solmajer / exponential desolvation
// derivatives, used once per FIRE search (calcgradient.cl:109-1003).  Forces
// are float; intra forces use LDS float atomics of one team.
// ---------------------------------------------------------------------------
template <int TW, int NC, int MF, bool PL>
DEV void float_gradient(const EvalCtx<TW, NC>& X, const float (&gene)[64 / TW], float (&grad)[64 / TW]) {
    using TM = Team<TW>;
    const LigandDev* L = X.L;
    const GridDev& G = X.G;
    const TeamView& tv = X.tv;
    const SharedView& sv = X.sv;
    const int tl = TM::lane();
    const int T = X.ls.T, P = X.ls.P, NG = X.ls.NG;
    const bool has_lig = X.ls.has_lig;
    (void)L;
    float* ffx = reinterpret_cast<float*>(tv.fx);
    float* ffy = reinterpret_cast<float*>(tv.fy);
    float* ffz = reinterpret_cast<float*>(tv.fz);
    float* tacc = reinterpret_cast<float*>(tv.gi);

    gene_trig<TW>(X.ls, sv, tv, gene);
#pragma unroll
    for (int k = 0; k < NC; ++k) {
        const uint32_t o = X.A.slot[k];
        *at(ffx, o) = 0.f; *at(ffy, o) = 0.f; *at(ffz, o) = 0.f;
    }
    for (int t = tl; t < T; t += TW) tacc[t] = 0.f;
    wave_sync();
    const Pose pose = read_pose(tv, has_lig);
    float3 c[NC];
    compute_coords<TW, NC, 1>(X, pose, c);   // by atom: first copies
    wave_sync();
    float3 gin[NC];
    const uint32_t g3 = G.g3, ne = (uint32_t)(G.nmaps - 2) * g3, nd = ne + g3;
#pragma unroll
    for (int k = 0; k < NC; ++k) {
        gin[k] = make_float3(0.f, 0.f, 0.f);
        if (X.A.ign[k]) continue;
        const float x = c[k].x, y = c[k].y, z = c[k].z;
        if (!((x >= 0.f) && (y >= 0.f) && (z >= 0.f) && (x < (float)(G.gx - 1)) && (y < (float)(G.gy - 1)) &&
              (z < (float)(G.gz - 1)))) {
            gin[k] = make_float3(16777216.0f, 16777216.0f, 16777216.0f);
            continue;
        }
        const uint32_t xl = (uint32_t)floorf(x), yl = (uint32_t)floorf(y), zl = (uint32_t)floorf(z);
        const uint32_t xh = (uint32_t)ceilf(x), yh = (uint32_t)ceilf(y), zh = (uint32_t)ceilf(z);
        const float dx = x - (float)xl, dy = y - (float)yl, dz = z - (float)zl;
        const uint32_t o[8] = {xl + yl * G.g1 + zl * G.g2, xl + yh * G.g1 + zl * G.g2, xl + yl * G.g1 + zh * G.g2,
                               xl + yh * G.g1 + zh * G.g2, xh + yl * G.g1 + zl * G.g2, xh + yh * G.g1 + zl * G.g2,
                               xh + yl * G.g1 + zh * G.g2, xh + yh * G.g1 + zh * G.g2};
        const uint32_t mb[3] = {X.A.mapoff[k], ne, nd};
        const float sc[3] = {1.0f, X.A.q[k], fabsf(X.A.q[k])};
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            float cb[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) cb[i] = load_pt<MF>(G.data, mb[m] + o[i]).x;
            const float vx0 = (1.0f - dy) * (cb[4] - cb[0]) + dy * (cb[5] - cb[1]);
            const float vx1 = (1.0f - dy) * (cb[6] - cb[2]) + dy * (cb[7] - cb[3]);
            const float vy0 = (1.0f - dx) * (cb[1] - cb[0]) + dx * (cb[5] - cb[4]);
            const float vy1 = (1.0f - dx) * (cb[3] - cb[2]) + dx * (cb[7] - cb[6]);
            const float vz0 = (1.0f - dx) * (cb[2] - cb[0]) + dx * (cb[6] - cb[4]);
            const float vz1 = (1.0f - dx) * (cb[3] - cb[1]) + dx * (cb[7] - cb[5]);
            gin[k].x += sc[m] * ((1.0f - dz) * vx0 + dz * vx1);
            gin[k].y += sc[m] * ((1.0f - dz) * vy0 + dz * vy1);
            gin[k].z += sc[m] * ((1.0f - dy) * vz0 + dy * vz1);
        }
    }
    const float spacing = G.spacing;
    const float half_smooth = X.ls.half_smooth;
    const float DA = -8.5525f, DB = 78.4f - (-8.5525f), DK = 7.7839f;
    const float DBH = DB * 0.003627f, DBHK = DBH * DK;
    for (int p = tl, r = tl; p < P; p += TW, r += pair_stride<TW, PL>) {
        const PairRec pr = compact_pairs(TW * NC, true) ? unpack(sv.pc[p]) : unpack(sv.pa[r], sv.pb[r]);
        // the pair's atoms in the list's order, first copies: float sums keep their order
        const uint32_t fl = sv.px[p].flags, atoms = sv.px[p].atoms;
        const int i = (int)(atoms & 0xffffu), j = (int)(atoms >> 16);
        const float sx = tv.cx[i] - tv.cx[j], sy = tv.cy[i] - tv.cy[j], sz = tv.cz[i] - tv.cz[j];
        const float dist = sqrtf(sx * sx + sy * sy + sz * sz);
        float d = dist * spacing;
        float sd;
        if (d <= pr.reqm - half_smooth) sd = d + half_smooth;
        else if (d < pr.reqm + half_smooth) sd = pr.reqm;
        else sd = d - half_smooth;
        const int m = (int)(fl & 0xffu), n = (int)((fl >> 8) & 0xffu);
        float pg = 0.f;
        if (d < 8.0f) {
            pg += (-(float)m * pr.ac) / powf(sd, (float)(m + 1));
            pg += ((float)n * pr.bd) / powf(sd, (float)(n + 1));
        }
        if (d < 20.48f) {
            if (d < X.ls.elec_min) d = X.ls.elec_min;
            const float ex = __expf(DBH * d);
            const float upper = DA * (ex + DK) * (ex + DK) + DB * ex * (DBHK * d + ex + DK);
            const float lw = DA * (ex + DK) + DB * ex;
            const float lower = d * d * lw * lw;
            pg += -pr.cq * (upper / lower);
            pg += pr.dsol * X.ls.coeff_desolv * -0.077160f * d * __expf(-0.038580f * d * d);
        }
        if (fl & kPairCgG0) pg += 50.0f;
        const float fx = pg * (-sx / dist), fy = pg * (-sy / dist), fz = pg * (-sz / dist);
        atomicAdd(&ffx[i], -fx); atomicAdd(&ffy[i], -fy); atomicAdd(&ffz[i], -fz);
        atomicAdd(&ffx[j], fx); atomicAdd(&ffy[j], fy); atomicAdd(&ffz[j], fz);
    }
    wave_sync();
    float3 F[NC];
    float sfx = 0.f, sfy = 0.f, sfz = 0.f, tx = 0.f, ty = 0.f, tz = 0.f;
    const float g0 = tv.pg[0], g1 = tv.pg[1], g2 = tv.pg[2];
#pragma unroll
    for (int k = 0; k < NC; ++k) {
        const int a = tl + TW * k;
        F[k] = make_float3(0.f, 0.f, 0.f);
        if (X.A.valid[k]) {
            F[k] = make_float3(gin[k].x / spacing + ffx[a], gin[k].y / spacing + ffy[a], gin[k].z / spacing + ffz[a]);
            if (X.A.lig[k]) {
                sfx += F[k].x; sfy += F[k].y; sfz += F[k].z;
                const float rx = (c[k].x - g0) * spacing, ry = (c[k].y - g1) * spacing, rz = (c[k].z - g2) * spacing;
                tx += ry * F[k].z - rz * F[k].y;
                ty += rz * F[k].x - rx * F[k].z;
                tz += rx * F[k].y - ry * F[k].x;
            }
        }
    }
    sfx = TM::sum(sfx); sfy = TM::sum(sfy); sfz = TM::sum(sfz);
    tx = TM::sum(tx); ty = TM::sum(ty); tz = TM::sum(tz);
    float gval = 0.f;
    if (tl < 3) gval = (tl == 0 ? sfx : tl == 1 ? sfy : sfz) * spacing;
    if (has_lig && tl >= 3 && tl < 6) {   // calcgradient.cl:714-873 (fmod)
        const float tlen = sqrtf(tx * tx + ty * ty + tz * tz);
        const bool small = tlen < 1e-3f;
        const float oscale = small ? 1.0f : tlen * (1.0f / 1e-3f);
        const float sc = small ? 0.5f - tlen * tlen / 48.0f : 0.0005f / tlen;
        const float4 qt = make_float4(tx * sc, ty * sc, tz * sc, small ? 1.0f - tlen * tlen * 0.125f : 0.99999988f);
        const float4 tq = qmul(qt, pose.q);
        const float cur_phi = fmod_pi2(kTwoPi + pose.phi);
        const float cur_theta = fmod_pi2(kTwoPi + pose.theta);
        const float cur_rot = fmod_pi2(kTwoPi + pose.rotangle);
        const float tgt_rot = 2.0f * fast_acos(tq.w);
        const float inv_sin = rsqrtf(1.0f - tq.w * tq.w);
        const float tgt_theta = kTwoPi + pose.is_theta_gt_pi * fast_acos(tq.z * inv_sin);
        const float tgt_phi = fmod_pi2(atan2f(pose.is_theta_gt_pi * tq.y, pose.is_theta_gt_pi * tq.x) + kTwoPi);
        const float corr = 4.0f * pose.sin_half * pose.sin_half;
        if (tl == 3) gval = oscale * (fmodf(tgt_phi - cur_phi + kPi, kTwoPi) - kPi) * pose.sin_theta * pose.sin_theta * corr * kDegToRad;
        if (tl == 4) gval = oscale * (fmodf(tgt_theta - cur_theta + kPi, kTwoPi) - kPi) * corr * kDegToRad;
        if (tl == 5) gval = oscale * (fmodf(tgt_rot - cur_rot + kPi, kTwoPi) - kPi) * kDegToRad;
    }
    for (int t = tl; t < T; t += TW) {
        const int2 ab = sv.tor_atoms[t];
        const float4 r0 = make_float4(tv.cx[ab.x], tv.cy[ab.x], tv.cz[ab.x], 0.f);
        const float ax = tv.cx[ab.y] - r0.x, ay = tv.cy[ab.y] - r0.y, az = tv.cz[ab.y] - r0.z;
        const float inv = rsqrtf(ax * ax + ay * ay + az * az);
        tv.tor[t].q = make_float4(ax * inv, ay * inv, az * inv, 0.f);
        tv.tor[t].r0 = r0;
    }
    wave_sync();
#pragma unroll
    for (int k = 0; k < NC; ++k) {
        for_bonds<TW, NC>(X, k, &TorRec::r0, [&](int t, const float4& ax, const float4& r0) {
            const float rx = (c[k].x - r0.x) * spacing, ry = (c[k].y - r0.y) * spacing, rz = (c[k].z - r0.z) * spacing;
            const float qx = ry * F[k].z - rz * F[k].y, qy = rz * F[k].x - rx * F[k].z, qz = rx * F[k].y - ry * F[k].x;
            atomicAdd(&tacc[t], (ax.x * qx + ax.y * qy + ax.z * qz) * kDegToRad);
        });
    }
    wave_sync();
    const float conv = spacing * spacing * 1.0f / (kDegToRad * kDegToRad);
#pragma unroll
    for (int j = 0; j < TM::kGPL; ++j) {
        const int g = tl + TW * j;
        float gv = 0.f;
        if (g < 6) gv = gval;
        else if (g < NG) gv = tacc[g - 6];
        if (g > 2) gv *= conv;
        grad[j] = g < NG ? gv : 0.f;
    }
}

// ---------------------------------------------------------------------------
// Kernel arguments and common prologue
// ---------------------------------------------------------------------------
struct Launch {
    const LigandDev* L;
    GridDev G;
    SearchDev S;
    JobBuffers B;
    const float* in_geno;
    int stride;          // floats from one genotype (and gradient) to the next
    float* out_e;
    float* out_g;
    int n;
    int mode;
    float lig_scale;     // SW: 1/sqrt(atoms)
    float gene_scale;    // SW: 1/sqrt(genes)
};

// A passed AutoStop test has ended the job: generation kernels do nothing.
#define JOB_STOPPED(b) ((b).stop != nullptr && *(b).stop != 0)

#define KERNEL_PROLOGUE(TW, NC, PL, GRAD)                                      \
    extern __shared__ __align__(16) char lds[];                                \
    using TM = Team<TW>;                                                       \
    constexpr int GPL = TM::kGPL;                                              \
    EvalCtx<TW, NC> X;                                                         \
    X.L = a.L;                                                                 \
    X.G = a.G;                                                                 \
    X.A.template load<PL, GRAD>(a.L, a.G);   /* its loads run beside the staging's */ \
    X.ls.load(a.L);                                                            \
    stage<TW, NC, PL, GRAD>(a.L, lds, X.sv, X.tv);                             \
    const int tl = TM::lane();                                                 \
    (void)tl;                                                                  \
    const int team_idx = (int)(blockIdx.x * (blockDim.x / TW) + threadIdx.x / TW); \
    (void)team_idx;

// Entity choice of every LS kernel (e.g. kernel3.cl:104-117): team lane 0
// draws from its own stream (state *st0) when le == 0.
template <int TW>
DEV int ls_entity(const SearchDev& S, int le, uint32_t* st0) {
    int ent = le;
    if (le == 0) {
        float r = 0.f;
        if (Team<TW>::lane() == 0) { uint32_t s = *st0; r = randf(s); *st0 = s; }
        r = Team<TW>::bcast(r, 0);
        if (100.0f * r > S.lsearch_rate) ent = S.num_ls;
    }
    // the reference reads entity num_ls even when num_ls == pop_size (the next
    // run's first entity, or past the buffer for the last run); clamp instead
    return ent < S.pop_size ? ent : S.pop_size - 1;
}

// ---------------------------------------------------------------------------
// Launch helpers
// ---------------------------------------------------------------------------
struct Shape {
    int tw, nc;
    bool pl;
    size_t lds;
    int threads;   // workgroup size (64 to 1024)
};

// LDS of a compute unit and the unit it is handed out in, and the wavefronts
// that fit on one at the kernels' register budget (four on each of its four
// SIMDs).
constexpr size_t kCuLds = 160 * 1024, kLdsUnit = 1280;
constexpr int kCuWaves = 16;
constexpr int kCus = 256;

// Workgroups of `threads` threads and `lds` bytes that fit on a compute unit.
inline int groups_per_cu(size_t lds, int threads) {
    const int by_lds = lds ? (int)(kCuLds / ((lds + kLdsUnit - 1) / kLdsUnit * kLdsUnit)) : kCuWaves;
    const int by_waves = kCuWaves / (threads / kWave);
    return by_lds < by_waves ? by_lds : by_waves;
}

// Chooses the team width and atom chunks for a ligand: the requested width,
// else 32-lane teams (two individuals per wavefront) up to 128 atoms and
// 64-lane teams beyond; 16-lane teams (four per wavefront) only for ligands
// of at most 32 atoms.  Jobs pass the width fixed when they start.  Pair
// records are staged in LDS while at least 12 wavefronts fit on a compute unit
// with them; beyond that they are read through L1/L2.  grad: the kernel
// evaluates gradients (KERNEL_PROLOGUE).
inline Shape choose_shape(const LigandDev& L, int team_width_hint, bool grad, int threads = kGroupThreads) {
    Shape s{};
    s.threads = threads;
    const int N = L.num_atoms;
    const int tw = team_lanes_for(N, team_width_hint);
    s.tw = tw;
    const int per = (N + tw - 1) / tw;
    s.nc = per <= 1 ? 1 : (per <= 2 ? 2 : 4);
    const size_t lds = lds_bytes_for(s.tw, s.nc, L.num_rotbonds, L.num_pairs, true, grad, threads);
    s.pl = groups_per_cu(lds, threads) * (threads / kWave) >= 12;
    s.lds = lds_bytes_for(s.tw, s.nc, L.num_rotbonds, L.num_pairs, s.pl, grad, threads);
    return s;
}

// Shape of a persistent local-search launch of so many searches.  All teams of
// a workgroup share one copy of the pair records, so the more threads it has,
// the more wavefronts a compute unit holds with the records in LDS.  Of the
// workgroups that can hold every search at once, the one that spreads them
// most evenly over the compute units; if none can, the one that puts most
// wavefronts on a compute unit; the smaller on ties, and never fewer than 12
// wavefronts where more are needed (the records then stay in memory).  M
// evals/s with the records in LDS by this rule against 256 threads and memory
// or fewer wavefronts: 54 atoms, ADAM, nrun 100 312 against 258; 64 atoms,
// FIRE, nrun 60 185 against 147, Solis-Wets 165 against 127.  A server's
// launches keep 256 threads: larger workgroups need half or all of a compute
// unit free at once, which the launches of other requests seldom leave (24
// ligands in 16 slots 0.56 s against 0.50 s).  So do ADADELTA's (uneven) of
// more searches than fit at once, unless 512 hold records that 256 leave in
// memory: a workgroup keeps its place until its last search ends, and
// ADADELTA's differ in length by ten times.  M evals/s in 256 threads against
// what other searches take there: 45 atoms, nrun 50 293 against 242 (on 126^3
// maps 330 against 367); 60 atoms, nrun 50 / 100 147 / 202 against 132 / 182;
// 72 atoms, nrun 50 86 against 73; 90 atoms, nrun 40 / 100 49 / 91 against 42 /
// 73.  54 atoms, in 512: nrun 50 / 100 221 / 288 against 230 / 269, on 126^3
// maps 283 / 311 against 260 / 278.
// fixed: the threads if they are not to be chosen, else 0.
inline Shape choose_ls_shape(const LaunchArgs& la, int searches, bool grad, int fixed, bool uneven = false) {
    const LigandDev& L = *la.lig_host;
    Shape s = choose_shape(L, la.team_hint, grad, fixed ? fixed : kGroupThreads);
    if (la.crowded || fixed) return s;
    // wavefronts of all the launches that share the device, were they like this one
    const int64_t need = ((int64_t)searches * s.tw + kWave - 1) / kWave * la.share;
    const bool small = s.pl || compact_pairs(s.tw * s.nc, grad);   // uneven searches stay in 256 threads
    int64_t best = INT64_MIN;
    for (int t = kGroupThreads; t <= 4 * kGroupThreads; t += kGroupThreads) {   // whole rounds of the four SIMDs
        const size_t lds = lds_bytes_for(s.tw, s.nc, L.num_rotbonds, L.num_pairs, true, grad, t);
        const int w = t / kWave, fit = groups_per_cu(lds, t);
        const int64_t groups = (need + w - 1) / w;
        const bool all = groups <= (int64_t)fit * kCus;
        if (!all && (fit * w < 12 || (uneven && (small || t > 2 * kGroupThreads)))) continue;
        // all at once: prefer few wavefronts on the fullest compute unit; else many in all
        const int64_t score = all ? 2 * kCuWaves - (groups + kCus - 1) / kCus * w : fit * w - kCuWaves;
        if (score > best) {
            best = score;
            s.pl = true;
            s.lds = lds;
            s.threads = t;
        }
    }
    return s;
}

// Dispatches a kernel template over (TW, NC, MF, PL).  KT must be a
// template<int TW, int NC, int MF, bool PL> __global__ function.
#define ADGPU_DISPATCH(KT, shape, mf, body)                                                     \
    do {                                                                                        \
        auto go_ = [&](auto tw_, auto nc_, auto mf_, auto pl_) {                                 \
            constexpr int TW_ = decltype(tw_)::value, NC_ = decltype(nc_)::value;               \
            constexpr int MF_ = decltype(mf_)::value;                                           \
            constexpr bool PL_ = decltype(pl_)::value;                                          \
            auto kfn = KT<TW_, NC_, MF_, PL_>;                                                  \
            body;                                                                               \
        };                                                                                      \
        auto mf_sel = [&](auto tw_, auto nc_, auto pl_) {                                       \
            if ((mf) == ADGPU_MAP_F16) go_(tw_, nc_, std::integral_constant<int, ADGPU_MAP_F16>{}, pl_); \
            else if ((mf) == ADGPU_MAP_BF16) go_(tw_, nc_, std::integral_constant<int, ADGPU_MAP_BF16>{}, pl_); \
            else go_(tw_, nc_, std::integral_constant<int, ADGPU_MAP_F32>{}, pl_);             \
        };                                                                                      \
        auto pl_sel = [&](auto tw_, auto nc_) {                                                 \
            if ((shape).pl) mf_sel(tw_, nc_, std::true_type{});                                 \
            else mf_sel(tw_, nc_, std::false_type{});                                           \
        };                                                                                      \
        using I16 = std::integral_constant<int, 16>;                                            \
        using I32 = std::integral_constant<int, 32>;                                            \
        using I64 = std::integral_constant<int, 64>;                                            \
        using N1 = std::integral_constant<int, 1>;                                              \
        using N2 = std::integral_constant<int, 2>;                                              \
        using N4 = std::integral_constant<int, 4>;                                              \
        if ((shape).tw == 16) {                                                                 \
            if ((shape).nc == 1) pl_sel(I16{}, N1{});                                           \
            else pl_sel(I16{}, N2{});                                                           \
        } else if ((shape).tw == 32) {                                                          \
            if ((shape).nc == 1) pl_sel(I32{}, N1{});                                           \
            else if ((shape).nc == 2) pl_sel(I32{}, N2{});                                      \
            else pl_sel(I32{}, N4{});                                                           \
        } else {                                                                                \
            if ((shape).nc == 1) pl_sel(I64{}, N1{});                                           \
            else if ((shape).nc == 2) pl_sel(I64{}, N2{});                                      \
            else pl_sel(I64{}, N4{});                                                           \
        }                                                                                       \
    } while (0)

}  // namespace adgpu
