// Device code of the Fletcher TTI time step for gfx950 (CDNA4, wave64).
//
// One time step updates the coupled pseudo-acoustic fields p, q (reference
// original/sample.h:32-90 and der1der1/sample.h:35-123):
//   pp <- 2 pc - pp + dt^2 rhsp(pc, qc),   qp <- 2 qc - qp + dt^2 rhsq(pc, qc)
// over iz,iy,ix in [bord, s-bord) (original/OpenMP/openmp_propagate.c:27-29).
//
// Device layout of the wavefields: each time level is one array of (p, q) pairs,
// cell c = (z*sy + y)*px + x with the row pitch px >= sx a multiple of 16 cells
// (128-byte rows), p at 2c and q at 2c+1.  A step reads the current level (stencil) and
// the previous one (own cell) and overwrites the previous one; the roles then swap.
// The coefficients are records of one cell each, at the same pitched cell index.
//
// Kernels here (the z-marching step kernels are in fl_step.h, fl_step2.h and fl_step_batch.h):
//   direct_dercross  the reference's direct 64-point DerCross form
//       (original/derivatives.h:59-68), z-marching through LDS planes.
//   der1_pass        pass 1 of the two-pass form (der1der1/OpenMP/openmp_propagate.c:24-76).
//   insert_source    p[i] += s, q[i] += s (original/OpenMP/openmp_insertsource.c:7-12).
//   field_pack / field_unpack   one field between the reference layout and a level.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace fl {

// 8th-order weights: the reference's float literals (original/derivatives.h:13-41).
#define FL_L1 0.8f
#define FL_L2 -0.2f
#define FL_L3 0.0380952380952381f
#define FL_L4 -0.0035714285714285713f
#define FL_L11 0.64f
#define FL_L12 -0.16f
#define FL_L13 0.03047619047619047618f
#define FL_L14 -0.00285714285714285713f
#define FL_L22 0.04f
#define FL_L23 -0.00761904761904761904f
#define FL_L24 0.00071428571428571428f
#define FL_L33 0.00145124716553287981f
#define FL_L34 -0.00013605442176870748f
#define FL_L44 0.00001275510204081632f
#define FL_K0 -2.84722222222222222222f
#define FL_K1 1.6f
#define FL_K2 -0.2f
#define FL_K3 0.02539682539682539682f
#define FL_K4 -0.00178571428571428571f

// Coefficient storage modes.
enum CoefMode : int {
    CM_F32 = 0,   // 10 FP32 volumes, precomp.h layout
    CM_BF16 = 1,  // 10 BF16 volumes; v2* pre-multiplied by dt^2
    CM_F16 = 2,   // 10 FP16 volumes; v2* pre-multiplied by dt^2
    CM_F16R = 3,  // 4 FP16 velocity factors (times dt^2) and theta, phi as u16 turns
    CM_F32R = 4,  // 4 FP32 velocity factors (precomp.h values) and theta, phi as FP32 turns
    CM_Q16R = 5,  // 4 velocity factors (times dt^2) in per-cell block floating point (15-bit
                  // mantissas, shared exponent), theta, phi as u16 turns
};

// Bytes of one cell's coefficient record.
__host__ __device__ constexpr int rec_bytes(int cm)
{
    return cm == CM_F32 ? 40 : (cm == CM_F16R || cm == CM_Q16R) ? 12 : cm == CM_F32R ? 24 : 20;
}

// Order of the precomp.h coefficients (0 ch1dxx, 1 ch1dyy, 2 ch1dzz, 3 ch1dxy, 4 ch1dyz,
// 5 ch1dxz, 6 v2px, 7 v2pz, 8 v2sz, 9 v2pn) within a stored record: slot s holds
// coefficient REC_ORDER[s].  The step kernel has the two lanes of a cell (p and q) load
// one half of the record each and broadcast it to the pair:
//   FP32 (40 B):        p lane {0 1 2 3 6}, q lane {4 5 7 8 9}; the fifth value is the
//                       lane's own v2px / v2pn.  On the device the record is held in two
//                       arrays of the pitched cells (fp32_part2): 32 bytes {0 1 2 3 4 5 7 8}
//                       at 32 c, then, after all cells, 8 bytes {6 9} at 32 np + 8 c.  A
//                       lane's two loads (16 and 4 bytes) then each read whole lines
//                       across the wave, which lets them stream non-temporally.
//   BF16 / FP16 (20 B): p lane {0 1 2 3}, q lane {4 5 7 8}, both {6 9}.
// The recompute inputs are v2px, v2pz, v2sz, v2pn, theta, phi (0..5), stored as
//   FP16 and block floating-point recompute (12 B): words (v2px, v2pn), (v2pz, v2sz),
//                          (theta, phi), loaded whole by both lanes;
//   FP32 recompute (24 B): p lane {v2px, v2pz, theta}, q lane {v2pn, v2sz, phi}.
__host__ __device__ constexpr int rec_order32(int s)
{
    constexpr int o[10] = {0, 1, 2, 3, 6, 4, 5, 7, 8, 9};
    return o[s];
}
// Byte offset of the 8-byte part of the FP32 records of a grid of np pitched cells.
__host__ __device__ constexpr long long fp32_part2(long long np) { return np * 32; }

__host__ __device__ constexpr int rec_order16(int s)
{
    constexpr int o[10] = {0, 1, 2, 3, 4, 5, 7, 8, 6, 9};
    return o[s];
}
__host__ __device__ constexpr int rec_order_r16(int s)
{
    constexpr int o[6] = {0, 3, 1, 2, 4, 5};
    return o[s];
}
__host__ __device__ constexpr int rec_order_r32(int s)
{
    constexpr int o[6] = {0, 1, 4, 3, 2, 5};
    return o[s];
}

struct StepArgs {
    float *prev;          // level read at the own cell and overwritten (pp, qp)
    const float *cur;     // level read with the stencil (pc, qc)
    const void *coef;     // coefficient records: per cell its values, consecutive
    const float *dvx, *dvy;  // TWOPASS: (pDx, qDx) and (pDy, qDy) pair volumes
    float dxxinv, dyyinv, dzzinv, dxinv, dyinv, dzinv, dt;
    float vq;             // CM_Q16R: 2^ebase, the unit of the block exponent 0
    int sx, sy, sz, bord, px;
    int ntx, nty, zt, nblk;  // tiles along x, y; z chunk depth; logical blocks
    int sw;                  // tile columns per strip of the workgroup order (tile_of)
    int xorg;                // x of the first tile column (0 or bord)
    // step index it: it_host for a plain launch.  Inside a multi-step run, run points at
    // the run's control block {k0, k1, it_base, src_n}: the step reads its counter
    // k = run[par], takes it = it_base + 1 + k and publishes run[1 - par] = k + 1 for the
    // following step, so a captured graph replays for any start step and run length.
    int it_host;
    int *run;
    int par;
    // source of the next step added to this step's output (multi-step runs): src_tab[k+1]
    // while k + 1 < src_n; src_idx is the pitched cell index
    const float *src_tab;
    long long src_idx;
    // receiver plane: slot it/rec_every-1 of trace when it % rec_every == 0
    float *trace;
    int rec_iz, rec_every, rec_slots;
};

// Per-launch scalars resolved from StepArgs at kernel entry.
struct StepCtl {
    float *trace;   // plane to write this step, or nullptr
    float src_add;
    bool do_src;
    int it;         // step index
};

// Wave-uniform copies (readfirstlane) of values the compiler computes or loads in vector
// registers although every lane holds the same value: integer divisions by runtime values
// (VALU only) and loads from memory the kernel also writes.  Without them such values
// occupy VGPRs for the whole tile.
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ float uni(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
}
__device__ __forceinline__ long long uni(long long v)
{
    const unsigned long long u = (unsigned long long)v;
    const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)u);
    const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(u >> 32));
    return (long long)(((unsigned long long)hi << 32) | lo);
}
// Pointers into device memory: rebuilt as global (address space 1) pointers, so that
// accesses through them stay global_* instructions.  A generic pointer would make them
// flat_* instructions, which may complete out of order with the buffer loads and make the
// compiler drain the whole load queue (s_waitcnt vmcnt(0)) before the next use of any load.
template <class T>
__device__ __forceinline__ T *uni(T *p)
{
    typedef __attribute__((address_space(1))) T global_t;
    return (T *)(global_t *)(uintptr_t)uni((long long)(uintptr_t)p);
}

// Control block of a multi-step run (StepArgs.run, BatchArgs.run).
enum { RUN_K0 = 0, RUN_K1 = 1, RUN_IT_BASE = 2, RUN_SRC_N = 3, RUN_WORDS = 4 };

__device__ __forceinline__ StepCtl step_ctl(const StepArgs &a)
{
    StepCtl c;
    int k = 0, it = a.it_host, src_n = 0;
    if (a.run) {
        k = a.run[a.par];
        it = a.run[RUN_IT_BASE] + 1 + k;
        src_n = a.run[RUN_SRC_N];
    }
    c.do_src = a.src_tab && (k + 1) < src_n;
    c.src_add = c.do_src ? a.src_tab[k + 1] : 0.0f;
    c.trace = nullptr;
    if (a.trace && a.rec_every > 0 && it % a.rec_every == 0) {
        const int slot = it / a.rec_every - 1;
        if (slot >= 0 && slot < a.rec_slots)
            c.trace = a.trace + (long long)slot * (a.sx - 2 * a.bord) * (a.sy - 2 * a.bord);
    }
    c.trace = uni(c.trace);
    c.src_add = uni(c.src_add);
    c.it = uni(it);
    return c;
}

// The step kernels are compiled with -ffp-contract=off and fuse multiply-adds explicitly,
// so every copy of an expression rounds identically (results do not depend on tile or
// chunk shapes).  The sums keep the reference association order (derivatives.h:47,53):
// ((w1 d1 + w2 d2) + w3 d3) + w4 d4, each step one FMA.
// SC = false leaves the sum unscaled (dinv unused): the caller applies the grid spacing
// once to the combination instead.
template <bool SC = true>
__device__ __forceinline__ float fd1(float d1, float d2, float d3, float d4, float dinv)
{
    float t = FL_L1 * d1;
    t = __builtin_fmaf(FL_L2, d2, t);
    t = __builtin_fmaf(FL_L3, d3, t);
    t = __builtin_fmaf(FL_L4, d4, t);
    return SC ? t * dinv : t;
}
template <bool SC = true>
__device__ __forceinline__ float fd2(float c, float s1, float s2, float s3, float s4, float d2inv)
{
    float t = FL_K0 * c;
    t = __builtin_fmaf(FL_K1, s1, t);
    t = __builtin_fmaf(FL_K2, s2, t);
    t = __builtin_fmaf(FL_K3, s3, t);
    t = __builtin_fmaf(FL_K4, s4, t);
    return SC ? t * d2inv : t;
}

template <bool SC = true>
__device__ __forceinline__ float der1_lds(const float *p, int s, float dinv)
{
    return fd1<SC>(p[s] - p[-s], p[2 * s] - p[-2 * s], p[3 * s] - p[-3 * s], p[4 * s] - p[-4 * s], dinv);
}

template <bool SC = true>
__device__ __forceinline__ float der2_lds(const float *p, int s, float d2inv)
{
    return fd2<SC>(p[0], p[s] + p[-s], p[2 * s] + p[-2 * s], p[3 * s] + p[-3 * s], p[4 * s] + p[-4 * s],
               d2inv);
}

// Both derivatives along one axis from the same neighbours (c the own value), each sum as above.
template <bool SC>
__device__ __forceinline__ void der12_lds(const float *p, int s, float c, float dinv, float d2inv, float &d1, float &d2)
{
    const float a1 = p[s], b1 = p[-s], a2 = p[2 * s], b2 = p[-2 * s], a3 = p[3 * s], b3 = p[-3 * s];
    const float a4 = p[4 * s], b4 = p[-4 * s];
    d1 = fd1<SC>(a1 - b1, a2 - b2, a3 - b3, a4 - b4, dinv);
    d2 = fd2<SC>(c, a1 + b1, a2 + b2, a3 + b3, a4 + b4, d2inv);
}

// q[0..8] = values at z-4..z+4
template <bool SC = true>
__device__ __forceinline__ float der1_q(const float *q, float dinv)
{
    return fd1<SC>(q[5] - q[3], q[6] - q[2], q[7] - q[1], q[8] - q[0], dinv);
}

template <bool SC = true>
__device__ __forceinline__ float der2_q(const float *q, float d2inv)
{
    return fd2<SC>(q[4], q[5] + q[3], q[6] + q[2], q[7] + q[1], q[8] + q[0], d2inv);
}

__device__ __forceinline__ float bf16_to_f32(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
__device__ __forceinline__ float f16_to_f32(uint16_t h)
{
    _Float16 v = __builtin_bit_cast(_Float16, h);
    return (float)v;
}

// The 10 per-cell coefficients, in precomp.h order; v2* include dt^2 when `scaled`.
struct Coef {
    float c[10];
};

// Coefficient combination + leapfrog, association order of original/sample.h:46-86.
template <int CM>
__device__ __forceinline__ void combine(const Coef &k, float dt, float pxx, float pyy, float pzz,
                                        float pxy, float pyz, float pxz, float qxx, float qyy,
                                        float qzz, float qxy, float qyz, float qxz, float pc,
                                        float qc, float &pp, float &qp)
{
    const float h1p = k.c[0] * pxx + k.c[1] * pyy + k.c[2] * pzz + k.c[3] * pxy + k.c[5] * pxz +
                      k.c[4] * pyz;
    const float h2p = pxx + pyy + pzz - h1p;
    const float h1q = k.c[0] * qxx + k.c[1] * qyy + k.c[2] * qzz + k.c[3] * qxy + k.c[5] * qxz +
                      k.c[4] * qyz;
    const float h2q = qxx + qyy + qzz - h1q;
    const float h1pmq = h1p - h1q;
    const float h2pmq = h2p - h2q;
    const float rhsp = k.c[6] * h2p + k.c[7] * h1q + k.c[8] * h1pmq;
    const float rhsq = k.c[9] * h2p + k.c[7] * h1q - k.c[8] * h2pmq;
    if constexpr (CM == CM_F32) {
        pp = 2.0f * pc - pp + rhsp * dt * dt;
        qp = 2.0f * qc - qp + rhsq * dt * dt;
    } else {  // dt^2 folded into the stored v2* factors
        pp = 2.0f * pc - pp + rhsp;
        qp = 2.0f * qc - qp + rhsq;
    }
}

// Logical block id from the hardware one.  Workgroups are dealt to the 8 XCDs
// round-robin (block b runs on XCD b%8); this gives each XCD a contiguous range of
// logical tiles so neighbouring tiles (shared halos) meet in the same L2.
__device__ __forceinline__ int xcd_remap(int b, int g)
{
    return (b & 7) * (g >> 3) + (b >> 3);
}

// Odd steps take the logical blocks in reverse (t -> nblk-1-t) and march each z chunk from
// its top plane down: a step then starts on the tiles, and in each tile on the planes, that
// the step before ended on, whose levels were the last to pass through the memory-side
// cache.  Each tile's result does not depend on the order or the direction.  At 344^3 the
// reversed order made the FP32 step 1.2% faster (12-row tiles) and the downward march another
// 0.8%; FP16 recompute (8-row tiles, both fields per lane) 1.6% and 0.9%.
__device__ __forceinline__ int step_order(int t, int n, int it) { return (it & 1) ? n - 1 - t : t; }
__device__ __forceinline__ bool step_down(int it) { return (it & 1) != 0; }

// Tile (tx, ty, tz) of logical block t: z chunks outermost; inside a chunk, strips of sw
// tile columns (the last one narrower) walked row by row.  The tiles an XCD holds at once
// (consecutive t) then form a compact block of the plane instead of part of one long row,
// so the halos they share meet in that XCD's L2.  sw >= ntx is the plain row-major order.
__device__ __forceinline__ void tile_of(int t, int ntx, int nty, int sw, int &tx, int &ty, int &tz)
{
    const int per = ntx * nty;
    tz = t / per;
    const int r = t - tz * per;
    const int x0 = r / (sw * nty) * sw;
    const int w = min(sw, ntx - x0);
    const int u = r - x0 * nty;
    ty = u / w;
    tx = x0 + (u - ty * w);
}

// ---------------------------------------------------------------------------------
// Kernels launched by the driver translation unit only (the kernel instantiation units
// define FL_NO_AUX_KERNELS).
#ifndef FL_NO_AUX_KERNELS

struct DirectArgs {
    float *prev;
    const float *cur;
    const float *coef;    // FP32 records (the two arrays of rec_order32's note)
    long long np;         // pitched cells of the grid
    float dxxinv, dyyinv, dzzinv, dxyinv, dxzinv, dyzinv, dt;
    int sx, sy, sz, bord, px, zt;
    int ntx, nty, nblk;   // tiles of DX_TX x DX_TY cells along x, y; z chunks of zt planes
    float *trace;
    int rec_iz;
};

// Four consecutive cells along x of one field: one expression evaluates four derivatives with
// the same operations in the same order.
typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint32_t u2v __attribute__((ext_vector_type(2)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));

// Der2 of derivatives.h:53 in the reference's association order: g(m) is the values m cells
// along the axis.
template <class G>
__device__ __forceinline__ f4 der2_f4(G g, float d2inv)
{
    return (FL_K0 * g(0) + FL_K1 * (g(1) + g(-1)) + FL_K2 * (g(2) + g(-2)) + FL_K3 * (g(3) + g(-3)) +
            FL_K4 * (g(4) + g(-4))) *
           d2inv;
}

// The running sum over the ten coefficient groups of DerCross (derivatives.h:59-68), g(m, n)
// the sum of group (m, n): the same additions in the same order.
template <class G>
__device__ __forceinline__ f4 cross_sum(G g, float dinv)
{
    f4 s = FL_L11 * g(1, 1);
    s = s + FL_L12 * g(1, 2);
    s = s + FL_L13 * g(1, 3);
    s = s + FL_L14 * g(1, 4);
    s = s + FL_L22 * g(2, 2);
    s = s + FL_L23 * g(2, 3);
    s = s + FL_L24 * g(2, 4);
    s = s + FL_L33 * g(3, 3);
    s = s + FL_L34 * g(3, 4);
    s = s + FL_L44 * g(4, 4);
    return s * dinv;
}

// The 12 values x-4 .. x+7 around four cells (three aligned 16-byte LDS reads): at(u) the
// four cells displaced by u.
struct XLine {
    float w[12];
    __device__ __forceinline__ explicit XLine(const float *p)
    {
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const f4 v = *(const f4 *)(p + 4 * (k - 1));
            w[4 * k] = v[0]; w[4 * k + 1] = v[1]; w[4 * k + 2] = v[2]; w[4 * k + 3] = v[3];
        }
    }
    __device__ __forceinline__ f4 at(int u) const { return f4{w[4 + u], w[5 + u], w[6 + u], w[7 + u]}; }
};

// DerCross whose first axis is x: line(v) points at the own cells displaced by v along the
// second axis.  Lines +-m feed the first half of the groups (m, n >= m) and the second half of
// the groups (k < m, m), so each line is read once and every group still adds up in its order:
// h(n, m) - h(-n, m) - h(n, -m) + h(-n, -m), then for n != m the same with m and n exchanged.
template <class L>
__device__ __forceinline__ f4 dercross_x(L line, float dinv)
{
    f4 g[5][5];
#pragma unroll
    for (int m = 1; m <= 4; m++) {
        const XLine a(line(m)), b(line(-m));
#pragma unroll
        for (int k = 1; k < m; k++) g[k][m] = g[k][m] + a.at(k) - a.at(-k) - b.at(k) + b.at(-k);
#pragma unroll
        for (int n = m; n <= 4; n++) g[m][n] = a.at(n) - a.at(-n) - b.at(n) + b.at(-n);
        __builtin_amdgcn_sched_barrier(0);  // two lines in flight
    }
    return cross_sum([&](int m, int n) { return g[m][n]; }, dinv);
}

// DerCross over an accessor h(a, b): the own cells a along the first axis and b along the second.
template <class H>
__device__ __forceinline__ f4 dercross_h(H h, float dinv)
{
    return cross_sum(
        [&](int m, int n) {
            f4 v = h(n, m) - h(-n, m) - h(n, -m) + h(-n, -m);
            if (m != n) v = v + h(m, n) - h(-m, n) - h(m, -n) + h(-m, -n);
            __builtin_amdgcn_sched_barrier(0);
            return v;
        },
        dinv);
}

// Direct 64-point DerCross form (original/sample.h:32-90) staged through LDS.  A workgroup
// of 8 waves owns 64 x 16 cells of a z chunk.  A lane forms the derivatives of four
// consecutive cells of one field (lanes 0-31 p, 32-63 q; 16 lanes a row, two rows a wave);
// the halves of a wave then exchange them (v_permlane32_swap) so that each lane has both
// fields of two cells, and update those.  The 9 planes of the stencil (tile + 4-cell halo,
// one array a field) sit in a ring of DX_NP plane slots; the next plane is loaded before the
// derivatives and stored after them into the slot that no step of the current plane reads, so
// one barrier a plane suffices.  Every derivative, the coefficient combination and the
// leapfrog keep the reference's association order: the results are those of the reference's
// loop, bit for bit.
//
// Bound by both units at two waves a SIMD, neither of them full: on a 192 x 240 x 216 array the VALU
// is busy 65% of the time (573 operations a cell, none of them fused, in the reference's order), the
// LDS 59% (half of that bank conflicts of the 16-byte reads), and waves wait 37% of theirs; HBM traffic is
// 2.7 TB/s.  A lane reads 131 16-byte values a plane, 1048 bytes a cell with
// both fields, where one cell a lane with both fields read 217 pairs, 1736 bytes.  That form,
// which also waited for the next plane's loads at the end of each plane, took 414 us on a
// 192 x 240 x 216 array and 2141 us on 384^3; this one 217 and 1182 us (the VALU operations
// alone 116 and 775 us).  The LDS ring holds one workgroup a CU.
constexpr int DX_TX = 64, DX_TY = 16, DX_NW = DX_TY / 2, DX_NT = 64 * DX_NW, DX_NP = 10;
constexpr int DX_HX = DX_TX + 8, DX_HY = DX_TY + 8, DX_PL = DX_HX * DX_HY;  // cells per staged plane
constexpr int DX_NLD = (DX_PL + DX_NT - 1) / DX_NT;                         // staging loads per thread
constexpr int DX_PER_CU = 1;                                                // resident workgroups a CU
constexpr uint32_t DX_OOB = 0x80000000u;  // beyond every plane (planes hold < 2^31 bytes)

__device__ __forceinline__ __amdgpu_buffer_rsrc_t dx_rsrc(const void *p, uint32_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ float dx_f(uint32_t v) { return __uint_as_float(v); }

// grid: nblk rounded up to whole XCD rounds; block (64, DX_NW).  Fields are (p, q) pairs at
// the pitched cell index.
__global__ __launch_bounds__(DX_NT) __attribute__((amdgpu_waves_per_eu(DX_PER_CU * DX_NW / 4)))
void direct_dercross(const DirectArgs a)
{
    __shared__ __attribute__((aligned(16))) float lds[DX_NP][2][DX_PL];
    const int t = xcd_remap(blockIdx.x, gridDim.x);
    if (t >= a.nblk) return;
    const int tx = t % a.ntx, rest = t / a.ntx, ty = rest % a.nty, tz = rest / a.nty;
    const int x0 = a.bord + tx * DX_TX, y0 = a.bord + ty * DX_TY;
    const int zlo = a.bord + tz * a.zt, zhi = min(zlo + a.zt, a.sz - a.bord);
    const int f0 = zlo - 4;  // first staged plane
    const int lane = threadIdx.x, wv = uni((int)threadIdx.y), tid = wv * 64 + lane;
    const int fld = lane >> 5, row = 2 * wv + ((lane >> 4) & 1), c4 = (lane & 15) * 4;
    const uint32_t pxy = (uint32_t)a.px * (uint32_t)a.sy;

    // the two cells this lane updates, and their byte offsets within a plane of pairs (the
    // records are at 4 times, and at 1 times, these offsets)
    const int y = y0 + row, x = x0 + c4 + 2 * fld;
    uint32_t o8[2];
#pragma unroll
    for (int k = 0; k < 2; k++)
        o8[k] = (x + k < a.sx - a.bord && y < a.sy - a.bord) ? (uint32_t)(y * a.px + x + k) * 8u : DX_OOB;

    // staging: cell e of a staged plane is (row e / DX_HX, column e % DX_HX) of the window
    // whose corner is (x0 - 4, y0 - 4); cells outside the array read as zero.  Loads are
    // unconditional (out of range offsets read zero), so the waits for them count exactly.
    uint32_t goff[DX_NLD];
#pragma unroll
    for (int k = 0; k < DX_NLD; k++) {
        const int e = k * DX_NT + tid, r = e / DX_HX, gx = x0 - 4 + e - r * DX_HX, gy = y0 - 4 + r;
        goff[k] = (e < DX_PL && gx < a.sx && gy < a.sy) ? (uint32_t)(gy * a.px + gx) * 8u : DX_OOB;
    }
    auto fetch = [&](int zp, u2v *v) {  // a plane beyond the array: the last one (not read)
        const __amdgpu_buffer_rsrc_t rs = dx_rsrc(a.cur + 2ll * min(zp, a.sz - 1) * pxy, pxy * 8u);
#pragma unroll
        for (int k = 0; k < DX_NLD; k++) v[k] = __builtin_amdgcn_raw_buffer_load_b64(rs, goff[k], 0, 0);
    };
    auto stage = [&](int slot, const u2v *v) {
#pragma unroll
        for (int k = 0; k < DX_NLD; k++) {
            const int e = k * DX_NT + tid;
            const uint32_t p = v[k][0], q = v[k][1];
            if (e < DX_PL) {
                lds[slot][0][e] = dx_f(p);
                lds[slot][1][e] = dx_f(q);
            }
        }
    };
    {
        u2v v[9][DX_NLD];
#pragma unroll
        for (int i = 0; i < 9; i++) fetch(f0 + i, v[i]);
#pragma unroll
        for (int i = 0; i < 9; i++) stage(i, v[i]);
    }
    __syncthreads();

    const int own = (row + 4) * DX_HX + c4 + 4;  // own cells in a staged plane
    for (int z = zlo; z < zhi; z++) {
        const int j = z - zlo;
        u2v nxt[DX_NLD];
        fetch(z + 5, nxt);
        // records (slots 0-3, 5-8 and 4, 9) and previous level of the two cells, used at the end
        const __amdgpu_buffer_rsrc_t r_c1 = dx_rsrc(a.coef + (long long)z * pxy * 8, pxy * 32u);
        const __amdgpu_buffer_rsrc_t r_c2 =
            dx_rsrc((const char *)a.coef + fp32_part2(a.np) + (long long)z * pxy * 8, pxy * 8u);
        const __amdgpu_buffer_rsrc_t r_pv = dx_rsrc(a.prev + 2ll * z * pxy, pxy * 8u);
        u4v k1[2], k2[2];
        u2v k3[2], pv[2];
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const uint32_t o32 = o8[k] == DX_OOB ? DX_OOB : o8[k] * 4u;
            k1[k] = __builtin_amdgcn_raw_buffer_load_b128(r_c1, o32, 0, 0);
            k2[k] = __builtin_amdgcn_raw_buffer_load_b128(r_c1, o32, 16, 0);
            k3[k] = __builtin_amdgcn_raw_buffer_load_b64(r_c2, o8[k], 0, 0);
            pv[k] = __builtin_amdgcn_raw_buffer_load_b64(r_pv, o8[k], 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        const float *pl[9];
#pragma unroll
        for (int k = 0; k < 9; k++) pl[k] = &lds[(j + k) % DX_NP][fld][own];
        auto v4 = [](const float *p) { return *(const f4 *)p; };
        // xx, yy, zz, xy, yz, xz and the centre
        f4 d[7];
        {
            const XLine l(pl[4]);
            d[6] = l.at(0);
            d[0] = der2_f4([&](int m) { return l.at(m); }, a.dxxinv);
            d[1] = der2_f4([&](int m) { return m ? v4(pl[4] + m * DX_HX) : d[6]; }, a.dyyinv);
            __builtin_amdgcn_sched_barrier(0);
            d[2] = der2_f4([&](int m) { return m ? v4(pl[4 + m]) : d[6]; }, a.dzzinv);
        }
        __builtin_amdgcn_sched_barrier(0);
        d[3] = dercross_x([&](int v) { return pl[4] + v * DX_HX; }, a.dxyinv);
        d[4] = dercross_h([&](int u, int v) { return v4(pl[4 + v] + u * DX_HX); }, a.dyzinv);
        d[5] = dercross_x([&](int v) { return pl[4 + v]; }, a.dxzinv);
        __builtin_amdgcn_sched_barrier(0);
        // lanes 0-31 keep cells 0, 1 and lanes 32-63 cells 2, 3, each with both fields
        float p[7][2], q[7][2];
#pragma unroll
        for (int i = 0; i < 7; i++)
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const float lo = d[i][k], hi = d[i][k + 2];
                const u2v r = __builtin_amdgcn_permlane32_swap(__float_as_uint(lo), __float_as_uint(hi), false, false);
                const uint32_t rp = r[0], rq = r[1];
                p[i][k] = dx_f(rp);
                q[i][k] = dx_f(rq);
            }
#pragma unroll
        for (int k = 0; k < 2; k++) {
            Coef kc;
            const u4v ka = k1[k], kb = k2[k];
            const uint32_t w[10] = {ka[0], ka[1], ka[2], ka[3], k3[k][0], kb[0], kb[1], kb[2], kb[3], k3[k][1]};
#pragma unroll
            for (int s = 0; s < 10; s++) kc.c[rec_order32(s)] = dx_f(w[s]);
            const uint32_t op = pv[k][0], oq = pv[k][1];
            float np = dx_f(op), nq = dx_f(oq);
            combine<CM_F32>(kc, a.dt, p[0][k], p[1][k], p[2][k], p[3][k], p[4][k], p[5][k], q[0][k], q[1][k], q[2][k],
                            q[3][k], q[4][k], q[5][k], p[6][k], q[6][k], np, nq);
            if (a.trace && z == a.rec_iz && o8[k] != DX_OOB)
                a.trace[(long long)(y - a.bord) * (a.sx - 2 * a.bord) + (x + k - a.bord)] = np;
            __builtin_amdgcn_raw_buffer_store_b64(u2v{__float_as_uint(np), __float_as_uint(nq)}, r_pv, o8[k], 0, 0);
        }
        stage((j + 9) % DX_NP, nxt);  // the slot that no step of this plane reads
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------------
// Pass 1 of the two-pass form: Dx of pc,qc over ix in [bord, sx-bord), all iy;
// Dy over iy in [bord, sy-bord), ix in [bord, sx); every plane iz in [0, sz).
// dvx, dvy: (pDx, qDx), (pDy, qDy) pairs at the pitched cell index.  The association order
// is that of derivatives.h:47.
//
// Bound by memory: 8 bytes read and 16 written a cell.  A thread takes two cells along x (16-byte
// loads and stores) and D1_ROWS rows, which it walks with the nine rows of its own columns in
// registers: 32 16-byte loads for 8 cells, most from L1, where one cell a thread made sixteen
// 8-byte loads a cell and scattered 4-byte stores.  Threads are numbered along x first, so no
// lane idles on rows that are not multiples of 64, and the blocks of a plane stay on one XCD
// (xcd_remap), whose L2 holds the shared halo rows.  The four volumes are read back only
// after the whole pass: stored non-temporally (default policy: 183 against 171 us a two-pass step).
// Measured: 224 x 208 x 192 array 74 -> 51 us, 384^3 491 -> 294 us (4.6 TB/s).  Rows a thread: 4 is
// as fast as 8 and 16 on large arrays and faster on small ones (two-pass step on 104 x 110 x 100:
// 29.4, 31.3, 36.0 us with 4, 8, 16).
//
// grid: ceil(((sx+1)/2 * ceil(sy/D1_ROWS)) / 256) * sz blocks, rounded up to whole XCD rounds.
constexpr int D1_ROWS = 4;
__device__ __forceinline__ f4 der1_f4(f4 m4, f4 m3, f4 m2, f4 m1, f4 p1, f4 p2, f4 p3, f4 p4, float dinv)
{
    return (FL_L1 * (p1 - m1) + FL_L2 * (p2 - m2) + FL_L3 * (p3 - m3) + FL_L4 * (p4 - m4)) * dinv;
}
__device__ __forceinline__ u4v f4_bits(f4 v)
{
    const float a = v[0], b = v[1], c = v[2], d = v[3];
    return u4v{__float_as_uint(a), __float_as_uint(b), __float_as_uint(c), __float_as_uint(d)};
}
__global__ __launch_bounds__(256) void der1_pass(const float *__restrict__ cur, float *dvx, float *dvy, int sx, int sy,
                                                 int sz, int px, int bord, int nbx, float dxinv, float dyinv)
{
    const int b = xcd_remap(blockIdx.x, gridDim.x);
    const int z = uni(b / nbx), nxp = (sx + 1) >> 1;
    if (z >= sz) return;
    const int t = (b - z * nbx) * 256 + (int)threadIdx.x;
    const int yc = t / nxp, x = 2 * (t - yc * nxp), y0 = yc * D1_ROWS;
    if (y0 >= sy) return;
    const uint32_t pxy = (uint32_t)px * (uint32_t)sy, pb8 = pxy * 8u;
    const __amdgpu_buffer_rsrc_t rc = dx_rsrc(cur + 2ll * z * pxy, pb8);
    const __amdgpu_buffer_rsrc_t rx = dx_rsrc(dvx + 2ll * z * pxy, pb8), ry = dx_rsrc(dvy + 2ll * z * pxy, pb8);
    // two cells of row y displaced by dx; outside the plane they read as zero (not used)
    auto row = [&](int y, int dx) {
        const uint32_t o = (y >= 0 && y < sy) ? (uint32_t)(y * px + x + dx) * 8u : DX_OOB;
        const u4v v = __builtin_amdgcn_raw_buffer_load_b128(rc, o, 0, 0);
        const uint32_t v0 = v[0], v1 = v[1], v2 = v[2], v3 = v[3];
        return f4{dx_f(v0), dx_f(v1), dx_f(v2), dx_f(v3)};
    };
    // both cells with one store, or the one that is in the range
    auto put = [&](__amdgpu_buffer_rsrc_t r, f4 d, uint32_t o, bool c0, bool c1) {
        const u4v v = f4_bits(d);
        __builtin_amdgcn_raw_buffer_store_b128(v, r, c0 && c1 ? o : DX_OOB, 0, 2);
        if (c0 != c1) {
            const uint32_t v0 = v[0], v1 = v[1], v2 = v[2], v3 = v[3];
            __builtin_amdgcn_raw_buffer_store_b64(c0 ? u2v{v0, v1} : u2v{v2, v3}, r, c0 ? o : o + 8u, 0, 2);
        }
    };
    const bool x0 = x >= bord && x < sx - bord, x1 = x + 1 >= bord && x + 1 < sx - bord;
    const bool w0 = x >= bord && x < sx, w1 = x + 1 >= bord && x + 1 < sx;
    f4 q[9];  // rows y-4 .. y+4 of the own columns, row r in slot r % 9
#pragma unroll
    for (int k = 0; k < 8; k++) q[k] = row(y0 - 4 + k, 0);
#pragma unroll
    for (int j = 0; j < D1_ROWS; j++) {
        const int y = y0 + j;
        q[(j + 8) % 9] = row(y + 4, 0);
        const f4 a = row(y, -4), b2 = row(y, -2), c = q[(j + 4) % 9], d = row(y, 2), e = row(y, 4);
        const uint32_t o = (uint32_t)(y * px + x) * 8u;
        // cells x-4..x+5 are a, b2, c, d, e; the neighbours at an odd distance straddle two of them
        auto odd = [](f4 l, f4 r) { return f4{l[2], l[3], r[0], r[1]}; };
        const f4 gx = der1_f4(a, odd(a, b2), b2, odd(b2, c), odd(c, d), d, odd(d, e), e, dxinv);
        const f4 gy = der1_f4(q[j % 9], q[(j + 1) % 9], q[(j + 2) % 9], q[(j + 3) % 9], q[(j + 5) % 9], q[(j + 6) % 9],
                              q[(j + 7) % 9], q[(j + 8) % 9], dyinv);
        const bool in = y < sy, iny = y >= bord && y < sy - bord;
        put(rx, gx, o, in && x0, in && x1);
        put(ry, gy, o, iny && w0, iny && w1);
    }
}

// Source insertion at pitched cell c of a level: p += s, q += s.
__global__ void insert_source(float *lv, long long c, float s)
{
    if (threadIdx.x == 0) {
        lv[2 * c] += s;
        lv[2 * c + 1] += s;
    }
}

// Component fld of a pitched volume of ST values a cell (a level: ST 2, fld 0 p, 1 q; a model
// volume: ST 1) <-> m consecutive cells in the reference layout, the first one cell x0 of
// row row0.  grid: ceil(m/256); block 256
template <int ST>
__global__ __launch_bounds__(256) void field_pack(const float *__restrict__ lin, float *vol, int fld, int m, int x0,
                                                  long long row0, int sx, int px)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= m) return;
    const int r = (x0 + i) / sx;
    vol[ST * ((row0 + r) * px + (x0 + i - r * sx)) + fld] = lin[i];
}
template <int ST>
__global__ __launch_bounds__(256) void field_unpack(const float *__restrict__ vol, float *lin, int fld, int m, int x0,
                                                    long long row0, int sx, int px)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= m) return;
    const int r = (x0 + i) / sx;
    lin[i] = vol[ST * ((row0 + r) * px + (x0 + i - r * sx)) + fld];
}

#endif  // FL_NO_AUX_KERNELS

}  // namespace fl
