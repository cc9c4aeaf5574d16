// Forward projector (exact adjoint of the backprojection), analytic phantom images,
// and volume index-order / byte-order conversion for the writer.
//
// The forward projector has no counterpart in the reference; it transposes the
// voxel-driven backprojection of Ct/CtVolume.cpp:979-1039 term by term: every voxel that
// the backprojection would read through taps (u0,v0),(u0+1,v0),(u0,v0+1),(u0+1,v0+1) with
// weight U^2 and bilinear weights instead adds U^2 * f * weight into those pixels, under
// the same cylinder and window masks.  A workgroup owns a pixel column of one projection and
// collects the voxel columns that land on it: fp_rows_kernel, fp_entry_kernel for small
// volumes, or fp_gather_kernel where the geometry rules those out.
#include "ctg_internal.h"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <type_traits>

namespace ctg {
namespace {

struct FpArgs {
    int W, H, nx, ny, nzs, z0, nproj;
    int zstride;  // slices per voxel column of the volume buffer (nzs of them from z0 are projected)
    int cblock;   // pixel columns per unit of fp_rows_kernel's numbering
    float xpre, ypre, zpre, upre, vpre;
    float r2, fcd, uoff, ulo, uhi, vlo, vhi;
};

// Gather form of the projector.  No global or LDS float atomics: scattering splats
// costs LDS float atomics (about 30x an LDS read here) or global ones that contend
// across workgroups.  A workgroup owns one detector column c of one projection.
//  - The voxel columns that can feed column c are exactly those whose ray lands within
//    [c - 1, c + 1) on the detector (u0 = c takes weight 1 - fu, u0 = c - 1 takes fu).
//    Along a line of constant outer coordinate u is monotonic in the inner one, so the
//    two rays from the source through u = c - 1 and u = c + 1 (plus 0.05 pixel) bound
//    the candidates up to rounding; a 0.01-voxel margin covers that.
//  - The per-column work (cylinder and window tests, U, the tap weight) is done once per
//    candidate: the lanes fill a compacted list of candidates in LDS, in walk order.
//    The v-window test (v = (z + h) U inside [vLo, vHi]) is monotonic in z for U > 0, so
//    the fill also turns it, intersected with the slab, into an exact interval of z
//    (found by evaluating the backprojection's own expression at the boundaries);
//    candidates whose interval is empty are dropped.
//  - The waves then walk items of up to four consecutive 64-voxel z chunks of a
//    candidate (one voxel per lane and chunk), dealt round-robin, with the
//    backprojection's anchored row index, and add the two row taps of each voxel into
//    the wave's own row accumulators in LDS.  Chunks start at multiples of 32 in grid z,
//    so a lane's row anchor and its offset from it are fixed per lane.  Rows of voxels k
//    slices apart differ by at least k*U - 1, so lanes are split by residue modulo
//    ceil(2/U), rounded up to 2 or 4 (which divide the chunk length), between two row
//    copies per wave and, for 4, two passes: taps that meet never share a row, and the
//    read-modify-writes need no atomics.
//  - At the end the four waves' rows are summed into the image.
// Every (voxel, tap) pair is added exactly once, and the order of all additions is fixed:
// the result does not depend on scheduling.
constexpr int kGThreads = 256, kGWaves = kGThreads / 64;
constexpr int kSlots = 512;  // candidate slots per pass (16 B each)
constexpr int kMaxRowsFp = 4096;  // detector rows held in LDS per wave
constexpr int kFpZBits = 14;      // z interval bounds in a candidate record (relative to the run base)
constexpr int kFpMaxSlab = (1 << kFpZBits) - 2 * kRowAnchor;  // slices per launch
static_assert(kFpMaxSlab % (2 * kRowAnchor) == 0, "the next launch starts on a chunk");

// Raw buffer resource over `bytes` bytes of global memory: a 4-byte load at an offset at
// or past the end returns zero.  The builtins exist only in the device pass.
#if defined(__HIP_DEVICE_COMPILE__)
using vbuf = __amdgpu_buffer_rsrc_t;
__device__ inline vbuf make_vbuf(const float* base, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, bytes, 0x00020000);
}
__device__ inline float vbuf_load(vbuf rs, unsigned off) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, (int)off, 0, 0));
}
// a + b in a vector register, opaque to the compiler, so that a constant part of the
// sum is not moved into a load's immediate offset
__device__ inline unsigned vadd_sv(int a, unsigned b) {
    unsigned r;
    asm("v_add_u32 %0, %1, %2" : "=v"(r) : "s"(a), "v"(b));
    return r;
}
#else
__device__ inline unsigned vadd_sv(int a, unsigned b) { return (unsigned)a + b; }
struct vbuf {};
__device__ inline vbuf make_vbuf(const float*, int) { return {}; }
__device__ inline float vbuf_load(vbuf, unsigned) { return 0.0f; }
#endif

__global__ __launch_bounds__(kGThreads) void fp_gather_kernel(FpArgs a, const float4* __restrict__ pp,
                                                              const float* __restrict__ vol,
                                                              float* __restrict__ proj) {
    __shared__ int4 slots[kSlots];
    __shared__ int wave_cnt[kGWaves];
    // kGWaves x 2 copies of (H + 4) rows: row r at index r + 2; rows -2, -1, H, H + 1
    // absorb taps off the image.  Even lanes of a wave add into its first copy, odd
    // lanes into its second.
    extern __shared__ float rows_lds[];
    const int c = blockIdx.x;
    const int p = blockIdx.y;
    const int tid = (int)threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int H = a.H, pitch = a.H + 4;
    float* myrows = rows_lds + (size_t)(2 * wv + (lane & 1)) * pitch;
    for (int i = tid; i < 2 * kGWaves * pitch; i += kGThreads) rows_lds[i] = 0.0f;
    __syncthreads();

    const float4 g = pp[p];
    const float sn = g.x, cs = g.y, h = g.z;
    // source and detector points in world xy (voxel units; the virtual detector passes
    // through the axis, lateral coordinate u)
    const float Sx = a.fcd * cs + a.uoff * sn, Sy = a.fcd * sn - a.uoff * cs;
    const float ulo = (float)c - 1.05f - a.upre, uhi = (float)c + 1.05f - a.upre;
    const float q0x = -(ulo - a.uoff) * sn, q0y = (ulo - a.uoff) * cs;
    const float q1x = -(uhi - a.uoff) * sn, q1y = (uhi - a.uoff) * cs;
    const float umid = (float)c - a.upre - a.uoff;
    const bool xmajor = fabsf(-umid * sn - Sx) >= fabsf(umid * cs - Sy);
    const int n_out = xmajor ? a.nx : a.ny, n_in = xmajor ? a.ny : a.nx;
    const float pre_out = xmajor ? a.xpre : a.ypre, pre_in = xmajor ? a.ypre : a.xpre;
    const float So = xmajor ? Sx : Sy, Si = xmajor ? Sy : Sx;
    const float k0 = ((xmajor ? q0y : q0x) - Si) / ((xmajor ? q0x : q0y) - So);
    const float k1 = ((xmajor ? q1y : q1x) - Si) / ((xmajor ? q1x : q1y) - So);
    const float R = sqrtf(a.r2);
    const int o_lo = max(0, (int)floorf(pre_out - R) - 1), o_hi = min(n_out - 1, (int)ceilf(pre_out + R) + 1);
    const int zend = a.z0 + a.nzs - 1;  // last grid z index of the slab
    const int zrb = a.z0 & ~(kRowAnchor - 1);  // run base: chunks start at zrb + 64 k

    // lateral candidates of depth step o: [jl, jh]
    auto jrange = [&](int o, int& jl, int& jh) {
        const float ow = (float)o - pre_out;
        const float i0 = Si + (ow - So) * k0, i1 = Si + (ow - So) * k1;
        jl = max(0, (int)ceilf(fminf(i0, i1) + pre_in - 0.01f));
        jh = min(n_in - 1, (int)floorf(fmaxf(i0, i1) + pre_in + 0.01f));
    };
    // slots per depth step: the wedge width |i1 - i0| is linear in the depth and the
    // source lies outside the volume, so it peaks at an end of the depth range; the
    // count of integers in a window of width w + 0.02 is at most floor(w) + 2
    auto width = [&](int o) {
        const float ow = (float)o - pre_out;
        return fabsf((ow - So) * (k1 - k0));
    };
    const int jm = (int)fmaxf(width(o_lo), width(o_hi)) + 2;
    const int jm_pass = min(jm, kSlots);
    const int per_pass = max(1, kSlots / jm_pass);

    for (int ob = o_lo; ob <= o_hi; ob += per_pass) {
        const int no = min(per_pass, o_hi - ob + 1);
        for (int jb = 0; jb < jm; jb += jm_pass) {
            const int nj = min(jm_pass, jm - jb);
            const int nslot = no * nj;
            // fill: slot (o - ob) * nj + jj covers lateral candidate jl + jb + jj of depth o;
            // the candidates that pass the tests are stored compacted, in slot order
            // (a ballot prefix within each wave, wave totals through LDS)
            int ncand = 0;
            for (int sbase = 0; sbase < nslot; sbase += kGThreads) {
                const int sidx = sbase + tid;
                const int oi = sidx / nj, jj = sidx - oi * nj;
                const int o = ob + oi;
                int jl = 0, jh = -1;
                if (sidx < nslot) jrange(o, jl, jh);
                const int j = jl + jb + jj;
                int4 rec = make_int4(-1, 0, 0, 0);
                if (sidx < nslot && j <= jh) {
                    const int xi = xmajor ? o : j, yi = xmajor ? j : o;
                    // per-voxel arithmetic identical to the backprojection's
                    const float x = (float)xi - a.xpre, y = (float)yi - a.ypre;
                    if (x * x + y * y < a.r2) {
                        float t = (-1.0f) * x * g.x + y * g.y;
                        t += a.uoff;
                        const float s = x * g.y + y * g.x;
                        const float U = cone_magnification(a.fcd, s);
                        const float u = t * U;
                        if (u >= a.ulo && u <= a.uhi) {
                            const float uIdx = u + a.upre;
                            const int u0 = (int)uIdx;
                            if (u0 == c || u0 == c - 1) {
                                const float fu = uIdx - (float)u0;
                                const float wc = U * U * (u0 == c ? 1.0f - fu : fu);
                                // z interval of the window test v = (zk + h) U in [vLo, vHi]:
                                // v is non-decreasing in z (U > 0, monotone rounding), so the
                                // passing z form an interval; estimate its ends, then settle
                                // them with the backprojection's own expression
                                // (the estimate is within about 1e-2 of the true end for grids
                                // of up to 65536 slices, so its ceiling or floor is off by at
                                // most one)
                                auto v_of = [&](int zi) { const float zk = (float)zi - a.zpre; return (zk + h) * U; };
                                const float iU = __builtin_amdgcn_rcpf(U);
                                const float zlo_f = fminf(fmaxf(a.vlo * iU - h + a.zpre, (float)(a.z0 - 4)), (float)(zend + 4));
                                const float zhi_f = fminf(fmaxf(a.vhi * iU - h + a.zpre, (float)(a.z0 - 4)), (float)(zend + 4));
                                int lo = (int)ceilf(zlo_f), hi = (int)floorf(zhi_f);
#pragma unroll
                                for (int it = 0; it < 2; ++it) {
                                    if (lo > a.z0 && v_of(lo - 1) >= a.vlo) --lo;
                                    if (hi < zend && v_of(hi + 1) <= a.vhi) ++hi;
                                }
#pragma unroll
                                for (int it = 0; it < 2; ++it) {
                                    if (lo <= zend && !(v_of(lo) >= a.vlo)) ++lo;
                                    if (hi >= a.z0 && !(v_of(hi) <= a.vhi)) --hi;
                                }
                                lo = max(lo, a.z0);
                                hi = min(hi, zend);
                                if (lo <= hi) {
                                    // ceil(2/U) passes, rounded up to a power of two (a
                                    // multiple of ceil(2/U) passes is as safe); U > 1/1.9
                                    // keeps it at most 4
                                    const int np0 = (int)ceilf(2.0f * __builtin_amdgcn_rcpf(U) + 1e-3f);
                                    const int npass = np0 <= 1 ? 1 : (np0 == 2 ? 2 : 4);
                                    rec = make_int4(xi * a.ny + yi, __float_as_int(U), __float_as_int(wc),
                                                    (lo - zrb) | ((hi - zrb) << kFpZBits) | (npass << (2 * kFpZBits)));
                                }
                            }
                        }
                    }
                }
                const unsigned long long m = __ballot(rec.x >= 0);
                const int below = __popcll(m & ((1ull << lane) - 1ull));
                if (lane == 0) wave_cnt[wv] = __popcll(m);
                __syncthreads();
                int base = ncand;
                for (int w = 0; w < wv; ++w) base += wave_cnt[w];
                int total = 0;
                for (int w = 0; w < kGWaves; ++w) total += wave_cnt[w];
                if (rec.x >= 0) slots[base + below] = rec;
                ncand += total;
                __syncthreads();  // wave_cnt is rewritten by the next round
            }
            // walk: a voxel's taps go to rows v0, v0 + 1 of the wave's own accumulators.
            // Chunks start at zrb + 64 k (multiples of 32 in grid z), so lane l's voxel
            // lies (l & 31) slices past its row anchor, which is (l & 32) slices past the
            // chunk start.  Lanes outside the candidate's z interval load zero and send
            // their (zero) taps to the absorbing rows H, H + 1: their own rows could meet
            // an active lane's, because truncation folds (-1, 1) onto row 0.  A lane whose
            // voxel is zero may do the same, as its taps are zero too.
            const float lane_k = (float)(lane & 31), anchor_off = (float)(lane & 32);
            const float* colbase = vol + (zrb - a.z0);  // voxel (column, z) at column * zstride + z - zrb
            auto tap = [&](float zcw, float xv, float U, float wc, float& ta, float& tb) -> int {
                const float vA = det_row_anchor(zcw + anchor_off, h, U, a.vpre);
                const float vI = det_row_index(lane_k, U, vA);
                const int v0 = (int)vI;
                const float fv = vI - (float)v0;
                const float val = wc * xv;
                tb = fv * val;
                ta = val - tb;
                return (xv != 0.0f ? v0 : H) + 2;  // in-window rows are 0 .. H - 2 (checked on the host)
            };
            // a candidate record: column, U, weight, and z interval [lo, hi] relative to
            // zrb with the residue pass count in the top bits.  The column's voxels in
            // [lo, hi] are read through a buffer resource covering exactly them: a load
            // outside it returns zero, which is the mask of the window and the slab.
            struct Item {
                vbuf rs;
                float U, wc;
                int lo, npass;
            };
            // past the last candidate an item still issues its loads, over an empty
            // resource (they return zero without touching memory): every slot then has
            // the same loads in flight and the walk waits for exactly its own
            auto item_of = [&](int ci, bool valid) {
                const int4 r = slots[valid ? ci : 0];
                Item it;
                const int w = __builtin_amdgcn_readfirstlane(r.w);
                it.lo = w & ((1 << kFpZBits) - 1);
                const int hi = (w >> kFpZBits) & ((1 << kFpZBits) - 1);
                it.rs = make_vbuf(colbase + (size_t)__builtin_amdgcn_readfirstlane(r.x) * a.zstride + it.lo,
                                  valid ? (hi - it.lo + 1) * (int)sizeof(float) : 0);
                it.U = __int_as_float(__builtin_amdgcn_readfirstlane(r.y));
                it.wc = __int_as_float(__builtin_amdgcn_readfirstlane(r.z));
                it.npass = (unsigned)w >> (2 * kFpZBits);
                return it;
            };
            // this lane's voxel of the chunk starting at zc (relative to zrb).  The byte
            // offset is formed in one register per chunk: lanes before the interval get
            // an offset that wraps to a huge value, which the resource's range check
            // rejects.  With the chunk's distance in the load's immediate offset instead,
            // a wrapped register offset plus the immediate was measured to read zeros
            // where the sum lands at the start of the resource.
            const unsigned lane4 = (unsigned)lane * (unsigned)sizeof(float);
            auto load = [&](const Item& it, int zc) -> float {
                return vbuf_load(it.rs, vadd_sv((zc - it.lo) * (int)sizeof(float), lane4));
            };
            auto zworld = [&](int zc) { return (float)(zrb + zc) - a.zpre; };
            const int nzr = zend - zrb + 1;  // slices from the run base to the slab end
            if (ncand == 0) {
                __syncthreads();
                continue;
            }
            // Items are (candidate, group of G consecutive 64-voxel chunks), in walk order,
            // dealt to the four waves round-robin: item q = ci * ngrp + j goes to wave
            // q mod 4.  With n = ceil(2/U) rounded up to 1, 2 or 4, voxels n or more slices
            // apart have rows at least two apart.  Lanes of one parity add into one of the
            // wave's two row copies, and for n = 4 in two passes by (lane >> 1) & 1: lanes
            // l and l' of any two chunks of an item (chunks are 64 slices apart) meet in a
            // copy and pass only if their z differ by a nonzero multiple of 2 (n <= 2) or
            // 4, so a pass's read-modify-writes touch distinct rows.  Each wave walks its
            // items through S slots: the voxels of the next S - 1 items are in flight
            // while the current one is processed (the slots are named, not rotated, so that
            // no in-flight register is copied).
            const int nch = (nzr + 63) / 64;
            auto walk = [&](auto g_const) {
                constexpr int G = decltype(g_const)::value;
                constexpr int S = G == 1 ? 3 : 2;
                const int ngrp = (nch + G - 1) / G;
                const int dci = kGWaves / ngrp, dj = kGWaves - dci * ngrp;
                int ci_f = 0, j_f = wv;  // next item to fetch
                while (j_f >= ngrp) { j_f -= ngrp; ++ci_f; }
                struct Slot { Item it; int zc; float x[G]; };
                auto next = [&](Slot& s) -> bool {
                    const bool valid = ci_f < ncand;
                    s.it = item_of(ci_f, valid);
                    s.zc = 64 * G * j_f;
#pragma unroll
                    for (int k = 0; k < G; ++k) s.x[k] = load(s.it, s.zc + 64 * k);
                    ci_f += dci;
                    j_f += dj;
                    if (j_f >= ngrp) { j_f -= ngrp; ++ci_f; }
                    __builtin_amdgcn_sched_barrier(0);  // keep the slots' loads in walk order
                    return valid;
                };
                auto process = [&](const Slot& s) {
                    float ta[G], tb[G];
                    int ix[G];
                    // world z of the chunks: exact half-integers, so chunk k's is chunk 0's + 64 k
                    const float zw0 = zworld(s.zc);
#pragma unroll
                    for (int k = 0; k < G; ++k) ix[k] = tap(zw0 + (float)(64 * k), s.x[k], s.it.U, s.it.wc, ta[k], tb[k]);
                    // loads before stores: the 2G rows of a pass are distinct
                    auto rmw = [&]() {
                        float r0[G], r1[G];
#pragma unroll
                        for (int k = 0; k < G; ++k) { r0[k] = myrows[ix[k]]; r1[k] = myrows[ix[k] + 1]; }
#pragma unroll
                        for (int k = 0; k < G; ++k) { myrows[ix[k]] = r0[k] + ta[k]; myrows[ix[k] + 1] = r1[k] + tb[k]; }
                    };
                    if (s.it.npass <= 2) {
                        rmw();  // the lane parity picks the copy: one pass
                    } else {
                        const int pid = (lane >> 1) & 1;
                        for (int ps = 0; ps < 2; ++ps) {
                            if (pid == ps) rmw();
                            __builtin_amdgcn_wave_barrier();
                        }
                    }
                };
                if constexpr (S == 3) {
                    Slot sa, sb, sc;
                    bool ha = next(sa), hb = next(sb), hc = next(sc);
                    while (ha) {
                        process(sa);
                        ha = next(sa);
                        if (!hb) break;
                        process(sb);
                        hb = next(sb);
                        if (!hc) break;
                        process(sc);
                        hc = next(sc);
                    }
                } else {
                    Slot sa, sb;
                    bool ha = next(sa), hb = next(sb);
                    while (ha) {
                        process(sa);
                        ha = next(sa);
                        if (!hb) break;
                        process(sb);
                        hb = next(sb);
                    }
                }
            };
            if (nch >= 4) walk(std::integral_constant<int, 4>{});
            else if (nch == 3) walk(std::integral_constant<int, 3>{});
            else if (nch == 2) walk(std::integral_constant<int, 2>{});
            else walk(std::integral_constant<int, 1>{});
            __syncthreads();
        }
    }
    // both row copies of the four waves, summed in a fixed order, into the image
    for (int r = tid; r < H; r += kGThreads) {
        float sum = rows_lds[r + 2];
        for (int w = 1; w < 2 * kGWaves; ++w) sum += rows_lds[(size_t)w * pitch + r + 2];
        proj[((size_t)p * H + r) * a.W + c] += sum;
    }
}

struct FpWin {
    int wz0;     // first grid slice of the window (a multiple of 64 past the run base)
    int rbase;   // first row any voxel of the window can reach
    int span;    // rows per copy
    int stride;  // rows between copies
    int first;   // 1: the workgroup's column of sums is written, 0: added to
};

// -------------------------------------------------------- entry-space projector
//
// The backprojection evaluates a voxel's value from ONE coefficient entry (A, dU, dV, dUV)
// at (u0, v0): val = A + fu dU + fv (dV + fu dUV), weighted by w = U^2.  Its transpose
// therefore adds (w x, w x fu, w x fv, w x fu fv) into one entry gradient per (voxel,
// projection), and the transpose of the layout (A = q00, dU = q10 - q00, dV = q01 - q00,
// dUV = q11 - q10 - q01 + q00) turns entry gradients into pixels:
//     q00 += gA - gdU - gdV + gdUV,  q01 += gdV - gdUV,  q10 += gdU - gdUV,  q11 += gdUV.
//
// fp_entry_kernel<G>: candidates, windows, lanes and voxel reads as in fp_rows_kernel below,
// but every voxel is added into its entry as it comes, with one LDS read and one write of 16
// bytes, in two private copies per wave (even and odd lanes: same-parity lanes of an item are
// two or more slices apart, so their rows differ).  Each round of 256 slots is walked at once,
// candidate ci by wave ci mod 4.  At the end the eight copies are summed in a fixed order.
//
// What bounds it: the LDS (a 16-byte read and write take 18 cycles per wave and CU), a third
// more per update than fp_rows_kernel at 512^3, but it has no runs to begin and end.  It is the
// faster one where columns are short (see the launch): 59 against 64 us at 96^2 x 72 from 48
// projections of 103 x 83, 296 against 311 at 128^3 from 200, but 217 against 207 at 200^2 x
// 128 from 60 and 428 against 302 at 160^3 from 100, where a third window is begun.
constexpr int kEntryMaxSpan = 320;  // entry rows per copy (three workgroups per CU)
constexpr int kEntryMaxSide = 160;  // voxels
// Windows whose runs would be shorter than this many candidates take the entry form too, two
// chunks at a time: a run end then costs as much as it saves.  200^2 x 200 (a window of 256
// slices) from 250 projections and a source 1.2, 1.4 detector widths away, runs of 1.6, 1.9: rows
// 2.04, 1.93 ms, entries 1.77, 1.73; 150^2 x 223, 2 widths, 2.0: 0.83, 0.88; 200^2 x 256, 1.6
// widths, 2.5: 1.06, 1.24; 125^2 x 223, 2.5 widths, 2.2: 0.64, 0.66.
// Heights that spread over many rows take that away, as every copy holds the rows of all of them
// (109^2 x 223, 2.5 widths, 1.9: 0.48 and 0.48 ms, with heights of -22 to 22 0.52 and 0.58).
constexpr double kMinRun = 1.95, kMinRunHeights = 16.0;

__device__ inline int flr_i32(float x) {
    int r;
    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(r) : "v"(x));
    return r;
}

template <int G, bool CHECK>
__global__ __launch_bounds__(kGThreads) void fp_entry_kernel(FpArgs a, FpWin win, const float4* __restrict__ pp,
                                                             const float* __restrict__ vol,
                                                             float2* __restrict__ ps) {
    // column, U, w fu and the z interval relative to the run base (w = U^2 is recomputed
    // from U): one 16-byte LDS read per item
    __shared__ int4 slots[kGThreads];
    __shared__ int wave_cnt[kGWaves];
    // [wave][parity][row], copies `stride` entries apart, a multiple of 16.  On gfx950 a ds_write_b128 occupies the LDS for about
    // 13.5 cycles per wave instruction whatever its lane mask and a conflict-free
    // ds_read_b128 about 4 (16 lanes per cycle); of the copy offsets 0, 2, 5, 6, 8 and 13
    // entries modulo 16, 0 was the fastest on the 512^3 x 360 workload.
    extern __shared__ float4 entry_lds[];
    const int c = blockIdx.x;
    const int p = blockIdx.y;
    const int tid = (int)threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int span = win.span, stride = win.stride;
    const float4 g = pp[p];
    const float sn = g.x, cs = g.y, h = g.z;
    const float Sx = a.fcd * cs + a.uoff * sn, Sy = a.fcd * sn - a.uoff * cs;
    const float ulo = (float)c - 0.05f - a.upre, uhi = (float)c + 1.05f - a.upre;
    const float q0x = -(ulo - a.uoff) * sn, q0y = (ulo - a.uoff) * cs;
    const float q1x = -(uhi - a.uoff) * sn, q1y = (uhi - a.uoff) * cs;
    const float umid = (float)c + 0.5f - a.upre - a.uoff;
    const bool xmajor = fabsf(-umid * sn - Sx) >= fabsf(umid * cs - Sy);
    const int n_out = xmajor ? a.nx : a.ny, n_in = xmajor ? a.ny : a.nx;
    const float pre_out = xmajor ? a.xpre : a.ypre, pre_in = xmajor ? a.ypre : a.xpre;
    const float So = xmajor ? Sx : Sy, Si = xmajor ? Sy : Sx;
    const float k0 = ((xmajor ? q0y : q0x) - Si) / ((xmajor ? q0x : q0y) - So);
    const float k1 = ((xmajor ? q1y : q1x) - Si) / ((xmajor ? q1x : q1y) - So);
    const float R = sqrtf(a.r2);
    const int o_lo = max(0, (int)floorf(pre_out - R) - 1), o_hi = min(n_out - 1, (int)ceilf(pre_out + R) + 1);
    const int zend = a.z0 + a.nzs - 1;
    const int zrb = a.z0 & ~(kRowAnchor - 1);
    // the slices of this window inside the slab
    const int wlo = max(a.z0, win.wz0), whi = min(zend, win.wz0 + 64 * G - 1);

    auto jrange = [&](int o, int& jl, int& jh) {
        const float ow = (float)o - pre_out;
        const float i0 = Si + (ow - So) * k0, i1 = Si + (ow - So) * k1;
        jl = max(0, (int)ceilf(fminf(i0, i1) + pre_in - 0.01f));
        jh = min(n_in - 1, (int)floorf(fmaxf(i0, i1) + pre_in + 0.01f));
    };
    // lateral slots per depth step: the wedge width |i1 - i0| is linear in the depth and
    // the source lies outside the volume, so it peaks at an end of the depth range; a
    // window of width w + 0.02 holds at most floor(w) + 2 integers
    auto width = [&](int o) {
        const float ow = (float)o - pre_out;
        return fabsf((ow - So) * (k1 - k0));
    };
    const int jm = (int)fmaxf(width(o_lo), width(o_hi)) + 2;
    const int nslot = (o_hi - o_lo + 1) * jm;

    // per lane and chunk: world z of the slice's row anchor plus the height (the
    // backprojection's zwa + h), and the slice's offset from the anchor
    float zh[G];
#pragma unroll
    for (int k = 0; k < G; ++k) zh[k] = ((float)(win.wz0 + 64 * k + (lane & 32)) - a.zpre) + h;
    const float lane_k = (float)(lane & 31);
    // LDS byte address of entry row v0 in this lane's copy: v0 * 16 + lane_base
    int lane_base = (wv * 2 + (lane & 1)) * stride * 16 - win.rbase * 16;
    // opaque to the optimiser, so that v0 * 16 + lane_base stays one shift-and-add per
    // voxel instead of being re-associated around rbase
    asm volatile("" : "+v"(lane_base));
    char* acc_bytes = reinterpret_cast<char*>(entry_lds);
    const float* colbase = vol + (zrb - a.z0);
    const int zc = win.wz0 - zrb;  // the window's first slice relative to the run base
    const unsigned lane4 = (unsigned)lane * (unsigned)sizeof(float);

    // An infinite voxel makes NaN of the pixels' differences of entry sums, and of pixels that it
    // has no weight in.  CHECK: a column with sums that are not finite is computed again, tap by
    // tap (small volumes do without: the check and its code take 5 to 14 % of a small launch).
    int by_tap = 0;
again:
    for (int i = tid; i < 2 * kGWaves * stride; i += kGThreads) entry_lds[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    __syncthreads();

    int ncand = 0;
    for (int sbase = 0; sbase < nslot && wlo <= whi; sbase += kGThreads) {
        // fill, step 1: the cheap tests for 256 slots, survivors compacted (ballot prefix
        // within each wave, wave totals through LDS)
        const int sidx = sbase + tid;
        int4 rec = make_int4(-1, 0, 0, 0);
        if (sidx < nslot) {
            const int oi = sidx / jm, jj = sidx - oi * jm;
            const int o = o_lo + oi;
            int jl, jh;
            jrange(o, jl, jh);
            const int j = jl + jj;
            if (j <= jh) {
                const int xi = xmajor ? o : j, yi = xmajor ? j : o;
                // per-voxel arithmetic identical to the backprojection's
                const float x = (float)xi - a.xpre, y = (float)yi - a.ypre;
                if (x * x + y * y < a.r2) {
                    float t = (-1.0f) * x * g.x + y * g.y;
                    t += a.uoff;
                    const float s = x * g.y + y * g.x;
                    const float U = cone_magnification(a.fcd, s);
                    const float u = t * U;
                    if (u >= a.ulo && u <= a.uhi) {
                        const float uIdx = u + a.upre;
                        const int u0 = (int)uIdx;
                        if (u0 == c) rec = make_int4(xi * a.ny + yi, __float_as_int(U), __float_as_int(uIdx - (float)u0), 0);
                    }
                }
            }
        }
        {
            const unsigned long long m = __ballot(rec.x >= 0);
            const int below = __popcll(m & ((1ull << lane) - 1ull));
            if (lane == 0) wave_cnt[wv] = __popcll(m);
            __syncthreads();
            int base = ncand;
            for (int w = 0; w < wv; ++w) base += wave_cnt[w];
            int total = 0;
            for (int w = 0; w < kGWaves; ++w) total += wave_cnt[w];
            if (rec.x >= 0) slots[base + below] = rec;
            __syncthreads();  // the slots are complete; wave_cnt is rewritten below
            // fill, step 2: one lane per new survivor settles its z interval and writes its
            // final record (candidates with an empty interval keep an empty one)
            const int ci = ncand + tid;
            if (tid < total) {
                const int4 r = slots[ci];
                const float U = __int_as_float(r.y), fu = __int_as_float(r.z);
                auto v_of = [&](int zi) { const float zk = (float)zi - a.zpre; return (zk + h) * U; };
                int lo = wlo, hi = whi;
                if (!(v_of(wlo) >= a.vlo && v_of(whi) <= a.vhi)) {
                    // the passing z of v = (zk + h) U in [vLo, vHi] form an interval (v is
                    // non-decreasing in z): estimate its ends, then settle them with the
                    // backprojection's own expression
                    const float iU = __builtin_amdgcn_rcpf(U);
                    const float zlo_f = fminf(fmaxf(a.vlo * iU - h + a.zpre, (float)(wlo - 4)), (float)(whi + 4));
                    const float zhi_f = fminf(fmaxf(a.vhi * iU - h + a.zpre, (float)(wlo - 4)), (float)(whi + 4));
                    lo = (int)ceilf(zlo_f);
                    hi = (int)floorf(zhi_f);
#pragma unroll
                    for (int it = 0; it < 2; ++it) {
                        if (lo > wlo && v_of(lo - 1) >= a.vlo) --lo;
                        if (hi < whi && v_of(hi + 1) <= a.vhi) ++hi;
                    }
#pragma unroll
                    for (int it = 0; it < 2; ++it) {
                        if (lo <= whi && !(v_of(lo) >= a.vlo)) ++lo;
                        if (hi >= wlo && !(v_of(hi) <= a.vhi)) --hi;
                    }
                    lo = max(lo, wlo);
                    hi = min(hi, whi);
                }
                const float w = U * U;
                // an empty interval [lo, hi] with hi < lo becomes a zero-length resource
                slots[ci] = make_int4(r.x, r.y, __float_as_int(w * fu),
                                      (lo - zrb) | (max(hi, lo - 1) - zrb + 1) << kFpZBits);
            }
            ncand += total;
            __syncthreads();  // records complete; wave_cnt free again
        }
        if (ncand > 0) {
            struct Item {
                vbuf rs;
                float U, w, wfu;
                int lo;
            };
            // past the last candidate an item still issues its loads, over an empty
            // resource (they return zero without touching memory)
            auto item_of = [&](int ci, bool valid) {
                const int4 r = slots[valid ? ci : 0];
                const int zb = __builtin_amdgcn_readfirstlane(r.w);
                Item it;
                it.lo = zb & ((1 << kFpZBits) - 1);
                const int hi1 = (zb >> kFpZBits) & ((1 << kFpZBits) - 1);  // one past the last slice
                it.rs = make_vbuf(colbase + (size_t)__builtin_amdgcn_readfirstlane(r.x) * a.zstride + it.lo,
                                  valid ? (hi1 - it.lo) * (int)sizeof(float) : 0);
                // the same value in every lane: kept in vector registers (operands of the
                // per-voxel arithmetic), where moving them to scalars would cost a
                // readfirstlane each
                it.U = __int_as_float(r.y);
                it.w = it.U * it.U;  // as in the fill: the weight is U^2
                it.wfu = __int_as_float(r.z);
                return it;
            };
            // Candidate ci goes to wave ci mod 4.  Three named slots keep the next two
            // candidates' voxels in flight while one is accumulated.
            struct Slot { Item it; float x[G]; };
            int ci_f = wv;
            auto next = [&](Slot& sl) -> bool {
                const bool valid = ci_f < ncand;
                sl.it = item_of(ci_f, valid);
#pragma unroll
                for (int k = 0; k < G; ++k)
                    sl.x[k] = vbuf_load(sl.it.rs, vadd_sv((zc + 64 * k - sl.it.lo) * (int)sizeof(float), lane4));
                ci_f += kGWaves;
                __builtin_amdgcn_sched_barrier(0);  // keep the slots' loads in walk order
                return valid;
            };
            // The G chunks of one item touch distinct entries of each copy (same-parity
            // lanes of the item are two or more slices apart, so their rows differ), so
            // all G reads are issued before the first write: one LDS round trip per item
            // instead of one per chunk.
            auto process = [&](const Slot& sl) {
                float4* e[G];
                float4 v[G];
                float fv[G];
#pragma unroll
                for (int k = 0; k < G; ++k) {
                    const float vA = fmaf(-zh[k], sl.it.U, a.vpre);  // det_row_anchor(zwa, h, U, vpre)
                    const float vI = det_row_index(lane_k, sl.it.U, vA);
                    const int v0 = flr_i32(vI);
                    fv[k] = __builtin_amdgcn_fractf(vI);
                    e[k] = reinterpret_cast<float4*>(acc_bytes + (v0 * 16 + lane_base));
                    v[k] = *e[k];
                }
#pragma unroll
                for (int k = 0; k < G; ++k) {
                    const float t = sl.it.w * sl.x[k], tu = sl.it.wfu * sl.x[k];
                    v[k].x += t;
                    v[k].y += tu;
                    v[k].z = fmaf(t, fv[k], v[k].z);
                    v[k].w = fmaf(tu, fv[k], v[k].w);
                    *e[k] = v[k];
                }
            };
            if (CHECK && opaque_uniform(by_tap)) {
                for (int ci = wv; ci < ncand; ci += kGWaves) {
                    const int4 r = slots[ci];
                    const int lo = r.w & ((1 << kFpZBits) - 1), hi1 = (r.w >> kFpZBits) & ((1 << kFpZBits) - 1);
                    const float U = __int_as_float(r.y), ws = __int_as_float(r.z), wo = U * U - ws;
                    for (int k = 0; k < G; ++k) {
                        const int z = zc + 64 * k + lane;
                        const float vI = det_row_index(lane_k, U, fmaf(-zh[k], U, a.vpre)), v0 = floorf(vI);
                        const bool on = z >= lo && z < hi1;
                        const float x = on ? colbase[(size_t)r.x * a.zstride + z] : 0.0f;
                        float4* const e = reinterpret_cast<float4*>(acc_bytes + ((int)v0 * 16 + lane_base));
                        for (int j = 0; j < 2; ++j) {
                            const float wr = j ? vI - v0 : 1.0f - (vI - v0);
                            float4 o = e[j];
                            o.x += wo * wr * x;
                            o.y += ws * wr * x;
                            if (on) e[j] = o;
                            // the next row of one lane may be the row of another
                            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                            __builtin_amdgcn_wave_barrier();
                        }
                    }
                }
            } else {
                Slot sa, sb, sc;
                bool ha = next(sa), hb = next(sb), hc = next(sc);
                while (ha) {
                    process(sa);
                    ha = next(sa);
                    if (!hb) break;
                    process(sb);
                    hb = next(sb);
                    if (!hc) break;
                    process(sc);
                    hc = next(sc);
                }
            }
            ncand = 0;
            __syncthreads();  // every wave is done with the slots
        }
    }
    // sum the eight copies per entry row (waves in order, even before odd) and turn the
    // entry gradients into pixel partials: own column (q00 at row v, q01 at v + 1) and
    // the next column (q10 at v, q11 at v + 1); pixel row rbase + r takes entry rows r
    // and r - 1 (tap by tap: its own row's sums)
    float2* col = ps + ((size_t)p * a.W + c) * a.H;
    auto entry = [&](int r) {
        float4 sum = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (r >= 0 && r < span) {
            for (int w = 0; w < kGWaves; ++w)
                for (int par = 0; par < 2; ++par) {
                    const float4 e = entry_lds[(w * 2 + par) * stride + r];
                    sum.x += e.x; sum.y += e.y; sum.z += e.z; sum.w += e.w;
                }
        }
        return sum;
    };
    if constexpr (CHECK) {
        bool bad = false;
        for (int r = tid; r < span; r += kGThreads) {
            const float4 e = entry(r);
            bad |= !((fabsf(e.x) + fabsf(e.y)) + (fabsf(e.z) + fabsf(e.w)) <= 3.402823466e38f);
        }
        if (__builtin_amdgcn_readfirstlane(__syncthreads_or(bad)) && !by_tap) {
            by_tap = 1;
            goto again;
        }
    }
    const int row0 = win.first ? 0 : max(win.rbase, 0), row1 = win.first ? a.H - 1 : min(win.rbase + span, a.H - 1);
    for (int row = row0 + tid; row <= row1; row += kGThreads) {
        const int r = row - win.rbase;
        const float4 e0 = entry(r), e1 = entry(r - 1);  // entries at rows v = row and v = row - 1
        float own = ((e0.x - e0.y) - e0.z + e0.w) + (e1.z - e1.w);
        float side = (e0.y - e0.w) + e1.w;
        if (CHECK && by_tap) {
            own = e0.x;
            side = e0.y;
        }
        float2 o = win.first ? make_float2(0.0f, 0.0f) : col[row];
        o.x += own;
        o.y += side;
        col[row] = o;
    }
}

// ------------------------------------------------------------ row-run projector
//
// Every voxel adds its two row taps to pixel columns c = u0 and c + 1, with weights
// w (1 - fu) and w fu, w = U^2.  The voxel columns that feed one c lie along a ray, and from
// one to the next the detector row of a given slice moves by (z + h) dU, a small part of a
// pixel.  So a lane keeps one slice (per chunk of 64) and walks the candidates in depth
// order: over a run of candidates whose rows of the window's outermost slice stay within one
// pixel, its taps fall on three rows R, R + 1, R + 2, whose six sums (three rows, two pixel
// columns) stay in registers.  Each row's weight is the hat 1 - |vIndex - row| clamped at 0,
// from the backprojection's own vIndex (exactly 1 - fv and fv on the two rows of a tap).
// Only the end of a run touches LDS.
//
// fp_rows_kernel<G>: a workgroup owns pixel column c of one projection within one
// window of 64 G slices (grid z [wz0, wz0 + 64 G), wz0 - zrb a multiple of 64).
//  - Candidates are the voxel columns with u0 == c that pass the cylinder and u window
//    tests, between the two fan rays through u = c - 0.05 and u = c + 1.05 (plus a
//    0.01-voxel margin).  Each lane tests the lateral slots of one depth step and the
//    survivors (column, U, fu) go compacted into LDS in depth order; then one lane each
//    settles its z interval of the v-window test (exactly, with the backprojection's
//    expression), intersected with the slab and the window, and writes the final record.
//  - Each wave walks a quarter of the list.  A candidate is one item of G chunks of 64
//    slices: lane l takes slices wz0 + 64 k + l, whose row anchor is (l & 32) slices past
//    the chunk start and whose offset from it is l & 31, as in the backprojection.  The
//    voxels come through a buffer resource covering the candidate's interval (zero outside
//    it, which is the window, slab and v-window mask).
//  - A run is the most of the next 16 candidates whose magnifications span [Umin, Umax] with (Umax - Umin) |z + h| <= 0.98 over the window; R is the row below the
//    smaller of vIndex(Umin) and vIndex(Umax), less 0.002 for the rounding of either.
//  - At the end of a run each lane adds its sums into its wave's rows in LDS, kept in two
//    copies (even and odd lanes): lanes two slices apart have rows at least 2U - 1e-3 > 1
//    apart (U > 2/3 whenever the cylinder radius is below half the FCD, checked on the
//    host), and chunks are 64 slices apart, so no two lanes of one copy touch one row in an
//    instruction and the read-modify-writes need no atomics.  The host bounds the rows that
//    any slice of the window can reach for every candidate U and height, [rbase, rbase +
//    span), so lanes outside their interval (adding zero) stay inside their own copy.
//  - At the end the eight copies are summed in a fixed order (if a sum is infinite or NaN, the
//    workgroup starts again and adds every voxel's two taps by themselves, so that such voxels
//    reach their own two rows only) and added into the workgroup's own float2 column ps[p][c][*] of a column-major buffer (own column c, next column).
//    Windows run one after another on one stream; fp_finish_kernel then adds ps[p][c][r].x +
//    ps[p][c-1][r].y into the row-major image.
// The order of every addition is fixed: the result does not depend on scheduling.
//
// What bounds it: VALU issue, then the memory: 92 % of the time remains at 512^3 when every
// voxel read hits L2 (85 % of a 768^3 iteration with 60 projections per call).  At 512^3 x 360
// projections of 512 x 512 (5.9e8 wave-updates inside the cylinder) it issues 1.07e10 VALU
// instructions, 18 per update: 11 for the update, 2 for its candidate, 3 to end a run and
// start the next (9.6 candidates per run), the rest to fill the list.  16.3 ms.  Twice the row
// sums in LDS, |e| instead of max(e, 0) and runs of any length to 16 instead of powers of two
// took 18.3 ms to 16.9, column sums and images written instead of cleared and added to the rest
// (at 4 waves per SIMD: 134 VGPRs, 6 too many without being told, cost 2 ms).  A form that added each voxel's two rows to LDS as it came (one 16-byte
// read-modify-write per update, LDS-bound) took 24.8 ms; with its column-by-column order 1 %
// of the voxel reads hit the L2, with fp_item's units 53 %.
constexpr int kJ = 3;  // lateral slots per lane and round
constexpr int kESlots = (kJ + 1) * kGThreads;  // a round always fits behind 256 candidates
constexpr int kEMaxSpan = 512;  // rows per copy

// min and max over a lane and the `S` before it in its row of 16 lanes (fewer at the row's
// start).  On the bits of positive floats, which order like integers (no canonicalisation).
template <int S>
__device__ inline void dpp_minmax(int& mn, int& mx) {
#if defined(__HIP_DEVICE_COMPILE__)
    mn = min(mn, __builtin_amdgcn_update_dpp(mn, mn, 0x110 + S, 0xf, 0xf, false));  // row_shr:S
    mx = max(mx, __builtin_amdgcn_update_dpp(mx, mx, 0x110 + S, 0xf, 0xf, false));
#endif
}
// A scalar that the optimiser knows nothing about.
__device__ inline int opaque_scalar(int v) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+s"(v));
#endif
    return v;
}
// acc += x |e|, in place (see fmac)
__device__ inline void fma_abs(float& acc, float x, float e) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm("v_fma_f32 %0, %1, |%2|, %0" : "+v"(acc) : "v"(x), "v"(e));
#else
    acc = fmaf(x, fabsf(e), acc);
#endif
}
// x = v, keeping x in its register (see fmac)
__device__ inline void set_in_place(float& x, float v) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm("v_mov_b32 %0, %1" : "+v"(x) : "v"(v));
#else
    x = v;
#endif
}
__device__ inline float lane_value(int x, int lane) { return __int_as_float(__builtin_amdgcn_readlane(x, lane)); }

// The workgroups that an XCD runs together (dispatch is round-robin over 8 XCDs) should read
// the same voxels: a voxel column is read once per projection, by the column it falls on, and
// for neighbouring projections by neighbouring columns.  So the work is cut into units of
// kPBlock projections x cblock columns, dealt to the XCDs in turn (columns vary slowest, so
// that short rays at the edges spread over the XCDs), and inside a unit the projections vary
// fastest.  Units of the rounded-up grid beyond it exit, and the last workgroups of a unit that
// reaches past the last projection or column (not every fourth: an XCD deals workgroups to its
// shader engines in turn, and one projection of 384^3 took 182 us so, with work on one engine).
//
// Columns per unit: 64, halved down to 8 while there are fewer than 64 units, that is eight for
// each XCD: 40 projections of 50 columns are 10 units of 64, two of them for two of the XCDs.
constexpr int kPBlock = 4, kCBlock = 64, kMinCBlock = 8;
__host__ __device__ inline unsigned fp_units(int W, int nproj, int cblock) {
    return (unsigned)((W + cblock - 1) / cblock) * (unsigned)((nproj + kPBlock - 1) / kPBlock);
}
__device__ inline bool fp_item(const FpArgs& a, int& c, int& p) {
    const unsigned per = (unsigned)(kPBlock * a.cblock);
    const unsigned xcd = blockIdx.x & 7u, k = blockIdx.x >> 3;
    const unsigned unit = (k / per) * 8u + xcd, r = k % per;
    const unsigned npb = (unsigned)((a.nproj + kPBlock - 1) / kPBlock);
    const unsigned cb = unit / npb, pb = unit - cb * npb;
    const unsigned np = (unsigned)min(kPBlock, a.nproj - (int)pb * kPBlock);  // projections of this unit
    const unsigned cl = np == kPBlock ? r / kPBlock : r / np;
    c = (int)(cb * a.cblock + cl);
    p = (int)(pb * kPBlock + (r - cl * np));
    return cl < (unsigned)a.cblock && c < a.W;
}

template <int G>
__global__ __launch_bounds__(kGThreads) __attribute__((amdgpu_waves_per_eu(4))) void fp_rows_kernel(FpArgs a, FpWin win, const float4* __restrict__ pp,
                                                            const float* __restrict__ vol,
                                                            float2* __restrict__ ps) {
    // column, U, w fu and the z interval relative to the run base (w = U^2 is recomputed
    // from U): one 16-byte LDS read per item
    __shared__ int4 slots[kESlots];
    __shared__ int wave_cnt[kGWaves];
    // [wave][parity][row]: (own column, next column)
    extern __shared__ float2 acc_lds[];
    int c, p;
    if (!fp_item(a, c, p)) return;
    const int tid = (int)threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int span = win.span, stride = win.stride;
    const float4 g = pp[p];
    const float sn = g.x, cs = g.y, h = g.z;
    const float Sx = a.fcd * cs + a.uoff * sn, Sy = a.fcd * sn - a.uoff * cs;
    const float ulo = (float)c - 0.05f - a.upre, uhi = (float)c + 1.05f - a.upre;
    const float q0x = -(ulo - a.uoff) * sn, q0y = (ulo - a.uoff) * cs;
    const float q1x = -(uhi - a.uoff) * sn, q1y = (uhi - a.uoff) * cs;
    const float umid = (float)c + 0.5f - a.upre - a.uoff;
    const bool xmajor = fabsf(-umid * sn - Sx) >= fabsf(umid * cs - Sy);
    const int n_out = xmajor ? a.nx : a.ny, n_in = xmajor ? a.ny : a.nx;
    const float pre_out = xmajor ? a.xpre : a.ypre, pre_in = xmajor ? a.ypre : a.xpre;
    const float So = xmajor ? Sx : Sy, Si = xmajor ? Sy : Sx;
    // (divided: the slopes' error is multiplied by the distance to the source, and a hardware
    // reciprocal one ulp off its rounded value loses voxel columns from 6e5 pixels on)
    const float k0 = ((xmajor ? q0y : q0x) - Si) / ((xmajor ? q0x : q0y) - So);
    const float k1 = ((xmajor ? q1y : q1x) - Si) / ((xmajor ? q1x : q1y) - So);
    const float R = sqrtf(a.r2);
    const int o_lo = max(0, (int)floorf(pre_out - R) - 1), o_hi = min(n_out - 1, (int)ceilf(pre_out + R) + 1);
    const int zend = a.z0 + a.nzs - 1;
    const int zrb = a.z0 & ~(kRowAnchor - 1);
    // the slices of this window inside the slab
    const int wlo = max(a.z0, win.wz0), whi = min(zend, win.wz0 + 64 * G - 1);

    auto jrange = [&](int o, int& jl, int& jh) {
        const float ow = (float)o - pre_out;
        const float i0 = Si + (ow - So) * k0, i1 = Si + (ow - So) * k1;
        jl = max(0, (int)ceilf(fminf(i0, i1) + pre_in - 0.01f));
        jh = min(n_in - 1, (int)floorf(fmaxf(i0, i1) + pre_in + 0.01f));
    };
    // lateral slots per depth step: the wedge width |i1 - i0| is linear in the depth and
    // the source lies outside the volume, so it peaks at an end of the depth range; a
    // window of width w + 0.02 holds at most floor(w) + 2 integers
    auto width = [&](int o) {
        const float ow = (float)o - pre_out;
        return fabsf((ow - So) * (k1 - k0));
    };
    const int jm = (int)fmaxf(width(o_lo), width(o_hi)) + 2;

    // per lane and chunk: world z of the slice's row anchor plus the height (the
    // backprojection's zwa + h), and the slice's offset from the anchor
    float zh[G];
#pragma unroll
    for (int k = 0; k < G; ++k) zh[k] = ((float)(win.wz0 + 64 * k + (lane & 32)) - a.zpre) + h;
    const float lane_k = (float)(lane & 31);
    // the window's largest |z + h|
    const float zm = fmaxf(fabsf(((float)win.wz0 - a.zpre) + h), fabsf(((float)(win.wz0 + 64 * G - 1) - a.zpre) + h));
    float2* const my_rows = acc_lds + (wv * 2 + (lane & 1)) * stride - win.rbase;
    // A candidate's voxels are read from the window's first slice inside the slab, zs (relative
    // to the run base).  Lanes of chunk 0 before it wrap to a huge offset, past every
    // resource; an immediate added to that was measured to read zeros where the sum lands inside
    // it, so the later chunks start from a register of their own, which the compiler may add
    // immediates to but not fold into chunk 0's.
    const int zs = max(wlo - zrb, win.wz0 - zrb);
    const float* colbase = vol + (zrb - a.z0) + zs;
    const unsigned off0 = (unsigned)((lane - (zs - (win.wz0 - zrb))) * (int)sizeof(float));
    const unsigned off1 = vadd_sv(256, off0);

    // An infinite or NaN voxel makes all three rows of its run infinite or NaN, and sums past half
    // the largest float overflow where they are held twice: a column with such sums is computed
    // again, tap by tap, into rows that hold the sums once.
    int by_tap = 0;
again:
    for (int i = tid; i < 2 * kGWaves * stride; i += kGThreads) acc_lds[i] = make_float2(0.0f, 0.0f);
    __syncthreads();

    // Rounds: 256 depth steps (one per lane) times kJ lateral slots, all laterals of a block of
    // depth steps before the next block.
    int ncand = 0;
    for (int ob = o_lo, jb = 0; ob <= o_hi && wlo <= whi;) {
        // fill, step 1: the cheap tests of this lane's slots; survivors are compacted in
        // depth order (ballot prefix within each wave, wave totals through LDS)
        int4 rec[kJ];
        int cnt = 0;  // survivors of this lane: rec[0 .. cnt)
        const int o = ob + tid;
        if (o <= o_hi) {
            int jl, jh;
            jrange(o, jl, jh);
#pragma unroll
            for (int jj = 0; jj < kJ; ++jj) {
                const int j = jl + jb + jj;
                if (j > jh) continue;
                const int xi = xmajor ? o : j, yi = xmajor ? j : o;
                // per-voxel arithmetic identical to the backprojection's
                const float x = (float)xi - a.xpre, y = (float)yi - a.ypre;
                if (!(x * x + y * y < a.r2)) continue;
                float t = (-1.0f) * x * g.x + y * g.y;
                t += a.uoff;
                const float s = x * g.y + y * g.x;
                const float U = cone_magnification(a.fcd, s);
                const float u = t * U;
                if (!(u >= a.ulo && u <= a.uhi)) continue;
                const float uIdx = u + a.upre;
                const int u0 = (int)uIdx;
                if (u0 != c) continue;
                const int4 r = make_int4(xi * a.ny + yi, __float_as_int(U), __float_as_int(uIdx - (float)u0), 0);
#pragma unroll
                for (int q = 0; q < kJ; ++q)
                    if (q == cnt) rec[q] = r;
                ++cnt;
            }
        }
        const bool last_round = jb + kJ >= jm && ob + kGThreads > o_hi;
        if (jb + kJ >= jm) {
            jb = 0;
            ob += kGThreads;
        } else {
            jb += kJ;
        }
        {
            static_assert(kJ <= 3, "two ballots count the survivors of a lane");
            const unsigned long long m1 = __ballot(cnt & 1), m2 = __ballot(cnt & 2), lt = (1ull << lane) - 1ull;
            if (lane == 0) wave_cnt[wv] = __popcll(m1) + 2 * __popcll(m2);
            __syncthreads();
            int base = ncand + __popcll(m1 & lt) + 2 * __popcll(m2 & lt);
            for (int w = 0; w < wv; ++w) base += wave_cnt[w];
            int total = 0;
            for (int w = 0; w < kGWaves; ++w) total += wave_cnt[w];
#pragma unroll
            for (int q = 0; q < kJ; ++q)
                if (q < cnt) slots[base + q] = rec[q];
            __syncthreads();  // the slots are complete; wave_cnt is rewritten below
            // fill, step 2: one lane per new survivor settles its z interval and writes its
            // final record (candidates with an empty interval keep an empty one)
            for (int ci = ncand + tid; ci < ncand + total; ci += kGThreads) {
                const int4 r = slots[ci];
                const float U = __int_as_float(r.y), fu = __int_as_float(r.z);
                auto v_of = [&](int zi) { const float zk = (float)zi - a.zpre; return (zk + h) * U; };
                int lo = wlo, hi = whi;
                if (!(v_of(wlo) >= a.vlo && v_of(whi) <= a.vhi)) {
                    // the passing z of v = (zk + h) U in [vLo, vHi] form an interval (v is
                    // non-decreasing in z): estimate its ends, then settle them with the
                    // backprojection's own expression
                    const float iU = __builtin_amdgcn_rcpf(U);
                    const float zlo_f = fminf(fmaxf(a.vlo * iU - h + a.zpre, (float)(wlo - 4)), (float)(whi + 4));
                    const float zhi_f = fminf(fmaxf(a.vhi * iU - h + a.zpre, (float)(wlo - 4)), (float)(whi + 4));
                    lo = (int)ceilf(zlo_f);
                    hi = (int)floorf(zhi_f);
#pragma unroll
                    for (int it = 0; it < 2; ++it) {
                        if (lo > wlo && v_of(lo - 1) >= a.vlo) --lo;
                        if (hi < whi && v_of(hi + 1) <= a.vhi) ++hi;
                    }
#pragma unroll
                    for (int it = 0; it < 2; ++it) {
                        if (lo <= whi && !(v_of(lo) >= a.vlo)) ++lo;
                        if (hi >= wlo && !(v_of(hi) <= a.vhi)) --hi;
                    }
                    lo = max(lo, wlo);
                    hi = min(hi, whi);
                }
                const float w = U * U;
                // an empty interval [lo, hi] with hi < lo becomes a zero-length resource
                slots[ci] = make_int4(r.x, r.y, __float_as_int(w * fu),
                                      (lo - zrb) | (max(hi, lo - 1) - zrb + 1) << kFpZBits);
            }
            ncand += total;
            __syncthreads();  // records complete; wave_cnt free again
        }
        // walk when another fill round might not fit, and after the last round
        if (ncand > kESlots - kJ * kGThreads || last_round) {
            // this wave's part of the list
            const int per_wave = (ncand + kGWaves - 1) / kGWaves;
            const int c_begin = min(wv * per_wave, ncand), c_end = min(c_begin + per_wave, ncand);
            struct Item {
                vbuf rs;
                float U, wo, ws;  // weights of the own and the next column
                int lo;
            };
            // past the last candidate an item still issues its loads, over an empty
            // resource (they return zero without touching memory)
            auto item_of = [&](int ci, bool valid) {
                const int4 r = slots[valid ? ci : 0];
                const int zb = __builtin_amdgcn_readfirstlane(r.w);
                Item it;
                it.lo = zb & ((1 << kFpZBits) - 1);
                const int hi1 = zb >> kFpZBits;  // one past the last slice
                it.rs = make_vbuf(colbase + (size_t)__builtin_amdgcn_readfirstlane(r.x) * a.zstride,
                                  valid && hi1 > it.lo ? (hi1 - zs) * (int)sizeof(float) : 0);
                // the same value in every lane: kept in vector registers (operands of the
                // per-voxel arithmetic), where moving them to scalars would cost a
                // readfirstlane each
                it.U = __int_as_float(r.y);
                it.ws = __int_as_float(r.z);
                it.wo = it.U * it.U - it.ws;
                return it;
            };
            // Three named slots keep the next two candidates' voxels in flight while one is
            // accumulated.
            struct Slot { Item it; float x[G]; };
            int ci_f = c_begin;
            auto next = [&](Slot& sl) {
                sl.it = item_of(ci_f, ci_f < c_end);
#pragma unroll
                for (int k = 0; k < G; ++k)
                    sl.x[k] = vbuf_load(sl.it.rs, k == 0 ? off0 : off1 + 256u * (unsigned)(k - 1));
                ++ci_f;
                __builtin_amdgcn_sched_barrier(0);  // keep the slots' loads in walk order
            };
            const float vpre_run = a.vpre - 0.002f;
            // sums S0, S1, S2 over a run of x, x e and x |e|, e = vIndex - (R + 1), for the own
            // and the next column: row R takes (S2 - S1) / 2, R + 1 S0 - S2, R + 2 (S2 + S1) / 2
            // (the LDS rows hold twice that)
            float acc[G][6];
            float row1[G];   // R + 1
            float2* at[G];   // row R in this lane's copy
#pragma unroll
            for (int k = 0; k < G; ++k) {
                row1[k] = (float)(win.rbase + 1);
                at[k] = my_rows + win.rbase;
#pragma unroll
                for (int j = 0; j < 6; ++j) acc[k][j] = 0.0f;
            }
            auto flush = [&]() {
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    // The G rows of a lane and those of the other lanes are distinct; row j + 1
                    // of one lane may be row j of another, so the compiler must keep the
                    // three steps apart (a wave's LDS operations then run in order).
                    float2 o[G];
#pragma unroll
                    for (int k = 0; k < G; ++k) o[k] = at[k][j];
#pragma unroll
                    for (int k = 0; k < G; ++k) {
                        const float* S = acc[k];
                        o[k].x = j == 0 ? o[k].x + (S[4] - S[2]) : j == 1 ? fmaf(2.0f, S[0] - S[4], o[k].x) : o[k].x + (S[4] + S[2]);
                        o[k].y = j == 0 ? o[k].y + (S[5] - S[3]) : j == 1 ? fmaf(2.0f, S[1] - S[5], o[k].y) : o[k].y + (S[5] + S[3]);
                        at[k][j] = o[k];
                    }
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                }
#pragma unroll
                for (int k = 0; k < G; ++k)
#pragma unroll
                    for (int j = 0; j < 6; ++j) set_in_place(acc[k][j], 0.0f);
            };
            // starts a run at candidate ci; returns its length
            auto start_run = [&](int ci) -> int {
                // lane l of a row: the extremes of the next l + 1 magnitudes
                int mn = slots[min(ci + (lane & 15), c_end - 1)].y, mx = mn;
                dpp_minmax<1>(mn, mx);
                dpp_minmax<2>(mn, mx);
                dpp_minmax<4>(mn, mx);
                dpp_minmax<8>(mn, mx);
                const unsigned over = (unsigned)__ballot(!((__int_as_float(mx) - __int_as_float(mn)) * zm <= 0.98f));
                const int n = __builtin_ctz((over & 0xfffeu) | 0x10000u);
                const float umin = lane_value(mn, n - 1), umax = lane_value(mx, n - 1);
#pragma unroll
                for (int k = 0; k < G; ++k) {
                    // within 0.001 of vIndex of the lanes whose row is on the detector
                    const float y = zh[k] + lane_k;
                    const float R = floorf(fminf(fmaf(-y, umin, vpre_run), fmaf(-y, umax, vpre_run)));
                    set_in_place(row1[k], R + 1.0f);
                    at[k] = my_rows + (int)R;
                }
                return n;
            };
            int ci_p = c_begin, left = 0;
            auto process = [&](Slot& sl) {
                if (opaque_scalar(left) == 0) {
                    if (opaque_scalar(ci_p) != c_begin) flush();
                    left = start_run(ci_p);
                }
                --left;
                ++ci_p;
                if (sl.it.lo > zs) {
                    // the v window starts inside the window: slices before it are masked
                    // here (those past its end are past the resource's)
#pragma unroll
                    for (int k = 0; k < G; ++k)
                        if (win.wz0 - zrb + 64 * k + lane < sl.it.lo) sl.x[k] = 0.0f;
                }
#pragma unroll
                for (int k = 0; k < G; ++k) {
                    const float vA = fmaf(-zh[k], sl.it.U, a.vpre);  // det_row_anchor(zwa, h, U, vpre)
                    const float e = det_row_index(lane_k, sl.it.U, vA) - row1[k];
                    const float xo = sl.it.wo * sl.x[k], xs = sl.it.ws * sl.x[k];
                    acc[k][0] += xo;
                    acc[k][1] += xs;
                    fmac(acc[k][2], xo, e);
                    fmac(acc[k][3], xs, e);
                    fma_abs(acc[k][4], xo, e);
                    fma_abs(acc[k][5], xs, e);
                }
            };
            // Three items at a time, whatever is left (items past the last add zeros): with
            // a way out between them the compiler no longer knows which loads are older
            // and waits for all of them at each item.
            if (opaque_uniform(by_tap)) {
                for (int ci = c_begin; ci < c_end; ++ci) {
                    const int4 r = slots[ci];
                    const int zb = r.w, lo = zb & ((1 << kFpZBits) - 1), hi1 = zb >> kFpZBits;
                    const float U = __int_as_float(r.y), ws = __int_as_float(r.z), wo = U * U - ws;
                    for (int k = 0; k < G; ++k) {
                        const int z = win.wz0 - zrb + 64 * k + lane;
                        const float zk = ((float)(win.wz0 + 64 * k + (lane & 32)) - a.zpre) + h;
                        const float vI = det_row_index(lane_k, U, fmaf(-zk, U, a.vpre)), v0 = floorf(vI);
                        const bool on = z >= lo && z < hi1;
                        const float x = on ? colbase[(size_t)r.x * a.zstride + (z - zs)] : 0.0f;
                        float2* const at0 = my_rows + (int)v0;
                        for (int j = 0; j < 2; ++j) {
                            const float wr = j ? vI - v0 : 1.0f - (vI - v0);
                            float2 o = at0[j];
                            o.x += wo * wr * x;
                            o.y += ws * wr * x;
                            if (on) at0[j] = o;
                            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                            __builtin_amdgcn_wave_barrier();
                        }
                    }
                }
            } else if (c_begin < c_end) {
                Slot sa, sb, sc;
                next(sa);
                next(sb);
                next(sc);
                do {
                    process(sa);
                    next(sa);
                    process(sb);
                    next(sb);
                    process(sc);
                    next(sc);
                } while (ci_p < c_end);
                flush();
            }
            ncand = 0;
            __syncthreads();  // every wave is done with the slots
        }
    }
    // sum the eight copies per row (waves in order, even before odd)
    bool bad = false;
    for (int r = tid; r < span; r += kGThreads) {
        const int row = win.rbase + r;
        if (row < 0 || row >= a.H) continue;
        float2 o = acc_lds[r];
        for (int w = 1; w < 2 * kGWaves; ++w) {
            const float2 e = acc_lds[w * stride + r];
            o.x += e.x;
            o.y += e.y;
        }
        bad |= !(fabsf(o.x) + fabsf(o.y) <= 3.402823466e38f);
        acc_lds[r] = o;
    }
    if (__builtin_amdgcn_readfirstlane(__syncthreads_or(bad)) && !by_tap) {
        by_tap = 1;
        goto again;
    }
    const float share = by_tap ? 1.0f : 0.5f;
    float2* col = ps + ((size_t)p * a.W + c) * a.H;
    const int row0 = win.first ? 0 : max(win.rbase, 0), row1 = win.first ? a.H - 1 : min(win.rbase + span - 1, a.H - 1);
    for (int row = row0 + tid; row <= row1; row += kGThreads) {
        const int r = row - win.rbase;
        const float2 s2 = r >= 0 && r < span ? acc_lds[r] : make_float2(0.0f, 0.0f);
        float2 o = win.first ? make_float2(0.0f, 0.0f) : col[row];
        o.x = fmaf(share, s2.x, o.x);
        o.y = fmaf(share, s2.y, o.y);
        col[row] = o;
    }
}

// img[p][r][c] = or += ps[p][c][r].x + ps[p][c - 1][r].y: column-major partials into the
// row-major images, through a 32 x 33 tile per (row, column) block.
__global__ __launch_bounds__(256) void fp_finish_kernel(const float2* __restrict__ ps, int W, int H,
                                                        int accumulate, float* __restrict__ img) {
    __shared__ float2 tile[33][33];  // [column - c0 + 1][row - r0]
    const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
    const size_t p = blockIdx.z;
    const int tl = threadIdx.x & 31;
    for (int i = threadIdx.x >> 5; i < 33; i += 8) {
        const int cc = c0 - 1 + i, r = r0 + tl;
        tile[i][tl] = (cc >= 0 && cc < W && r < H) ? ps[(p * W + cc) * H + r] : make_float2(0.0f, 0.0f);
    }
    __syncthreads();
    for (int i = threadIdx.x >> 5; i < 32; i += 8) {
        const int r = r0 + i, cc = c0 + tl;
        if (cc < W && r < H) {
            float* o = img + (p * H + r) * W + cc;
            *o = (accumulate ? *o : 0.0f) + (tile[tl + 1][i].x + tile[tl][i].y);
        }
    }
}

// ------------------------------------------------------------------ phantom

struct EllDev {
    double c[3];
    double M[9];  // D^-1 R^T (rows)
    double mu;
};

__device__ inline uint64_t splitmix64(uint64_t& s) {
    uint64_t z = (s += 0x9e3779b97f4a7c15ull);
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}
__device__ inline double uniform01(uint64_t& s) { return (double)(splitmix64(s) >> 11) * 0x1.0p-53; }

// Poisson sample: inversion by sequential multiplication for small means, Hormann's
// transformed rejection (PTRS, 1993) otherwise.  The rejection loop is bounded; a draw
// that has not been accepted after 64 rounds returns the rounded mean.
__device__ double poisson(double lam, uint64_t& s) {
    if (lam <= 0.0) return 0.0;
    if (lam < 10.0) {
        const double L = exp(-lam);
        double prod = uniform01(s);
        int k = 0;
        while (prod > L && k < 1000) { prod *= uniform01(s); ++k; }
        return (double)k;
    }
    const double slam = sqrt(lam), loglam = log(lam);
    const double b = 0.931 + 2.53 * slam;
    const double a = -0.059 + 0.02483 * b;
    const double invalpha = 1.1239 + 1.1328 / (b - 3.4);
    const double vr = 0.9277 - 3.6224 / (b - 2.0);
    for (int it = 0; it < 64; ++it) {
        const double U = uniform01(s) - 0.5;
        const double V = uniform01(s);
        const double us = 0.5 - fabs(U);
        const double k = floor((2.0 * a / us + b) * U + lam + 0.43);
        if (us >= 0.07 && V <= vr) return k;
        if (k < 0.0 || (us < 0.013 && V > us)) continue;
        if (log(V) + log(invalpha) - log(a / (us * us) + b) <= -lam + k * loglam - lgamma(k + 1.0)) return k;
    }
    return floor(lam + 0.5);
}

__global__ __launch_bounds__(256) void phantom_kernel(int W, int H, int nproj, int p0, double fcd, double uoff,
                                                      double upre, double vpre, const double4* __restrict__ pp,
                                                      const EllDev* __restrict__ ell, int n_ell, double photons,
                                                      double full_scale, uint64_t seed,
                                                      uint16_t* __restrict__ img, float* __restrict__ lin) {
    const int c = blockIdx.x * 256 + threadIdx.x;
    const int r = blockIdx.y;
    const int pl = blockIdx.z;
    if (c >= W) return;
    const double4 g = pp[p0 + pl];
    const double sn = g.x, cs = g.y, h = g.z;
    const double S[3] = {fcd * cs + uoff * sn, fcd * sn - uoff * cs, -h};
    const double u = (double)c - upre, v = vpre - (double)r;
    const double tq = u - uoff;
    const double Q[3] = {-tq * sn, tq * cs, v - h};
    double d[3] = {Q[0] - S[0], Q[1] - S[1], Q[2] - S[2]};
    const double dn = sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
    d[0] /= dn; d[1] /= dn; d[2] /= dn;
    double acc = 0.0;
    for (int e = 0; e < n_ell; ++e) {
        const EllDev E = ell[e];
        const double o[3] = {S[0] - E.c[0], S[1] - E.c[1], S[2] - E.c[2]};
        double q0[3], q1[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            q0[i] = E.M[3 * i] * o[0] + E.M[3 * i + 1] * o[1] + E.M[3 * i + 2] * o[2];
            q1[i] = E.M[3 * i] * d[0] + E.M[3 * i + 1] * d[1] + E.M[3 * i + 2] * d[2];
        }
        const double A = q1[0] * q1[0] + q1[1] * q1[1] + q1[2] * q1[2];
        const double B = q0[0] * q1[0] + q0[1] * q1[1] + q0[2] * q1[2];
        const double C = q0[0] * q0[0] + q0[1] * q0[1] + q0[2] * q0[2] - 1.0;
        const double disc = B * B - A * C;
        if (disc > 0.0) acc += E.mu * 2.0 * sqrt(disc) / A;
    }
    const size_t idx = ((size_t)pl * H + r) * W + c;
    if (lin) lin[idx] = (float)acc;
    if (img) {
        double val;
        if (photons > 0.0) {
            uint64_t st = seed ^ (0xd1b54a32d192ed03ull * ((uint64_t)(p0 + pl) * H * W + (uint64_t)r * W + c + 1));
            splitmix64(st);
            val = poisson(photons * exp(-acc), st);
        } else {
            val = floor(full_scale * exp(-acc) + 0.5);
        }
        val = fmin(fmax(val, 0.0), 65535.0);
        img[idx] = (uint16_t)val;
    }
}

// --------------------------------------------------------------- conversion

__device__ inline uint32_t maybe_swap(float v, int swap) {
    uint32_t b = __float_as_uint(v);
    return swap ? __builtin_bswap32(b) : b;
}

// Sum over a workgroup of 256, in thread 0, in a fixed order.
__device__ inline double block_sum(double v) {
    __shared__ double part[4];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    return (part[0] + part[1]) + (part[2] + part[3]);
}

// Sums of squares in FP64, one partial per workgroup, then their sum by one workgroup.  Bound
// by the one read of x: 0.34 ms for 768^3 values (5.3 TB/s) where it took 5.5 as library operations,
// two conversions to FP64, a product and a sum.
constexpr unsigned kSumBlocks = CTG_SUM_WORK - 1;
__global__ __launch_bounds__(256) void sum_squares_kernel(const float* __restrict__ x, size_t n, double* __restrict__ part) {
    const size_t i0 = blockIdx.x * (size_t)256 + threadIdx.x, step = gridDim.x * (size_t)256;
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    size_t done = 0;
    if (((uintptr_t)x & 15) == 0) {
        const float4* __restrict__ x4 = reinterpret_cast<const float4*>(x);
        const size_t n4 = n / 4;
        auto add = [&](float4 v) {
            s[0] = fma((double)v.x, (double)v.x, s[0]);
            s[1] = fma((double)v.y, (double)v.y, s[1]);
            s[2] = fma((double)v.z, (double)v.z, s[2]);
            s[3] = fma((double)v.w, (double)v.w, s[3]);
        };
        size_t i = i0;
        for (; i + 3 * step < n4; i += 4 * step) {
            const float4 a = x4[i], b = x4[i + step], c = x4[i + 2 * step], d = x4[i + 3 * step];
            add(a);
            add(b);
            add(c);
            add(d);
        }
        for (; i < n4; i += step) add(x4[i]);
        done = n4 * 4;
    }
    for (size_t i = done + i0; i < n; i += step) s[0] = fma((double)x[i], (double)x[i], s[0]);
    const double sum = block_sum((s[0] + s[1]) + (s[2] + s[3]));
    if (threadIdx.x == 0) part[blockIdx.x] = sum;
}
__global__ __launch_bounds__(256) void sum_partials_kernel(const double* __restrict__ part, unsigned n, double* __restrict__ out) {
    double s = 0.0;
    for (unsigned i = threadIdx.x; i < n; i += 256) s += part[i];
    s = block_sum(s);
    if (threadIdx.x == 0) *out = s;
}

// Z_FASTEST [x][y][z] -> X_FASTEST [z][y][x] through a 32x32 LDS tile per (x,z) block.
__global__ __launch_bounds__(256) void to_xfastest_kernel(const float* __restrict__ in, int nx, int ny, int nz,
                                                          int swap, uint32_t* __restrict__ out) {
    __shared__ float tile[32][33];
    const int z0 = blockIdx.x * 32, x0 = blockIdx.y * 32, y = blockIdx.z;
    const int tl = threadIdx.x & 31;
    for (int i = threadIdx.x >> 5; i < 32; i += 8) {
        const int x = x0 + i, z = z0 + tl;
        tile[i][tl] = (x < nx && z < nz) ? in[((size_t)x * ny + y) * nz + z] : 0.0f;
    }
    __syncthreads();
    for (int i = threadIdx.x >> 5; i < 32; i += 8) {
        const int z = z0 + i, x = x0 + tl;
        if (x < nx && z < nz) out[((size_t)z * ny + y) * nx + x] = maybe_swap(tile[tl][i], swap);
    }
}

__global__ __launch_bounds__(256) void copy_swap_kernel(const float* __restrict__ in, size_t n, int swap,
                                                        uint32_t* __restrict__ out) {
    for (size_t i = blockIdx.x * (size_t)256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
        out[i] = maybe_swap(in[i], swap);
}

}  // namespace

namespace {

// Rows that the slices [wz0, wz0 + nsl) of any voxel column can reach: vIndex =
// vPre - (z + h) U over every world z of the window, every height of the launch's
// projections and every magnification of the cylinder.  A run's first row lies up to two
// below and its last up to two above the rows that its voxels fall in; one more on either
// side covers the rounding of the kernel's anchored expression.
void window_rows(const ctg_geometry& g, double hmin, double hmax, double Umin, double Umax, int wz0, int nsl,
                 int& rbase, int& span) {
    const double ylo = (double)wz0 - g.z_pre + hmin, yhi = (double)(wz0 + nsl - 1) - g.z_pre + hmax;
    const double c[4] = {ylo * Umin, ylo * Umax, yhi * Umin, yhi * Umax};
    const double mn = std::min(std::min(c[0], c[1]), std::min(c[2], c[3]));
    const double mx = std::max(std::max(c[0], c[1]), std::max(c[2], c[3]));
    rbase = (int)std::floor(g.v_pre - mx) - 3;
    const int rtop = (int)std::floor(g.v_pre - mn) + 3;
    span = rtop - rbase + 1;
}

}  // namespace

ctg_status launch_forward_project(const ctg_geometry& g, const float4* d_params, const float4* h_params,
                                  const float* d_volume, int z0, int nz, int nproj, float* d_proj, DevBuf& work,
                                  int accumulate, hipStream_t st) {
    const size_t pixels = (size_t)nproj * g.det_width * g.det_height;
    if (nproj <= 0) return CTG_OK;
    if (nz <= 0) return accumulate ? CTG_OK : fill_u32(d_proj, 0u, pixels, st);
    FpArgs a{};
    a.W = g.det_width; a.H = g.det_height; a.nx = g.nx; a.ny = g.ny; a.nzs = nz; a.z0 = z0; a.nproj = nproj;
    a.xpre = g.x_pre; a.ypre = g.y_pre; a.zpre = g.z_pre; a.upre = g.u_pre; a.vpre = g.v_pre;
    a.r2 = g.radius * g.radius; a.fcd = g.fcd; a.uoff = g.u_offset;
    a.ulo = g.u_lo; a.uhi = g.u_hi; a.vlo = g.v_lo; a.vhi = g.v_hi;
    a.zstride = nz;
    if (a.H > kMaxRowsFp) return fail(CTG_ERROR_UNSUPPORTED, "forward projection of more than %d detector rows", kMaxRowsFp);
    // the candidate z intervals are settled from an estimate accurate to about 1e-2
    // slices for grids of up to 65536 slices
    if (g.nz > 65536 || std::fabs(g.z_pre) > 65536.0f)
        return fail(CTG_ERROR_UNSUPPORTED, "forward projection of more than 65536 slices");
    // U = FCD / (FCD - s) with |s| < radius stays in (1/1.9, 10): at most 4 residue passes
    if (!(g.radius < 0.9f * g.fcd))
        return fail(CTG_ERROR_UNSUPPORTED, "forward projection needs the reconstruction cylinder within 0.9 FCD");
    // a voxel inside the v window reads rows v0, v0 + 1 with 0 <= v0 <= H - 2 (vIndex =
    // vPre - v within about 1e-3 of rounding); the kernel indexes its row accumulators
    // with v0 unclamped
    if (!(g.v_pre - g.v_hi >= -0.5f && g.v_pre - g.v_lo <= (float)g.det_height - 1.05f))
        return fail(CTG_ERROR_UNSUPPORTED, "forward projection needs the v window inside the detector rows");
    dim3 grid((unsigned)a.W, (unsigned)nproj);
    if (grid.y > 65535u) return fail(CTG_ERROR_UNSUPPORTED, "forward projection grid too large");

    // Row-run form (fp_rows_kernel) when the windows' rows fit the LDS copies: it
    // needs U > 2/3 (radius below half the FCD) and host parameters for the row bounds.
    int G = 0;
    double hmin = 0.0, hmax = 0.0;
    const double R = g.radius, F = g.fcd;
    const double Umin = F / (F + R) * (1.0 - 1e-5), Umax = F / (F - R) * (1.0 + 1e-5);
    // Candidates per run of a window's outermost slice: neighbours along a ray are a voxel apart in
    // depth, so their magnifications differ by about 1 / FCD, and a run spans 0.98 rows.
    auto run_of = [&](int w0, int chunks) {
        const double y = w0 - g.z_pre + 0.5 * (hmin + hmax);
        return 0.98 * F / std::max(std::fabs(y), std::fabs(y + 64 * chunks - 1));
    };
    const bool entry_ok = h_params != nullptr && R < 0.5 * F && !std::getenv("CTG_FP_GATHER");
    if (entry_ok) {
        hmin = hmax = h_params[0].z;
        for (int i = 1; i < nproj; ++i) {
            hmin = std::min(hmin, (double)h_params[i].z);
            hmax = std::max(hmax, (double)h_params[i].z);
        }
        const int zrb = z0 & ~(kRowAnchor - 1);
        // CTG_FP_MAXSPAN overrides the rows per copy the window height may need (tuning;
        // at most 800, which keeps the eight copies within 52 KB of LDS)
        int max_span = kEMaxSpan;
        if (const char* e = std::getenv("CTG_FP_MAXSPAN")) max_span = std::max(16, std::min(800, std::atoi(e)));
        // as few windows as chunks of 64 slices allow at four per window, equally deep
        const int nch = (z0 + nz - zrb + 63) / 64;
        const int deep = (nch + (nch + 3) / 4 - 1) / ((nch + 3) / 4);
        for (int cand = deep; cand >= 1 && G == 0; --cand) {
            bool fits = true;
            for (int s = 0; s < nz; s += kFpMaxSlab)
                for (int w0 = zrb + s; w0 < z0 + std::min(s + kFpMaxSlab, nz) && fits; w0 += 64 * cand) {
                    int rb, sp;
                    window_rows(g, hmin, hmax, Umin, Umax, w0, 64 * cand, rb, sp);
                    fits = sp <= max_span;
                }
            if (fits) G = cand;
        }
        // Windows of a single chunk with short runs, where the rows of one column span too much for
        // more, have neither form's advantage: 656^2 x 1015 from a source 1.3 detector widths away
        // takes 15.2 ms so, 11.6 in the gather form; 48^2 x 2000 from 2.5 widths 0.30 and 0.26.
        if (G == 1 && deep > 1 && std::min(run_of(zrb, 1), run_of(z0 + nz - 64, 1)) < kMinRun) G = 0;
    }
    if (G > 0) {
        // the first window writes the column sums and fp_finish_kernel the images, so neither is
        // cleared first
        CTG_TRY(work.reserve(pixels * sizeof(float2)));
        float2* ps = work.as<float2>();
        a.cblock = kCBlock;
        while (a.cblock > kMinCBlock && fp_units(a.W, nproj, a.cblock) < 64) a.cblock /= 2;
        const unsigned long long blocks = (unsigned long long)((fp_units(a.W, nproj, a.cblock) + 7) / 8) * 8 * kPBlock * a.cblock;
        if (blocks > 0x7fffffffull) return fail(CTG_ERROR_UNSUPPORTED, "forward projection grid too large");
        const dim3 rgrid((unsigned)blocks);
        auto window = [&](int w0, int chunks) {
            FpWin win{};
            win.wz0 = w0;
            window_rows(g, hmin, hmax, Umin, Umax, w0, 64 * chunks, win.rbase, win.span);
            return win;
        };
        // windows whose rows all lie off the detector are left out
        auto off = [&](const FpWin& win) { return win.rbase >= a.H || win.rbase + win.span <= 0; };
        int first = 1;  // the first window to run writes the column sums
        // Volumes of at most two chunks of slices (one window) and short rays go to the entry
        // form: its time per update is larger, but it spends less per column (figures there).
        const bool small = z0 + nz - (z0 & ~(kRowAnchor - 1)) <= 128 && std::max(g.nx, g.ny) <= kEntryMaxSide;
        // the candidate records hold z relative to the launch's run base in kFpZBits bits
        for (int s = 0; s < nz; s += kFpMaxSlab) {
            a.z0 = z0 + s;
            a.nzs = std::min(kFpMaxSlab, nz - s);
            const int zend = a.z0 + a.nzs;
            for (int w0 = a.z0 & ~(kRowAnchor - 1); w0 < zend; w0 += 64 * G) {
                FpWin win = window(w0, G);
                if (off(win)) continue;
                bool entries = small || (hmax - hmin <= kMinRunHeights && run_of(w0, G) < kMinRun);
                for (int e0 = w0; e0 < std::min(w0 + 64 * G, zend) && entries; e0 += 128)
                    entries = window(e0, std::min(2, (zend - e0 + 63) / 64)).span <= kEntryMaxSpan;
                for (int e0 = w0; e0 < std::min(w0 + 64 * G, zend) && entries; e0 += 128) {
                    const int chunks = std::min({2, (zend - e0 + 63) / 64, G - (e0 - w0) / 64});
                    FpWin part = window(e0, chunks);
                    if (off(part)) continue;
                    part.stride = (part.span + 15) & ~15;
                    part.first = first;
                    const size_t lds = sizeof(float4) * 2 * kGWaves * (size_t)part.stride;
#define CTG_ENTRY(G, CHECK) \
    hipLaunchKernelGGL((fp_entry_kernel<G, CHECK>), grid, dim3(kGThreads), lds, st, a, part, d_params, d_volume + s, ps)
                    if (small && chunks == 2) CTG_ENTRY(2, false);
                    else if (small) CTG_ENTRY(1, false);
                    else if (chunks == 2) CTG_ENTRY(2, true);
                    else CTG_ENTRY(1, true);
#undef CTG_ENTRY
                    CTG_HIP(hipGetLastError());
                    first = 0;
                }
                if (entries) continue;
                win.stride = (win.span + 1) & ~1;
                win.first = first;
                first = 0;
                const size_t lds = sizeof(float2) * 2 * kGWaves * (size_t)win.stride;
                if (G == 4) hipLaunchKernelGGL(fp_rows_kernel<4>, rgrid, dim3(kGThreads), lds, st, a, win, d_params, d_volume + s, ps);
                else if (G == 3) hipLaunchKernelGGL(fp_rows_kernel<3>, rgrid, dim3(kGThreads), lds, st, a, win, d_params, d_volume + s, ps);
                else if (G == 2) hipLaunchKernelGGL(fp_rows_kernel<2>, rgrid, dim3(kGThreads), lds, st, a, win, d_params, d_volume + s, ps);
                else hipLaunchKernelGGL(fp_rows_kernel<1>, rgrid, dim3(kGThreads), lds, st, a, win, d_params, d_volume + s, ps);
                CTG_HIP(hipGetLastError());
            }
        }
        if (first) return accumulate ? CTG_OK : fill_u32(d_proj, 0u, pixels, st);  // no voxel is seen
        dim3 fg((unsigned)((a.W + 31) / 32), (unsigned)((a.H + 31) / 32), (unsigned)nproj);
        hipLaunchKernelGGL(fp_finish_kernel, fg, dim3(256), 0, st, ps, a.W, a.H, accumulate, d_proj);
        CTG_HIP(hipGetLastError());
        return CTG_OK;
    }

    if (!accumulate) CTG_TRY(fill_u32(d_proj, 0u, pixels, st));
    const size_t lds = sizeof(float) * (size_t)(2 * kGWaves) * (a.H + 4);
    // the candidate records hold z relative to the launch's run base in kFpZBits bits
    for (int s = 0; s < nz; s += kFpMaxSlab) {
        a.z0 = z0 + s;
        a.nzs = std::min(kFpMaxSlab, nz - s);
        hipLaunchKernelGGL(fp_gather_kernel, grid, dim3(kGThreads), lds, st, a, d_params, d_volume + s, d_proj);
        CTG_HIP(hipGetLastError());
    }
    return CTG_OK;
}

ctg_status launch_phantom(const ctg_geometry& g, const double4* d_params, const double* h_ell, int n_ell,
                          int nproj, int p0, double photons, double full_scale, uint64_t seed, uint16_t* d_img,
                          float* d_lineint, DevBuf& ell_buf, hipStream_t st) {
    std::vector<EllDev> e(n_ell > 0 ? n_ell : 1);
    for (int i = 0; i < n_ell; ++i) {
        const double* E = h_ell + 10 * i;
        const double c1 = std::cos(E[6]), s1 = std::sin(E[6]), c2 = std::cos(E[7]), s2 = std::sin(E[7]);
        const double c3 = std::cos(E[8]), s3 = std::sin(E[8]);
        // R = Rz(phi) Ry(theta) Rz(psi), row-major; columns are the ellipsoid axes
        const double R[9] = {c1 * c2 * c3 - s1 * s3, -c1 * c2 * s3 - s1 * c3, c1 * s2,
                             s1 * c2 * c3 + c1 * s3, -s1 * c2 * s3 + c1 * c3, s1 * s2,
                             -s2 * c3,               s2 * s3,                c2};
        for (int a = 0; a < 3; ++a) {
            e[i].c[a] = E[a];
            for (int b = 0; b < 3; ++b) e[i].M[3 * a + b] = R[3 * b + a] / E[3 + a];
        }
        e[i].mu = E[9];
    }
    CTG_TRY(ell_buf.reserve(sizeof(EllDev) * e.size()));
    CTG_HIP(hipMemcpyAsync(ell_buf.ptr, e.data(), sizeof(EllDev) * e.size(), hipMemcpyHostToDevice, st));
    dim3 grid((unsigned)((g.det_width + 255) / 256), (unsigned)g.det_height, (unsigned)nproj);
    hipLaunchKernelGGL(phantom_kernel, grid, dim3(256), 0, st, g.det_width, g.det_height, nproj, p0, (double)g.fcd,
                       (double)g.u_offset, (double)g.u_pre, (double)g.v_pre, d_params, (const EllDev*)ell_buf.ptr,
                       n_ell, photons, full_scale, seed, d_img, d_lineint);
    CTG_HIP(hipGetLastError());
    // the host vector must outlive the asynchronous copy
    CTG_HIP(hipStreamSynchronize(st));
    return CTG_OK;
}

ctg_status launch_sum_squares(const float* d_x, size_t n, double* d_work, hipStream_t st) {
    const unsigned blocks = (unsigned)std::min<size_t>(kSumBlocks, std::max<size_t>(1, (n + 4095) / 4096));
    hipLaunchKernelGGL(sum_squares_kernel, dim3(blocks), dim3(256), 0, st, d_x, n, d_work + 1);
    CTG_HIP(hipGetLastError());
    hipLaunchKernelGGL(sum_partials_kernel, dim3(1), dim3(256), 0, st, d_work + 1, blocks, d_work);
    CTG_HIP(hipGetLastError());
    return CTG_OK;
}

ctg_status launch_convert_volume(const ctg_geometry& g, const float* d_vol, int nz, ctg_index_order order,
                                 ctg_byte_order bo, void* d_out, hipStream_t st) {
    const int swap = bo == CTG_BIG_ENDIAN ? 1 : 0;
    if (order == CTG_Z_FASTEST) {
        const size_t n = (size_t)g.nx * g.ny * nz;
        const unsigned blocks = (unsigned)std::min<size_t>((n + 255) / 256, 65535 * 8);
        hipLaunchKernelGGL(copy_swap_kernel, dim3(blocks ? blocks : 1), dim3(256), 0, st, d_vol, n, swap,
                           (uint32_t*)d_out);
    } else {
        dim3 grid((unsigned)((nz + 31) / 32), (unsigned)((g.nx + 31) / 32), (unsigned)g.ny);
        hipLaunchKernelGGL(to_xfastest_kernel, grid, dim3(256), 0, st, d_vol, g.nx, g.ny, nz, swap,
                           (uint32_t*)d_out);
    }
    CTG_HIP(hipGetLastError());
    return CTG_OK;
}

}  // namespace ctg
