// Voxel-driven FDK backprojection for gfx950.
//
// Per voxel and projection the arithmetic is the reference's (Ct/CtVolume.cpp:979-1039,
// Ct/cuda_ct.cu:234-283): cylinder test x^2+y^2 < R^2; t = -x sin + y cos + uOffset,
// s = x cos + y sin, U = FCD/(FCD-s), u = t U; window test on u; v = (z+h) U and window
// test on v; uIndex = u + uPre, vIndex = vPre - v; bilinear tap of the filtered
// projection; vol += U^2 * value.
//
// Organisation (MI355X-first, not the reference's one-launch-per-projection):
//  - one launch covers many projections; every lane owns one (x,y) voxel column and a
//    run of ZPL consecutive z, accumulating in registers across all projections, so the
//    volume slab is written once per launch (z-fastest, each lane stores ZPL*4 bytes);
//  - projections arrive as bilinear-coefficient entries (A, dU, dV, dUV) stored
//    column-major, so one voxel-update is one LDS read of one entry and
//    val = A + fu*dU + fv*(dV + fu*dUV): 3 FMAs, plus 1 FMA into the accumulator;
//  - a workgroup (256 lanes = 16x16 columns) stages, per projection, the bounding box of
//    its voxel block's detector footprint into LDS with global->LDS DMA (buffer loads
//    to LDS), one detector column per DMA burst, double-buffered so that the DMA of
//    projection p+1 runs under the compute of p (the two buffers reach the compute as
//    __restrict__ pointers, without which the compiler waits for the DMA before the
//    first LDS read); a box's detector columns sit at an LDS pitch of +1 or -1 mod 16
//    entries, chosen per box against bank conflicts;
//  - per z the lane does one FMA for vIndex, v_cvt_flr/v_fract, one address op, the LDS
//    read and 4 FMAs, with the reads software-pipelined in small groups; the
//    per-column geometry (one reciprocal) is amortised over the run;
//  - a step runs in one of three forms: unmasked where the tile's run lies inside the
//    detector window (8 VALU instructions per update and 22 per column), masked by groups
//    of four slices where part of it does not, and voxel by voxel from global memory where
//    the box does not fit the LDS;
//  - boxes are computed by wave 0 for 64 projections at a time (one lane per projection);
//    a projection whose box exceeds the tile capacity reads entries from global memory
//    instead, so any geometry stays correct;
//  - workgroups are numbered so that each XCD (dispatch is round-robin over 8 XCDs)
//    receives contiguous ranges of tiles, in 4x4 blocks of tiles, and shares detector
//    footprints in its own L2, with an equal part of every layer (tile_of).
//
// What bounds it (1024^3 x 720 x 1024^2, MI355X, 160 ms FP32 and 130 ms FP16): with FP32 entries
// the traffic of boxes that miss L2 (658 GB per backprojection, 4.1 TB/s, 39 % L2 hits; an earlier
// form of 162 ms took 137 with every line a hit), then the LDS (a ds_read_b128 takes 4.8 cycles
// per wave and CU, a staging DMA instruction 17 whatever its lane mask); with 8-byte entries VALU
// issue (116 of 133 ms remained without any staging).  Accumulators updated in place, three forms
// per step and tests left out where a box lies inside the window took FP32 from 177 to 163 ms and
// FP16 from 147 to 133, launches of about 240 projections the rest; with the numbering of the tiles
// a 256^3 x 360 scan went from 2.67 to 1.55 ms.
#include "ctg_internal.h"

#include <hip/hip_fp16.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>

namespace ctg {
namespace bp_detail {

constexpr int kTX = 16, kTY = 16, kThreads = 256, kWaves = kThreads / 64;
constexpr int kMaxTileBytes = 36 * 1024;  // per LDS buffer (two buffers per workgroup)
constexpr int kStaticLds = 4112;
// LDS reads per software-pipeline group: with 8-byte entries 4 takes 133.5 ms at 1024^3 x 720
// where 2 takes 134.5 (both fit 96 VGPRs), with FP32 ones 4 is as much as fits.
constexpr int kGrp = 4;
// Detector pixels added around a footprint box's corner bounds: the corner and voxel
// expressions round differently by about 1e-4 pixel at most.
constexpr float kBoxMargin = 0.05f;

constexpr int kMaxStrips = 64;  // strips of a layer

struct BpArgs {
    int W, H, nx, ny, nzs, z0;
    float xpre, ypre, zpre, upre, vpre;
    float r2, fcd, uoff, ulo, uhi, vlo, vhi;
    int nproj, ntx, nty, nzb, cap, accumulate, vec4;
    int resume;              // the sums go on from the volume's values
    int zshift;              // z0 mod ZPL: runs start at grid z multiples of ZPL, zshift voxels before the slab
    int dma16;               // 8-byte entries staged with 16-byte DMA (H even: rows start even)
    int pitch_mod, pitch_rem;  // LDS column pitch = rows rounded up to pitch_rem mod pitch_mod (a power of two)
    int pitch_adapt;           // per box, -pitch_rem mod pitch_mod where the footprint slants the other way
    int pitch_alt;             // remainder for boxes that do not fit with pitch_rem (pitch_rem: none)
    // numbering of the tiles (tile_of)
    int strip_h, nstrips, blk;  // tile rows per strip, tile columns per block
    unsigned nwork, nidle;     // tiles of one layer inside / outside the strips' ranges
    unsigned chunk, extra;     // rounds of 8 chunks, the first `extra` chunks of chunk + 1 tiles, the others of chunk
    unsigned long_rounds, work_wgs;  // rounds of eight chunks with longer ones among them; working tiles' workgroups of an XCD
    unsigned before[kMaxStrips + 1];  // working tiles of the strips before each
    int first[kMaxStrips];            // first working tile column of each strip
};

// Tile of this workgroup; false for the surplus of the rounded-up grid.  A layer (one run of
// slices) is cut into strips of strip_h tile rows, each with the range of tile columns inside
// the reconstruction cylinder; a strip is numbered in blocks of blk columns, so that
// consecutive numbers are neighbours along every ray direction.  The working tiles of all
// layers, in that order, are cut into chunks of equal size (to one tile), eight per layer
// (number_chunks), that go to the XCDs in turn (dispatch is round-robin over 8 XCDs).  So an XCD works on a
// contiguous region, whose footprints its own L2 holds, and yet has an equal share of every
// layer and, since the turn shifts by three per layer, of every part of the layers: outer
// layers and tiles leave the detector window and are cheaper.  The tiles outside the
// cylinder only store; they come last.  No workgroup in between has nothing to do: an XCD deals
// its workgroups to its shader engines in turn, and where most chunks held a tile less than the
// longest, every chunk's last workgroup was such a one (198^2 x 81 from 289 projections, 661
// columns: 698 us, 620 so).
//
// One contiguous range of all tiles per XCD (outer layers all on two of them) took 2.21 ms for
// a 256^3 scan of 360 projections of 256 x 192 and 12.6 ms for 512^3 of 512 x 512, this
// numbering 1.56 and 11.05 ms; 1024^3 does not depend on it (160 ms FP32, 130 FP16), nor on two
// or half a chunk per layer, strips of 2 rows, by more than 3 %; single blocks dealt in turn
// take 171 and 140 ms there, and blocks numbered column by column 132 with FP16.
__device__ inline bool tile_of(const BpArgs& a, int& zbi, int& tx, int& ty) {
    const unsigned xcd = blockIdx.x & 7u, k = blockIdx.x >> 3;
    const bool work = k < a.work_wgs;
    unsigned n;
    if (work) {
        const unsigned big = a.long_rounds * (a.chunk + 1u), size = k < big ? a.chunk + 1u : a.chunk;
        const unsigned kr = k < big ? k : k - big, mr = kr / size, w = kr - mr * size;
        const unsigned m = k < big ? mr : a.long_rounds + mr, i = m * 8u + ((xcd + 3u * m) & 7u);
        if (w >= a.chunk + (i < a.extra ? 1u : 0u)) return false;  // (in the last long round only)
        n = i * a.chunk + min(i, a.extra) + w;
    } else {
        n = (k - a.work_wgs) * 8u + xcd;
        if (n >= a.nidle * (unsigned)a.nzb) return false;
    }
    const unsigned layer = work ? a.nwork : a.nidle;
    zbi = (int)(n / layer);
    unsigned t = n - (unsigned)zbi * layer;
    // the last strip that starts at or before t
    auto start = [&](int s) { return work ? a.before[s] : (unsigned)(a.ntx * a.strip_h * s) - a.before[s]; };
    int lo = 0, hi = a.nstrips;  // start(lo) <= t < start(hi)
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (start(mid) <= t) lo = mid;
        else hi = mid;
    }
    t -= start(lo);
    const int h = min(a.strip_h, a.nty - lo * a.strip_h);
    const int n_in = (int)(a.before[lo + 1] - a.before[lo]) / h;  // working columns
    if (work) {
        const int hb = a.blk * h, b = (int)t / hb, w = (int)t - b * hb;
        const int bw = min(a.blk, n_in - a.blk * b), y = w / bw;
        tx = a.first[lo] + a.blk * b + (w - y * bw);
        ty = lo * a.strip_h + y;
    } else {
        const int c = (int)t / h;
        tx = c < a.first[lo] ? c : c + n_in;
        ty = lo * a.strip_h + ((int)t - c * h);
    }
    return true;
}

// Entry formats: FP32 (16 B), FP16 and BF16 (8 B: {A,dU} {dV,dUV} as 16-bit pairs).
struct EF32 {
    using T = float4;
    static constexpr int kBytes = 16;
    static constexpr int kMinWaves = 4;  // 127 VGPRs; the LDS may allow only 3
    __device__ static float eval(const T& e, float fu, float fv) {
        return fmaf(fv, fmaf(fu, e.w, e.z), fmaf(fu, e.y, e.x));
    }
};
struct EF16 {
    using T = uint2;
    static constexpr int kBytes = 8;
    static constexpr int kMinWaves = 5;  // VALU-bound: 5 waves per SIMD (at most 96 VGPRs)
    __device__ static float lo(uint32_t e) { return __half2float(__ushort_as_half((unsigned short)(e & 0xffffu))); }
    __device__ static float hi(uint32_t e) { return __half2float(__ushort_as_half((unsigned short)(e >> 16))); }
    __device__ static float eval(const T& e, float fu, float fv) {
        return fmaf(fv, fmaf(fu, hi(e.y), lo(e.y)), fmaf(fu, hi(e.x), lo(e.x)));
    }
};
struct EBF16 {
    using T = uint2;
    static constexpr int kBytes = 8;
    static constexpr int kMinWaves = 5;
    __device__ static float lo(uint32_t e) { return __uint_as_float(e << 16); }
    __device__ static float hi(uint32_t e) { return __uint_as_float(e & 0xffff0000u); }
    __device__ static float eval(const T& e, float fu, float fv) {
        return fmaf(fv, fmaf(fu, hi(e.y), lo(e.y)), fmaf(fu, hi(e.x), lo(e.x)));
    }
};

// Global->LDS DMA through a buffer resource: B bytes (4 or 16) per lane from byte
// offset soff + voff of the resource into lds + lane*B.  The buffer form matters: an
// outstanding global_load_lds is modelled by the compiler as a flat access to memory
// and LDS, after which it waits for every outstanding LDS read (lgkmcnt(0)) at each LDS
// use and the read pipeline collapses; a buffer load to LDS is tracked by the memory
// counter only.  Offsets past the resource's size read zeros.  The builtins exist only
// in the device pass.
#if defined(__HIP_DEVICE_COMPILE__)
using dma_rsrc = __amdgpu_buffer_rsrc_t;
__device__ inline dma_rsrc make_dma_rsrc(const void* base, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, bytes, 0x00020000);
}
template <int B>
__device__ inline void lds_dma(dma_rsrc rs, unsigned voff, int soff, void* lds_wave_base) {
    auto* l = (__attribute__((address_space(3))) void*)lds_wave_base;
    if constexpr (B == 16) __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, l, 16, voff, soff, 0, 0);
    else __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, l, 4, voff, soff, 0, 0);
}
#else
struct dma_rsrc {};
__device__ inline dma_rsrc make_dma_rsrc(const void*, int) { return {}; }
template <int B>
__device__ inline void lds_dma(dma_rsrc, unsigned, int, void*) {}
#endif

__device__ inline int cvt_flr(float x) {
    int r;
    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(r) : "v"(x));
    return r;
}

// box: x = first entry column, y = first row, w = rows, z = ncols | flags.
// bits 28-29: 0 the block cannot hit the detector, 1 staged in LDS, 2 global reads;
// bit 27: the unmasked path may be used; bit 26: it may be used without any test, because
// the whole tile and run lie inside the detector window; bit 25: the box covers the whole run
// where the slab holds a part of it.
__device__ inline int box_kind(int4 b) { return ((unsigned)b.z >> 28) & 3; }
__device__ inline bool box_fast(int4 b) { return (b.z >> 27) & 1; }
__device__ inline bool box_inside(int4 b) { return (b.z >> 26) & 1; }
__device__ inline bool box_full(int4 b) { return (b.z >> 25) & 1; }
__device__ inline int box_nc(int4 b) { return b.z & 0x01ffffff; }
__device__ inline int box_nr(int4 b) { return b.w & 0xffff; }
__device__ inline int box_pitch(int4 b) { return (unsigned)b.w >> 16; }

// DMA: bytes per lane of the global->LDS staging (16, or 4 for 8-byte entries).  A
// compile-time width keeps the staging loop free of a run-time choice between the two
// DMA forms, which measured markedly slower for the 8-byte entries.
template <int ZPL, class E, int DMA>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(E::kMinWaves))) void bp_kernel(BpArgs a, const float4* __restrict__ pp,
                                                      const float* __restrict__ scales,
                                                      const void* __restrict__ proj_raw,
                                                      float* __restrict__ vol) {
    using T = typename E::T;
    const T* __restrict__ proj = reinterpret_cast<const T*>(proj_raw);
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int4 boxes[2][64];  // with params and zero_entry kStaticLds bytes
    // per projection: sin, cos, height, and the entry scale in w (written with the boxes)
    __shared__ float4 params[2][64];
    __shared__ float4 zero_entry;  // what columns that add nothing read

    int zbi, tx, ty;
    if (!tile_of(a, zbi, tx, ty)) return;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int xi = tx * kTX + (tid & (kTX - 1));
    const int yi = ty * kTY + (tid / kTX);
    // runs start at grid z indices that are multiples of ZPL (the slab begins zshift
    // voxels into the first run); run-local k is stored when zfirst <= k < zlast
    const int zb = zbi * ZPL;
    const int zfirst = a.zshift - zb;
    const int zlast = a.nzs + a.zshift - zb;
    const bool colvol = xi < a.nx && yi < a.ny;
    // lanes past the grid take its last column, so that every lane's ray stays inside the
    // tile's footprint; what they and lanes outside the cylinder add up is dropped at the end
    const float x = (float)min(xi, a.nx - 1) - a.xpre, y = (float)min(yi, a.ny - 1) - a.ypre;
    const bool incyl = colvol && (x * x + y * y < a.r2);

    const float cxa = (float)(tx * kTX) - a.xpre;
    const float cxb = (float)min(tx * kTX + kTX - 1, a.nx - 1) - a.xpre;
    const float cya = (float)(ty * kTY) - a.ypre;
    const float cyb = (float)min(ty * kTY + kTY - 1, a.ny - 1) - a.ypre;
    // the z-run always spans ZPL voxels (those outside the slab are computed, never
    // stored), so boxes and the fast-path test cover the full run.  Detector rows are
    // taken from the run's 32-slice anchor (det_row_index): k + koff slices past it.
    static_assert(ZPL == kRowAnchor || ZPL == kRowAnchor / 2, "a run lies inside one row anchor block");
    const int zrun = a.z0 - a.zshift + zb;
    const float zw0 = (float)zrun - a.zpre;
    // The slices a step has to cover: the whole run, unless the slab holds at most two thirds of it
    // and the run leaves the detector's rows: masked (by groups of four, 1.5 to 2.3 times the time
    // per slice) those slices alone are then cheaper.  72 slices in runs of 32 at 96^2 x 48
    // projections took 99 us with a whole last run of 8 slices, 88 so; 221^2 x 21 from 111
    // projections, inside the rows, 155 us whole and 232 masked.
    const int valid = min(zlast, ZPL) - max(zfirst, 0);
    const bool whole = valid * 3 > ZPL * 2;
    const int kfirst = whole ? 0 : max(zfirst, 0), klast = whole ? ZPL - 1 : min(zlast, ZPL) - 1;
    const float zwf = zw0 + (float)kfirst, zwl = zw0 + (float)klast;
    const int koff = ZPL == kRowAnchor ? 0 : (zrun & (kRowAnchor - 1));
    const float zwa = (float)(zrun - koff) - a.zpre;

    float acc[ZPL];
#pragma unroll
    for (int k = 0; k < ZPL; ++k) acc[k] = 0.0f;
    float* const col = vol + ((size_t)xi * a.ny + yi) * a.nzs;
    const bool whole_vec = a.vec4 && zfirst <= 0 && zlast >= ZPL;
    if (a.resume && colvol) {
        // the sums of the launch before
        if (whole_vec) {
            const float4* s4 = reinterpret_cast<const float4*>(col + zb);
#pragma unroll
            for (int k = 0; k < ZPL; k += 4) {
                const float4 v = s4[k >> 2];
                acc[k] = v.x; acc[k + 1] = v.y; acc[k + 2] = v.z; acc[k + 3] = v.w;
            }
        } else {
#pragma unroll
            for (int k = 0; k < ZPL; ++k)
                if (k >= zfirst && k < zlast) acc[k] = col[zb - a.zshift + k];
        }
    }

    // nearest point of the tile's xy rectangle to the axis
    const float ndx = cxa > 0.0f ? cxa : (cxb < 0.0f ? cxb : 0.0f);
    const float ndy = cya > 0.0f ? cya : (cyb < 0.0f ? cyb : 0.0f);
    const bool any_cyl = ndx * ndx + ndy * ndy < a.r2;

    if (any_cyl) {
        auto box_for = [&](int p) -> int4 {
            const float4 g = pp[p];
            float umin = INFINITY, umax = -INFINITY, vmin = INFINITY, vmax = -INFINITY;
            // changes of uIdx and vIdx along x (the lanes of a 16-lane row), summed over
            // the tile's two y edges and the run's two z ends
            float du = 0.0f, dv = 0.0f;
            float runlo = INFINITY, runhi = -INFINITY;  // rows of the whole run
            bool bad = false;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const float cx = (c & 1) ? cxb : cxa;
                const float cy = (c & 2) ? cyb : cya;
                float t = (-1.0f) * cx * g.x + cy * g.y;
                t += a.uoff;
                const float s = cx * g.y + cy * g.x;
                const float den = a.fcd - s;
                bad |= !(den > 0.0f);
                const float U = a.fcd / den;
                const float ui = t * U + a.upre;
                const float va = fmaf(-(zwf + g.z), U, a.vpre);
                const float vb = fmaf(-(zwl + g.z), U, a.vpre);
                umin = fminf(umin, ui); umax = fmaxf(umax, ui);
                vmin = fminf(vmin, fminf(va, vb)); vmax = fmaxf(vmax, fmaxf(va, vb));
                if (!whole) {
                    const float fa = fmaf(-(zw0 + g.z), U, a.vpre), fb = fmaf(-(zw0 + (float)(ZPL - 1) + g.z), U, a.vpre);
                    runlo = fminf(runlo, fminf(fa, fb)); runhi = fmaxf(runhi, fmaxf(fa, fb));
                }
                du += (c & 1) ? ui : -ui;
                dv += (c & 1) ? va + vb : -(va + vb);
            }
            int4 b = make_int4(0, 0, 2 << 28, 0);
            if (bad || !(umin == umin) || !(vmin == vmin)) return b;
            if (umax < -1.0f || umin > (float)a.W || vmax < -1.0f || vmin > (float)a.H) {
                b.z = 0;
                return b;
            }
            // A voxel reads the one entry at (floor(uIdx), floor(vIdx)).  uIdx and vIdx are
            // projective in the voxel's position, so over the tile and run they lie between
            // the corners' values; kBoxMargin covers the rounding of either expression.
            const int us0 = (int)floorf(umin - kBoxMargin);
            const int us = max(us0, 0);
            const int ue = min((int)floorf(umax + kBoxMargin), a.W - 1);
            const int nc = ue - us + 1;
            const int vmask = a.dma16 ? ~1 : ~0;
            // every slice of the run on the detector's rows: the unmasked path for all of them,
            // if their box fits the LDS
            auto rows_in = [&](float lo, float hi) {
                return lo - kBoxMargin >= fmaxf(a.vpre - a.vhi, 0.0f) && hi + kBoxMargin <= fminf(a.vpre - a.vlo, (float)(a.H - 1));
            };
            bool full = false;
            if (!whole && rows_in(runlo, runhi)) {
                const int n = (int)floorf(runhi + kBoxMargin) - ((int)floorf(runlo - kBoxMargin) & vmask) + 2;
                full = nc * (n + ((a.pitch_alt - n) & (a.pitch_mod - 1))) <= a.cap;
            }
            if (full) {
                vmin = runlo;
                vmax = runhi;
            }
            const int vs0 = (int)floorf(vmin - kBoxMargin);
            const int vs = max(vs0, 0) & vmask;
            const int ve = min((int)floorf(vmax + kBoxMargin), a.H - 1);
            const int nr = ve - vs + 1;
            if (nc <= 0 || nr <= 0) { b.z = 0; return b; }
            // LDS column pitch: the rows the DMA writes (an even count when 16-byte lanes
            // carry two 8-byte entries) rounded up to pitch_rem mod pitch_mod (a power of
            // two, so a mask: a division here would raise the kernel's register peak), so
            // that neighbouring detector columns start in different LDS bank groups
            const int wr = (DMA == 16 && E::kBytes == 8) ? (nr + 1) & ~1 : nr;
            // A 16-lane row of voxels reads entries whose column and row both drift along
            // x.  With the pitch at +1 mod 16 a lane's bank group is column + row, and two
            // lanes whose column step is undone by a row step share one; where the column
            // and row drift in opposite directions the pitch -1 mod 16 (row - column)
            // avoids that.  Taken only where the box still fits the buffer.
            const bool minus = a.pitch_adapt && du * dv < 0.0f;
            auto pitch_of = [&](int rem) {
                const int p = wr + ((rem - wr) & (a.pitch_mod - 1));
                const int m = wr + ((a.pitch_mod - rem - wr) & (a.pitch_mod - 1));
                return minus && nc * m <= a.cap ? m : p;
            };
            int pitch = pitch_of(a.pitch_rem);
            if (nc * pitch > a.cap) pitch = pitch_of(a.pitch_alt);
            b.x = us; b.y = vs; b.w = nr | (pitch << 16);
            // the fused vIndex of the fast path may round a hair below 0 at the top edge
            const int fast = vs0 >= 0 ? 1 : 0;
            // no voxel of the tile and run can fail a window test (by more than either
            // expression's rounding), and no entry is clipped away
            const bool in = (whole || full) && fast && us0 >= 0 && umin - kBoxMargin >= a.ulo + a.upre &&
                            umax + kBoxMargin <= fminf(a.uhi + a.upre, (float)(a.W - 1)) && rows_in(vmin, vmax);
            b.z = nc | ((full ? 1 : 0) << 25) | ((in ? 1 : 0) << 26) | (fast << 27) | ((nc * pitch <= a.cap ? 1 : 2) << 28);
            return b;
        };

        // Stage the box of projection p into LDS buffer `buf`: wave w copies detector
        // columns w, w+4, ...; a column's entries are contiguous in global memory and in
        // LDS.  All addresses are wave-uniform (SGPR arithmetic); each lane moves DMA bytes.
        const int wave_u = __builtin_amdgcn_readfirstlane(wave);
        auto stage = [&](unsigned char* dst, int p, int4 bx) {
            const int us = bx.x, vs = bx.y, nr = box_nr(bx), nc = box_nc(bx), pitch = box_pitch(bx);
            static_assert(DMA == 16 || (DMA == 4 && E::kBytes == 8), "16-byte entries stage 16 bytes per lane");
            constexpr bool wide = DMA == 16;
            constexpr int ub = DMA;  // bytes per lane per DMA
            const int units = wide ? (nr * E::kBytes + 15) / 16 : nr * (E::kBytes / 4);
            // one resource per projection image (its size is below 2^31 bytes, checked by
            // launch_backproject before the launch); the column offsets are wave-uniform
            const int img_bytes = a.W * a.H * E::kBytes;
            const dma_rsrc rs = make_dma_rsrc(reinterpret_cast<const char*>(proj) + (size_t)p * img_bytes, img_bytes);
            const int col0 = (us * a.H + vs) * E::kBytes;
            const unsigned lane_off = (unsigned)lane * ub;
            const int gstep = kWaves * a.H * E::kBytes, lstep = kWaves * pitch * E::kBytes;
            // A DMA instruction costs about the same whatever its lane mask, and the loop
            // around it is scalar work: every column takes `full` unmasked instructions,
            // then the columns' partial tails share one lane mask, set once per box.
            const int full = units >> 6, tail = units & 63;
            for (int j = 0; j < full; ++j) {
                int gcol = col0 + wave_u * a.H * E::kBytes + j * 64 * ub;
                unsigned char* lcol = dst + (size_t)wave_u * pitch * E::kBytes + (size_t)j * 64 * ub;
                for (int c = wave_u; c < nc; c += kWaves, gcol += gstep, lcol += lstep) lds_dma<ub>(rs, lane_off, gcol, lcol);
            }
            if (tail > 0 && lane < tail) {
                int gcol = col0 + wave_u * a.H * E::kBytes + full * 64 * ub;
                unsigned char* lcol = dst + (size_t)wave_u * pitch * E::kBytes + (size_t)full * 64 * ub;
                for (int c = wave_u; c < nc; c += kWaves, gcol += gstep, lcol += lstep) lds_dma<ub>(rs, lane_off, gcol, lcol);
            }
        };

        auto compute = [&](const T* tile, int p, int4 bx, float4 g, float sc) {
            const int kind = box_kind(bx);
            if (kind == 0) return;
            float t = (-1.0f) * x * g.x + y * g.y;
            t += a.uoff;
            const float s = x * g.y + y * g.x;
            const float U = cone_magnification(a.fcd, s);
            const float u = t * U;
            const float uIdx = u + a.upre;
            const int u0 = (int)uIdx;
            const float fu = uIdx - (float)u0;
            const float w = U * U * sc;
            const float vA = det_row_anchor(zwa, g.z, U, a.vpre);
            const int us = bx.x, vs = bx.y, pitch = box_pitch(bx);
            const bool cv = incyl && u >= a.ulo && u <= a.uhi;
            float Ue = U, we = w, fue = fu, vAe = vA;
            const char* tile_b = reinterpret_cast<const char*>(tile) - (us * pitch + vs) * E::kBytes;
            const char* col = tile_b + __mul24(u0, pitch * E::kBytes);
            // a column that adds nothing reads an entry of zeros for every slice, with zero weight
            // (not an entry of the box, which may be infinite or NaN, and so its product with 0)
            auto idle = [&]() {
                Ue = we = fue = 0.0f;
                vAe = (float)vs;
                col = reinterpret_cast<const char*>(&zero_entry) - vs * E::kBytes;
            };
            // how the step runs: 1 unmasked from LDS, 2 masked by groups of slices from LDS,
            // 3 voxel by voxel from global memory
            int mode = kind == 1 ? 1 : 3;
            if (kind == 1 && !box_inside(bx)) {
                const bool lane_full = !cv || ((zw0 + g.z) * U >= a.vlo && (zwl + g.z) * U <= a.vhi);
                if (!((whole || box_full(bx)) && box_fast(bx) && __all(lane_full))) mode = 2;
                else if (!cv) idle();
            }
            // The three forms follow one another, each under its own opaque condition: as
            // alternatives of one branch the compiler keeps the accumulators of each in
            // registers of its own and copies them together on every step.
            if (opaque_uniform(mode) == 1) {
                const T* tb = reinterpret_cast<const T*>(col);
                // software pipeline in groups of kGrp: the LDS reads of group g+1 are
                // issued before the arithmetic of group g, and scheduling barriers
                // keep the compiler from trading those in-flight reads for hoisted
                // row-index arithmetic
                T e[2][kGrp];
                float fv[2][kGrp];
                auto fetch = [&](int g0, int slot) {
#pragma unroll
                    for (int j = 0; j < kGrp; ++j) {
                        const float vI = det_row_index((float)(g0 + j + koff), Ue, vAe);
                        e[slot][j] = tb[cvt_flr(vI)];
                        fv[slot][j] = __builtin_amdgcn_fractf(vI);
                    }
                };
                fetch(0, 0);
#pragma unroll
                for (int g0 = 0; g0 < ZPL; g0 += kGrp) {
                    const int slot = (g0 / kGrp) & 1;
                    if (g0 + kGrp < ZPL) fetch(g0 + kGrp, slot ^ 1);
#pragma unroll
                    for (int j = 0; j < kGrp; ++j)
                        fmac(acc[g0 + j], we, E::eval(e[slot][j], fue, fv[slot][j]));
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            if (opaque_uniform(mode) == 2) {
                // Some column leaves the window within the run.  v = (z + h) U is
                // non-decreasing in z (U > 0, monotone rounding), so the slices that pass the
                // window test form an interval [lo, hi]: estimated by division, then settled
                // with the test's own expression.
                auto v_of = [&](int k) { return ((zw0 + (float)k) + g.z) * U; };
                const float iU = __builtin_amdgcn_rcpf(U), zo = zw0 + g.z;
                int lo = (int)ceilf(fminf(fmaxf(a.vlo * iU - zo, -4.0f), (float)(ZPL + 4)));
                int hi = (int)floorf(fminf(fmaxf(a.vhi * iU - zo, -4.0f), (float)(ZPL + 4)));
#pragma unroll
                for (int it = 0; it < 2; ++it) {
                    if (v_of(lo - 1) >= a.vlo) --lo;
                    if (v_of(hi + 1) <= a.vhi) ++hi;
                }
#pragma unroll
                for (int it = 0; it < 2; ++it) {
                    if (!(v_of(lo) >= a.vlo)) ++lo;
                    if (!(v_of(hi) <= a.vhi)) --hi;
                }
                lo = max(lo, kfirst);
                hi = min(hi, klast);
                const bool act = cv && lo <= hi && v_of(lo) >= a.vlo && v_of(hi) <= a.vhi;
                if (!act) idle();
                const T* tb = reinterpret_cast<const T*>(col);
                const int ve = vs + box_nr(bx) - 1;
                // groups of four slices: skipped where no column is in the window, unmasked
                // where every column is (by one slice at the upper end, where the fused row
                // index may round a hair below row 0), else each voxel masked and its row
                // clamped into the box
#pragma unroll
                for (int g0 = 0; g0 < ZPL; g0 += 4) {
                    int form = 0;
                    if (__any(act && lo <= g0 + 3 && hi >= g0)) form = __all(!act || (lo <= g0 && hi > g0 + 3)) ? 1 : 2;
                    if (opaque_uniform(form) == 1) {
                        T e[4];
                        float fv[4];
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            const float vI = det_row_index((float)(g0 + j + koff), Ue, vAe);
                            e[j] = tb[cvt_flr(vI)];
                            fv[j] = __builtin_amdgcn_fractf(vI);
                        }
#pragma unroll
                        for (int j = 0; j < 4; ++j) fmac(acc[g0 + j], we, E::eval(e[j], fue, fv[j]));
                    }
                    if (opaque_uniform(form) == 2) {
                        T e[4];
                        float fv[4];
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            const float vI = det_row_index((float)(g0 + j + koff), Ue, vAe);
                            const int v0 = (int)vI;
                            e[j] = tb[min(max(v0, vs), ve)];
                            fv[j] = vI - (float)v0;
                        }
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            const float q = E::eval(e[j], fue, fv[j]);
                            fmac(acc[g0 + j], we, lo <= g0 + j && hi >= g0 + j ? q : 0.0f);
                        }
                    }
                }
            }
            if (opaque_uniform(mode) == 3) {
                const T* src = proj + ((size_t)p * a.W + u0) * a.H;
#pragma unroll
                for (int k = 0; k < ZPL; ++k) {
                    const float zk = zw0 + (float)k;
                    const float v = (zk + g.z) * U;
                    if (cv && v >= a.vlo && v <= a.vhi) {
                        const float vI = det_row_index((float)(k + koff), U, vA);
                        const int v0 = (int)vI;
                        const T e = src[v0];
                        fmac(acc[k], w, E::eval(e, fu, vI - (float)v0));
                    }
                }
            }
        };

        // Buffer p&1 holds projection p while it is computed.  The box of p+1 is always
        // produced at least one barrier before it is staged (batches are computed one
        // batch ahead by wave 0).
        // wave 0 fills one batch of 64 projections: footprint boxes and parameters
        auto fill_batch = [&](int slot, int pn) {
            boxes[slot][tid] = pn < a.nproj ? box_for(pn) : make_int4(0, 0, 0, 0);
            float4 g = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (pn < a.nproj) {
                g = pp[pn];
                g.w = scales ? scales[pn] : 1.0f;
            }
            params[slot][tid] = g;
        };
        if (tid < 64) fill_batch(0, tid);
        if (tid == 0) zero_entry = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        __syncthreads();
        auto buffer = [&](int p) { return smem + (size_t)(p & 1) * a.cap * E::kBytes; };
        if (a.nproj > 0) {
            const int4 b0 = boxes[0][0];
            if (box_kind(b0) == 1) stage(buffer(0), 0, b0);
        }
        // One projection step: stage projection p+1 into `nxt` (LDS DMA) and accumulate
        // projection p from `cur`.  The buffers are disjoint; declaring them __restrict__
        // lets the compiler issue the LDS reads of p while the DMA of p+1 is in flight
        // (otherwise it waits for all outstanding DMA before the first read).
        auto step = [&](const T* __restrict__ cur, unsigned char* __restrict__ nxt, int p, int4 bx, int4 bn,
                        float4 g, float sc) {
            if (box_kind(bn) == 1) stage(nxt, p + 1, bn);
            __builtin_amdgcn_sched_barrier(0);  // the DMA is issued before the compute
            compute(cur, p, bx, g, sc);
        };
        auto uniform_box = [](int4 b) {
            return make_int4(__builtin_amdgcn_readfirstlane(b.x), __builtin_amdgcn_readfirstlane(b.y),
                             __builtin_amdgcn_readfirstlane(b.z), __builtin_amdgcn_readfirstlane(b.w));
        };
        auto uniform_f = [](float v) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v))); };
        auto uniform_f4 = [&](float4 v) {
            return make_float4(uniform_f(v.x), uniform_f(v.y), uniform_f(v.z), uniform_f(v.w));
        };
        // The box and parameters of projection p+1 are read from LDS during step p, so a
        // step starts without waiting for memory other than its own staging DMA.
        int4 bx = uniform_box(boxes[0][0]);
        float4 g = uniform_f4(params[0][0]);
        for (int p = 0; p < a.nproj; ++p) {
            // this wave's DMA for projection p has landed; the barrier publishes every
            // wave's and guarantees that nobody still reads buffer (p+1)&1 or the box
            // batch about to be overwritten
            __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
            __syncthreads();
            if ((p & 63) == 0 && tid < 64) fill_batch(((p >> 6) + 1) & 1, p + 64 + tid);
            const int q = p + 1;
            // (past the last projection the batch holds empty boxes)
            const int4 bl = boxes[(q >> 6) & 1][q & 63];
            const float4 gl = params[(q >> 6) & 1][q & 63];
            const int4 bn = uniform_box(bl);
            const float4 gn = uniform_f4(gl);
            step(reinterpret_cast<const T*>(buffer(p)), buffer(p + 1), p, bx, bn, g, g.w);
            bx = bn;
            g = gn;
        }
    }

    if (!incyl) {
#pragma unroll
        for (int k = 0; k < ZPL; ++k) acc[k] = 0.0f;
    }
    if (colvol) {
        if (whole_vec) {
            float4* d4 = reinterpret_cast<float4*>(col + zb);
#pragma unroll
            for (int k = 0; k < ZPL; k += 4) {
                float4 v = make_float4(acc[k], acc[k + 1], acc[k + 2], acc[k + 3]);
                if (a.accumulate) {
                    const float4 o = d4[k >> 2];
                    v.x += o.x; v.y += o.y; v.z += o.z; v.w += o.w;
                }
                d4[k >> 2] = v;
            }
        } else {
#pragma unroll
            for (int k = 0; k < ZPL; ++k) {
                if (k >= zfirst && k < zlast) {
                    float* d = col + (zb - a.zshift + k);
                    *d = a.accumulate ? *d + acc[k] : acc[k];
                }
            }
        }
    }
}

// FP64 backprojection from row-major double images (the GPU error yardstick).
// One thread per voxel column and run of 16 z; the same masks as the FP32 path,
// evaluated in double.
__global__ __launch_bounds__(256) void bp_f64_kernel(BpArgs a, const double4* __restrict__ pp,
                                                     const double* __restrict__ rows,
                                                     double* __restrict__ vol) {
    constexpr int ZR = 16;
    const int xi = blockIdx.x * 16 + (threadIdx.x & 15);
    const int yi = blockIdx.y * 16 + (threadIdx.x >> 4);
    const int zb = blockIdx.z * ZR;
    if (xi >= a.nx || yi >= a.ny) return;
    const int zc = min(ZR, a.nzs - zb);
    double acc[ZR];
#pragma unroll
    for (int k = 0; k < ZR; ++k) acc[k] = 0.0;
    const double x = (double)xi - a.xpre, y = (double)yi - a.ypre;
    const double r2 = (double)a.r2;
    if (x * x + y * y < r2) {
        for (int p = 0; p < a.nproj; ++p) {
            const double4 g = pp[p];
            const double sn = g.x, cs = g.y, h = g.z;
            const double t = -x * sn + y * cs + (double)a.uoff;
            const double s = x * cs + y * sn;
            const double U = (double)a.fcd / ((double)a.fcd - s);
            const double u = t * U;
            if (u < (double)a.ulo || u > (double)a.uhi) continue;
            const double w = U * U;
            const double uI = u + (double)a.upre;
            const int u0 = (int)uI;
            const double fu = uI - u0;
            const double* img = rows + (size_t)p * a.W * a.H;
#pragma unroll
            for (int k = 0; k < ZR; ++k) {
                if (k >= zc) break;
                const double v = ((double)(a.z0 + zb + k) - (double)a.zpre + h) * U;
                if (v < (double)a.vlo || v > (double)a.vhi) continue;
                const double vI = -v + (double)a.vpre;
                const int v0 = (int)vI;
                const double fv = vI - v0;
                const double* r0 = img + (size_t)v0 * a.W;
                const double* r1 = r0 + a.W;
                const double ta = (1.0 - fu) * r0[u0] + fu * r0[u0 + 1];
                const double tb = (1.0 - fu) * r1[u0] + fu * r1[u0 + 1];
                acc[k] += w * ((1.0 - fv) * ta + fv * tb);
            }
        }
    }
    double* dst = vol + ((size_t)xi * a.ny + yi) * a.nzs + zb;
    for (int k = 0; k < zc; ++k) dst[k] = acc[k];
}

BpArgs make_args(const ctg_geometry& g, int nproj, int z0, int nz, int accumulate) {
    BpArgs a{};
    a.W = g.det_width;
    a.H = g.det_height;
    a.nx = g.nx;
    a.ny = g.ny;
    a.nzs = nz;
    a.z0 = z0;
    a.xpre = g.x_pre;
    a.ypre = g.y_pre;
    a.zpre = g.z_pre;
    a.upre = g.u_pre;
    a.vpre = g.v_pre;
    a.r2 = g.radius * g.radius;
    a.fcd = g.fcd;
    a.uoff = g.u_offset;
    a.ulo = g.u_lo;
    a.uhi = g.u_hi;
    a.vlo = g.v_lo;
    a.vhi = g.v_hi;
    a.nproj = nproj;
    a.accumulate = accumulate;
    return a;
}

bool tile_in_cylinder(const ctg_geometry& g, int tx, int ty) {
    const float cxa = (float)(tx * kTX) - g.x_pre, cxb = (float)std::min(tx * kTX + kTX - 1, g.nx - 1) - g.x_pre;
    const float cya = (float)(ty * kTY) - g.y_pre, cyb = (float)std::min(ty * kTY + kTY - 1, g.ny - 1) - g.y_pre;
    const float ndx = cxa > 0.0f ? cxa : (cxb < 0.0f ? cxb : 0.0f);
    const float ndy = cya > 0.0f ? cya : (cyb < 0.0f ? cyb : 0.0f);
    return ndx * ndx + ndy * ndy < g.radius * g.radius;
}

// Largest footprint box (entries) over a sample of tiles and projections, with the
// same construction as box_for on the device.  Boxes that exceed the resulting
// capacity at run time take the global-memory path, so sampling only affects speed.
// x: with the column pitch at prem mod pmod, y: at palt.
int2 sample_max_box(const ctg_geometry& g, const float4* hp, int nproj, int z0, int nz, int zpl, int dma16,
                    int pmod, int prem, int palt) {
    const int ntx = (g.nx + kTX - 1) / kTX, nty = (g.ny + kTY - 1) / kTY, nzb = (nz + zpl - 1) / zpl;
    // about 16 projections: boxes change slowly with the angle, and the capacity keeps a
    // margin above the largest sampled box
    const int pstep = std::max(1, nproj / 16);
    int2 best = make_int2(0, 0);
    const int zblocks[3] = {0, nzb / 2, nzb - 1};
    for (int zi = 0; zi < 3; ++zi) {
        const int zb = zblocks[zi] * zpl;
        const float zw0 = (float)(z0 + zb) - g.z_pre, zw1 = zw0 + (float)(zpl - 1);
        for (int ty = 0; ty < nty; ++ty) {
            for (int tx = 0; tx < ntx; ++tx) {
                const float cxa = (float)(tx * kTX) - g.x_pre;
                const float cxb = (float)std::min(tx * kTX + kTX - 1, g.nx - 1) - g.x_pre;
                const float cya = (float)(ty * kTY) - g.y_pre;
                const float cyb = (float)std::min(ty * kTY + kTY - 1, g.ny - 1) - g.y_pre;
                if (!tile_in_cylinder(g, tx, ty)) continue;
                for (int p = 0; p < nproj; p += pstep) {
                    const float4 q = hp[p];
                    float umin = INFINITY, umax = -INFINITY, vmin = INFINITY, vmax = -INFINITY;
                    bool bad = false;
                    for (int c = 0; c < 4; ++c) {
                        const float cx = (c & 1) ? cxb : cxa, cy = (c & 2) ? cyb : cya;
                        float t = (-1.0f) * cx * q.x + cy * q.y;
                        t += g.u_offset;
                        const float s = cx * q.y + cy * q.x;
                        const float den = g.fcd - s;
                        if (!(den > 0.0f)) bad = true;
                        const float U = g.fcd / den;
                        const float ui = t * U + g.u_pre;
                        const float va = std::fma(-(zw0 + q.z), U, g.v_pre);
                        const float vb = std::fma(-(zw1 + q.z), U, g.v_pre);
                        umin = std::min(umin, ui); umax = std::max(umax, ui);
                        vmin = std::min(vmin, std::min(va, vb)); vmax = std::max(vmax, std::max(va, vb));
                    }
                    if (bad) continue;
                    const int us = std::max((int)std::floor(umin - kBoxMargin), 0);
                    const int ue = std::min((int)std::floor(umax + kBoxMargin), g.det_width - 1);
                    const int vs = std::max((int)std::floor(vmin - kBoxMargin), 0) & (dma16 ? ~1 : ~0);
                    const int ve = std::min((int)std::floor(vmax + kBoxMargin), g.det_height - 1);
                    if (ue >= us && ve >= vs) {
                        const int nr = ve - vs + 1;
                        const int wr = dma16 ? (nr + 1) & ~1 : nr;
                        best.x = std::max(best.x, (ue - us + 1) * (wr + ((prem - wr) & (pmod - 1))));
                        best.y = std::max(best.y, (ue - us + 1) * (wr + ((palt - wr) & (pmod - 1))));
                    }
                }
            }
        }
    }
    return best;
}

// sample_max_box behind a small per-thread cache: callers that backproject the same
// projections into the same slab again (iterative methods, slab by slab) pay the host
// sampling once.  The key hashes the geometry, the projection parameters and the slab;
// a collision can only mis-size the LDS tile, which costs speed, not correctness
// (boxes beyond the capacity read global memory).
int2 cached_max_box(const ctg_geometry& g, const float4* hp, int nproj, int z0, int nz, int zpl, int dma16, int pmod,
                    int prem, int palt) {
    uint64_t h = 1469598103934665603ull;
    auto mix = [&](const void* p, size_t n) {
        const unsigned char* b = static_cast<const unsigned char*>(p);
        for (size_t i = 0; i < n; ++i) h = (h ^ b[i]) * 1099511628211ull;
    };
    const int keys[8] = {nproj, z0, nz, zpl, dma16, pmod, prem, palt};
    mix(&g, sizeof(g));
    mix(keys, sizeof(keys));
    mix(hp, sizeof(float4) * (size_t)nproj);
    struct Entry { uint64_t key; int2 cap; bool used; };
    static thread_local Entry cache[16] = {};
    static thread_local int next = 0;
    for (const Entry& e : cache)
        if (e.used && e.key == h) return e.cap;
    const int2 cap = sample_max_box(g, hp, nproj, z0, nz, zpl, dma16, pmod, prem, palt);
    cache[next] = {h, cap, true};
    next = (next + 1) % 16;
    return cap;
}

// Strips of the tile numbering (tile_of).
void number_tiles(const ctg_geometry& g, BpArgs& a) {
    // blocks of 4 x 4 tiles; CTG_BP_BLOCK=n sets their edge, 0 takes single rows (tuning)
    int edge = 4;
    if (const char* e = std::getenv("CTG_BP_BLOCK")) edge = std::max(0, std::min(64, std::atoi(e)));
    a.strip_h = std::max(edge, 1);
    a.blk = edge > 0 ? edge : a.ntx;
    while ((a.nty + a.strip_h - 1) / a.strip_h > kMaxStrips) a.strip_h *= 2;
    a.nstrips = (a.nty + a.strip_h - 1) / a.strip_h;
    a.before[0] = 0;
    for (int s = 0; s < a.nstrips; ++s) {
        const int y0 = s * a.strip_h, h = std::min(a.strip_h, a.nty - y0);
        int lo = a.ntx, hi = -1;
        for (int ty = y0; ty < y0 + h; ++ty)
            for (int tx = 0; tx < a.ntx; ++tx)
                if (tile_in_cylinder(g, tx, ty)) {
                    lo = std::min(lo, tx);
                    hi = std::max(hi, tx);
                }
        if (hi < lo) lo = 0;
        a.first[s] = lo;
        a.before[s + 1] = a.before[s] + (unsigned)((hi - lo + 1) * h);
    }
    a.nwork = a.before[a.nstrips];
    a.nidle = (unsigned)(a.ntx * a.nty) - a.nwork;
}

// Its chunks: eight per layer, but of at least 16 tiles where a layer holds at most 20, so that
// neighbours still share an L2 (FP32 and FP16, chunks of at least 1 and 16 tiles: 48^2 x 2000 from
// 40 projections, 9 tiles per layer, 359 and 321, 301 and 278 us; 32^2 x 1000 from 100, 4 tiles,
// 491 and 424, 420 and 362; 160^3 from 200, 100 tiles, no difference).
void number_chunks(BpArgs& a) {
    const unsigned total = a.nwork * (unsigned)a.nzb, least = a.nwork <= 20 ? 16 : 1;
    const unsigned rounds = std::max(1u, std::min((unsigned)a.nzb, total / (8u * least)));
    a.chunk = total / (8u * rounds);
    a.extra = total - a.chunk * 8u * rounds;
    a.long_rounds = (a.extra + 7u) / 8u;
    a.work_wgs = rounds * a.chunk + a.long_rounds;
}

// Launches of `step` projections that go on from each other's sums.  One set of tiles and buffers
// serves all of them: boxes are sampled over the whole scan, once (sampled launch by launch, a
// scan of more launches than cached_max_box keeps took its samples anew on every call).
template <int ZPL>
ctg_status launch_zpl(const BpLaunch& L, BpArgs a, int step, hipStream_t st) {
    const ctg_geometry& g = *L.g;
    const int ebytes = L.store == CTG_STORE_F32 ? 16 : 8;
    a.zshift = L.z0 & (ZPL - 1);
    // whole runs store 16-byte vectors when the slab starts on a run boundary
    a.vec4 = (a.zshift == 0 && L.nz % 4 == 0 && ((uintptr_t)L.d_volume % 16) == 0) ? 1 : 0;
    a.nzb = (L.nz + a.zshift + ZPL - 1) / ZPL;
    // 8-byte entries are staged 16 bytes (two rows) per lane when the detector height is
    // even, so that the first row of every box can be even and each lane's 16 bytes are
    // aligned in global memory: one DMA instruction per column of up to 128 rows instead
    // of two beyond 32.  A DMA instruction costs about the same whatever it moves, and the
    // LDS side needs only 8-byte alignment, so the odd pitch stays.  CTG_BP_DMA16=0
    // selects 4 bytes per lane (tuning).
    const char* dma_env = std::getenv("CTG_BP_DMA16");
    a.dma16 = (ebytes == 8 && g.det_height % 2 == 0 && !(dma_env && std::atoi(dma_env) == 0)) ? 1 : 0;
    // column pitch: rows rounded up to 1 mod 16.  CTG_BP_PITCH="mod,rem" overrides (tuning).
    a.pitch_mod = 16;
    a.pitch_rem = 1;
    // per-box choice of +1 or -1 mod 16 for 16-byte entries (FP32 179.4 -> 174.8 ms at
    // 1024^3 x 720; no change for 8-byte entries, which keep +1).  CTG_BP_PITCH_ADAPT=0/1
    // overrides (tuning).
    a.pitch_adapt = ebytes == 16 ? 1 : 0;
    if (const char* env = std::getenv("CTG_BP_PITCH_ADAPT")) a.pitch_adapt = std::atoi(env) != 0;
    if (const char* env = std::getenv("CTG_BP_PITCH")) {
        int m = 0, r = 0;
        if (std::sscanf(env, "%d,%d", &m, &r) == 2 && m >= 1 && (m & (m - 1)) == 0 && r >= 0) {
            a.pitch_mod = m;
            a.pitch_rem = r % m;
        }
    }
    // Boxes that do not fit with the pitch at 1 mod 16 (1.11 passes per LDS read on average) may
    // take 11 mod 16 (1.21 passes, up to 6 rows less on a column); the buffers are sized for that
    // where it lets more workgroups into a CU's 160 KB.  512^3 x 360 in batches of 64, FP32: 3
    // workgroups and 11.3 ms with 1, 4 and 10.0 with 11; 1024^3 x 720, where both leave 3: 164.3
    // and 166.7 ms.
    a.pitch_alt = a.pitch_mod == 16 && a.pitch_rem == 1 ? 11 : a.pitch_rem;
    const int2 most = L.h_params ? cached_max_box(g, L.h_params, L.nproj, L.z0 - a.zshift, L.nz + a.zshift, ZPL,
                                                  a.dma16, a.pitch_mod, a.pitch_rem, a.pitch_alt)
                                 : make_int2(0, 0);
    // keeps the second buffer and every column start 16-byte aligned
    auto capacity = [&](int n) { return std::min(n + n / 32 + 16, kMaxTileBytes / ebytes) & ~7; };
    auto per_cu = [&](int n) { return std::min((160 * 1024) / (2 * capacity(n) * ebytes + kStaticLds), ebytes == 16 ? EF32::kMinWaves : EF16::kMinWaves); };
    const bool tight = per_cu(most.y) > per_cu(most.x);
    if (!tight) a.pitch_alt = a.pitch_rem;
    const int cap = capacity(tight ? most.y : most.x);
    a.cap = cap;
    const size_t lds = (size_t)2 * cap * ebytes;
    if ((long long)a.ntx * a.nty * a.nzb > 0x7fffffffll) return fail(CTG_ERROR_UNSUPPORTED, "backprojection grid too large");
    number_chunks(a);
    const long long grid = 8ll * ((long long)a.work_wgs + ((long long)a.nidle * a.nzb + 7) / 8);
    if (grid > 0x7fffffffll) return fail(CTG_ERROR_UNSUPPORTED, "backprojection grid too large");
    const size_t img_bytes = (size_t)g.det_width * g.det_height * ebytes;
    for (int p = 0; p < std::max(L.nproj, 1); p += step) {
        a.nproj = std::min(step, L.nproj - p);
        a.resume = p > 0;
        const float* scales = L.d_scales ? L.d_scales + p : nullptr;
        const void* filtered = (const char*)L.d_filtered + p * img_bytes;
#define CTG_BP_LAUNCH(E, DMA)                                                                                  \
    hipLaunchKernelGGL((bp_kernel<ZPL, E, DMA>), dim3((unsigned)grid), dim3(kThreads), lds, st, a, L.d_params + p, \
                       scales, filtered, L.d_volume)
        switch (L.store) {
            case CTG_STORE_F32:
                CTG_BP_LAUNCH(EF32, 16);
                break;
            case CTG_STORE_F16:
                if (a.dma16) CTG_BP_LAUNCH(EF16, 16);
                else CTG_BP_LAUNCH(EF16, 4);
                break;
            case CTG_STORE_BF16:
                if (a.dma16) CTG_BP_LAUNCH(EBF16, 16);
                else CTG_BP_LAUNCH(EBF16, 4);
                break;
            default:
                return fail(CTG_ERROR_INVALID_ARGUMENT, "unknown store type %d", (int)L.store);
        }
#undef CTG_BP_LAUNCH
        CTG_HIP(hipGetLastError());
    }
    return CTG_OK;
}

}  // namespace bp_detail

using namespace bp_detail;

ctg_status launch_backproject(const BpLaunch& L, hipStream_t st) {
    const ctg_geometry& g = *L.g;
    if (L.nz <= 0 || g.nx <= 0 || g.ny <= 0) return CTG_OK;
    if (((uintptr_t)L.d_filtered % 16) != 0)
        return fail(CTG_ERROR_INVALID_ARGUMENT, "filtered projections must be 16-byte aligned");
    // The staging DMA addresses one projection through a buffer resource whose size and
    // column offsets are 32-bit: a projection's entries must stay below 2^31 bytes.
    const long long img_bytes = (long long)g.det_width * g.det_height * (L.store == CTG_STORE_F32 ? 16 : 8);
    if (img_bytes > 0x7fffffffll)
        return fail(CTG_ERROR_UNSUPPORTED,
                    "detector %dx%d: %lld bytes of backprojection entries per projection exceed the 2^31-byte limit",
                    g.det_width, g.det_height, img_bytes);
    BpArgs a = make_args(g, L.nproj, L.z0, L.nz, L.accumulate);
    a.ntx = (g.nx + kTX - 1) / kTX;
    a.nty = (g.ny + kTY - 1) / kTY;
    number_tiles(g, a);
    // Slices per lane: 32, but 16 where the working tiles are then still at most one per CU (256
    // of them): every tile runs alone on its CU, so shorter ones end sooner (96^2 x 72 from 48
    // projections: 88 us with 32, 75 with 16).  From there on both take the same (128^3: 95 and
    // 86, 160^3: 89 and 89, 200^3: 187 and 185 us), and on a full chip 16 takes 15 % longer.
    // CTG_BP_ZPL=16 or 32 overrides (tuning).
    const char* env = std::getenv("CTG_BP_ZPL");
    const long long short_runs = (long long)a.nwork * ((L.nz + (L.z0 & 15) + 15) / 16);
    const int zpl = env ? (std::atoi(env) == 16 ? 16 : 32) : (short_runs <= 256 ? 16 : 32);
    // The tiles that run at one time are spread over all projections of the launch, so a large
    // scan's entries pass through the Infinity Cache without being met again.  Launches of about
    // 240 projections that go on from each other's sums (the same additions in the same order)
    // keep to fewer images at a time: 1024^3 x 720 162.0 -> 160.1 ms (FP16 131.2 -> 129.1), 768^3
    // x 720 72.8 -> 71.4, 512^3 x 1440 44.2 -> 42.6, though each writes and reads the volume;
    // 512^3 x 720 does not change.  At least 8192 tiles, so that a launch's last ones are few, and
    // not where the sums are to be added to the volume.
    const bool large = (long long)a.nwork * ((L.nz + (L.z0 & 31) + 31) / 32) >= 8192;
    const int parts = large && !L.accumulate ? std::max(1, L.nproj / 240) : 1;
    const int step = std::max(1, (L.nproj + parts - 1) / parts);
    return zpl == 16 ? launch_zpl<16>(L, a, step, st) : launch_zpl<32>(L, a, step, st);
}

ctg_status launch_backproject_f64(const ctg_geometry& g, const double4* d_params, const double* d_rows,
                                  int nproj, double* d_volume, int z0, int nz, hipStream_t st) {
    if (nz <= 0) return CTG_OK;
    BpArgs a = make_args(g, nproj, z0, nz, 0);
    dim3 grid((unsigned)((g.nx + 15) / 16), (unsigned)((g.ny + 15) / 16), (unsigned)((nz + 15) / 16));
    hipLaunchKernelGGL(bp_f64_kernel, grid, dim3(256), 0, st, a, d_params, d_rows, d_volume);
    CTG_HIP(hipGetLastError());
    return CTG_OK;
}

}  // namespace ctg
