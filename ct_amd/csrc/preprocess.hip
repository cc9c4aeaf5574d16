// Projection preprocessing on gfx950: intensity -> line integral, Feldkamp weight,
// ramp-family row filter, and conversion into the backprojection layout.
//
// Reference behaviour restated (not translated):
//  - log forms: Ct/CtVolume.cpp:802-812 + 860-866 (CPU) and :892-904 (GPU);
//  - Feldkamp weight D/sqrt(D^2+u^2+v^2): Ct/CtVolume.cpp:814-830, Ct/cuda_ct.cu:102-131;
//  - row filter: real DFT of length W without padding, bins 0..W/2 scaled by the
//    window with r = k/(W/2+1), unnormalised real inverse: Ct/CtVolume.cpp:41-101,
//    832-858, 910-917 and Ct/cuda_ct.cu:48-100.
//
// Design: two rows are filtered at once as the real and imaginary parts of one complex
// sequence (the response is real and even, so real rows stay real).
//  - Powers of two transform at their own length.  For other W the row's circular
//    convolution with the filter kernel g (length W) is the middle of a linear convolution
//    with g extended periodically to 2W - 1 taps, done in a power-of-two transform of
//    length M >= 2W - 1 (no wrap-around reaches the W outputs kept).
//  - W = 256..2048, powers of two (FP32): one wave per row pair, values in registers,
//    Stockham radix-16/8/4 passes exchanging through the wave's LDS region
//    (rows_fft_kernel).
//  - Padded rows and W = 4096, 8192, 16384 (FP32, M from 256): radix-2 stages, decimation in time
//    forward and in frequency back, several at a time in registers (rows_r2_kernel).
//  - Shorter transforms and the FP64 yardstick: the same radix-2 stages one at a time in
//    LDS, one workgroup per row pair (rows_kernel).
#include "ctg_internal.h"

#include <hip/hip_fp16.h>

#include <cmath>
#include <complex>
#include <vector>

namespace ctg {
namespace {

constexpr int kRowThreads = 256;
constexpr double kPi = 3.14159265358979323846;

template <typename T>
struct Cx {
    T re, im;
};

struct PreArgs {
    int W, H, log2W;
    long long nrows;  // total rows (nproj * H for images)
    float la, lb, lk;  // p = -log((I * la + lb) * lk)
    double dla, dlb, dlk;
    float fcd, upre, vpre;
    int pow2;
    int M, log2M;  // transform length: W for powers of two, else the padded length
};

__device__ inline float dlog(float x) { return logf(x); }
__device__ inline double dlog(double x) { return log(x); }
__device__ inline float dsqrt(float x) { return sqrtf(x); }
__device__ inline double dsqrt(double x) { return sqrt(x); }

// Feldkamp weight D / sqrt(D^2 + u^2 + v^2), u = column - uPre, v = vPre - row
template <typename T>
__device__ inline T feldkamp(const PreArgs& a, int r, int c) {
    const T u = (T)c - (T)a.upre;
    const T v = (T)(-r) + (T)a.vpre;
    const T D = (T)a.fcd;
    return D / dsqrt(D * D + u * u + v * v);
}

// an intensity's line integral, Feldkamp weighted, or the value of a filter-only row
template <typename T, typename Tin>
__device__ inline T load_pixel(const Tin* __restrict__ raw, const float* __restrict__ lin, size_t idx,
                               const PreArgs& a, int r, int c) {
    if (raw == nullptr) return (T)lin[idx];
    const T I = (T)raw[idx];
    T x;
    if constexpr (sizeof(T) == 4) x = -dlog(fmaf((float)I, a.la, a.lb) * a.lk);
    else x = -dlog((I * (T)a.dla + (T)a.dlb) * (T)a.dlk);
    return x * feldkamp<T>(a, r, c);
}

template <typename T>
__device__ void fft_dit(T* re, T* im, int W, int log2W, const Cx<T>* __restrict__ tw) {
    for (int lh = 0; lh < log2W; ++lh) {
        const int half = 1 << lh;
        const int sh = log2W - lh - 1;
        __syncthreads();
        for (int j = threadIdx.x; j < (W >> 1); j += blockDim.x) {
            int k = j & (half - 1);
            int i0 = ((j - k) << 1) + k, i1 = i0 + half;
            Cx<T> w = tw[k << sh];
            T br = re[i1], bi = im[i1];
            T xr = br * w.re - bi * w.im;
            T xi = br * w.im + bi * w.re;
            T ar = re[i0], ai = im[i0];
            re[i1] = ar - xr; im[i1] = ai - xi;
            re[i0] = ar + xr; im[i0] = ai + xi;
        }
    }
    __syncthreads();
}

template <typename T>
__device__ void fft_dif(T* re, T* im, int W, int log2W, const Cx<T>* __restrict__ tw) {
    for (int lh = log2W - 1; lh >= 0; --lh) {
        const int half = 1 << lh;
        const int sh = log2W - lh - 1;
        __syncthreads();
        for (int j = threadIdx.x; j < (W >> 1); j += blockDim.x) {
            int k = j & (half - 1);
            int i0 = ((j - k) << 1) + k, i1 = i0 + half;
            Cx<T> w = tw[k << sh];
            T ar = re[i0], ai = im[i0], br = re[i1], bi = im[i1];
            re[i0] = ar + br; im[i0] = ai + bi;
            T dr = ar - br, di = ai - bi;
            re[i1] = dr * w.re - di * w.im;
            im[i1] = dr * w.im + di * w.re;
        }
    }
    __syncthreads();
}

__device__ inline unsigned bitrev(unsigned n, int bits) { return __brev(n) >> (32 - bits); }

__device__ inline float wave_max(float v) {
    for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
    return v;
}

// The maxima of a workgroup's rows, folded into their images' maxima: one atomic of the
// workgroup where all its rows are of one image, else one per wave and image.  Atomics to one
// cache line run one after another, about 10 ns each: with one per wave and the counters of 32
// images in a line, 40 images of 1944 x 1536 spent 1.17 ms on them, so every image's has a line of
// its own.  A look at the maximum before the atomic leaves most out where the waves of an
// image end one after another, but the workgroup waits for it (360 images of 512 x 512: 1060
// us, 344 with an atomic per wave, 235 so; 360 of 256 x 192: 350 and 50 us).
struct BlockMax {
    unsigned bits, waves;
};
// Before the workgroup's first barrier.
__device__ inline void block_max_init(BlockMax& s) {
    if (threadIdx.x == 0) s = BlockMax{0u, 0u};
}
// Once by every wave that handles rows, `waves` of them; rows [first, last] are the workgroup's,
// ma and mb this lane's maxima of rows a and b, of images pa and pb (they may differ when H is odd).
__device__ inline void block_max(BlockMax& s, unsigned waves, long long first, long long last, int H, unsigned* maxabs,
                                 long long pa, long long pb, float ma, float mb) {
    const bool lane0 = (threadIdx.x & 63) == 0;
    if (first / H == last / H) {
        const float m = wave_max(fmaxf(ma, mb));
        if (lane0) {
            // the bits of non-negative floats order like unsigned integers; the last wave to
            // come sees the others' values
            __hip_atomic_fetch_max(&s.bits, __float_as_uint(m), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            if (__hip_atomic_fetch_add(&s.waves, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP) == waves - 1)
                atomicMax(&maxabs[first / H * kMaxStride], __hip_atomic_load(&s.bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
        }
    } else if (pa == pb) {
        const float m = wave_max(fmaxf(ma, mb));
        if (lane0) atomicMax(&maxabs[pa * kMaxStride], __float_as_uint(m));
    } else {
        ma = wave_max(ma);
        mb = wave_max(mb);
        if (lane0) {
            atomicMax(&maxabs[pa * kMaxStride], __float_as_uint(ma));
            atomicMax(&maxabs[pb * kMaxStride], __float_as_uint(mb));
        }
    }
}

// One workgroup per row pair.  Output rows (T) row-major; for float output the
// per-image max |value| is folded into maxabs with an atomic max on the bits.
template <typename T, typename Tin>
__global__ __launch_bounds__(kRowThreads) void rows_kernel(PreArgs a, const Tin* __restrict__ raw,
                                                          const float* __restrict__ lin,
                                                          const T* __restrict__ resp,
                                                          const Cx<T>* __restrict__ tw,
                                                          const Cx<T>* __restrict__ pad_resp,
                                                          T* __restrict__ out,
                                                          unsigned* __restrict__ maxabs) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ BlockMax bmax;
    block_max_init(bmax);  // (the transforms begin with a barrier)
    T* re = reinterpret_cast<T*>(smem_raw);
    T* im = re + a.M;
    const int W = a.W, M = a.M;
    const long long ra = 2ll * blockIdx.x;
    const long long rb = ra + 1;
    const bool hasb = rb < a.nrows;
    const int rin_a = (int)(ra % a.H), rin_b = (int)(rb % a.H);
    const size_t offa = (size_t)ra * W, offb = (size_t)rb * W;

    // padded: y[n] = sum_m x[m] g[(n - m) mod W] = (x * h)[n + W - 1] with h[j] = g[(j - W + 1)
    // mod W], j < 2W - 1: x zero-padded to M, times the M-point transform of h (over M,
    // precomputed), outputs read at n + W - 1
    for (int n = threadIdx.x; n < M; n += blockDim.x) {
        T xa = (T)0, xb = (T)0;
        if (n < W) {
            xa = load_pixel<T, Tin>(raw, lin, offa + n, a, rin_a, n);
            if (hasb) xb = load_pixel<T, Tin>(raw, lin, offb + n, a, rin_b, n);
        }
        unsigned pos = bitrev((unsigned)n, a.log2M);
        re[pos] = xa;
        im[pos] = xb;
    }
    fft_dit<T>(re, im, M, a.log2M, tw);
    // multiply by the response (real and even, complex when padded) and conjugate:
    // IDFT(Z) = conj(DFT(conj Z))
    for (int k = threadIdx.x; k < M; k += blockDim.x) {
        const T xr = re[k], xi = im[k];
        if (a.pow2) {
            const T h = resp[k];
            re[k] = xr * h;
            im[k] = -xi * h;
        } else {
            const Cx<T> h = pad_resp[k];
            re[k] = xr * h.re - xi * h.im;
            im[k] = -(xr * h.im + xi * h.re);
        }
    }
    fft_dif<T>(re, im, M, a.log2M, tw);

    // filtered outputs sit in bit-reversed order (at n + W - 1 for padded widths)
    const int out_shift = a.pow2 ? 0 : W - 1;
    float ma = 0.0f, mb = 0.0f;
    for (int n = threadIdx.x; n < W; n += blockDim.x) {
        const unsigned pos = bitrev((unsigned)(n + out_shift), a.log2M);
        const T ya = re[pos];
        const T yb = -im[pos];
        out[offa + n] = ya;
        if (hasb) out[offb + n] = yb;
        ma = fmaxf(ma, fabsf((float)ya));
        if (hasb) mb = fmaxf(mb, fabsf((float)yb));
    }
    if (sizeof(T) == 4 && maxabs != nullptr) {
        const long long last = hasb ? rb : ra;
        block_max(bmax, kRowThreads / 64, ra, last, a.H, maxabs, ra / a.H, last / a.H, ma, mb);
    }
}

// Feldkamp weight in place, one lane per pixel.
__global__ __launch_bounds__(256) void weight_kernel(PreArgs a, float* __restrict__ img) {
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= a.W) return;
    for (long long r = blockIdx.y; r < a.nrows; r += gridDim.y) {
        float* px = img + (size_t)r * a.W + c;
        *px = *px * feldkamp<float>(a, (int)(r % a.H), c);
    }
}

// ---------------------------------------------------------------------------------
// Register-resident row filter for W = 256, 512, 1024, 2048 (FP32).
//
// One wave owns one row pair (rows a and b as the real and imaginary parts), each lane
// holds P = W/64 complex values, and the transform is a Stockham autosort FFT of 3-4
// passes with radix 16/8/4 butterflies evaluated in registers; between passes the wave
// exchanges values through its own LDS region (no workgroup barrier: a wave's LDS
// operations execute in order).  Pass i, radix R, stride NS: butterfly j reads
// x[j + r*W/R], multiplies by exp(-2 pi i (j mod NS) r / (NS R)) and writes the R-point
// DFT to y[(j / NS) NS R + j mod NS + r NS]; the output ends in natural order.  The
// filtered rows are the conjugate of the forward transform of conj(X * H), so the same
// forward passes run twice; the first pass reads the raw pixels from global memory and
// the last writes the filtered rows.
//
// What bounds it (MI355X, N = 2048): VALU issue 50 % busy and the vector memory unit 43 %
// at 2 waves per SIMD.  A twiddle gather holds that unit about 16 cycles, so pass 1 takes
// its twiddles from a table in LDS and short transforms keep the last pass's in registers
// for both directions: 48 images of 2048 x 1536 in 0.38 ms instead of 0.53.
namespace fftw {

__host__ __device__ constexpr int passes(int N) { return N == 256 ? 4 : 3; }
__host__ __device__ constexpr int radix(int N, int i) {
    return N == 256 ? 4 : (N == 512 ? 8 : (i < 2 ? 16 : (N == 1024 ? 4 : 8)));
}
__host__ __device__ constexpr int stride(int N, int i) { return i == 0 ? 1 : stride(N, i - 1) * radix(N, i - 1); }
// entries of pass 1's twiddle table
__host__ __device__ constexpr int ltw_size(int N) { return radix(N, 0) * radix(N, 1); }
// LDS position of element i: one float2 of padding per 16 spreads the strided writes
__device__ inline int lds_pos(int i) { return i + (i >> 4); }

struct F2 {
    float x, y;
};
__device__ inline F2 add(F2 a, F2 b) { return {a.x + b.x, a.y + b.y}; }
__device__ inline F2 sub(F2 a, F2 b) { return {a.x - b.x, a.y - b.y}; }
__device__ inline F2 mul(F2 a, F2 w) { return {fmaf(a.x, w.x, -(a.y * w.y)), fmaf(a.x, w.y, a.y * w.x)}; }
__device__ inline F2 mul_mi(F2 a) { return {a.y, -a.x}; }  // a * (-i)

// in-place forward DFTs (kernel exp(-2 pi i n k / R)), natural order in and out
__device__ inline void dft4(F2& a0, F2& a1, F2& a2, F2& a3) {
    const F2 t0 = add(a0, a2), t1 = sub(a0, a2), t2 = add(a1, a3), t3 = mul_mi(sub(a1, a3));
    a0 = add(t0, t2);
    a2 = sub(t0, t2);
    a1 = add(t1, t3);
    a3 = sub(t1, t3);
}
__device__ inline void dft8(F2* a) {
    constexpr float h = 0.70710678118654752440f;
    F2 e0 = a[0], e1 = a[2], e2 = a[4], e3 = a[6];
    F2 o0 = a[1], o1 = a[3], o2 = a[5], o3 = a[7];
    dft4(e0, e1, e2, e3);
    dft4(o0, o1, o2, o3);
    o1 = mul(o1, F2{h, -h});
    o2 = mul_mi(o2);
    o3 = mul(o3, F2{-h, -h});
    a[0] = add(e0, o0); a[4] = sub(e0, o0);
    a[1] = add(e1, o1); a[5] = sub(e1, o1);
    a[2] = add(e2, o2); a[6] = sub(e2, o2);
    a[3] = add(e3, o3); a[7] = sub(e3, o3);
}
__device__ inline void dft16(F2* a) {
    // 16 = 4 x 4: DFT4 over n_a of a[4 n_a + n_b], twiddle exp(-2 pi i n_b k_a / 16),
    // DFT4 over n_b; X[k_a + 4 k_b]
    constexpr float c1 = 0.92387953251128675613f, s1 = 0.38268343236508977173f, h = 0.70710678118654752440f;
    F2 t[4][4];
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) {
        t[nb][0] = a[nb]; t[nb][1] = a[4 + nb]; t[nb][2] = a[8 + nb]; t[nb][3] = a[12 + nb];
        dft4(t[nb][0], t[nb][1], t[nb][2], t[nb][3]);
    }
    t[1][1] = mul(t[1][1], F2{c1, -s1});
    t[1][2] = mul(t[1][2], F2{h, -h});
    t[1][3] = mul(t[1][3], F2{s1, -c1});
    t[2][1] = mul(t[2][1], F2{h, -h});
    t[2][2] = mul_mi(t[2][2]);
    t[2][3] = mul(t[2][3], F2{-h, -h});
    t[3][1] = mul(t[3][1], F2{s1, -c1});
    t[3][2] = mul(t[3][2], F2{-h, -h});
    t[3][3] = mul(t[3][3], F2{-c1, s1});
#pragma unroll
    for (int ka = 0; ka < 4; ++ka) {
        F2 y0 = t[0][ka], y1 = t[1][ka], y2 = t[2][ka], y3 = t[3][ka];
        dft4(y0, y1, y2, y3);
        a[ka] = y0; a[ka + 4] = y1; a[ka + 8] = y2; a[ka + 12] = y3;
    }
}
template <int R>
__device__ inline void dft(F2* a) {
    if constexpr (R == 4) dft4(a[0], a[1], a[2], a[3]);
    else if constexpr (R == 8) dft8(a);
    else dft16(a);
}

// orders the wave's LDS stores and loads around a cross-lane exchange
__device__ inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// LDS element that value b*R + r of a pass's inputs (load) or outputs (store) lives at
template <int N, int I>
__device__ inline int load_at(int lane, int i) {
    constexpr int R = radix(N, I);
    return lds_pos(lane + 64 * (i / R) + (i % R) * (N / R));
}
template <int N, int I>
__device__ inline int store_at(int lane, int i) {
    constexpr int R = radix(N, I), NS = stride(N, I);
    const int j = lane + 64 * (i / R);
    return lds_pos((j / NS) * NS * R + (j % NS) + (i % R) * NS);
}

// Moves the values through LDS from where `from` puts them to where `to` takes them.
template <int N, class From, class To>
__device__ inline void exchange(F2* __restrict__ buf, F2 (&v)[N / 64], From from, To to) {
    constexpr int P = N / 64;
#pragma unroll
    for (int i = 0; i < P; ++i) buf[from(i)] = v[i];
    wave_sync();
#pragma unroll
    for (int i = 0; i < P; ++i) v[i] = buf[to(i)];
    wave_sync();
}

// Twiddles of pass I: w[b*R + r] = exp(-2 pi i (j mod NS) r / (NS R)), r > 0.
template <int N, int I>
__device__ inline void load_twiddles(F2 (&w)[N / 64], int lane, const Cx<float>* __restrict__ tw) {
    constexpr int R = radix(N, I), NS = stride(N, I), B = N / 64 / R;
#pragma unroll
    for (int b = 0; b < B; ++b) {
        const int jm = (lane + 64 * b) % NS;
#pragma unroll
        for (int r = 1; r < R; ++r) {
            const Cx<float> t = tw[jm * r * (N / (NS * R))];
            w[b * R + r] = F2{t.re, t.im};
        }
    }
}

// Passes I.. of one forward transform.  On entry v holds pass I's inputs; on return v holds
// the last pass's outputs: value b*R + r is X[lane + 64 b + r * NS_last].  Twiddles: pass 1
// reads the short table ltw (exp(-2 pi i q / (NS R)), in LDS), the last pass takes `last`
// (KEEP: registers, the same for both transforms), other passes read the global table.
template <int N, int I, bool KEEP>
__device__ inline void passes_from(F2 (&v)[N / 64], const F2 (&last)[N / 64], F2* __restrict__ buf,
                                   const F2* __restrict__ ltw, int lane, const Cx<float>* __restrict__ tw) {
    constexpr int R = radix(N, I), NS = stride(N, I), B = N / 64 / R;
    if constexpr (I == 1) {
#pragma unroll
        for (int b = 0; b < B; ++b)
#pragma unroll
            for (int r = 1; r < R; ++r) v[b * R + r] = mul(v[b * R + r], ltw[(lane + 64 * b) % NS * r]);
    } else if constexpr (KEEP && I == passes(N) - 1) {
#pragma unroll
        for (int b = 0; b < B; ++b)
#pragma unroll
            for (int r = 1; r < R; ++r) v[b * R + r] = mul(v[b * R + r], last[b * R + r]);
    } else if constexpr (I > 0) {
        // an opaque zero offset: loaded where they are used instead of being hoisted and
        // kept live across both transforms
        int zero = 0;
        asm volatile("" : "+s"(zero));
        F2 w[N / 64];
        load_twiddles<N, I>(w, lane, tw + zero);
#pragma unroll
        for (int b = 0; b < B; ++b)
#pragma unroll
            for (int r = 1; r < R; ++r) v[b * R + r] = mul(v[b * R + r], w[b * R + r]);
    }
#pragma unroll
    for (int b = 0; b < B; ++b) dft<R>(v + b * R);
    if constexpr (I + 1 < passes(N)) {
        exchange<N>(buf, v, [=](int i) { return store_at<N, I>(lane, i); }, [=](int i) { return load_at<N, I + 1>(lane, i); });
        passes_from<N, I + 1, KEEP>(v, last, buf, ltw, lane, tw);
    }
}

}  // namespace fftw

// row pairs (waves) per workgroup; LDS is (N + N/16) float2 per wave, and pass 1's table
__host__ __device__ constexpr int fft_waves(int N) { return N >= 2048 ? 2 : 4; }

template <int N, typename Tin>
__global__ __launch_bounds__(64 * fft_waves(N)) void rows_fft_kernel(PreArgs a, const Tin* __restrict__ raw,
                                                                  const float* __restrict__ lin,
                                                                  const float* __restrict__ resp,
                                                                  const Cx<float>* __restrict__ tw,
                                                                  float* __restrict__ out,
                                                                  unsigned* __restrict__ maxabs) {
    using namespace fftw;
    constexpr int P = N / 64;
    constexpr int LAST = passes(N) - 1;
    constexpr int R0 = radix(N, 0), RL = radix(N, LAST), NSL = stride(N, LAST);
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ BlockMax bmax;
    block_max_init(bmax);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    F2* buf = reinterpret_cast<F2*>(smem_raw) + (size_t)wave * (N + N / 16);
    F2* ltw = reinterpret_cast<F2*>(smem_raw) + (size_t)fft_waves(N) * (N + N / 16);
    constexpr int S = ltw_size(N);
    for (int q = threadIdx.x; q < S; q += 64 * fft_waves(N)) {
        const Cx<float> t = tw[q * (N / S)];
        ltw[q] = F2{t.re, t.im};
    }
    __syncthreads();
    const long long pair = (long long)blockIdx.x * fft_waves(N) + wave;
    const long long ra = 2 * pair, rb = ra + 1;
    if (ra >= a.nrows) return;  // waves share nothing more, so a finished wave may leave
    const bool hasb = rb < a.nrows;
    const int rin_a = (int)(ra % a.H), rin_b = (int)(rb % a.H);
    const size_t offa = (size_t)ra * N, offb = (size_t)rb * N;

    F2 v[P];
    // pass 0 inputs straight from the images: x[lane + 64 b + r N/R0].  All loads are
    // issued first (a missing row b re-reads row a and is zeroed below).
    const size_t offb_ld = hasb ? offb : offa;
    auto col = [&](int i) { return lane + 64 * (i / R0) + (i % R0) * (N / R0); };
    if (raw != nullptr) {
#pragma unroll
        for (int i = 0; i < P; ++i) {
            v[i].x = (float)raw[offa + col(i)];
            v[i].y = (float)raw[offb_ld + col(i)];
        }
#pragma unroll
        for (int i = 0; i < P; ++i) {
            v[i].x = -logf(fmaf(v[i].x, a.la, a.lb) * a.lk) * feldkamp<float>(a, rin_a, col(i));
            v[i].y = -logf(fmaf(v[i].y, a.la, a.lb) * a.lk) * feldkamp<float>(a, rin_b, col(i));
        }
    } else {
#pragma unroll
        for (int i = 0; i < P; ++i) {
            v[i].x = lin[offa + col(i)];
            v[i].y = lin[offb_ld + col(i)];
        }
    }
    if (!hasb) {
#pragma unroll
        for (int i = 0; i < P; ++i) v[i].y = 0.0f;
    }
    // where the registers hold them beside the values without spilling
    constexpr bool KEEP = N <= 512;
    F2 last[P];
    if constexpr (KEEP) load_twiddles<N, LAST>(last, lane, tw);
    passes_from<N, 0, KEEP>(v, last, buf, ltw, lane, tw);
    // multiply by the real even response and conjugate; back to pass 0's distribution
#pragma unroll
    for (int i = 0; i < P; ++i) {
        const float h = resp[lane + 64 * (i / RL) + (i % RL) * NSL];
        v[i] = F2{v[i].x * h, -(v[i].y * h)};
    }
    exchange<N>(buf, v, [=](int i) { return lds_pos(lane + 64 * (i / RL) + (i % RL) * NSL); },
                [=](int i) { return load_at<N, 0>(lane, i); });
    passes_from<N, 0, KEEP>(v, last, buf, ltw, lane, tw);

    float ma = 0.0f, mb = 0.0f;
#pragma unroll
    for (int i = 0; i < P; ++i) {
        const int n = lane + 64 * (i / RL) + (i % RL) * NSL;
        const float ya = v[i].x, yb = -v[i].y;
        out[offa + n] = ya;
        if (hasb) out[offb + n] = yb;
        ma = fmaxf(ma, fabsf(ya));
        mb = fmaxf(mb, fabsf(yb));
    }
    if (maxabs != nullptr) {
        const long long first = 2ll * fft_waves(N) * blockIdx.x, last = min(first + 2 * fft_waves(N), a.nrows) - 1;
        block_max(bmax, (unsigned)((last - first) / 2 + 1), first, last, a.H, maxabs, ra / a.H,
                  hasb ? rb / a.H : ra / a.H, ma, hasb ? mb : 0.0f);
    }
}

// ---------------------------------------------------------------------------------
// Register-resident radix-2 row filter (FP32): padded rows, and W = 4096 ... 16384.
//
// The stages and their arithmetic are rows_kernel's (a radix-2 decimation in time, the
// response, a decimation in frequency back), product by product, so the rows are the same
// bit for bit whichever kernel filters them.  What differs is where values live: T lanes
// hold P = M/T of them each and run s stages at a time in registers.  A pass over stages
// [a, a + s) takes groups of 2^s elements pos = hi 2^(a+s) + m 2^a + k (m < 2^s, k < 2^a);
// between passes the values move through LDS, within one wave without a workgroup barrier.
//  - Pass 0 (s = log2 P, k = 0): lane t holds positions P rev(t) + m, whose natural
//    indices rev(m) M/P + t are consecutive over the lanes, on the way in and out.
//  - The last pass runs its stages, the response and its stages of the way back in one
//    stay in registers, on one set of twiddles.
//  - Padded rows fill less than half of M: odd m of pass 0 are zero, whatever W.
// One float2 of padding per 2^(L-5) positions and, in pass 1, five low bits of hi before k
// in the lane number make the LDS accesses conflict-free (up to two-way at 9, 13 and 14).
//
// What bounds it (MI355X, M = 4096): VALU issue and the vector memory unit, each about
// half busy, at 16 waves per CU (35 KB of LDS per row pair).  40 images of 1944 x 1536:
// 2.67 ms one stage at a time in LDS, 0.51 ms here.
namespace r2 {

using fftw::F2;

__host__ __device__ constexpr int lanes(int L) { return L == 8 ? 16 : (L == 9 || L == 10) ? 64 : (1 << L) / 16; }
__host__ __device__ constexpr int values(int L) { return (1 << L) / lanes(L); }
__host__ __device__ constexpr int passes(int L) { return L == 8 ? 2 : (L <= 12 ? 3 : 4); }
// stages of pass i
__host__ __device__ constexpr int stages(int L, int i) {
    return L == 9 ? 3 : i == 0 ? 4 : (L == 10 || L == 13) ? 3 : (L == 11 ? (i == 1 ? 4 : 3) : (L == 14 ? (i == 1 ? 4 : 3) : 4));
}
__host__ __device__ constexpr int first(int L, int i) { return i == 0 ? 0 : first(L, i - 1) + stages(L, i - 1); }
__host__ __device__ constexpr int pad_shift(int L) { return L == 8 ? 3 : L == 9 ? 4 : (L <= 12 ? L - 5 : L - 6); }
// row pairs and lanes per workgroup, LDS per pair (float2) and per workgroup (bytes; the
// second part is pass 1's twiddle table)
__host__ __device__ constexpr int pairs(int L) { return lanes(L) <= 64 ? 256 / lanes(L) : 1; }
__host__ __device__ constexpr int threads(int L) { return lanes(L) * pairs(L); }
__host__ __device__ constexpr int pair_lds(int L) { return (1 << L) + ((1 << L) >> pad_shift(L)); }
__host__ __device__ constexpr int ltw_size(int L) { return 1 << (first(L, 1) + stages(L, 1) - 1); }
__host__ __device__ constexpr int lds_bytes(int L) { return (pairs(L) * pair_lds(L) + ltw_size(L)) * 8; }

__host__ __device__ constexpr int rev(int x, int bits) {
    int r = 0;
    for (int i = 0; i < bits; ++i) r |= ((x >> i) & 1) << (bits - 1 - i);
    return r;
}

// k and hi of group b of a lane in pass I > 0
template <int L, int I>
__device__ inline void group_of(int lane, int b, int& k, int& hi) {
    constexpr int a = first(L, I), nh = L - stages(L, I) - a;
    const int g = lane + lanes(L) * b;
    if constexpr (I == 1 && I < passes(L) - 1) {
        constexpr int h1 = nh < 5 ? nh : 5;
        hi = (g & ((1 << h1) - 1)) | ((g >> (h1 + a)) << h1);
        k = (g >> h1) & ((1 << a) - 1);
    } else {
        k = g & ((1 << a) - 1);
        hi = g >> a;
    }
}

// LDS place of value i of a lane in pass I
template <int L, int I>
__device__ inline int place(int lane, int i) {
    constexpr int s = stages(L, I), a = first(L, I);
    int pos;
    if constexpr (I == 0) {
        pos = ((int)(__brev((unsigned)lane) >> (32 - (L - s))) << s) + i;
    } else {
        int k, hi;
        group_of<L, I>(lane, i >> s, k, hi);
        pos = (hi << (a + s)) + ((i & ((1 << s) - 1)) << a) + k;
    }
    return pos + (pos >> pad_shift(L));
}

template <int L>
__device__ inline void pair_sync() {
    if constexpr (lanes(L) > 64) __syncthreads();
    else fftw::wave_sync();
}

template <int L, int I, int J>
__device__ inline void exchange(F2 (&v)[values(L)], F2* __restrict__ buf, int lane) {
#pragma unroll
    for (int i = 0; i < values(L); ++i) buf[place<L, I>(lane, i)] = v[i];
    pair_sync<L>();
#pragma unroll
    for (int i = 0; i < values(L); ++i) v[i] = buf[place<L, J>(lane, i)];
    pair_sync<L>();
}

__device__ inline F2 cmul(F2 b, F2 w) { return {b.x * w.x - b.y * w.y, b.x * w.y + b.y * w.x}; }

// b exp(-2 pi i mm / 2^(j+1)), the twiddles of pass 0 (those off the axes as the table
// rounds them)
template <int J>
__device__ inline F2 cmul_const(F2 b, int mm) {
    constexpr float c1 = 0.92387953251128675613f, s1 = 0.38268343236508977173f, h = 0.70710678118654752440f;
    switch (mm << (3 - J)) {  // sixteenths of a turn
        case 0: return b;
        case 1: return cmul(b, F2{c1, -s1});
        case 2: return cmul(b, F2{h, -h});
        case 3: return cmul(b, F2{s1, -c1});
        case 4: return F2{b.y, -b.x};
        case 5: return cmul(b, F2{-s1, -c1});
        case 6: return cmul(b, F2{-h, -h});
        default: return cmul(b, F2{-c1, -s1});
    }
}

// stage J of a group of 2^S; twiddle mm of stage j is w[2^j - 1 + mm] (CONST: pass 0)
template <int S, int J, bool CONST, bool HALF>
__device__ inline void dit_from(F2* v, const F2* w) {
    if constexpr (J < S) {
#pragma unroll
        for (int m = 0; m < (1 << S); ++m) {
            if (m & (1 << J)) continue;
            const int mm = m & ((1 << J) - 1);
            F2 &x = v[m], &y = v[m + (1 << J)];
            if constexpr (HALF && J == 0) {
                y = x;  // y is zero
            } else {
                F2 t;
                if constexpr (CONST) t = cmul_const<J>(y, mm);
                else t = cmul(y, w[(1 << J) - 1 + mm]);
                y = fftw::sub(x, t);
                x = fftw::add(x, t);
            }
        }
        dit_from<S, J + 1, CONST, HALF>(v, w);
    }
}
template <int S, int J, bool CONST>
__device__ inline void dif_from(F2* v, const F2* w) {
    if constexpr (J >= 0) {
#pragma unroll
        for (int m = 0; m < (1 << S); ++m) {
            if (m & (1 << J)) continue;
            const int mm = m & ((1 << J) - 1);
            F2 &x = v[m], &y = v[m + (1 << J)];
            const F2 d = fftw::sub(x, y);
            x = fftw::add(x, y);
            if constexpr (CONST) y = cmul_const<J>(d, mm);
            else y = cmul(d, w[(1 << J) - 1 + mm]);
        }
        dif_from<S, J - 1, CONST>(v, w);
    }
}

// Twiddles of pass I > 0: the short LDS table for pass 1, else the global table.
template <int L, int I>
__device__ inline void load_twiddles(F2 (&w)[values(L)], int lane, const F2* __restrict__ ltw,
                                     const Cx<float>* __restrict__ tw) {
    constexpr int s = stages(L, I), a = first(L, I), B = values(L) >> s;
#pragma unroll
    for (int b = 0; b < B; ++b) {
        int k, hi;
        group_of<L, I>(lane, b, k, hi);
#pragma unroll
        for (int j = 0; j < s; ++j)
#pragma unroll
            for (int mm = 0; mm < (1 << j); ++mm) {
                F2& d = w[(b << s) + (1 << j) - 1 + mm];
                if constexpr (I == 1) {
                    d = ltw[(k + (mm << a)) << (s - 1 - j)];
                } else {
                    const Cx<float> t = tw[(k + (mm << a)) << (L - 1 - a - j)];
                    d = F2{t.re, t.im};
                }
            }
    }
}

// Passes I.. there, the response, and back to pass I - 1's distribution.
template <int L, int I, class Response>
__device__ inline void passes_from(F2 (&v)[values(L)], F2* __restrict__ buf, const F2* __restrict__ ltw, int lane,
                                   const Cx<float>* __restrict__ tw, Response response) {
    constexpr int s = stages(L, I), B = values(L) >> s;
    constexpr bool last = I == passes(L) - 1;
    exchange<L, I - 1, I>(v, buf, lane);
    {
        F2 w[values(L)];
        load_twiddles<L, I>(w, lane, ltw, tw);
#pragma unroll
        for (int b = 0; b < B; ++b) dit_from<s, 0, false, false>(v + (b << s), w + (b << s));
        if constexpr (last) {
            response(v);
#pragma unroll
            for (int b = 0; b < B; ++b) dif_from<s, s - 1, false>(v + (b << s), w + (b << s));
        }
    }
    if constexpr (!last) {
        passes_from<L, I + 1>(v, buf, ltw, lane, tw, response);
        // an opaque zero offset: the twiddles are read again instead of being kept live
        int zero = 0;
        asm volatile("" : "+s"(zero));
        F2 w[values(L)];
        load_twiddles<L, I>(w, lane, ltw + zero, tw + zero);
#pragma unroll
        for (int b = 0; b < B; ++b) dif_from<s, s - 1, false>(v + (b << s), w + (b << s));
    }
    exchange<L, I, I - 1>(v, buf, lane);
}

}  // namespace r2

template <int L, bool PAD, typename Tin>
__global__ __launch_bounds__(r2::threads(L)) __attribute__((amdgpu_waves_per_eu(4))) void rows_r2_kernel(
    PreArgs a, const Tin* __restrict__ raw, const float* __restrict__ lin, const float* __restrict__ resp,
    const Cx<float>* __restrict__ pad_resp, const Cx<float>* __restrict__ tw, float* __restrict__ out,
    unsigned* __restrict__ maxabs) {
    using namespace r2;
    constexpr int M = 1 << L, T = lanes(L), P = values(L), S0 = stages(L, 0), LAST = passes(L) - 1;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ BlockMax bmax;
    block_max_init(bmax);
    const int slot = threadIdx.x / T, lane = threadIdx.x % T;
    F2* buf = reinterpret_cast<F2*>(smem_raw) + (size_t)slot * pair_lds(L);
    F2* ltw = reinterpret_cast<F2*>(smem_raw) + (size_t)pairs(L) * pair_lds(L);
    for (int q = threadIdx.x; q < ltw_size(L); q += threads(L)) {
        const Cx<float> t = tw[q * (M / (2 * ltw_size(L)))];
        ltw[q] = F2{t.re, t.im};
    }
    __syncthreads();
    // lanes of a pair past the end re-read the last row and store nothing
    const long long ra0 = 2 * ((long long)blockIdx.x * pairs(L) + slot);
    const bool hasa = ra0 < a.nrows, hasb = ra0 + 1 < a.nrows;
    const long long ra = hasa ? ra0 : a.nrows - 1, rb = hasb ? ra0 + 1 : ra;
    const int W = a.W;
    const int rin_a = (int)(ra % a.H), rin_b = (int)(rb % a.H);
    const size_t offa = (size_t)ra * W, offb = (size_t)rb * W;

    // natural index of value m in pass 0
    auto col = [&](int m) { return rev(m, S0) * (M / P) + lane; };
    auto used = [](int m) { return !PAD || (m & 1) == 0; };
    F2 v[P];
    // all loads are issued first (columns past the row re-read its last one); what does not
    // exist is zeroed below
    if (raw != nullptr) {
#pragma unroll
        for (int m = 0; m < P; ++m) {
            if (!used(m)) continue;
            const int n = PAD ? min(col(m), W - 1) : col(m);
            v[m].x = (float)raw[offa + n];
            v[m].y = (float)raw[offb + n];
        }
#pragma unroll
        for (int m = 0; m < P; ++m) {
            if (!used(m)) continue;
            v[m].x = -logf(fmaf(v[m].x, a.la, a.lb) * a.lk) * feldkamp<float>(a, rin_a, col(m));
            v[m].y = -logf(fmaf(v[m].y, a.la, a.lb) * a.lk) * feldkamp<float>(a, rin_b, col(m));
        }
    } else {
#pragma unroll
        for (int m = 0; m < P; ++m) {
            if (!used(m)) continue;
            const int n = PAD ? min(col(m), W - 1) : col(m);
            v[m].x = lin[offa + n];
            v[m].y = lin[offb + n];
        }
    }
#pragma unroll
    for (int m = 0; m < P; ++m) {
        if (!used(m) || (PAD && col(m) >= W)) v[m] = F2{0.0f, 0.0f};
        if (!hasb) v[m].y = 0.0f;
    }
    dit_from<S0, 0, true, PAD>(v, nullptr);
    passes_from<L, 1>(v, buf, ltw, lane, tw, [&](F2(&z)[P]) {
        // multiply by the response (real and even, complex when padded) and conjugate
        constexpr int s = stages(L, LAST), f = first(L, LAST);
#pragma unroll
        for (int i = 0; i < P; ++i) {
            const int k = lane + T * (i >> s) + ((i & ((1 << s) - 1)) << f);
            if constexpr (PAD) {
                const Cx<float> h = pad_resp[k];
                const F2 y = cmul(z[i], F2{h.re, h.im});
                z[i] = F2{y.x, -y.y};
            } else {
                const float h = resp[k];
                z[i] = F2{z[i].x * h, -z[i].y * h};
            }
        }
    });
    dif_from<S0, S0 - 1, true>(v, nullptr);

    const int shift = PAD ? W - 1 : 0;
    float ma = 0.0f, mb = 0.0f;
#pragma unroll
    for (int m = 0; m < P; ++m) {
        const int n = col(m) - shift;
        if (!hasa || (PAD && (n < 0 || n >= W))) continue;
        const float ya = v[m].x, yb = -v[m].y;
        out[offa + n] = ya;
        ma = fmaxf(ma, fabsf(ya));
        if (hasb) {
            out[offb + n] = yb;
            mb = fmaxf(mb, fabsf(yb));
        }
    }
    if (maxabs != nullptr) {
        const long long first = 2ll * pairs(L) * blockIdx.x, last = min(first + 2 * pairs(L), a.nrows) - 1;
        if (T >= 64 || first / a.H == last / a.H) {
            // (a pair past the end adds zeros to the last row's image)
            block_max(bmax, threads(L) / 64, first, last, a.H, maxabs, ra / a.H, rb / a.H, ma, mb);
        } else {
            // several pairs per wave, of more than one image
            for (int off = T / 2; off > 0; off >>= 1) {
                ma = fmaxf(ma, __shfl_xor(ma, off, 64));
                mb = fmaxf(mb, __shfl_xor(mb, off, 64));
            }
            if (lane == 0 && hasa) {
                atomicMax(&maxabs[ra / a.H * kMaxStride], __float_as_uint(ma));
                if (hasb) atomicMax(&maxabs[rb / a.H * kMaxStride], __float_as_uint(mb));
            }
        }
    }
}

// Row-major FP32 images -> backprojection layout.  Entry (u, v) of image p holds the
// bilinear coefficients of the cell whose top-left texel is (u, v):
//   A = q[v][u], dU = q[v][u+1] - A, dV = q[v+1][u] - A, dUV = q[v+1][u+1] - q[v+1][u] - dU
// (texels past the last column or row are 0), so that the interpolated value at
// (u + fu, v + fv) is A + fu*dU + fv*(dV + fu*dUV).  Entries are stored column-major
// (v fastest): a detector column is contiguous, and one voxel-update reads one entry.
//
// Bound by memory: a tile of TS x TS texels goes through LDS; 64 instead of 32 doubles the
// contiguous run of a column's stores (512 bytes of 8-byte entries) and halves the texels read
// twice, and 8-byte entries go out two rows per lane.  48 images of 2048 x 1536 to FP16: 0.48
// -> 0.41 ms (4.4 TB/s), 359 of 1001 x 763 (odd height, one row per lane): 0.80 -> 0.73 ms.
//
// The tiles of an image are rotated by its number, except large images (over 64 tiles) in tiles of
// 64: dispatch deals workgroups to the 8 XCDs in turn, and where the tiles of an image are a
// multiple of 4 or 8 the same XCDs would take the partly filled ones at the edge of every image
// (FP32, 300 images of 250 x 201 in 4 x 4 tiles: 91 us, 78 rotated; 120 of 341 x 196 in 6 x 4: 34
// and 29; 240 of 1024 x 1024 in tiles of 32: 1035 and 1001).
__device__ inline uint32_t pack_f16(float a, float b) {
    __half ha = __float2half_rn(a), hb = __float2half_rn(b);
    return (uint32_t)__half_as_ushort(ha) | ((uint32_t)__half_as_ushort(hb) << 16);
}
__device__ inline uint32_t f2bf(float x) {
    uint32_t u = __float_as_uint(x);
    u += 0x7fffu + ((u >> 16) & 1u);
    return u >> 16;
}
__device__ inline uint32_t pack_bf16(float a, float b) { return f2bf(a) | (f2bf(b) << 16); }

template <int STORE, int TS>
__global__ __launch_bounds__(256) void layout_kernel(const float* __restrict__ rows, int W, int H,
                                                     const unsigned* __restrict__ maxabs, int mstride, int pairs,
                                                     void* __restrict__ out, float* __restrict__ scales) {
    __shared__ float tile[TS + 1][TS + 1];
    constexpr int kStep = 256 / TS;  // rows loaded, then columns stored, at a time
    const size_t p = blockIdx.z;
    unsigned tx = blockIdx.x, ty = blockIdx.y;
    if (blockIdx.z > 0 && (TS == 32 || gridDim.x * gridDim.y <= 64)) {
        tx = (tx + blockIdx.z) % gridDim.x;
        ty = (ty + blockIdx.z / gridDim.x) % gridDim.y;
    }
    const int u0 = tx * TS, v0 = ty * TS;
    const float* img = rows + p * (size_t)W * H;
    const int tl = threadIdx.x & (TS - 1), tr = threadIdx.x / TS;
    auto texel = [&](int vl, int ul) {
        const int v = v0 + vl, u = u0 + ul;
        return v < H && u < W ? img[(size_t)v * W + u] : 0.0f;
    };
    // (a small tile in one go over its 33 x 33 texels: as below it takes 2 to 10 % longer)
    if constexpr (TS == 32) {
        for (int i = threadIdx.x; i < (TS + 1) * (TS + 1); i += 256) {
            const int vl = i / (TS + 1), ul = i - vl * (TS + 1);
            tile[vl][ul] = texel(vl, ul);
        }
    } else {
#pragma unroll
        for (int i = 0; i < TS / kStep; ++i) tile[tr + i * kStep][tl] = texel(tr + i * kStep, tl);
        // the row below and the column to the right
        if (threadIdx.x < TS) tile[TS][threadIdx.x] = texel(TS, threadIdx.x);
        else if (threadIdx.x < 2 * TS + 1) tile[threadIdx.x - TS][TS] = texel(threadIdx.x - TS, TS);
    }
    __syncthreads();
    float scale = 1.0f, inv = 1.0f;
    if (STORE != CTG_STORE_F32) {
        float m = __uint_as_float(maxabs[p * mstride]);
        if (m > 0.0f && m < INFINITY) {
            int e;
            frexpf(m, &e);
            scale = ldexpf(1.0f, e);
            inv = ldexpf(1.0f, -e);
        }
    }
    if (tx == 0 && ty == 0 && threadIdx.x == 0 && scales != nullptr) scales[p] = scale;
    auto coeffs = [&](int vl, int ul) {
        const float A = tile[vl][ul] * inv, B = tile[vl][ul + 1] * inv;
        const float C = tile[vl + 1][ul] * inv, D = tile[vl + 1][ul + 1] * inv;
        const float dU = B - A, dV = C - A;
        return make_float4(A, dU, dV, (D - C) - dU);
    };
    auto pack = [&](float4 c) {
        return STORE == CTG_STORE_F16 ? make_uint2(pack_f16(c.x, c.y), pack_f16(c.z, c.w))
                                      : make_uint2(pack_bf16(c.x, c.y), pack_bf16(c.z, c.w));
    };
    if (STORE != CTG_STORE_F32 && TS == 64 && pairs) {
        // two rows of 8-byte entries per lane
        const int vl = 2 * (threadIdx.x & 31), v = v0 + vl;
        for (int ul = threadIdx.x >> 5; ul < TS; ul += 8) {
            const int u = u0 + ul;
            if (u < W && v < H) {
                const uint2 a = pack(coeffs(vl, ul)), b = pack(coeffs(vl + 1, ul));
                reinterpret_cast<uint4*>(out)[((p * (size_t)W + u) * H + v) >> 1] = make_uint4(a.x, a.y, b.x, b.y);
            }
        }
        return;
    }
    for (int ul = tr; ul < TS; ul += kStep) {
        const int u = u0 + ul, v = v0 + tl;
        if (u < W && v < H) {
            const size_t idx = (p * (size_t)W + u) * H + v;
            const float4 c = coeffs(tl, ul);
            if (STORE == CTG_STORE_F32) reinterpret_cast<float4*>(out)[idx] = c;
            else reinterpret_cast<uint2*>(out)[idx] = pack(c);
        }
    }
}

int ilog2_exact(int W) {
    int l = 0;
    while ((1 << l) < W) ++l;
    return (1 << l) == W ? l : -1;
}

// Transform length of the row filter: W itself for powers of two, otherwise the
// smallest power of two >= 2W - 1 (the padded linear convolution).
int filter_log2_length(int W) {
    const int l = ilog2_exact(W);
    if (l >= 0) return l;
    int m = 0;
    while ((1 << m) < 2 * W - 1) ++m;
    return m;
}

// the LDS row buffer holds transforms of up to `most` points
ctg_status check_transform(const PreArgs& a, int most) {
    if (a.M <= most) return CTG_OK;
    return fail(CTG_ERROR_UNSUPPORTED, "detector width %d (transform length %d) exceeds the LDS row buffer", a.W, a.M);
}

void set_transform(PreArgs& a) {
    a.pow2 = ilog2_exact(a.W) >= 0;
    a.log2M = filter_log2_length(a.W);
    a.M = 1 << a.log2M;
}

void fill_log_params(PreArgs& a, ctg_pixel_type pixel, float base, ctg_log_form form) {
    const double B = base;
    const double S = pixel == CTG_PIXEL_U8 ? 255.0 : (pixel == CTG_PIXEL_U16 ? 65535.0 : 1.0);
    if (form == CTG_LOG_CPU_FORM) {
        // convertTo32bit: integer images I/S + 1e-6*B (float images unchanged), then * 1/(B+1e-6*B)
        a.dla = (pixel == CTG_PIXEL_F32) ? 1.0 : 1.0 / S;
        a.dlb = (pixel == CTG_PIXEL_F32) ? 0.0 : 0.000001 * B;
        a.dlk = 1.0 / (B + 0.000001 * B);
    } else {
        // convertTo(alpha = (1-1e-6)/(S*B), beta = 1e-6), log, * -1
        a.dla = (1.0 - 0.000001) / (S * B);
        a.dlb = 0.000001;
        a.dlk = 1.0;
    }
    a.la = (float)a.dla;
    a.lb = (float)a.dlb;
    a.lk = (float)a.dlk;
}

// Launches KERNEL<..., Tin> for the pixel type of `raw` (float for filter-only rows).
#define CTG_ROWS_LAUNCH(KERNEL, ...)                                                                        \
    do {                                                                                                    \
        if (raw != nullptr && pixel == CTG_PIXEL_U8)                                                        \
            hipLaunchKernelGGL((KERNEL(uint8_t)), grid, block, lds, st, a, (const uint8_t*)raw, __VA_ARGS__);   \
        else if (raw != nullptr && pixel == CTG_PIXEL_U16)                                                  \
            hipLaunchKernelGGL((KERNEL(uint16_t)), grid, block, lds, st, a, (const uint16_t*)raw, __VA_ARGS__); \
        else                                                                                                \
            hipLaunchKernelGGL((KERNEL(float)), grid, block, lds, st, a, (const float*)raw, __VA_ARGS__);   \
    } while (0)

// workgroups for `pairs` row pairs, `per` in each
ctg_status row_blocks(long long pairs, int per, dim3& grid) {
    const long long blocks = (pairs + per - 1) / per;
    if (blocks > 0x7fffffffll) return fail(CTG_ERROR_UNSUPPORTED, "too many detector rows in one call");
    grid = dim3((unsigned)blocks);
    return CTG_OK;
}

template <int N>
ctg_status launch_rows_fft(const FilterTables& ft, const void* raw, ctg_pixel_type pixel, const float* lin,
                           const PreArgs& a, float* out, unsigned* maxabs, hipStream_t st) {
    constexpr int waves = fft_waves(N);
    dim3 grid;
    CTG_TRY(row_blocks((a.nrows + 1) / 2, waves, grid));
    const dim3 block(64 * waves);
    const size_t lds = ((size_t)waves * (N + N / 16) + fftw::ltw_size(N)) * sizeof(fftw::F2);
#define CTG_K(Tin) rows_fft_kernel<N, Tin>
    CTG_ROWS_LAUNCH(CTG_K, lin, ft.resp_f.as<float>(), ft.tw_f.as<Cx<float>>(), out, maxabs);
#undef CTG_K
    CTG_HIP(hipGetLastError());
    return CTG_OK;
}

template <int L, bool PAD>
ctg_status launch_rows_r2(const FilterTables& ft, const void* raw, ctg_pixel_type pixel, const float* lin,
                          const PreArgs& a, float* out, unsigned* maxabs, hipStream_t st) {
    dim3 grid;
    CTG_TRY(row_blocks((a.nrows + 1) / 2, r2::pairs(L), grid));
    const dim3 block(r2::threads(L));
    const size_t lds = r2::lds_bytes(L);
#define CTG_K(Tin) rows_r2_kernel<L, PAD, Tin>
    CTG_ROWS_LAUNCH(CTG_K, lin, ft.resp_f.as<float>(), ft.pad_f.as<Cx<float>>(), ft.tw_f.as<Cx<float>>(), out, maxabs);
#undef CTG_K
    CTG_HIP(hipGetLastError());
    return CTG_OK;
}

// Filters a.nrows rows of raw images (log, weight) or of line integrals `lin` into `out`.
// Every transform that fills a wave's registers takes a register kernel.  8192 rows of line
// integrals, one stage at a time in LDS against here: W = 90 19 / 9 us, 250 33 / 12 us,
// 1000 145 / 36 us, 1944 331 / 64 us, 3000 843 / 182 us; 4096 rows of 4096 191 / 42 us, of
// 8191 1431 / 261 us.
ctg_status launch_rows(ctg_context* ctx, const void* raw, ctg_pixel_type pixel, const float* lin, const PreArgs& a,
                       float* out, unsigned* maxabs, hipStream_t st) {
    const FilterTables& ft = ctx->ftab;
    CTG_TRY(check_transform(a, 16384));
    if (a.pow2) {
        switch (a.W) {
            case 256: return launch_rows_fft<256>(ft, raw, pixel, lin, a, out, maxabs, st);
            case 512: return launch_rows_fft<512>(ft, raw, pixel, lin, a, out, maxabs, st);
            case 1024: return launch_rows_fft<1024>(ft, raw, pixel, lin, a, out, maxabs, st);
            case 2048: return launch_rows_fft<2048>(ft, raw, pixel, lin, a, out, maxabs, st);
            case 4096: return launch_rows_r2<12, false>(ft, raw, pixel, lin, a, out, maxabs, st);
            case 8192: return launch_rows_r2<13, false>(ft, raw, pixel, lin, a, out, maxabs, st);
            case 16384: return launch_rows_r2<14, false>(ft, raw, pixel, lin, a, out, maxabs, st);
        }
    } else {
        switch (a.M) {
            case 256: return launch_rows_r2<8, true>(ft, raw, pixel, lin, a, out, maxabs, st);
            case 512: return launch_rows_r2<9, true>(ft, raw, pixel, lin, a, out, maxabs, st);
            case 1024: return launch_rows_r2<10, true>(ft, raw, pixel, lin, a, out, maxabs, st);
            case 2048: return launch_rows_r2<11, true>(ft, raw, pixel, lin, a, out, maxabs, st);
            case 4096: return launch_rows_r2<12, true>(ft, raw, pixel, lin, a, out, maxabs, st);
            case 8192: return launch_rows_r2<13, true>(ft, raw, pixel, lin, a, out, maxabs, st);
            case 16384: return launch_rows_r2<14, true>(ft, raw, pixel, lin, a, out, maxabs, st);
        }
    }
    // transforms of up to 128 points: a few LDS stages, not worth a register form
    dim3 grid;
    CTG_TRY(row_blocks((a.nrows + 1) / 2, 1, grid));
    const dim3 block(kRowThreads);
    const size_t lds = (size_t)a.M * sizeof(float) * 2;
#define CTG_K(Tin) rows_kernel<float, Tin>
    CTG_ROWS_LAUNCH(CTG_K, lin, ft.resp_f.as<float>(), ft.tw_f.as<Cx<float>>(), ft.pad_f.as<Cx<float>>(), out, maxabs);
#undef CTG_K
    CTG_HIP(hipGetLastError());
    return CTG_OK;
}

}  // namespace

ctg_status launch_preprocess_rows(ctg_context* ctx, const void* d_raw, ctg_pixel_type pixel, int nproj,
                                  float base, ctg_log_form form, ctg_filter filter, float* d_out,
                                  unsigned* d_maxabs, hipStream_t st) {
    const ctg_geometry& g = ctx->geom;
    PreArgs a{};
    a.W = g.det_width;
    a.H = g.det_height;
    a.nrows = (long long)nproj * a.H;
    fill_log_params(a, pixel, base, form);
    a.fcd = g.fcd;
    a.upre = g.u_pre;
    a.vpre = g.v_pre;
    set_transform(a);
    CTG_TRY(check_transform(a, 16384));
    CTG_TRY(ensure_filter_tables(ctx, a.W, filter));
    return launch_rows(ctx, d_raw, pixel, nullptr, a, d_out, d_maxabs, st);
}

ctg_status launch_feldkamp_weight(const ctg_geometry& g, float* d_images, int nproj, hipStream_t st) {
    PreArgs a{};
    a.W = g.det_width;
    a.H = g.det_height;
    a.nrows = (long long)nproj * a.H;
    a.fcd = g.fcd;
    a.upre = g.u_pre;
    a.vpre = g.v_pre;
    const dim3 grid((unsigned)((a.W + 255) / 256), (unsigned)std::min<long long>(a.nrows, 16384));
    hipLaunchKernelGGL(weight_kernel, grid, dim3(256), 0, st, a, d_images);
    CTG_HIP(hipGetLastError());
    return CTG_OK;
}

ctg_status launch_filter_rows_only(ctg_context* ctx, const float* d_in, float* d_out, int64_t rows,
                                   ctg_filter filter, hipStream_t st) {
    const ctg_geometry& g = ctx->geom;
    PreArgs a{};
    a.W = g.det_width;
    a.H = g.det_height > 0 ? g.det_height : 1;
    a.nrows = rows;
    set_transform(a);
    CTG_TRY(check_transform(a, 16384));
    CTG_TRY(ensure_filter_tables(ctx, a.W, filter));
    return launch_rows(ctx, nullptr, CTG_PIXEL_F32, d_in, a, d_out, nullptr, st);
}

ctg_status launch_preprocess_rows_f64(ctg_context* ctx, const void* d_raw, ctg_pixel_type pixel, int nproj,
                                      float base, ctg_filter filter, double* d_out, hipStream_t st) {
    const ctg_geometry& g = ctx->geom;
    PreArgs a{};
    a.W = g.det_width;
    a.H = g.det_height;
    a.nrows = (long long)nproj * a.H;
    fill_log_params(a, pixel, base, CTG_LOG_CPU_FORM);
    a.fcd = g.fcd;
    a.upre = g.u_pre;
    a.vpre = g.v_pre;
    set_transform(a);
    CTG_TRY(check_transform(a, 8192));
    CTG_TRY(ensure_filter_tables(ctx, a.W, filter));
    const FilterTables& ft = ctx->ftab;
    const size_t lds = (size_t)a.M * sizeof(double) * 2;
    dim3 grid;
    CTG_TRY(row_blocks((a.nrows + 1) / 2, 1, grid));
    const dim3 block(kRowThreads);
    const void* raw = d_raw;
#define CTG_K(Tin) rows_kernel<double, Tin>
    CTG_ROWS_LAUNCH(CTG_K, (const float*)nullptr, ft.resp_d.as<double>(), ft.tw_d.as<Cx<double>>(),
                    ft.pad_d.as<Cx<double>>(), d_out, (unsigned*)nullptr);
#undef CTG_K
    CTG_HIP(hipGetLastError());
    return CTG_OK;
}

ctg_status launch_layout(const ctg_geometry& g, const float* d_rows, int nproj, ctg_store store,
                         const unsigned* d_maxabs, int mstride, void* d_out, float* d_scales, hipStream_t st) {
    // one grid z index per projection; the grid's z extent is limited to 65535
    const size_t img = (size_t)g.det_width * g.det_height;
    const size_t ebytes = store == CTG_STORE_F32 ? 16 : 8;
    for (int p0 = 0; p0 < nproj; p0 += 65535) {
        const int np = std::min(65535, nproj - p0);
        const auto tiles = [&](int ts) { return dim3((unsigned)((g.det_width + ts - 1) / ts), (unsigned)((g.det_height + ts - 1) / ts), (unsigned)np); };
        const float* rows = d_rows + (size_t)p0 * img;
        const unsigned* mx = d_maxabs ? d_maxabs + (size_t)p0 * mstride : nullptr;  // not read for FP32 entries
        void* out = (char*)d_out + (size_t)p0 * img * ebytes;
        float* sc = d_scales ? d_scales + p0 : nullptr;
        const dim3 big = tiles(64), small = tiles(32);
        // 64 x 64 tiles where at least four per CU are left (one image of 256 x 192 takes 4.1 us
        // with its 48 tiles of 32, 7.6 with 12 of 64), where they cover at most 1.45 times the area
        // that tiles of 32 do (FP32, 600 images of 129 x 129, 1.44 times: 41 us and 42 in tiles of
        // 32; 720 of 70 x 70, 1.78 times: 23 and 16) and, with FP32 entries, where these about fit
        // the 256 MB Infinity Cache (in tiles of 64 and 32: 270 MiB, 360 of 256 x 192, 79 and 91 us;
        // 291 MiB, 107 of 1038 x 172, 95 and 91; 1144 MiB, 100 of 1000 x 750, 348 and 315; 8-byte
        // entries gain 2 to 9 % at all of these sizes)
        const bool wide = (long long)big.x * big.y * big.z >= 1024 && 400ll * big.x * big.y <= 145ll * small.x * small.y &&
                          (store != CTG_STORE_F32 || np * img * ebytes <= (size_t)280 << 20);
        // columns of an even height start 16-byte aligned if the buffer does
        const int pairs = g.det_height % 2 == 0 && (uintptr_t)out % 16 == 0;
        const dim3 grid = wide ? big : small;
#define CTG_LAYOUT(S, TS) \
    hipLaunchKernelGGL((layout_kernel<S, TS>), grid, dim3(256), 0, st, rows, g.det_width, g.det_height, mx, mstride, pairs, out, sc)
        if (store == CTG_STORE_F32) {
            if (wide) CTG_LAYOUT(CTG_STORE_F32, 64);
            else CTG_LAYOUT(CTG_STORE_F32, 32);
        } else if (store == CTG_STORE_F16) {
            if (wide) CTG_LAYOUT(CTG_STORE_F16, 64);
            else CTG_LAYOUT(CTG_STORE_F16, 32);
        } else {
            if (wide) CTG_LAYOUT(CTG_STORE_BF16, 64);
            else CTG_LAYOUT(CTG_STORE_BF16, 32);
        }
#undef CTG_LAYOUT
        CTG_HIP(hipGetLastError());
    }
    return CTG_OK;
}

// Host-side tables in double: window H(k) with the float/double evaluation of
// Ct/CtVolume.cpp:868-885 (N = W/2+1) and its real even extension; twiddles
// exp(-2 pi i m / M) for the transform length M; for other W the circular-convolution
// kernel g[m] = sum_k H(k) cos(2 pi k m / W), extended periodically to 2W - 1 taps,
// and its M-point transform over M.
ctg_status ensure_filter_tables(ctg_context* ctx, int W, int filter) {
    FilterTables& ft = ctx->ftab;
    if (ft.W == W && ft.filter == filter && ft.resp_f.ptr) return CTG_OK;
    const int nyq = W / 2 + 1;
    std::vector<double> h(nyq);
    const float N = (float)nyq;
    for (int k = 0; k < nyq; ++k) {
        float n = (float)k;
        float rl = n / N;
        float hv;
        if (filter == CTG_FILTER_SHEPP_LOGAN) {
            if (n == 0.0f) hv = 0.0f;
            else {
                double ang = (double)(rl * 0.5f) * kPi;
                hv = (float)((double)rl * std::sin(ang) / ang);
            }
        } else if (filter == CTG_FILTER_HANN) {
            hv = (float)((double)rl * (double)0.5f * (1.0 + std::cos(kPi * (double)rl)));
        } else {
            hv = rl;
        }
        h[k] = hv;
    }
    std::vector<double> resp(W);
    for (int k = 0; k < W; ++k) resp[k] = h[k <= W / 2 ? k : W - k];
    const bool pow2 = ilog2_exact(W) >= 0;
    const int log2M = filter_log2_length(W), M = 1 << log2M;
    std::vector<double> tw(2 * (size_t)M, 0.0);
    for (int m = 0; m < M / 2; ++m) {
        double ang = 2.0 * kPi * (double)m / (double)M;
        tw[2 * m] = std::cos(ang);
        tw[2 * m + 1] = -std::sin(ang);
        tw[2 * (m + M / 2)] = -tw[2 * m];
        tw[2 * (m + M / 2) + 1] = -tw[2 * m + 1];
    }
    std::vector<double> pad(2 * (size_t)M, 0.0);  // complex, interleaved
    if (!pow2) {
        std::vector<double> cosw(W), g(W);
        for (int j = 0; j < W; ++j) cosw[j] = std::cos(2.0 * kPi * (double)j / (double)W);
        for (int m = 0; m < W; ++m) {
            double s = 0.0;
            for (int k = 0, j = 0; k < W; ++k) {  // j = k m mod W
                s += resp[k] * cosw[j];
                j += m;
                if (j >= W) j -= W;
            }
            g[m] = s;
        }
        std::vector<std::complex<double>> z(M);
        for (int j = 0; j < 2 * W - 1; ++j) z[j] = g[((j - (W - 1)) % W + W) % W];
        // iterative radix-2 transform exp(-2 pi i jk / M), over M
        for (int i = 1, r = 0; i < M; ++i) {
            int bit = M >> 1;
            for (; r & bit; bit >>= 1) r ^= bit;
            r ^= bit;
            if (i < r) std::swap(z[i], z[r]);
        }
        for (int len = 2; len <= M; len <<= 1) {
            for (int i0 = 0; i0 < M; i0 += len) {
                for (int k = 0; k < len / 2; ++k) {
                    const int t = k * (M / len);
                    const std::complex<double> w(tw[2 * t], tw[2 * t + 1]);
                    const std::complex<double> u = z[i0 + k], v = z[i0 + k + len / 2] * w;
                    z[i0 + k] = u + v;
                    z[i0 + k + len / 2] = u - v;
                }
            }
        }
        for (int k = 0; k < M; ++k) {
            pad[2 * (size_t)k] = z[k].real() / (double)M;
            pad[2 * (size_t)k + 1] = z[k].imag() / (double)M;
        }
    }
    std::vector<float> resp_f(W), tw_f(tw.size()), pad_f(pad.size());
    for (int i = 0; i < W; ++i) resp_f[i] = (float)resp[i];
    for (size_t i = 0; i < tw.size(); ++i) tw_f[i] = (float)tw[i];
    for (size_t i = 0; i < pad.size(); ++i) pad_f[i] = (float)pad[i];
    CTG_TRY(ft.resp_f.reserve(sizeof(float) * W));
    CTG_TRY(ft.tw_f.reserve(sizeof(float) * tw_f.size()));
    CTG_TRY(ft.pad_f.reserve(sizeof(float) * pad_f.size()));
    CTG_TRY(ft.resp_d.reserve(sizeof(double) * W));
    CTG_TRY(ft.tw_d.reserve(sizeof(double) * tw.size()));
    CTG_TRY(ft.pad_d.reserve(sizeof(double) * pad.size()));
    CTG_HIP(hipMemcpy(ft.resp_f.ptr, resp_f.data(), sizeof(float) * W, hipMemcpyHostToDevice));
    CTG_HIP(hipMemcpy(ft.tw_f.ptr, tw_f.data(), sizeof(float) * tw_f.size(), hipMemcpyHostToDevice));
    CTG_HIP(hipMemcpy(ft.pad_f.ptr, pad_f.data(), sizeof(float) * pad_f.size(), hipMemcpyHostToDevice));
    CTG_HIP(hipMemcpy(ft.resp_d.ptr, resp.data(), sizeof(double) * W, hipMemcpyHostToDevice));
    CTG_HIP(hipMemcpy(ft.tw_d.ptr, tw.data(), sizeof(double) * tw.size(), hipMemcpyHostToDevice));
    CTG_HIP(hipMemcpy(ft.pad_d.ptr, pad.data(), sizeof(double) * pad.size(), hipMemcpyHostToDevice));
    ft.W = W;
    ft.filter = filter;
    return CTG_OK;
}

}  // namespace ctg
