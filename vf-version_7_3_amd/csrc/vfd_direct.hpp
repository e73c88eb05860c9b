// vfd_direct.hpp -- a tick of a separable field as a direct convolution (FP32).
//
// A separable spectrum K^(kz,ky,kx) = scale gz gy gx is, along each axis, the
// DFT of a real even window; where the three windows are short the tick
//   v = scale px py pz (hz * hy * hx * u)
// is the linear convolution of the data with them, and two passes over the
// unpadded data do it:
//   dir_xy : u -> w   x and y windows, plane by plane
//   dir_z  : w -> v   z window, decay, and the chem update / downsample epilogue
// 16 bytes per voxel instead of the 104 of the five FFT passes (whose arrays
// hold the padded half spectrum), and no padding is ever transformed.
//
// dir_classify decides from the tables themselves, on every call: it inverts
// the three tables to windows and keeps the direct form only where they
// reproduce the tables (see there).  Its record says so to every later launch
// of the tick; fields without the form go through the FFT passes.
//
// Reference semantics: the operator of fftDiffuse3D (src/Diffusion/Diffusion.cu:
// 1622-1934) with a zero pad.
#pragma once
#include "vfd_passes.hpp"

namespace vfd {

__device__ __forceinline__ DirRecord* dir_record(const FieldDesc& fd, const DirDims& d) {
    return d.rec_off < 0 ? (DirRecord*)const_cast<void*>(fd.kspec) : (DirRecord*)((char*)fd.work + d.rec_off);
}

// --------------------------------------------------------------- classify
// One work-group per (axis, field): the axis' table t[k] (x: the half k <= P/2;
// y, z: all P entries) back to its window,
//   h_j = (1/P) sum_k t[k] cos(2 pi j k / P),  j <= J = min(kDirMaxR, (P-1)/2),
// and forward again: the axis has the direct form of radius R (the last j with
// |h_j| > 1e-13 max|h|) when every entry is reproduced to 1e-12 of the largest
// (the tables of vfd_gauss_spectrum are, to about 1e-15), the table is even,
// and no tap wraps around the box (R <= P - n).  Everything else -- wider
// windows, uneven or arbitrary tables, NaN -- gets radius -1.
// FP64 throughout.  A latency chain in a tick's first launch: the table and the
// box's cosines are staged in LDS (one entry and one cospi per thread), then
// 1024 threads are 32 taps x 32 slices of the frequencies in the inverse and a
// frequency each forward.
constexpr int kDirTaps = kDirMaxR + 1, kDirSlices = 32, kClassifyThreads = kDirTaps * kDirSlices;
static_assert(kDirTaps == 32, "a record's taps are one half wave");

__global__ void __launch_bounds__(kClassifyThreads)
dir_classify_kernel(const FieldBatch fb, DirDims d) {
    __shared__ double tl[kDirHalfMax + 1], ct[kDirHalfMax + 1];  // entries; cos(2 pi m / P)
    __shared__ double part[kDirSlices][kDirTaps];
    __shared__ double h[kDirTaps];
    __shared__ int bad_s;
    constexpr int NK = (kDirHalfMax + kClassifyThreads) / kClassifyThreads;  // frequencies per thread
    const int ax = blockIdx.x;
    const FieldDesc& fd = fb.f[blockIdx.y];
    const double* tab = (const double*)fd.kspec;
    DirRecord* rec = dir_record(fd, d);
    const int P = ax == 0 ? d.px : ax == 1 ? d.py : d.pz;
    const int n = ax == 0 ? d.nx : ax == 1 ? d.ny : d.nz;
    const double* t = tab + 1 + (ax == 0 ? 0 : ax == 1 ? d.px / 2 + 1 : d.px / 2 + 1 + d.py);
    const int K = P / 2;  // frequencies 0 .. K
    const int J = min(kDirMaxR, (P - 1) / 2);
    const int tid = threadIdx.x, j = tid % kDirTaps, sl = tid / kDirTaps;
    auto wrap = [&](int m) { return m >= P ? m - P : m; };
    auto cosine = [&](int m) { return ct[m <= K ? m : P - m]; };  // 0 <= m < P
    if (tid == 0) bad_s = 0;
    // the mirrored entries of an even table agree: their mean stands for both,
    // their difference is checked below
    double asym[NK];
#pragma unroll
    for (int i = 0; i < NK; ++i) {
        const int k = tid + i * kClassifyThreads;
        asym[i] = 0.0;
        if (k <= K) {
            const double a = t[k], b = ax == 0 || k == 0 ? a : t[P - k];
            tl[k] = 0.5 * (a + b);
            ct[k] = cospi(2.0 * (double)k / (double)P);
            asym[i] = fabs(a - b);
        }
    }
    __syncthreads();
    {
        // slice sl holds the frequencies sl, sl + 32, ...
        int m = j * sl % P;
        const int step = j * kDirSlices % P;
        double acc = 0.0;
#pragma unroll 4
        for (int k = sl; k <= K; k += kDirSlices) {
            const double w = (k == 0 || 2 * k == P) ? tl[k] : 2.0 * tl[k];
            acc = fma(w, cosine(m), acc);
            m = wrap(m + step);
        }
        part[sl][j] = acc;
    }
    __syncthreads();
    if (tid < kDirTaps) {
        double v = 0.0;
#pragma unroll
        for (int w = 0; w < kDirSlices; ++w) v += part[w][tid];
        h[tid] = tid <= J ? v / (double)P : 0.0;
    }
    __syncthreads();
    // gmax bounds every entry of an even window with these taps
    double gmax = 0.0;
#pragma unroll
    for (int i = 0; i < kDirTaps; ++i) gmax += (i ? 2.0 : 1.0) * fabs(h[i]);
    const double tol = 1e-12 * gmax;
    bool bad = !(gmax <= 1e30);  // out of FP32's range, NaN
#pragma unroll
    for (int i = 0; i < NK; ++i) {
        const int k = tid + i * kClassifyThreads;
        if (k <= K) {
            double r = h[0];
            int m = k;
#pragma unroll 8
            for (int q = 1; q < kDirTaps; ++q) {
                r = fma(2.0 * h[q], cosine(m), r);
                m = wrap(m + k);
            }
            bad |= !(fabs(r - tl[k]) <= tol) || !(asym[i] <= tol);  // also NaN
        }
    }
    if (bad) bad_s = 1;
    __syncthreads();
    if (tid < kWave) {  // one wave: lanes 0 .. 31 hold a tap each
        // the taps go to FP32 with their sum near 1 (within 0.75 .. 1.5, where a
        // normalized window's is already), the power of two back into the gain: a
        // table may hold any part of the kernel's magnitude in any of its factors
        int e2 = 0;
        if (gmax > 0.0 && frexp(gmax, &e2) < 0.75) --e2;
        const double v = tid < kDirTaps ? ldexp(h[tid], -e2) : 0.0;
        double hmax = fabs(v);
        for (int m = kDirTaps / 2; m > 0; m >>= 1) hmax = fmax(hmax, __shfl_xor(hmax, m));
        const unsigned long long big = __ballot(fabs(v) > 1e-13 * hmax) & 0xffffffffull;
        const int R = big ? 63 - __builtin_clzll(big) : 0;
        const bool in = tid <= R;
        // taps rounded to FP32 sum to sr where the exact ones sum to se: the z
        // pass applies se / sr, so the window conserves mass (taps of one sign)
        const bool pos = __ballot(in && tid < kDirTaps && !(v >= 0.0)) == 0;
        double se = in && tid < kDirTaps ? (tid ? 2.0 : 1.0) * v : 0.0;
        double sr = in && tid < kDirTaps ? (tid ? 2.0 : 1.0) * (double)(float)v : 0.0;
        for (int m = kDirTaps / 2; m > 0; m >>= 1) {
            se += __shfl_xor(se, m);
            sr += __shfl_xor(sr, m);
        }
        if (tid < kDirTaps) rec->ax[ax].tap[tid] = in ? (float)v : 0.0f;
        if (tid == 0) {
            rec->ax[ax].gain = ldexp(pos && sr > 0.0 ? se / sr : 1.0, e2);
            rec->ax[ax].radius = !bad_s && R <= P - n ? R : -1;
            if (ax == 0) rec->scale = tab[0] * (double)d.px * (double)d.py * (double)d.pz;
        }
    }
}

// ------------------------------------------------------------- the passes
// Work-groups of 256 threads march along one axis (y, or z in dir_z) over a
// strip of TX columns, B = 2048 / TX rows a batch, 8 outputs per thread and
// batch.  The rows the march convolves sit in an LDS ring of B + 2 RB4 rows; a
// thread takes 8 outputs of one column from the 8 + 2 RB4 ring rows around
// them (conflict-free: a wave reads 64 columns of one row), so a ring value is
// read (8 + 2 RB4) / 8 times instead of 2 R + 1.  The taps are wave-uniform and
// stay in scalar registers; RB is the compile-time bound on the radius (the
// taps beyond R are zero), and RB4 = RB rounded up to 4 keeps every run of
// rows or columns 16-byte aligned.
constexpr int kDirThreads = 256;
constexpr int kDirOut = 8;  // outputs per thread and batch
constexpr int dir_r4(int rb) { return (rb + 3) / 4 * 4; }
constexpr int dir_batch(int tx) { return kDirThreads * kDirOut / tx; }
constexpr int dir_ring_rows(int tx, int rb) { return dir_batch(tx) + 2 * dir_r4(rb); }

// The radius bounds that form their outputs in pairs (DirTaps<RB, true>): where
// the pass is bound by its vector instructions.  x-y of 4 fields 512x512x128, one
// by one against in pairs: R = 6 235 / 233 us (the memory's time either way), 8
// 243 / 237, 12 295 / 262, 16 351 / 312, 20 450 / 404, 24 504 / 462, 31 615 / 573;
// z 212 / 211 at 12, 250 / 236 at 20, 310 / 281 at 31; a tick of 8 fields
// 1024x512x128 (R 6 - 19) 1950 -> 1811.  Windows narrower than 8 fall off too
// fast from tap to tap for their differences to be small: beside a value 1000
// times its own, an output at R = 1 lost 1e-5 of itself.  (A wide window with
// such a step errs by 1e-7 of the step times the largest value, as the FFT
// passes do.)  Against 64 bits a tick's rel-L2 is 6.2e-8 either way.
constexpr bool dir_pairs(int rb) { return rb >= 8; }

template <int RB, bool PAIRS = dir_pairs(RB)> struct DirTaps {
    float t[RB + 1];
    __device__ __forceinline__ void load(const DirAxis* a) {
#pragma unroll
        for (int j = 0; j <= RB; ++j)
            t[j] = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, a->tap[j])));
    }
};

// The 8 outputs of a thread, each as two partial sums: inputs arrive in order,
// so the taps first grow to the centre (lo) and then shrink (hi); one running
// sum would round every term after the centre at the full magnitude of the
// result (rel-L2 of a tick 1.0e-7 instead of 0.7e-7).
template <bool PAIRS> struct DirSums {
    float lo[kDirOut], hi[kDirOut];
    __device__ __forceinline__ DirSums() {
#pragma unroll
        for (int v = 0; v < kDirOut; ++v) lo[v] = hi[v] = 0.0f;
    }
    __device__ __forceinline__ float operator[](int v) const { return lo[v] + hi[v]; }
    __device__ __forceinline__ void pin() {
#pragma unroll
        for (int v = 0; v < kDirOut; ++v) asm volatile("" : "+v"(lo[v]), "+v"(hi[v]));
    }
    // input elements idx, idx + 1 (0 .. 7 + 2 RB4) of the run that starts RB4
    // before the first of the 8 outputs
    template <int RB> __device__ __forceinline__ void add(const DirTaps<RB>& tp, float i0, float i1, int idx) {
        add1<RB>(tp, i0, idx);
        add1<RB>(tp, i1, idx + 1);
    }
    template <int RB> __device__ __forceinline__ void add1(const DirTaps<RB>& tp, float in, int idx) {
        constexpr int RB4 = dir_r4(RB);
#pragma unroll
        for (int v = 0; v < kDirOut; ++v) {
            const int k = idx - RB4 - v;
            if (k < -RB || k > RB) continue;
            float& a = k <= 0 ? lo[v] : hi[v];
            a = fmaf(tp.t[k < 0 ? -k : k], in, a);
        }
    }
};

// Outputs are formed in pairs from pairs of inputs (e, o), o one after e: with
// h the window,
//   y[0] = sum h[2i] (e + o)[i] + sum (h[2i+1] - h[2i]) o[i]
//   y[1] = sum h[2i] (e + o)[i] + sum (h[2i-1] - h[2i]) e[i],
// of which the first sum is shared: 3 R + 2 products a pair and one sum an input
// pair instead of 4 R + 2 products.  The differences of an even window are two
// lists, of which the second sum runs one forwards and the third backwards.
template <int RB> struct DirTaps<RB, true> {
    static constexpr int NE = RB / 2 + 1, NB = (RB + 1) / 2;
    float e[NE];      // h[2i]
    float up[NE];     // h[2i+1] - h[2i]
    float dn[NB + 1]; // h[2i-1] - h[2i], i >= 1
    __device__ __forceinline__ void load(const DirAxis* a) {
        auto uni = [](float v) {
            return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
        };
        auto h = [&](int j) { return j <= RB ? a->tap[j] : 0.0f; };
#pragma unroll
        for (int i = 0; i < NE; ++i) {
            e[i] = uni(h(2 * i));
            up[i] = uni(h(2 * i + 1) - h(2 * i));
        }
        dn[0] = 0.0f;
#pragma unroll
        for (int i = 1; i <= NB; ++i) dn[i] = uni(h(2 * i - 1) - h(2 * i));
    }
};

// the outputs as 4 pairs: the shared sum in two parts, and the differences' sums
template <> struct DirSums<true> {
    float lo[kDirOut / 2], hi[kDirOut / 2], d[kDirOut];
    __device__ __forceinline__ DirSums() {
#pragma unroll
        for (int m = 0; m < kDirOut / 2; ++m) lo[m] = hi[m] = d[2 * m] = d[2 * m + 1] = 0.0f;
    }
    __device__ __forceinline__ float operator[](int v) const { return lo[v / 2] + hi[v / 2] + d[v]; }
    __device__ __forceinline__ void pin() {
#pragma unroll
        for (int m = 0; m < kDirOut / 2; ++m)
            asm volatile("" : "+v"(lo[m]), "+v"(hi[m]), "+v"(d[2 * m]), "+v"(d[2 * m + 1]));
    }
    // input elements idx, idx + 1 (idx even, 0 .. 6 + 2 RB4) of the run that
    // starts RB4 before the first of the 8 outputs
    template <int RB> __device__ __forceinline__ void add(const DirTaps<RB>& tp, float ev, float od, int idx) {
        constexpr int RB4 = dir_r4(RB);
        const int j = idx / 2 - RB4 / 2;
        const float s = ev + od;
#pragma unroll
        for (int m = 0; m < kDirOut / 2; ++m) {
            const int i = j - m, n = i < 0 ? -i : i;
            if (2 * n <= RB) {
                float& a = i <= 0 ? lo[m] : hi[m];
                a = fmaf(tp.e[n], s, a);
                float& u = i >= 0 ? d[2 * m] : d[2 * m + 1];
                u = fmaf(tp.up[n], i >= 0 ? od : ev, u);
                if (i == 0) d[2 * m + 1] = fmaf(tp.up[0], ev, d[2 * m + 1]);
            }
            if (n > 0 && 2 * n - 1 <= RB) {
                float& u = i < 0 ? d[2 * m] : d[2 * m + 1];
                u = fmaf(tp.dn[n], i < 0 ? od : ev, u);
            }
        }
    }
};

// 8 outputs of one ring column: `start` is the ring row of the first input
template <int TX, int RB>
__device__ __forceinline__ void dir_ring_conv(DirSums<dir_pairs(RB)>& acc, const DirTaps<RB>& tp, const float* ring, int start,
                                              int col) {
    constexpr int RB4 = dir_r4(RB), RS = dir_ring_rows(TX, RB), NB = (kDirOut + 2 * RB4) / 8;
    float in[2][8];
    auto fetch = [&](int blk) {
        int row = start + 8 * blk;  // wave-uniform; rings are whole 8-row blocks
        row = row >= RS ? row - RS : row;
        const float* p = ring + row * TX + col;
#pragma unroll
        for (int e = 0; e < 8; ++e) in[blk & 1][e] = p[e * TX];
    };
    fetch(0);
#pragma unroll
    for (int blk = 0; blk < NB; ++blk) {
        if (blk + 1 < NB) fetch(blk + 1);
#pragma unroll
        for (int e = 0; e < 8; e += 2) acc.template add<RB>(tp, in[blk & 1][e], in[blk & 1][e + 1], 8 * blk + e);
        // Sums formed here, reads one block ahead: left alone, the compiler forms
        // one output after the other (sinking the sums to their stores), with
        // the whole run's inputs live (122 VGPRs at radius 31 instead of 80).
        acc.pin();
    }
}

// four floats at element offset `off` of a row segment of which `left` elements
// are inside (<= 0: none); a chunk that is cut takes single loads
template <int A> __device__ __forceinline__ float4 dir_ld4(rsrc_t r, unsigned off, int left) {
    float4 q = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, left >= 4 ? off * 4u : kBufOOB, 0, A));
    if (left > 0 && left < 4) {
        q.x = BufOps<float>::ld_r<A>(r, off * 4u);
        q.y = BufOps<float>::ld_r<A>(r, left > 1 ? off * 4u + 4u : kBufOOB);
        q.z = BufOps<float>::ld_r<A>(r, left > 2 ? off * 4u + 8u : kBufOOB);
    }
    return q;
}

// x and y windows of one strip: TX columns from x0, rows [y0, y1) of plane z.
// Bound by vector instructions, 0.96 of its cycles: 8 fields 1024x512x128 (R 6 - 19)
// in 1.02 ms, 4.2 TB/s (1.12 ms one output at a time).
template <int TX, int RB>
__device__ __forceinline__ void dir_xy_strip(float* lds, const DirRecord* rec, rsrc_t rin, rsrc_t rw, const DirDims& d,
                                             int z, int x0, int y0, int y1) {
    constexpr int RB4 = dir_r4(RB), B = dir_batch(TX), RS = dir_ring_rows(TX, RB);
    constexpr int W4 = (TX + 2 * RB4) / 4;           // 16-byte chunks of a raw row
    constexpr int NLD = (B * W4 + kDirThreads - 1) / kDirThreads;
    constexpr int M0 = (2 * RB4 + B - 1) / B;        // batches before the first output
    // raw rows: the even chunks first, then the odd ones, so that the 16-byte
    // reads of threads 8 columns apart are adjacent
    float4* raw = (float4*)lds;
    float* ring = lds + B * W4 * 4;
    const int tid = threadIdx.x;
    DirTaps<RB> tx, ty;
    tx.load(&rec->ax[0]);
    ty.load(&rec->ax[1]);
    const int ylo = max(0, y0 - RB4), yhi = min(d.ny, y1 + RB4);
    int yb = y0 + RB4 - M0 * B;  // first input row of the batch; its outputs start at yb - RB4
    const int nb = M0 + (y1 - y0 + B - 1) / B;
    const unsigned plane = (unsigned)z * (unsigned)d.ny * (unsigned)d.nx;
    float4 q[NLD];
    // element offset of each chunk from the batch's first row, columns outside
    // the data (whole 16-byte chunks on the left, the row's end on the right)
    // masked once; where the whole batch is inside the chunk of rows a load is
    // this offset and the wave's scalar base
    unsigned voff[NLD];
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
        const int idx = tid + i * kDirThreads, r = idx / W4, x = x0 - RB4 + 4 * (idx % W4);
        voff[i] = (NLD * kDirThreads == B * W4 || r < B) && x >= 0 && x + 4 <= d.nx ? ((unsigned)(r * d.nx + x)) * 4u : kBufOOB;
    }
    const bool cut = x0 + TX + RB4 > d.nx && d.nx % 4 != 0;  // a chunk of the strip crosses the row's end
    auto fetch = [&](int yb) {
        if (yb >= ylo && yb + B <= yhi && !cut) {
            const int base = __builtin_amdgcn_readfirstlane((int)((plane + (unsigned)yb * (unsigned)d.nx) * 4u));
#pragma unroll
            for (int i = 0; i < NLD; ++i)
                q[i] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rin, voff[i], base, kCacheDefault));
            return;
        }
#pragma unroll
        for (int i = 0; i < NLD; ++i) {
            const int idx = tid + i * kDirThreads, r = idx / W4, c = idx % W4;
            const int y = yb + r, x = x0 - RB4 + 4 * c;
            const bool ok = (NLD * kDirThreads == B * W4 || r < B) && y >= ylo && y < yhi && x >= 0;
            q[i] = dir_ld4<kCacheDefault>(rin, ok ? plane + (unsigned)y * (unsigned)d.nx + (unsigned)x : 0u,
                                          ok ? d.nx - x : 0);
        }
    };
    const int xr = tid / (TX / 8), xt = tid % (TX / 8);          // x phase: row of the batch, 8 columns
    const int col = tid % TX, rg = __builtin_amdgcn_readfirstlane(tid / TX);  // y phase: column, 8 rows
    const unsigned xoff = x0 + col < d.nx ? (unsigned)(x0 + col) * 4u : kBufOOB;
    int pos = 0;  // ring row of the batch's first row
    fetch(yb);
    for (int b = 0; b < nb; ++b) {
#pragma unroll
        for (int i = 0; i < NLD; ++i) {
            const int idx = tid + i * kDirThreads, r = idx / W4, c = idx % W4;
            if (NLD * kDirThreads == B * W4 || r < B) raw[r * W4 + (c & 1) * (W4 / 2) + (c >> 1)] = q[i];
        }
        __syncthreads();
        if (b + 1 < nb) fetch(yb + B);
        {
            DirSums<dir_pairs(RB)> acc;
#pragma unroll
            for (int i = 0; i < (kDirOut + 2 * RB4) / 4; ++i) {
                const float4 u = raw[xr * W4 + (i & 1) * (W4 / 2) + xt + (i >> 1)];
                acc.template add<RB>(tx, u.x, u.y, 4 * i);
                acc.template add<RB>(tx, u.z, u.w, 4 * i + 2);
            }
            int row = pos + xr;
            row = row >= RS ? row - RS : row;
            float4* dst = (float4*)(ring + row * TX + 8 * xt);
            dst[0] = float4{acc[0], acc[1], acc[2], acc[3]};
            dst[1] = float4{acc[4], acc[5], acc[6], acc[7]};
        }
        __syncthreads();
        if (b >= M0) {
            int start = pos + 8 * rg - 2 * RB4;
            start = start < 0 ? start + RS : start >= RS ? start - RS : start;
            DirSums<dir_pairs(RB)> acc;
            dir_ring_conv<TX, RB>(acc, ty, ring, start, col);
            const int yo = yb - RB4 + 8 * rg;  // wave-uniform, as the rows' bases
            unsigned base = (plane + (unsigned)yo * (unsigned)d.nx) * 4u;
#pragma unroll
            for (int v = 0; v < kDirOut; ++v) {
                if (yo + v < y1)
                    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, acc[v]), rw, xoff, (int)base,
                                                          kCacheDefault);
                base += (unsigned)d.nx * 4u;
            }
        }
        yb += B;
        pos += B;
        pos = pos >= RS ? pos - RS : pos;
    }
}

// The radius bounds compiled: a field takes the smallest that holds its radius.
// An even step wastes at most one tap a side (the odd bounds as well: within 2 %
// either way); beyond 20 (the radius of
// D = 5 patch^2 a tick is 19) steps of 4.
#define VFD_DIR_RADII(X) X(2) X(4) X(6) X(8) X(10) X(12) X(14) X(16) X(18) X(20) X(24) X(28) X(31)

constexpr unsigned dir_xy_lds(int tx, int rb) {
    return (unsigned)(dir_batch(tx) * (tx + 2 * dir_r4(rb)) + dir_ring_rows(tx, rb) * tx) * 4u;
}
constexpr unsigned dir_z_lds(int tx, int rb) { return (unsigned)(dir_ring_rows(tx, rb) * tx) * 4u; }

template <int TX>
__global__ void __launch_bounds__(kDirThreads) dir_xy_kernel(const FieldBatch fb, DirDims d) {
    extern __shared__ __align__(16) float dir_lds[];
    // the x tiles of one (plane, y chunk, field) get ids 8 apart: ids are dealt
    // round-robin to the 8 XCDs, so tiles sharing halo columns share an L2
    const unsigned lin = blockIdx.x, nt = d.xtiles;
    const unsigned grp = lin / (8u * nt) * 8u + lin % 8u;
    const unsigned tile = lin / 8u % nt;
    const unsigned z = grp % (unsigned)d.nz, rest = grp / (unsigned)d.nz;
    const unsigned ch = rest % d.ychunks, f = rest / d.ychunks;
    if (f >= d.nfields) return;  // padding ids
    const FieldDesc& fd = fb.f[f];
    const DirRecord* rec = dir_record(fd, d);
    if (!dir_form(rec)) return;  // the FFT passes do it
    const int R = __builtin_amdgcn_readfirstlane(max(rec->ax[0].radius, rec->ax[1].radius));
    const rsrc_t rin = make_rsrc(fd.in, d.bytes), rw = make_rsrc(fd.work, d.bytes);
    const int x0 = (int)tile * TX, y0 = (int)ch * d.yrows, y1 = min(d.ny, y0 + d.yrows);
    if (R > d.max_radius) return;  // the launch's LDS holds windows up to max_radius
#define VFD_GO(RB) \
    if (R <= RB) return dir_xy_strip<TX, RB>(dir_lds, rec, rin, rw, d, (int)z, x0, y0, y1);
    VFD_DIR_RADII(VFD_GO)
#undef VFD_GO
}

// Bound by HBM: 8 fields 1024x512x128 in 0.82 ms, 5.2 TB/s of the 6.4 that a copy
// reaches (its loads and stores alone take 0.74).
// z window of TX columns of the flattened (y, x) plane from c0
template <int TX, int RB, bool VIS, int POL>
__device__ __forceinline__ void dir_z_strip(float* ring, const FieldDesc& fd, const DirRecord* rec, const DirDims& d,
                                            unsigned c0) {
    constexpr int RB4 = dir_r4(RB), B = dir_batch(TX), RS = dir_ring_rows(TX, RB);
    constexpr int W4 = TX / 4, NLD = B * W4 / kDirThreads;
    constexpr int M0 = (2 * RB4 + B - 1) / B;
    const int tid = threadIdx.x;
    const rsrc_t rw = make_rsrc(fd.work, d.bytes), rout = make_rsrc(fd.out, d.bytes);
    DirTaps<RB> tz;
    tz.load(&rec->ax[2]);
    // the decay (and the taps' power of two and FP32 rounding, see classify) as hi + lo
    const double fac = rec->scale * rec->ax[0].gain * rec->ax[1].gain * rec->ax[2].gain;
    const float fh = (float)fac, fl = (float)(fac - (double)fh);
    const unsigned np = (unsigned)d.ny * (unsigned)d.nx;
    const int lr = tid / W4, lc = tid % W4;  // loads: row, 16-byte chunk
    constexpr int LSTEP = kDirThreads / W4;
    const unsigned lcol = c0 + 4u * lc;
    const int left = lcol < np ? (int)min(np - lcol, 4u) : 0;
    float4 q[NLD];
    auto fetch = [&](int zb) {
#pragma unroll
        for (int i = 0; i < NLD; ++i) {
            const int z = zb + lr + i * LSTEP;
            const bool ok = z >= 0 && z < d.nz;
            q[i] = dir_ld4<POL>(rw, ok ? (unsigned)z * np + lcol : 0u, ok ? left : 0);
        }
    };
    const int cc = tid % TX, rg = __builtin_amdgcn_readfirstlane(tid / TX);
    const unsigned col = c0 + (unsigned)cc;
    const bool live = col < np;
    const bool upd = fd.delta != nullptr;
    const rsrc_t rdel = make_rsrc(fd.delta, upd ? d.bytes : 0ul);
    int vs = 1, vH = 0, vW = 0, vD = 0;
    unsigned vbase = 0;
    bool vcol = false;
    [[maybe_unused]] rsrc_t rvis = make_rsrc(nullptr, 0ul);
    if constexpr (VIS) {
        vs = fd.vis_stride;
        vD = d.nz / vs; vH = d.ny / vs; vW = d.nx / vs;
        const int y = (int)(col / (unsigned)d.nx), x = (int)(col % (unsigned)d.nx);
        vcol = live && y % vs == 0 && x % vs == 0 && y / vs < vH && x / vs < vW;
        vbase = vcol ? (unsigned)(y / vs) * (unsigned)vW + (unsigned)(x / vs) : 0u;
        rvis = make_rsrc(fd.vis, (unsigned long)vD * vH * vW * 4ul);
    }
    int zb = RB4 - M0 * B, pos = 0;
    const int nb = M0 + (d.nz + B - 1) / B;
    fetch(zb);
    for (int b = 0; b < nb; ++b) {
#pragma unroll
        for (int i = 0; i < NLD; ++i) {
            int row = pos + lr + i * LSTEP;
            row = row >= RS ? row - RS : row;
            ((float4*)(ring + row * TX))[lc] = q[i];
        }
        __syncthreads();
        if (b + 1 < nb) fetch(zb + B);
        const int zo = zb - RB4 + 8 * rg;
        if (b >= M0 && zo < d.nz) {
            int start = pos + 8 * rg - 2 * RB4;
            start = start < 0 ? start + RS : start >= RS ? start - RS : start;
            unsigned off = ((unsigned)zo * np + col) * 4u;
            // the deltas are on their way while the window is summed
            float dl[kDirOut];
            if (upd) {
#pragma unroll
                for (int v = 0; v < kDirOut; ++v)
                    dl[v] = BufOps<float>::ld_r<kStream>(rdel, live && zo + v < d.nz ? off + (unsigned)v * np * 4u : kBufOOB);
            }
            DirSums<dir_pairs(RB)> acc;
            dir_ring_conv<TX, RB>(acc, tz, ring, start, cc);
#pragma unroll
            for (int v = 0; v < kDirOut; ++v) {
                const bool ok = live && zo + v < d.nz;
                const float t = acc[v];
                float o = fmaf(fh, t, fl * t);
                if constexpr (VIS) {
                    if (vcol && ok && (zo + v) % vs == 0 && (zo + v) / vs < vD) {
                        float s = o * fd.vis_scale;
                        if (s > 1.0f) s = 1.0f;
                        BufOps<float>::st_r(s, rvis, ((unsigned)((zo + v) / vs) * (unsigned)vH * (unsigned)vW + vbase) * 4u);
                    }
                }
                if (upd) {
                    o = upd_level(dl[v], o, fd.decay);
                    BufOps<float>::st_r<kStream>(0.0f, rdel, ok ? off : kBufOOB);
                }
                BufOps<float>::st_r<kStream>(o, rout, ok ? off : kBufOOB);
                off += np * 4u;
            }
        }
        __syncthreads();
        zb += B;
        pos += B;
        pos = pos >= RS ? pos - RS : pos;
    }
}

// POL: cache policy of the loads (see launch_dir_z)
template <int TX, bool VIS, int POL>
__global__ void __launch_bounds__(kDirThreads) dir_z_kernel(const FieldBatch fb, DirDims d) {
    extern __shared__ __align__(16) float dir_lds[];
    const FieldDesc& fd = fb.f[blockIdx.y];
    const DirRecord* rec = dir_record(fd, d);
    if (!dir_form(rec)) return;  // the FFT passes do it
    const int R = __builtin_amdgcn_readfirstlane(rec->ax[2].radius);
    if (R > d.max_radius) return;
#define VFD_GO(RB) \
    if (R <= RB) return dir_z_strip<TX, RB, VIS, POL>(dir_lds, fd, rec, d, blockIdx.x * (unsigned)TX);
    VFD_DIR_RADII(VFD_GO)
#undef VFD_GO
}

}  // namespace vfd
