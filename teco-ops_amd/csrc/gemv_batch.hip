// gemv_batch.hip — weight products for a batch of rows of x: one stream of W
// for up to 64 rows.
//
//   y[b, n] = T( sum_k W[n, k] x[b, k] )            fp32 accumulation
//   y[b, n] = fp16( s[n] sum_k Wq[n, k] x[b, k] )   int8 weights
//
// gfx950 design: Y^T = W X^T on v_mfma_f32_16x16x32_{f16,bf16}; a wave owns
// WR rows of W and all XR columns (rows of x), so each W value is read
// from HBM once whatever the batch.  W and x go from memory straight into LDS
// (global_load_lds_dwordx4, no registers) in stages of 256 bytes per row of
// W, D stages in a ring, and the MFMA operands are 16-byte LDS reads.  What
// bounds it is HBM for W and, for few rows per workgroup, the L2 -> LDS
// traffic of x (every workgroup copies all of x); both want whole row
// segments per copy:
//   * a copy instruction moves four 256-byte row segments (1 KiB).  Loading
//     the operands straight from memory instead touches 16 rows x 64 bytes
//     per instruction: [28672, 4096] bf16, batch 16, 60-76 µs for that over
//     12 launch shapes, 40-53 µs with W copied and x loaded, 36-40 µs with
//     both copied; batch 64 112-170 / 85-140 / 43-48 µs.
//   * RS waves of a workgroup take different rows and share the x stage; KS
//     groups of waves take different ranges of K and add their sums through
//     LDS at the end, so that few rows still fill the chip with copies in
//     flight.
// The 16-byte chunk c of row r sits at chunk c ^ (r % 8) of its LDS row, so
// that the 16 rows a fragment read touches fall on distinct banks; the copy's
// source address carries the permutation.  Chunks past K are copied from a
// zero constant, for W and x alike, so any K in whole chunks works.
#include "gemv_batch.h"

#include "common.h"
#include "device.h"

namespace {

using namespace tecoops::dev;
using tecoops::gemv_batch_rows;

typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

template <typename T> struct Mma16;
template <> struct Mma16<f16> {
    static __device__ __forceinline__ f32x4_t run(u32x4_t a, u32x4_t b, f32x4_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a),
                                                      __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
    }
};
template <> struct Mma16<bf16> {
    static __device__ __forceinline__ f32x4_t run(u32x4_t a, u32x4_t b, f32x4_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                       __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
    }
};

// 16 zero bytes: the source of chunks past K.
__device__ __attribute__((aligned(16))) const uint32_t kZero16[4] = {0u, 0u, 0u, 0u};

// Global -> LDS with no register staging: 16 bytes per lane into
// dst + 16 * lane (dst wave-uniform, in M0).  STREAM: read once (W), so not
// to displace x in L2.  Inline assembly, so that the compiler does not wait
// for every copy in flight before each LDS read; the copies are ordered by
// wait_copies().  No other code of these kernels uses M0 (build.py checks
// it in the assembly).
template <bool STREAM>
__device__ __forceinline__ void dma16(const void *src, void *dst) {
    const uint32_t lds = static_cast<uint32_t>(
        reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) void *)(dst)));
    if constexpr (STREAM)
        asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off nt" ::"v"(src), "s"(lds)
                     : "memory");
    else
        asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds)
                     : "memory");
}

// Waits until this wave has at most N younger vector-memory operations in
// flight.  Every copy counts as one; any other load in flight only makes the
// wait stricter.
template <int N>
__device__ __forceinline__ void wait_copies() {
    static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
    __builtin_amdgcn_s_waitcnt(((N >> 4) << 14) | 0x0F70 | (N & 15));
    asm volatile("" ::: "memory");
}

// 16 int8 weights -> 16 fp16 values holding them exactly: bytes of w + 128
// under the exponent of 1024.0, then minus 1152.
__device__ __forceinline__ void widen_i8x16(u32x4_t q, u32x4_t &lo8, u32x4_t &hi8) {
    const half2_t bias = {static_cast<_Float16>(-1152.0f), static_cast<_Float16>(-1152.0f)};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint32_t u = q[e] ^ 0x80808080u;
        const half2_t a = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) + bias;
        const half2_t b = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) + bias;
        u32x4_t &d = e < 2 ? lo8 : hi8;
        d[2 * (e & 1)] = __builtin_bit_cast(uint32_t, a);
        d[2 * (e & 1) + 1] = __builtin_bit_cast(uint32_t, b);
    }
}

// Sizes of a workgroup's stages.  XR: rows of x staged; WR: rows of W per wave.
template <bool I8, int XR, int WR, int RS, int KS>
struct Shape {
    static constexpr int NW = RS * KS;
    static constexpr int CT = (XR + 15) / 16;      // column tiles of 16
    static constexpr int RT = (WR + 15) / 16;      // row tiles of 16
    static constexpr int WB = WR * 256;            // W bytes of a wave's stage
    static constexpr int WC = WR / 4;              // W copies of a wave and stage
    static constexpr int XROW = I8 ? 512 : 256;    // x bytes of a row and stage
    static constexpr int XB = XR * XROW;           // x bytes of a K part's stage
    static constexpr int SB = NW * WB + KS * XB;   // bytes of a stage
    static constexpr int XN = XB / 1024;           // x copies of a K part and stage
    static constexpr int XC = (XN + RS - 1) / RS;  // ... of a wave
    static constexpr int PER = WC + XC;            // copies of a wave and stage
    static constexpr int FIT = static_cast<int>(tecoops::kLdsMax) / SB;
    static constexpr int D = FIT > 4 ? 4 : FIT;    // stages in the ring
    static constexpr int RED = NW * RT * CT * 1024;  // partial sums (KS > 1)
    static constexpr size_t LDS = D * SB > RED ? D * SB : RED;
    static_assert(XR == 4 || XR == 8 || XR % 16 == 0, "whole column tiles, or part of one");
    static_assert(WR == 8 || WR % 16 == 0, "whole row tiles, or half of one");
    static_assert(D < 3 || (D - 2) * PER < 64, "vmcnt");
};

// The wave's copies of stage i + D - 1 are issued while stage i is consumed.
// With RS > 1 one barrier per stage publishes the x copies of the other waves
// and, since every wave passes it after reading stage i - 1, frees the slot
// the next copies go to.  With RS = 1 a wave reads only what it copied.
template <typename T, bool I8, int XR, int WR, int RS, int KS>
__global__ void __launch_bounds__(RS * KS * 64)
gemv_batch_kernel(const char *__restrict__ W, const uint16_t *__restrict__ scales,
                  const char *__restrict__ x, uint16_t *__restrict__ y, int N, int K, int B,
                  int pairs) {
    using S = Shape<I8, XR, WR, RS, KS>;
    constexpr int NW = S::NW, CT = S::CT, RT = S::RT, D = S::D, WC = S::WC, XC = S::XC, PER = S::PER;
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rs = wave % RS, kp = wave / RS;
    const int n0 = (blockIdx.x * RS + rs) * WR;
    const int g = lane >> 4, c = lane & 15;
    const int kw = I8 ? K / 16 : K / 8, kx = K / 8;  // 16-byte chunks of a row of W / x
    constexpr int XCH = I8 ? 32 : 16;                // x chunks of a row and stage
    const int nst = ((kw + 15) / 16 + KS - 1) / KS;  // stages of a K part
    // W copy m: rows 4m + lane / 16, chunk slot lane % 16
    const char *wsrc[WC];
    int wch[WC];
#pragma unroll
    for (int m = 0; m < WC; ++m) {
        const int row = 4 * m + (lane >> 4);
        wsrc[m] = W + static_cast<long long>(min(n0 + row, N - 1)) * kw * 16;
        wch[m] = kp * nst * 16 + ((lane & 15) ^ (row & 7));
    }
    // x copy q: rows (1024 / XROW) q + lane / XCH, slot lane % XCH; a K part's
    // copies are dealt to its RS waves (the last ones repeated to fill up)
    const char *xsrc[XC];
    int xch[XC], xdst[XC];
#pragma unroll
    for (int m = 0; m < XC; ++m) {
        const int q = (rs + m * RS) % S::XN;
        const int row = (1024 / S::XROW) * q + lane / XCH;
        xsrc[m] = x + static_cast<long long>(min(row, B - 1)) * kx * 16;
        xch[m] = kp * nst * XCH + ((lane % XCH) ^ (row & 7));
        xdst[m] = q * 1024;
    }
    f32x4_t acc[RT][CT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int t = 0; t < CT; ++t) acc[r][t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    // Workgroups start their sweep of K at different stages, so that the
    // requests in flight spread over the HBM channels (rows a power of two
    // bytes apart start on the same one).  The step is odd: nst mostly is a
    // power of two, and an even step would leave most starts unused (bf16
    // batch 8, steps of 2 / 3 stages: [16384, 8192] 81.0 / 47.6 µs, [32768,
    // 4096] 44.3 / 42.8; steps of 8 / 9 at 128 rows [32768, 4096] 51.2 / 43.1).
    const int rot = (blockIdx.x * (RS | 1) + (RS == 1 ? wave : 0)) % nst;
    char *wbuf = lds + wave * S::WB;
    char *xbuf = lds + NW * S::WB + kp * S::XB;
    const auto slot = [&](int i) { return __builtin_amdgcn_readfirstlane((i % D) * S::SB); };
    const auto load = [&](int i) {
        const int st = i + rot < nst ? i + rot : i + rot - nst;
        const int so = slot(i);
#pragma unroll
        for (int m = 0; m < XC; ++m) {
            const int q = xch[m] + XCH * st;
            dma16<false>(q < kx ? static_cast<const void *>(xsrc[m] + 16 * q)
                                : static_cast<const void *>(kZero16),
                         xbuf + so + xdst[m]);
        }
#pragma unroll
        for (int m = 0; m < WC; ++m) {
            const int q = wch[m] + 16 * st;
            dma16<true>(q < kw ? static_cast<const void *>(wsrc[m] + 16 * q)
                               : static_cast<const void *>(kZero16),
                        wbuf + so + m * 1024);
        }
    };
    // this lane's fragment rows: W row c of a row tile, x row c of a column
    // tile (in a tile of fewer rows the lanes past them repeat its rows, and
    // what they produce is never stored)
    const int wc = WR < 16 ? c & 7 : c, xc = XR < 16 ? c & (XR - 1) : c;
    const int wsw = wc & 7, xsw = xc & 7;
    const char *wl = wbuf + wc * 256, *xl = xbuf + xc * S::XROW;
#pragma unroll
    for (int d = 0; d < D - 1; ++d)
        if (d < nst) load(d);
    for (int i = 0; i < nst; ++i) {
        // stages i + 1 .. min(i + D - 2, nst - 1) may still be in flight
        if (D > 3 && i + 2 < nst) wait_copies<(D > 3 ? 2 : 1) * PER>();
        else if (D > 2 && i + 1 < nst) wait_copies<PER>();
        else wait_copies<0>();
        if constexpr (RS > 1) __syncthreads();
        if (i + D - 1 < nst) load(i + D - 1);
        const int so = slot(i);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            u32x4_t a[RT];
#pragma unroll
            for (int r = 0; r < RT; ++r)
                a[r] = *reinterpret_cast<const u32x4_t *>(wl + so + r * 4096 + 16 * ((4 * u + g) ^ wsw));
            if constexpr (I8) {
                u32x4_t b0[CT], b1[CT];
#pragma unroll
                for (int t = 0; t < CT; ++t) {
                    const char *p = xl + so + t * 16 * S::XROW;
                    b0[t] = *reinterpret_cast<const u32x4_t *>(p + 16 * ((8 * u + 2 * g) ^ xsw));
                    b1[t] = *reinterpret_cast<const u32x4_t *>(p + 16 * ((8 * u + 2 * g + 1) ^ xsw));
                }
#pragma unroll
                for (int r = 0; r < RT; ++r) {
                    u32x4_t a0, a1;
                    widen_i8x16(a[r], a0, a1);
#pragma unroll
                    for (int t = 0; t < CT; ++t) {
                        acc[r][t] = Mma16<T>::run(a0, b0[t], acc[r][t]);
                        acc[r][t] = Mma16<T>::run(a1, b1[t], acc[r][t]);
                    }
                }
            } else {
                u32x4_t b[CT];
#pragma unroll
                for (int t = 0; t < CT; ++t)
                    b[t] = *reinterpret_cast<const u32x4_t *>(xl + so + t * 16 * S::XROW +
                                                              16 * ((4 * u + g) ^ xsw));
#pragma unroll
                for (int r = 0; r < RT; ++r)
#pragma unroll
                    for (int t = 0; t < CT; ++t) acc[r][t] = Mma16<T>::run(a[r], b[t], acc[r][t]);
            }
        }
        // the reads of stage i are done before its slot is copied over
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    // lane l holds column l % 16 of rows 4 (l / 16) .. + 3 of each tile
    const auto put = [&](int n, int col, f32x4_t s) {
        if (col >= B || n >= N || (WR < 16 && g >= WR / 4)) return;
        if constexpr (I8) {
#pragma unroll
            for (int v = 0; v < 4; ++v) s[v] *= h2f(scales[min(n + v, N - 1)]);
        }
        uint16_t *dst = y + static_cast<long long>(col) * N + n;
        if (pairs) {  // N % 4 == 0 and y 8-byte aligned
            *reinterpret_cast<uint2 *>(dst) = make_uint2(pack<T>(s[0], s[1]), pack<T>(s[2], s[3]));
        } else {
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (n + v < N) dst[v] = Cvt<T>::from(s[v]);
        }
    };
    if constexpr (KS > 1) {
        __syncthreads();  // every wave is done with the ring
        float *red = reinterpret_cast<float *>(lds);
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int t = 0; t < CT; ++t)
                *reinterpret_cast<f32x4_t *>(red + (((wave * RT + r) * CT + t) * 64 + lane) * 4) = acc[r][t];
        __syncthreads();
        for (int q = wave; q < RS * RT * CT; q += NW) {
            const int rr = q / (RT * CT), r = q / CT % RT, t = q % CT;
            f32x4_t s = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int p = 0; p < KS; ++p)
                s += *reinterpret_cast<const f32x4_t *>(
                    red + ((((p * RS + rr) * RT + r) * CT + t) * 64 + lane) * 4);
            put((blockIdx.x * RS + rr) * WR + 16 * r + 4 * g, 16 * t + c, s);
        }
    } else {
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int t = 0; t < CT; ++t) put(n0 + 16 * r + 4 * g, 16 * t + c, acc[r][t]);
    }
}

template <typename T, bool I8, int XR, int WR, int RS, int KS>
bool launch(const void *W, const void *sc, const void *x, void *y, int B, int N, int K,
            hipStream_t s) {
    using S = Shape<I8, XR, WR, RS, KS>;
    static_assert(S::D >= 2, "two stages fit in LDS");
    auto *kern = &gemv_batch_kernel<T, I8, XR, WR, RS, KS>;
    if (!tecoops::reserve_lds(reinterpret_cast<const void *>(kern), S::LDS)) return false;
    const int pairs = N % 4 == 0 && tecoops::aligned(y, 8);
    hipLaunchKernelGGL(kern, dim3(tecoops::ceil_div(N, WR * RS)), dim3(S::NW * 64), S::LDS, s,
                       static_cast<const char *>(W), static_cast<const uint16_t *>(sc),
                       static_cast<const char *>(x), static_cast<uint16_t *>(y), N, K, B, pairs);
    return true;
}

// The waves of each size (gemv_batch_rows): K split over as many groups of
// waves as leave two stages or more in LDS.  A wave's stages are a serial chain
// of copies, LDS reads and MFMAs, so that where few rows leave a CU few waves,
// more groups of shorter ranges are faster, as long as a group has enough
// stages to run through:
//   * 16 rows split K eight ways where that leaves each group 4 stages or more
//     and x is short ([4096, 14336] batch 8, four / eight ways: fp16 21.0 /
//     20.0, int8 13.1 / 12.4 µs; int8 [4096, 4096], 2 stages a group: 5.5 / 6.3);
//   * 8 rows of int8 W with short x likewise, from 2 stages a group ([256,
//     8192] batch 3, four / eight ways 7.0 / 6.0 µs, [1024, 13824] 10.7 / 8.5,
//     [2048, 4096] 5.3 / 5.1);
//   * 32 rows of int8 W with short x four ways where at most three quarters of
//     the CUs have a workgroup ([5120, 13824] two / four ways: batch 3 19.1 /
//     17.0, batch 8 20.2 / 18.1, [5120, 4096] 7.8 / 7.8, 8.1 / 7.6; two of the
//     smaller workgroups share a CU, so full grids lose: [8192, 8192] batch 4
//     14.1 / 15.9).
// 64 rows: two waves of 32 for 16-bit W (one LDS read of x serves two row
// tiles), four of 16 for int8 ([14336, 4096] batch 8: fp16 19.1 / 21.6, int8
// 13.6 / 12.3 µs).
template <typename T, bool I8, int XR>
bool launch_rows(const void *W, const void *sc, const void *x, void *y, int B, int N, int K,
                 hipStream_t s) {
    // int8 stages hold twice the x: above 32 rows of x two of them fit only
    // with K split two ways, and 16 rows of W per workgroup are then no
    // faster than 32 ([4096, 14336] batch 64: 43.4 / 41.8 µs)
    constexpr bool kShortX = I8 && XR > 32;
    const int stages = (K / (I8 ? 16 : 8) + 15) / 16;
    const int cus = tecoops::device_cus();
    switch (gemv_batch_rows(N, K, B, I8, cus)) {
        case 8:
            if constexpr (I8 && XR <= 8)
                if (stages >= 16) return launch<T, I8, XR, 8, 1, 8>(W, sc, x, y, B, N, K, s);
            if constexpr (!kShortX) return launch<T, I8, XR, 8, 1, 4>(W, sc, x, y, B, N, K, s);
            return false;
        case 16:
            if constexpr (XR <= 8)
                if (stages >= 32) return launch<T, I8, XR, 16, 1, 8>(W, sc, x, y, B, N, K, s);
            if constexpr (!kShortX) return launch<T, I8, XR, 16, 1, 4>(W, sc, x, y, B, N, K, s);
            return false;
        case 32:
            if constexpr (I8 && XR <= 8)
                if (stages >= (XR <= 4 ? 32 : 16) && N <= 24 * cus)
                    return launch<T, I8, XR, 16, 2, 4>(W, sc, x, y, B, N, K, s);
            return launch<T, I8, XR, 16, 2, 2>(W, sc, x, y, B, N, K, s);
        case 48:
            if constexpr (XR <= 8) return launch<T, I8, XR, 16, 3, 2>(W, sc, x, y, B, N, K, s);
            return false;
        case 64:
            if constexpr (I8)
                return launch<T, I8, XR, 16, 4, (kShortX ? 1 : 2)>(W, sc, x, y, B, N, K, s);
            else
                return launch<T, I8, XR, 32, 2, 2>(W, sc, x, y, B, N, K, s);
        case 96: return launch<T, I8, XR, 16, 6, 1>(W, sc, x, y, B, N, K, s);
        case 112: return launch<T, I8, XR, 16, 7, 1>(W, sc, x, y, B, N, K, s);
        default: return launch<T, I8, XR, 16, 8, 1>(W, sc, x, y, B, N, K, s);
    }
}

template <typename T, bool I8>
bool launch_batch(const void *W, const void *sc, const void *x, void *y, int B, int N, int K,
                  hipStream_t s) {
    if (B <= 4) return launch_rows<T, I8, 4>(W, sc, x, y, B, N, K, s);
    if (B <= 8) return launch_rows<T, I8, 8>(W, sc, x, y, B, N, K, s);
    if (B <= 16) return launch_rows<T, I8, 16>(W, sc, x, y, B, N, K, s);
    if (B <= 32) return launch_rows<T, I8, 32>(W, sc, x, y, B, N, K, s);
    if (B <= 48) return launch_rows<T, I8, 48>(W, sc, x, y, B, N, K, s);
    return launch_rows<T, I8, 64>(W, sc, x, y, B, N, K, s);
}

}  // namespace

tecoopsStatus_t tecoops::gemv_batch(hipStream_t s, const void *W, const void *scales,
                                    const void *x, void *y, int batch, int n, int k,
                                    tecoopsDataType_t dataType, bool i8) {
    constexpr int kSlice = 64;
    for (int b0 = 0; b0 < batch; b0 += kSlice) {
        const int nb = batch - b0 < kSlice ? batch - b0 : kSlice;
        const void *xb = static_cast<const uint16_t *>(x) + static_cast<long long>(b0) * k;
        void *yb = static_cast<uint16_t *>(y) + static_cast<long long>(b0) * n;
        const bool ok = i8 ? launch_batch<f16, true>(W, scales, xb, yb, nb, n, k, s)
                        : dataType == TECOOPS_DATA_HALF
                            ? launch_batch<f16, false>(W, nullptr, xb, yb, nb, n, k, s)
                            : launch_batch<bf16, false>(W, nullptr, xb, yb, nb, n, k, s);
        if (!ok) return TECOOPS_STATUS_INTERNAL_ERROR;
        TECO_CHECK_LAUNCH("gemv");
    }
    return TECOOPS_STATUS_SUCCESS;
}
