// gemv.hip — decode-time matrix-vector products that stream the weight
// matrix at HBM rate.
//
// No reference implementation: GEMV is absent from the reference library.
//   fp16 / bf16:  y[b, n] = T( sum_k W[n, k] * x[b, k] )            fp32 acc
//   int8:         y[b, n] = fp16( s[n] * sum_k float(Wq[n, k]) * x[b, k] )
//
// gfx950 design, by batch size (rows of x):
//   * 2-8 with int8 W at the numbers of rows per CU in b8_takes() and K a
//     multiple of 256: the 4x4x4 matrix-core path ("4x4x4 MFMA path" below).
//     Each wave streams 4 whole rows of W in 256-byte row segments, x is copied
//     into LDS straight from memory, and the waves start their sweeps of K at
//     staggered offsets.
//   * 3 and more (16-bit W), 2 and more (int8 W) otherwise, K in whole
//     16-byte chunks of W: gemv_batch.hip, which copies W and x through LDS
//     and streams W once for up to 64 rows of x.
//   * 1-2 and all other shapes: the VALU path, which streams W fastest when
//     there is little math per byte.  A workgroup of 4 waves owns 4*R
//     consecutive output rows and stages x ([B, K], up to the workgroup's
//     160 KiB) in LDS; x (and the int8 scales) are loaded before W, so that waiting for
//     them leaves W in flight.  Each wave streams R rows of W with 16-byte
//     loads, lane-interleaved
//     along K so that every load instruction reads a contiguous 1 KiB run of
//     a row; a lane issues the loads of CPL chunks of each row before using
//     any (a whole fp16 row, or one or two int8 rows, in flight per wave at
//     K = 4096), and keeps R x B fp32 partial sums; the products use
//     v_dot2_f32_{f16,bf16} (two MACs per instruction, fp32 accumulation).  A
//     wave reduction through DPP and permlane swaps (wave_sum, no LDS)
//     finishes each (row, batch) sum.
// int8 weights are widened exactly to fp16 with one v_perm_b32 (bytes of
// w+128 under the exponent of 1024.0) and one packed fp16 subtract of 1152 per
// weight pair; the per-row int8 scale is applied to the fp32 sum.
// HBM-bound: algorithmic bytes = |W| + |x| + |y| (+|s|).
#include "common.h"
#include "device.h"
#include "gemv_batch.h"

namespace {

using namespace tecoops::dev;

constexpr int kWaves = 4;
constexpr int kThreads = kWaves * 64;

template <typename T> struct Dot2;
template <> struct Dot2<f16> {
    static __device__ __forceinline__ float run(uint32_t a, uint32_t b, float c) {
        return __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, a),
                                      __builtin_bit_cast(half2_t, b), c, false);
    }
};
template <> struct Dot2<bf16> {
    static __device__ __forceinline__ float run(uint32_t a, uint32_t b, float c) {
        return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf162_t, a),
                                               __builtin_bit_cast(bf162_t, b), c, false);
    }
};

typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));

// Streaming 16-byte load of weight data that is read exactly once.
__device__ __forceinline__ uint4 load_stream(const uint4 *p) {
    const u32x4_t v = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t *>(p));
    return make_uint4(v.x, v.y, v.z, v.w);
}

// Copies x [B, K] (16-bit elements, K % 8 == 0, nvec 16-byte chunks) into
// LDS in two halves.  x_pre loads the first XP chunks of each thread into
// registers and is called before the W loads, so that waiting for x later
// leaves the younger W loads in flight (loads complete in order); x_post
// stores them, copies any remaining chunks and synchronises the workgroup.
template <int XP>
__device__ __forceinline__ void x_pre(uint4 (&xr)[XP], const uint4 *x, int nvec) {
    // Relaxed workgroup-scope atomic loads (plain global loads in the ISA):
    // the compiler neither sinks them to their use nor hoists the W loads
    // above them, as it does with ordinary loads of read-only memory.
#pragma unroll
    for (int j = 0; j < XP; ++j) {
        const uint64_t *p = reinterpret_cast<const uint64_t *>(
            x + min(static_cast<int>(threadIdx.x + j * blockDim.x), nvec - 1));
        const uint64_t lo = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        const uint64_t hi = __hip_atomic_load(p + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        xr[j] = make_uint4(static_cast<uint32_t>(lo), static_cast<uint32_t>(lo >> 32),
                           static_cast<uint32_t>(hi), static_cast<uint32_t>(hi >> 32));
    }
}
template <int XP>
__device__ __forceinline__ void x_post(uint4 *xs, const uint4 (&xr)[XP], const uint4 *x, int nvec) {
    // unconditional (clamped) stores: a store under a branch lets the
    // compiler sink its load into that branch, behind the W loads; threads
    // past the end all write x's last chunk to its own place
#pragma unroll
    for (int j = 0; j < XP; ++j) xs[min(static_cast<int>(threadIdx.x + j * blockDim.x), nvec - 1)] = xr[j];
    for (int i = threadIdx.x + XP * blockDim.x; i < nvec; i += blockDim.x) xs[i] = x[i];
    __syncthreads();
}
// x chunks per thread loaded ahead of W: all of x for B = 1 and K <= 4096.
constexpr int x_pre_chunks(int B) { return B == 1 ? 2 : 4; }

// int8 weight dword (4 values) -> two packed fp16 pairs holding the exact values.
__device__ __forceinline__ void widen_i8(uint32_t w, uint32_t &p01, uint32_t &p23) {
    const uint32_t u = w ^ 0x80808080u;  // bytes now hold w + 128 in [0, 255]
    const half2_t bias = {static_cast<_Float16>(-1152.0f), static_cast<_Float16>(-1152.0f)};
    // 0x64XX as fp16 is 1024 + XX
    half2_t h01 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u));
    half2_t h23 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u));
    p01 = __builtin_bit_cast(uint32_t, h01 + bias);
    p23 = __builtin_bit_cast(uint32_t, h23 + bias);
}

// int8 weights, VALU path with the weight loads batched: each K step of a
// wave covers 64 * CPL 16-byte chunks of each of its R rows, and a lane issues
// all R * CPL of its loads before widening any of them, so every lane keeps
// R * CPL * 16 bytes in flight and a row needs K / (1024 * CPL) round trips.
template <int B, int R, int CPL, int NW>
__global__ void __launch_bounds__(NW * 64)
gemv_i8_kernel(const uint4 *__restrict__ W, const uint16_t *__restrict__ scales,
                       const uint4 *__restrict__ x, uint16_t *__restrict__ y, int N, int K) {
    extern __shared__ uint4 xs[];
    const int kx = K / 8;    // 16-byte chunks of an x row (8 fp16)
    const int kw = K / 16;   // 16-byte chunks of a W row (16 int8)
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int n0 = (blockIdx.x * NW + wave) * R;
    const uint4 *wrow[R];
#pragma unroll
    for (int r = 0; r < R; ++r) wrow[r] = W + static_cast<long long>(min(n0 + r, N - 1)) * kw;
    // the scales and x are loaded before W: they are waited for without
    // draining the W loads, and the scales are in registers by the end
    uint16_t sc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) sc[r] = scales[min(n0 + r, N - 1)];
    uint4 xr[x_pre_chunks(B)];
    x_pre(xr, x, B * kx);
    // W loads are unconditional (clamped to the row's last chunk) so that the
    // compiler waits for each one at its use rather than for all of them
    uint4 q[R][CPL];
#pragma unroll
    for (int u = 0; u < CPL; ++u)
#pragma unroll
        for (int r = 0; r < R; ++r) q[r][u] = load_stream(wrow[r] + min(lane + 64 * u, kw - 1));
    x_post(xs, xr, x, B * kx);
    if (n0 >= N) return;
    float acc[R][B];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int b = 0; b < B; ++b) acc[r][b] = 0.0f;
    for (int c0 = lane;; c0 += 64 * CPL) {
#pragma unroll
        for (int u = 0; u < CPL; ++u) {
            const int c = c0 + 64 * u;
            if (c < kw) {
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    uint32_t wh[8];  // 16 weights as 8 fp16 pairs
                    widen_i8(q[r][u].x, wh[0], wh[1]);
                    widen_i8(q[r][u].y, wh[2], wh[3]);
                    widen_i8(q[r][u].z, wh[4], wh[5]);
                    widen_i8(q[r][u].w, wh[6], wh[7]);
#pragma unroll
                    for (int b = 0; b < B; ++b) {
                        const uint4 x0 = xs[b * kx + 2 * c];
                        const uint4 x1 = xs[b * kx + 2 * c + 1];
                        const uint32_t xv[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
                        float s = acc[r][b];
#pragma unroll
                        for (int j = 0; j < 8; ++j) s = Dot2<f16>::run(wh[j], xv[j], s);
                        acc[r][b] = s;
                    }
                }
            }
        }
        const int cn = c0 + 64 * CPL;
        if (cn - lane >= kw) break;
#pragma unroll
        for (int u = 0; u < CPL; ++u)
#pragma unroll
            for (int r = 0; r < R; ++r) q[r][u] = load_stream(wrow[r] + min(cn + 64 * u, kw - 1));
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
        for (int b = 0; b < B; ++b) {
            const float s = wave_sum(acc[r][b]);
            if (lane == 0 && n0 + r < N)
                y[static_cast<long long>(b) * N + n0 + r] = f2h(h2f(sc[r]) * s);
        }
    }
}

// fp16 / bf16 weights, VALU path with batched loads (as gemv_i8_kernel).
template <typename T, int B, int R, int CPL, int NW>
__global__ void __launch_bounds__(NW * 64)
gemv16_kernel(const uint4 *__restrict__ W, const uint4 *__restrict__ x,
                      uint16_t *__restrict__ y, int N, int K) {
    extern __shared__ uint4 xs[];
    const int kv = K / 8;  // 16-byte chunks per row
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int n0 = (blockIdx.x * NW + wave) * R;
    const uint4 *wrow[R];
#pragma unroll
    for (int r = 0; r < R; ++r) wrow[r] = W + static_cast<long long>(min(n0 + r, N - 1)) * kv;
    uint4 xr[x_pre_chunks(B)];
    x_pre(xr, x, B * kv);
    uint4 q[R][CPL];
#pragma unroll
    for (int u = 0; u < CPL; ++u)
#pragma unroll
        for (int r = 0; r < R; ++r) q[r][u] = load_stream(wrow[r] + min(lane + 64 * u, kv - 1));
    x_post(xs, xr, x, B * kv);
    if (n0 >= N) return;
    float acc[R][B];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int b = 0; b < B; ++b) acc[r][b] = 0.0f;
    for (int c0 = lane;; c0 += 64 * CPL) {
#pragma unroll
        for (int u = 0; u < CPL; ++u) {
            const int c = c0 + 64 * u;
            if (c < kv) {
#pragma unroll
                for (int b = 0; b < B; ++b) {
                    const uint4 xv = xs[b * kv + c];
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        float s = acc[r][b];
                        s = Dot2<T>::run(q[r][u].x, xv.x, s);
                        s = Dot2<T>::run(q[r][u].y, xv.y, s);
                        s = Dot2<T>::run(q[r][u].z, xv.z, s);
                        s = Dot2<T>::run(q[r][u].w, xv.w, s);
                        acc[r][b] = s;
                    }
                }
            }
        }
        const int cn = c0 + 64 * CPL;
        if (cn - lane >= kv) break;
#pragma unroll
        for (int u = 0; u < CPL; ++u)
#pragma unroll
            for (int r = 0; r < R; ++r) q[r][u] = load_stream(wrow[r] + min(cn + 64 * u, kv - 1));
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int b = 0; b < B; ++b) {
            const float s = wave_sum(acc[r][b]);
            if (lane == 0 && n0 + r < N) y[static_cast<long long>(b) * N + n0 + r] = Cvt<T>::from(s);
        }
}

typedef _Float16 f16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

// Runs one wave's n steps (n wave-uniform) with the loads of each step issued
// D steps ahead of its use: load(j, i) fetches step j into ring slot i and
// use(j, i) consumes step j from slot i; start() runs once, after the first
// loads are issued and before the first use.  Slot indices are compile-time
// constants after unrolling, so the ring stays in registers, and the loads of
// the main loop are unconditional, so the waits before each use leave the
// younger loads in flight.
template <int D, typename Load, typename Use, typename Start>
__device__ __forceinline__ void ring_steps(int n, Load &&load, Use &&use, Start &&start) {
    if (n < D) {
        for (int j = 0; j < n; ++j) {
            load(j, 0);
            if (j == 0) start();
            use(j, 0);
        }
        if (n <= 0) start();
        return;
    }
#pragma unroll
    for (int i = 0; i < D; ++i) load(i, i);
    start();
    int j = 0;
    for (; j + 2 * D <= n; j += D) {
#pragma unroll
        for (int i = 0; i < D; ++i) {
            use(j + i, i);
            load(j + D + i, i);
            // keep this order: the scheduler would otherwise batch the loads
            // at the end of the iteration and drain the ring at its top
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // steps j .. j+D-1 are in the ring; j+D .. n-1 (fewer than D) are not
#pragma unroll
    for (int i = 0; i < D; ++i) {
        use(j + i, i);
        if (j + D + i < n) load(j + D + i, i);
    }
#pragma unroll
    for (int i = 0; i < D; ++i)
        if (j + D + i < n) use(j + D + i, i);
}

// ------------------------------------------------------ 4x4x4 MFMA path
//
// int8 W, batches of up to 8 rows of x: Y^T = W X^T on v_mfma_f32_4x4x4_16b_f16,
// which runs 16 independent 4x4x4 products (blocks) per instruction.
// Lane l = 4*blk + r supplies row r of block blk's A operand and column r of
// its B operand, and receives column r of its C block.  Each wave owns 4 whole
// rows of W: lane l loads the 16 bytes at chunk blk of every 16-chunk
// (256-byte) run of row n0 + r, so one load instruction reads four contiguous
// 256-byte row segments (the access pattern of the VALU path), and block blk
// accumulates those 4 rows against batch columns 4*cg + r over its own k
// values.  The 16 blocks hold partial sums over disjoint k; once the wave has
// covered K they are added across lanes l, l + 4, ..., l + 60 without LDS
// (DPP row rotations by 4 and 8, then the row-pair and half-wave permlane
// swaps).  No cross-wave reduction or barrier follows the staging of x.
//   x is staged in LDS as [4*NCG][K] 16-bit values with the 16-byte chunks of
//   row i XOR-swizzled by 4*(i % 4) inside each 256-byte run, so that the
//   128-bit B-operand reads of lanes 0-7 (rows 0-3, two chunks) hit distinct
//   banks.  int8 weights are widened exactly to fp16 (widen_i8) and feed 4
//   k-steps per 16-byte load; the per-row scale is applied to the fp32 sum.
typedef unsigned u32x2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ f32x4_t mma4(uint32_t a0, uint32_t a1, uint32_t b0, uint32_t b1,
                                        f32x4_t c) {
    const u32x2_t a = {a0, a1}, b = {b0, b1};
    return __builtin_amdgcn_mfma_f32_4x4x4f16(__builtin_bit_cast(f16x4_t, a),
                                              __builtin_bit_cast(f16x4_t, b), c, 0, 0, 0);
}

// 16 zero bytes: the source of staged x rows past the batch.
__device__ __attribute__((aligned(16))) const uint32_t kXZero16[4] = {0u, 0u, 0u, 0u};

// Global -> LDS with no register staging: 16 bytes per lane into
// dst + 16 * lane (dst wave-uniform, in M0).  Inline assembly so that the
// compiler does not count the copy among its own loads: through the builtin
// it would wait for every load in flight (the W ring included) before the
// first LDS read.  The copies are ordered by wait_vm() and the workgroup
// barrier after it.  No other code of these kernels uses M0 (build.py checks
// both in the assembly).
__device__ __forceinline__ void dma16(const void *src, void *dst) {
    const uint32_t lds = static_cast<uint32_t>(
        reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) void *)(dst)));
    asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds)
                 : "memory");
}

// s_waitcnt vmcnt(N): all but the N youngest vector-memory operations of the
// wave are done (expcnt and lgkmcnt not waited for).
template <int N>
__device__ __forceinline__ void wait_vm() {
    static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
    __builtin_amdgcn_s_waitcnt(((N >> 4) << 14) | 0x0F70 | (N & 15));
}

// LDS element offset of the 16-byte chunk c of staged x row `row`.
__device__ __forceinline__ int xs_chunk(int row, int c, int K) {
    return row * K + 8 * (c ^ (4 * (row & 3)));
}

// NCG: batch column groups of 4 (1 for B <= 4, else 2).  CPL: load steps a
// lane keeps in flight.
template <int NCG, int NW, int CPL>
__global__ void __launch_bounds__(NW * 64)
gemv_i8_b8_kernel(const uint4 *__restrict__ W, const uint16_t *__restrict__ scales,
                  const uint4 *__restrict__ x, uint16_t *__restrict__ y, int N, int K, int B) {
    extern __shared__ uint4 xs_raw[];
    uint16_t *xs = reinterpret_cast<uint16_t *>(xs_raw);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 3, blk = lane >> 2;
    const int n0 = (blockIdx.x * NW + wave) * 4;
    const int kw = K / 16;  // 16-byte chunks of a W row
    const int kx = K / 8;   // ... of an x row
    const int nl = kw / 16; // load steps per row
    const uint4 *wr = W + static_cast<long long>(min(n0 + r, N - 1)) * kw + blk;
    f32x4_t acc[NCG];
#pragma unroll
    for (int cg = 0; cg < NCG; ++cg) acc[cg] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    // The scales and x loads are issued first (unconditionally, clamped to
    // the last row), so that waiting for x leaves the younger W loads in
    // flight and the scales are in registers by the end.
    uint16_t sc[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) sc[v] = scales[min(n0 + v, N - 1)];
    // x goes straight into LDS (no registers, no LDS stores).  [14336, 4096]
    // batch 8, three alternating runs, us staged through registers / copied:
    // 12.57-12.91 / 12.10-12.43.  Copy m fills LDS chunks [64m, 64m + 64), so
    // lane l loads the x chunk stored at 64m + l (the swizzle flips bits 2-3
    // of the chunk index only, within the copy's 64); rows past the batch
    // copy zeros.
    for (int m = wave; m < NCG * 4 * kx / 64; m += NW) {
        const int slot = 64 * m + lane;
        const int row = slot / kx, cs = slot - row * kx;
        const void *src = row < B ? static_cast<const void *>(x + static_cast<long long>(row) * kx +
                                                              (cs ^ (4 * (row & 3))))
                                  : static_cast<const void *>(kXZero16);
        dma16(src, xs_raw + 64 * m);
    }
    // This lane's x chunks in LDS: chunk 32i + 2blk and the next of row 4cg +
    // r.  The swizzle xor (4r < 16) stays below the step's bits, so
    // xs_chunk(4cg + r, c0 + 32i, K) = xs_chunk(4cg + r, c0, K) + 256i (c0 =
    // 2blk), and rows 4 apart keep the same xor: one base address per lane.
    const uint16_t *xs_lane = xs + xs_chunk(r, 2 * blk, K);
    uint4 q[CPL];
    // Each wave starts its sweep of K at a different load step, so that the
    // requests in flight across the grid spread over all HBM channels instead
    // of every wave reading the same offset of its rows at the same time.
    const int rot = (blockIdx.x * NW + wave) % nl;
    const auto local = [&](int i) { return i + rot < nl ? i + rot : i + rot - nl; };
    // Every CU's x loads miss L2 together and, at HBM, queue behind the first
    // W loads of all waves, which start at the same moment, while no wave can
    // use its W before x is in LDS.  Pausing ~1000 cycles before the W loads
    // lets the x misses reach HBM first (batch 8 x [14336, 4096], A/B on two
    // boxes: 13.4 -> 12.9 us and 14.0 -> 13.8 us; waiting for x outright:
    // 14.0 us).  With 2 W steps in flight per lane, pauses of 0, 8, 16 and 32
    // (x 64 cycles) took 13.5-14.0, 13.4, 12.9-13.1 and 13.3 us on one box.
    // The best pause is about one vector L1 -> L2 read round trip of this
    // stream (865 cycles with one load in flight per lane, 1267 with two;
    // rocprofv3 TCP_TCC_READ_REQ_LATENCY / TCP_TCC_READ_REQ), i.e. long
    // enough for x's requests to leave the L1 and L2 queues before the W
    // requests fill them, and shorter than waiting for x's data (the HBM
    // round trip, ~2000 cycles once the stream saturates).
    if (gridDim.x >= 128) __builtin_amdgcn_s_sleep(16);
    // Waves past the last row still stage x and reach the barrier; their
    // loads read row N - 1 and their sums are never stored.
    ring_steps<CPL>(
        nl, [&](int i, int u) { q[u] = load_stream(wr + 16 * local(i)); },
        [&](int i0, int u) {
            const int i = local(i0);
            uint32_t p[8];
            widen_i8(q[u].x, p[0], p[1]);
            widen_i8(q[u].y, p[2], p[3]);
            widen_i8(q[u].z, p[4], p[5]);
            widen_i8(q[u].w, p[6], p[7]);
#pragma unroll
            for (int cg = 0; cg < NCG; ++cg) {
                const uint4 *xp = reinterpret_cast<const uint4 *>(xs_lane + cg * 4 * K) + 32 * i;
                const uint4 xa = xp[0];
                const uint4 xb = xp[1];
                f32x4_t c = acc[cg];
                c = mma4(p[0], p[1], xa.x, xa.y, c);
                c = mma4(p[2], p[3], xa.z, xa.w, c);
                c = mma4(p[4], p[5], xb.x, xb.y, c);
                c = mma4(p[6], p[7], xb.z, xb.w, c);
                acc[cg] = c;
            }
        },
        [&] {
            // This wave's copies are older than the CPL steps of W loads
            // ring_steps issues before start(), so waiting until at most
            // those are outstanding leaves them in flight.  The compiler
            // could legally sink a load of read-only memory below this wait,
            // which would make the count too large: build.py checks the
            // assembly of every such wait and fails the build if it ever
            // does.  A row with fewer steps (ring_steps' short path, K < 512)
            // waits for everything.  The barrier then covers every wave's
            // copies.
            if (nl >= CPL) wait_vm<CPL>();
            else wait_vm<0>();
            __syncthreads();
        });
    if (n0 >= N) return;
    // add the 16 blocks' partial sums (lanes r, r + 4, ..., r + 60: rotations
    // by 4 and 8 within each row of 16 lanes, then the row-pair and half-wave
    // swaps); lanes 0-3 then hold column r of rows n0 .. n0 + 3
#pragma unroll
    for (int cg = 0; cg < NCG; ++cg)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            float t = acc[cg][v];
            t += dpp<kDppRor4>(t);
            t += dpp<kDppRor8>(t);
            t = row_swap_sum(t);
            acc[cg][v] = half_swap_sum(t);
        }
    if (blk != 0) return;
#pragma unroll
    for (int cg = 0; cg < NCG; ++cg) {
        const int b = 4 * cg + r;
        if (b >= B) continue;
#pragma unroll
        for (int v = 0; v < 4; ++v)
            if (n0 + v < N) y[static_cast<long long>(b) * N + n0 + v] = f2h(acc[cg][v] * h2f(sc[v]));
    }
}

// Fallback for shapes the vector kernels do not take (K not a multiple of 8 /
// 16, misaligned pointers): one wave per (row, batch), element-wise.
template <typename T, bool INT8>
__global__ void __launch_bounds__(kThreads)
gemv_scalar_kernel(const void *__restrict__ Wv, const uint16_t *__restrict__ scales,
                   const uint16_t *__restrict__ x, uint16_t *__restrict__ y, int N, int K,
                   int batch) {
    const int lane = threadIdx.x & 63;
    const long long task = static_cast<long long>(blockIdx.x) * kWaves + (threadIdx.x >> 6);
    if (task >= static_cast<long long>(N) * batch) return;
    const int n = static_cast<int>(task % N), b = static_cast<int>(task / N);
    float s = 0.0f;
    for (int k = lane; k < K; k += 64) {
        const float w = INT8 ? static_cast<float>(static_cast<const int8_t *>(Wv)[static_cast<long long>(n) * K + k])
                             : Cvt<T>::to(static_cast<const uint16_t *>(Wv)[static_cast<long long>(n) * K + k]);
        s += w * Cvt<T>::to(x[static_cast<long long>(b) * K + k]);
    }
    s = wave_sum(s);
    if (lane == 0) {
        if (INT8) s *= h2f(scales[n]);
        y[static_cast<long long>(b) * N + n] = Cvt<T>::from(s);
    }
}

// x staged in LDS may fill a workgroup's whole LDS (reserve_lds sets the
// kernels' attribute above the default 64 KiB when it does).
constexpr long long kMaxLdsBytes = static_cast<long long>(tecoops::kLdsMax);

// Smallest batches that take the matrix cores.  16-bit W at batch 2 does above
// kBatch2MinK: the VALU path's 2 staged rows of x then leave fewer than 4
// workgroups per CU.  Batch 2 fp16, µs VALU / gemv_batch.hip: [4096, 4096]
// 7.5 / 7.3, [14336, 4096] 19.4 / 19.4, [28672, 4096] 36.2 / 37.0, [1024,
// 2048] 3.2 / 3.5; [4096, 14336] 23.1 / 19.2.  Batch 3 [14336, 4096]: 20.2
// with the 4x4x4 path / 19.1.  int8 batch 1, VALU / gemv_batch.hip: [14336,
// 4096] 10.5 / 12.7, [4096, 4096] 4.9 / 5.5.
constexpr int kBatchMin16 = 3, kBatch2MinK = 10240, kBatchMinI8 = 2;

// VALU path shapes (rows per wave R, 16-byte W chunks per lane per K step
// CPL), measured on the [14336, 4096] batch-1 shapes: fp16 one row per wave
// with the whole 8 KiB row in flight (19.5 us; 4 rows with one chunk in
// flight: 22.6 us), int8 two 4 KiB rows per wave (12.9 us; 15.5 us before).
// Fewer rows per wave beat deeper per-wave queues: 4 rows x 4 chunks of int8
// took 16.2 us, and 8 or 16 waves per workgroup were slower for both types.
constexpr int kR16 = 1, kCpl16 = 8;
constexpr int kRI8 = 2, kCplI8 = 4;
// int8 at batch 1 with rows of at most kRI8OneMaxK values and at least
// kRI8OneMinN rows: one row per wave (the whole 4 KiB row in flight, twice
// the workgroups, half the bytes in flight per wave).  Standalone sweep, 16
// rotating weight copies, µs two rows / one row per wave: [14336, 4096]
// 10.57-10.69 / 10.46-10.57 on four boxes, [28672, 4096] 18.5-19.2 /
// 18.1-19.0, [11008, 4096] 9.0-9.2 / 8.7; at fewer rows or longer rows two
// stay: [8192, 4096] 7.1-7.2 / 7.3, [4096, 4096] 4.7-5.0 / 5.2-5.5,
// [14336, 14336] 33.5-36.0 / 35.0-37.2, [8192, 28672] 40-43 / 47-50 (some
// shapes outside the rule gain: [8192, 8192] 13.3-13.7 / 12.4-12.8,
// [4096, 14336] 12.4-13.0 / 12.1-12.5).
constexpr int kRI8OneMaxK = 4096, kRI8OneMinN = 10240;

// 4x4x4 path: load steps in flight per lane.  x is staged in LDS once per
// workgroup, so workgroups are large (b8_waves picks their size).  Batch 8 on
// [14336, 4096], 1, 2, 3, 4, 8 and 16 steps in flight: 16.5, 12.6, 13.1, 14.9,
// 15.9 and 16.3 us (two groups of 4 rows per wave: 15.0-15.6 us).
constexpr int kB8CplI8 = 2, kB8MaxBatch = 8;

// Whether the 4x4x4 path takes an int8 product, with the staged x in LDS: where
// it still beats gemv_batch.hip.  Its waves are 4 rows each, so that its time
// follows N closely, and up to batch 4 it reads x with half the LDS traffic.  µs
// 4x4x4 / gemv_batch.hip at K = 4096: batch 4 [8192] 9.6 / 8.4, [9216] 9.9 /
// 10.4, [14336] 12.3 / 12.7, [18432] 16.1 / 16.9, [21504] 17.7 / 17.9, [22528]
// 19.0 / 18.5, [28672] 22.7 / 21.9, [34304] 27.1 / 28.8, [41984] 30.1 / 32.6,
// [45056] 33.4 / 34.1, [57344] 39.1 / 40.2; batch 8 [12288] 12.0 / 11.8, [15360]
// 13.5 / 14.1, [16384] 14.0 / 14.2, [17408] 20.8 / 17.0, [28672] 26.9 / 21.7.
bool b8_takes(int batch, int n, int k) {
    const long long cus = tecoops::device_cus();
    if (batch > kB8MaxBatch || k % 256 != 0) return false;
    if (batch <= 4 ? n <= 32 * cus || (n > 80 * cus && n <= 128 * cus)
                   : n <= 48 * cus || n > 64 * cus)
        return false;
    return (batch <= 4 ? 4 : 8) * 2LL * k <= kMaxLdsBytes;
}

// Waves per workgroup of the 4x4x4 path: of 16, 14, 12, 8 and 7, the one that
// leaves the busiest CU the fewest waves (ceil(workgroups / CUs) * waves; the
// first listed on ties), so that a grid just short of the CU count does not
// idle CUs: N = 14336 takes 14 waves and 256 workgroups (16 waves: 224).
int b8_waves(int N) {
    const long long cus = tecoops::device_cus();
    int best = 16;
    long long best_load = -1;
    for (int nw : {16, 14, 12, 8, 7}) {
        const long long wgs = tecoops::ceil_div(N, 4LL * nw);
        const long long load = (wgs + cus - 1) / cus * nw;
        if (best_load < 0 || load < best_load) {
            best_load = load;
            best = nw;
        }
    }
    return best;
}

template <int NCG, int NW>
bool launch_b8_nw(const void *W, const void *sc, const void *x, void *y, int B, int N, int K,
                  hipStream_t s) {
    const size_t lds = 4 * NCG * static_cast<size_t>(K) * 2;
    auto *kern = &gemv_i8_b8_kernel<NCG, NW, kB8CplI8>;
    if (!tecoops::reserve_lds(reinterpret_cast<const void *>(kern), lds)) return false;
    hipLaunchKernelGGL(kern, dim3(tecoops::ceil_div(N, 4 * NW)), dim3(NW * 64), lds, s,
                       static_cast<const uint4 *>(W), static_cast<const uint16_t *>(sc),
                       static_cast<const uint4 *>(x), static_cast<uint16_t *>(y), N, K, B);
    return true;
}

template <int NCG>
bool launch_b8(const void *W, const void *sc, const void *x, void *y, int B, int N, int K,
               hipStream_t s) {
    switch (b8_waves(N)) {
        case 14: return launch_b8_nw<NCG, 14>(W, sc, x, y, B, N, K, s);
        case 12: return launch_b8_nw<NCG, 12>(W, sc, x, y, B, N, K, s);
        case 8: return launch_b8_nw<NCG, 8>(W, sc, x, y, B, N, K, s);
        case 7: return launch_b8_nw<NCG, 7>(W, sc, x, y, B, N, K, s);
        default: return launch_b8_nw<NCG, 16>(W, sc, x, y, B, N, K, s);
    }
}

template <typename T, int B>
bool launch16(const void *W, const void *x, void *y, int N, int K, hipStream_t s) {
    const unsigned grid = tecoops::ceil_div(N, kWaves * kR16);
    auto *kern = &gemv16_kernel<T, B, kR16, kCpl16, kWaves>;
    if (!tecoops::reserve_lds(reinterpret_cast<const void *>(kern), B * static_cast<size_t>(K) * 2))
        return false;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(kThreads),
                       B * K * 2, s, static_cast<const uint4 *>(W), static_cast<const uint4 *>(x),
                       static_cast<uint16_t *>(y), N, K);
    return true;
}

template <int R>
bool launch_i8_r(const void *W, const void *sc, const void *x, void *y, int N, int K,
                 hipStream_t s) {
    const unsigned grid = tecoops::ceil_div(N, kWaves * R);
    auto *kern = &gemv_i8_kernel<1, R, kCplI8, kWaves>;
    if (!tecoops::reserve_lds(reinterpret_cast<const void *>(kern), static_cast<size_t>(K) * 2))
        return false;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(kThreads),
                       K * 2, s, static_cast<const uint4 *>(W),
                       static_cast<const uint16_t *>(sc), static_cast<const uint4 *>(x),
                       static_cast<uint16_t *>(y), N, K);
    return true;
}

bool launch_i8(const void *W, const void *sc, const void *x, void *y, int N, int K,
               hipStream_t s) {
    if (K <= kRI8OneMaxK && N >= kRI8OneMinN) return launch_i8_r<1>(W, sc, x, y, N, K, s);
    return launch_i8_r<kRI8>(W, sc, x, y, N, K, s);
}

}  // namespace

extern "C" tecoopsStatus_t tecoopsGemv(tecoopsHandle_t handle, const void *weight, const void *x,
                                       void *y, int batch, int n, int k,
                                       tecoopsDataType_t dataType) {
    if (handle == nullptr) return TECOOPS_STATUS_NOT_INITIALIZED;
    if (weight == nullptr || x == nullptr || y == nullptr) return TECOOPS_STATUS_BAD_PARAM;
    if (batch <= 0 || n <= 0 || k <= 0) return TECOOPS_STATUS_BAD_PARAM;
    if (!tecoops::is_16bit_float(dataType)) return TECOOPS_STATUS_BAD_PARAM;
    using tecoops::dev::bf16;
    using tecoops::dev::f16;
    hipStream_t s = handle->stream;
    const bool al = tecoops::aligned(weight, 16) && tecoops::aligned(x, 16);
    if ((batch >= kBatchMin16 || (batch == 2 && k > kBatch2MinK)) && k % 8 == 0 && al)
        return tecoops::gemv_batch(s, weight, nullptr, x, y, batch, n, k, dataType, false);
    // the VALU path: at most two rows of x, staged whole in LDS
    if (batch <= 2 && k % 8 == 0 && al && 2LL * batch * k <= kMaxLdsBytes) {
        const bool half = dataType == TECOOPS_DATA_HALF;
        const bool ok = batch == 1 ? (half ? launch16<f16, 1>(weight, x, y, n, k, s)
                                           : launch16<bf16, 1>(weight, x, y, n, k, s))
                                   : (half ? launch16<f16, 2>(weight, x, y, n, k, s)
                                           : launch16<bf16, 2>(weight, x, y, n, k, s));
        if (!ok) return TECOOPS_STATUS_INTERNAL_ERROR;
        TECO_CHECK_LAUNCH("gemv");
        return TECOOPS_STATUS_SUCCESS;
    }
    const unsigned grid = tecoops::ceil_div(static_cast<long long>(n) * batch, kWaves);
    if (dataType == TECOOPS_DATA_HALF)
        hipLaunchKernelGGL((gemv_scalar_kernel<f16, false>), dim3(grid), dim3(kThreads), 0, s,
                           weight, nullptr, static_cast<const uint16_t *>(x),
                           static_cast<uint16_t *>(y), n, k, batch);
    else
        hipLaunchKernelGGL((gemv_scalar_kernel<bf16, false>), dim3(grid), dim3(kThreads), 0, s,
                           weight, nullptr, static_cast<const uint16_t *>(x),
                           static_cast<uint16_t *>(y), n, k, batch);
    TECO_CHECK_LAUNCH("gemv");
    return TECOOPS_STATUS_SUCCESS;
}

extern "C" tecoopsStatus_t tecoopsGemvInt8(tecoopsHandle_t handle, const int8_t *weight,
                                           const void *scales, const void *x, void *y,
                                           int batch, int n, int k) {
    if (handle == nullptr) return TECOOPS_STATUS_NOT_INITIALIZED;
    if (weight == nullptr || scales == nullptr || x == nullptr || y == nullptr)
        return TECOOPS_STATUS_BAD_PARAM;
    if (batch <= 0 || n <= 0 || k <= 0) return TECOOPS_STATUS_BAD_PARAM;
    using tecoops::dev::f16;
    hipStream_t s = handle->stream;
    const bool al = tecoops::aligned(weight, 16) && tecoops::aligned(x, 16);
    if (batch >= kBatchMinI8 && k % 16 == 0 && al) {
        if (!b8_takes(batch, n, k))
            return tecoops::gemv_batch(s, weight, scales, x, y, batch, n, k, TECOOPS_DATA_HALF, true);
        if (!(batch <= 4 ? launch_b8<1>(weight, scales, x, y, batch, n, k, s)
                         : launch_b8<2>(weight, scales, x, y, batch, n, k, s)))
            return TECOOPS_STATUS_INTERNAL_ERROR;
        TECO_CHECK_LAUNCH("gemv_int8");
        return TECOOPS_STATUS_SUCCESS;
    }
    if (batch == 1 && k % 16 == 0 && al && 2LL * k <= kMaxLdsBytes) {
        if (!launch_i8(weight, scales, x, y, n, k, s)) return TECOOPS_STATUS_INTERNAL_ERROR;
        TECO_CHECK_LAUNCH("gemv_int8");
        return TECOOPS_STATUS_SUCCESS;
    }
    const unsigned grid = tecoops::ceil_div(static_cast<long long>(n) * batch, kWaves);
    hipLaunchKernelGGL((gemv_scalar_kernel<f16, true>), dim3(grid), dim3(kThreads), 0, s,
                       static_cast<const void *>(weight), static_cast<const uint16_t *>(scales),
                       static_cast<const uint16_t *>(x), static_cast<uint16_t *>(y), n, k, batch);
    TECO_CHECK_LAUNCH("gemv_int8");
    return TECOOPS_STATUS_SUCCESS;
}
