// flash_attention.hip — paged, varlen, causal, GQA attention on gfx950 MFMA.
//
// Semantics (teco/interface/ops/flash_attention.cpp:71-119,
// teco/ual/kernel/flash_attention/flash_attention.scpp:179-416, CPU baseline
// test/zoo/teco/flash_attention/flash_attention.py:79-140):
//   for sequence b with q_len L and kv_len S, query row i (0-based in its
//   chunk) sits at causal position q_start + i, q_start = max(S - L, 0)
//   (bottom-right alignment) and sees keys j <= q_start + i, j < S.  Head h
//   reads kv head h / (H / Hkv).  O = softmax(scale * Q K^T + mask) V with an
//   fp32 online softmax whose running max is clamped at >= 0 (scpp:149), P
//   rounded to the element type before the PV product (scpp:316-329), and
//   rows with no visible key written as 0 (scpp:388).
//   K/V are read from the paged caches [num_blocks, Hkv, block_size, D]
//   through block_table[b][j / block_size].
//
// gfx950 design (one wave = 64 lanes; v_mfma_f32_32x32x16_{bf16,f16}):
//   * Scores are computed transposed, S^T = K Q^T, so each lane owns one query
//     column (lane % 32) and 16 key rows per 32x32 block: the row max / sum of
//     the online softmax is a lane-local reduction plus one exchange with the
//     other half-wave.  P^T stays in registers and is directly the B operand
//     of O^T += V^T P^T (the key order inside an MFMA k-step is permuted
//     consistently on both operands).
//   * Prefill with D = 128 and a paged cache (block_size a multiple of 8):
//     K and V tiles go from HBM straight into LDS (global_load_lds_dwordx4,
//     no registers), two tiles ahead in a ring of three buffers, in a layout
//     of 4-row blocks (rows chunk-major, 64-byte pad per block) on which the
//     128-bit K reads and the transposing V reads (ds_read_b64_tr_b16, the A
//     operand of the PV product) are conflict-free.  Decode with D = 128
//     stages K and V row-major through registers (16- and 32-byte row pads),
//     with the same transposing V reads.  The other loaders stage K row-major
//     (16-byte pad) and V transposed (V^T[d][key], 4-element pad, two plain
//     64-bit reads).  Global -> register prefetch of the next tile overlaps
//     the current tile's MFMA work.
//   * Prefill (D = 128, block_size a multiple of 8): a workgroup of 12 waves
//     (3 per SIMD) shares each 96-key K/V tile among up to 4 query heads of
//     one GQA group (HW heads x (12/HW) row blocks of 32); other shapes use 4
//     waves and 64-key tiles.  The grid walks query tiles heaviest-first and
//     keeps all tiles of one (batch, kv head) on the same XCD (workgroup index
//     % 8 depends only on (b, kv head) when B*Hkv*groups is a multiple of 8),
//     so K/V are re-read from that XCD's L2.  MFMA-bound: 4*D*visible(q, k)
//     FLOP per (q row, head).  A wave issues MFMA and VALU work serially, so
//     the MFMA pipe is kept busy by the other waves of its SIMD: occupancy
//     (waves per SIMD) is the main lever.
//   * Decode (G * q_len <= 32): the 32 MFMA columns hold every (head, row) of
//     a GQA group; 4 waves split each 128-key tile and the key range is split
//     across workgroups (split-KV), partial (m, l, O) merged first in LDS and
//     then by a combine kernel.  HBM-bound: every cached K/V byte is read
//     once.
#include <algorithm>
#include <cmath>
#include <cstdio>

#include "fa_device.h"
#include "fa_grid.h"

namespace {

using tecoops::fa::FaCall;
using tecoops::fa::Plan;
using tecoops::fa::SplitArgs;
using tecoops::fa::turn_shift;
using tecoops::fa::turned_place;

// A kernel's FaParams argument where it lies, at the start of the kernel
// argument segment (constant address space): read through this pointer a
// callee gets the fields with scalar loads, and no copy of the argument is
// made on the stack.
// (The host pass only parses device code, and its target has no such
// address space.)
#if defined(__HIP_DEVICE_COMPILE__)
typedef const __attribute__((address_space(4))) FaParams KernargParams;
#else
typedef const FaParams KernargParams;
#endif

// The query tiles of (b, kv head kvh, head group hg) from first_tile on, in
// turn.  Not inlined: it runs only when max_seqlen_q understates a q length,
// and its loop keeps values live across tiles that would otherwise push the
// kernel's single-tile path past its register budget.
template <typename T, int D, int W, int HW, int QSUB, int BSM, int TILE>
__device__ __attribute__((noinline)) void prefill_rest(const KernargParams *pp, int b, int kvh,
                                                       int hg, int first_tile) {
    constexpr int QT = 32 * QSUB * (W / HW);
    extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
    const FaParams p = *pp;
    long long q_off;
    int L;
    seq_info(p, b, q_off, L);
    const int S = kv_len(p, b);
    for (int t = first_tile; t * QT < L; ++t)
        prefill_tile<T, D, W, HW, QSUB, BSM, TILE>(p, lds, b, kvh, hg, q_off, L, S, t * QT);
}

// Workgroup (b, kv head, head group, query tile) with W waves: wave w serves
// query head hg*HW + w % HW of the GQA group and query rows
// [q0 + (w / HW) * 32*QSUB, +32*QSUB).  K/V tiles of TILE keys rotate through
// the loader's LDS buffers (three for the HBM -> LDS copy, two for register
// staging; one barrier per tile) and are attended 32 * NKB keys at a time.
// W >= 12 asks for 3 waves per SIMD (168 VGPRs); head sizes above 128 with 4
// waves one (their 4-wave tiles fill the registers), else 2.
//
// The grid's tile rows are sized from max_seqlen_q, a bound the reference
// never reads (flash_attention.cpp:98-99).  The workgroup of tile 0, which
// is dispatched last, then takes every query tile past the grid in turn;
// with a bound that holds there is none.  A prefill is one launch whatever
// the bound.
template <typename T, int D, int W, int HW, int QSUB, int BSM, int TILE>
__global__ void __launch_bounds__(W * 64, (W >= 12 || TILE == 32) ? 3 : (D > 128 && W < 8 ? 1 : 2))
fa_prefill_kernel(FaParams p) {
    constexpr int QT = 32 * QSUB * (W / HW);
    extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
    if (blockIdx.x == 0 && blockIdx.y == 0) zero_tail_rows(p, D);
    const int ngroups = p.G / HW;
    const int hg = blockIdx.x % ngroups;
    const int kvh = (blockIdx.x / ngroups) % p.Hkv;
    const int b = turned_place(blockIdx.x / ngroups / p.Hkv, blockIdx.y, p.turn, p.batch);
    const int rows = gridDim.y;  // tile rows sized from max_seqlen_q
    long long q_off;
    int L;
    seq_info(p, b, q_off, L);
    const int S = kv_len(p, b);
    const int tile = rows - 1 - blockIdx.y;  // heaviest causal tiles first
    if (tile * QT < L)
        prefill_tile<T, D, W, HW, QSUB, BSM, TILE>(p, lds, b, kvh, hg, q_off, L, S, tile * QT);
    if (tile == 0 && rows * QT < L)
        prefill_rest<T, D, W, HW, QSUB, BSM, TILE>(
            (const KernargParams *)(__builtin_amdgcn_kernarg_segment_ptr()), b, kvh, hg, rows);
}

// ----------------------------------------------------------------- decode

constexpr int kDecTile = 128;

template <int D>
constexpr size_t decode_lds_bytes() {
    return sizeof(uint16_t) * kv_tile_elems<D, kDecTile>();
}

// The 4 waves of a decode workgroup attend keys [kv_lo, kv_hi) of (sequence
// b, kv head kvh) for the query rows [r0, r0 + rq): column c of the MFMA tile
// is (head c / rq, row r0 + c % rq) of the GQA group and wave w takes keys
// [32w, 32w + 32) of each 128-key tile.  Leaves each wave's partial state in
// LDS, after a barrier: max lm[4][32], sum ll[4][32] and unnormalised O
// lo[4][32][D] (fp32, over the tile buffers).
template <typename T, int D, int BSM>
__device__ __forceinline__ void decode_pass(const FaParams &p, uint16_t *smem, int b, int kvh,
                                            long long q_off, int L, int S, int kv_lo, int kv_hi,
                                            int rq, int r0) {
    using Loader = typename LoaderSel<D, kDecTile, 4, BSM, true>::type;
    constexpr int KP = Loader::KP, VP = Loader::VP, VR = Loader::VR;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int g = lane >> 5, r32 = lane & 31;
    const int hl = r32 / rq, row = r0 + r32 % rq;
    const bool col_ok = hl < p.G && row < L;
    const int h = kvh * p.G + min(hl, p.G - 1);
    const int q_start = p.causal ? max(S - L, 0) : 0;
    const int *bt_row = p.bt + b * p.bt_stride;
    const long long head_off = static_cast<long long>(kvh) * p.bs * D;

    u32x4 qf[1][D / 16];
    {
        const uint16_t *src = p.q + ((q_off + min(row, L - 1)) * p.H + h) * D;
#pragma unroll
        for (int ks = 0; ks < D / 16; ++ks) {
            const u32x4 x = *reinterpret_cast<const u32x4 *>(src + 16 * ks + 8 * g);
            const u32x4 zero = {0u, 0u, 0u, 0u};
            qf[0][ks] = col_ok ? x : zero;
        }
    }
    // keys visible to this column, and to the pass's first row (the fewest)
    const int vis = min(kv_hi, p.causal ? q_start + row + 1 : S);
    const int min_vis = min(kv_hi, p.causal ? q_start + r0 + 1 : S);

    float m[1] = {0.0f}, lsum[1] = {0.0f};
    f32x16_t oacc[1][D / 32];
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
        for (int v = 0; v < 16; ++v) oacc[0][db][v] = 0.0f;

    Loader ld;
    const int ntiles = (kv_hi - kv_lo + kDecTile - 1) / kDecTile;
    if (ntiles > 0) {
        ld.prefetch(p, bt_row, kv_lo, kv_hi);
        ld.load(p, bt_row, head_off, kv_lo, kv_hi);
    }
    for (int it = 0; it < ntiles; ++it) {
        const int j0 = kv_lo + it * kDecTile;
        __syncthreads();
        ld.store(smem);
        __syncthreads();
        if (it + 1 < ntiles) ld.load(p, bt_row, head_off, j0 + kDecTile, kv_hi);
        const int jw = j0 + 32 * wave;
        if (jw < kv_hi) {
            const int lim[1] = {vis - jw - 4 * g};
            if (jw + 32 > min_vis)
                wave_attend<T, D, KP, VP, VR, 1, 1, true>(smem, smem + Loader::VOFF, 32 * wave, qf,
                                                      oacc, m, lsum, lim, p.scale_log2,
                                                      p.inv_scale_log2);
            else
                wave_attend<T, D, KP, VP, VR, 1, 1, false>(smem, smem + Loader::VOFF, 32 * wave, qf,
                                                       oacc, m, lsum, lim, p.scale_log2,
                                                       p.inv_scale_log2);
        }
    }

    __syncthreads();
    float *lm = reinterpret_cast<float *>(smem);   // [4][32] max
    float *ll = lm + 4 * 32;                        // [4][32] sum
    float *lo = ll + 4 * 32;                        // [4][32][D] unnormalised O
    const float lt = half_swap_sum(lsum[0]);
    if (g == 0) {
        lm[wave * 32 + r32] = m[0];
        ll[wave * 32 + r32] = lt;
    }
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int d = 32 * db + 8 * (v >> 2) + 4 * g + (v & 3);
            lo[(wave * 32 + r32) * D + d] = oacc[0][db][v];
        }
    __syncthreads();
}

// Merges the 4 waves' partial states that decode_pass left in LDS, one thread
// per (column, d) of the first ncols columns: sink(c, d, O, m, l) receives the
// column's merged unnormalised O[d], max and sum.
template <int D, typename Sink>
__device__ __forceinline__ void merge_waves(const uint16_t *smem, int ncols, Sink sink) {
    const float *lm = reinterpret_cast<const float *>(smem);
    const float *ll = lm + 4 * 32;
    const float *lo = ll + 4 * 32;
    for (int task = threadIdx.x; task < ncols * D; task += blockDim.x) {
        const int c = task / D, d = task % D;
        float M = lm[c];
#pragma unroll
        for (int w = 1; w < 4; ++w) M = fmaxf(M, lm[w * 32 + c]);
        float acc = 0.0f, lsum_all = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const float f = __builtin_amdgcn_exp2f(lm[w * 32 + c] - M);
            acc += f * lo[(w * 32 + c) * D + d];
            lsum_all += f * ll[w * 32 + c];
        }
        sink(c, d, acc, M, lsum_all);
    }
}

// Workgroup (b, kv head, split): keys [split*split_len, +split_len), the last
// split also every key past the splits (the host sizes the splits from
// max_seqlen_k, which the reference never reads).  Its rows' partial (m, l, O)
// go to the workspace for fa_decode_combine_kernel.
//
// The host routes to this kernel when G * max_seqlen_q <= 32 and lays the
// columns out for rq = max_seqlen_q rows.  A sequence with more rows than
// that is attended here in full by its split-0 workgroup instead, 32 / G rows
// per pass over all its keys, which writes its output rows itself; the
// combine kernel leaves it alone.  So the output never depends on the host's
// bounds, only the speed does.
// q length of sequence b.
__device__ __forceinline__ int q_len_of(const FaParams &p, int b) {
    return p.q_lens != nullptr ? p.q_lens[b] : p.cu_q[b + 1] - p.cu_q[b];
}

// Split-KV work items of a sequence with q length L and kv length S: every
// split but the last is split_len keys long; the last holds the rest (up to
// the end of the sequence).  A sequence whose q length exceeds the decode
// bound rq, or that has no keys, is one item.
__device__ __forceinline__ int decode_items(const FaParams &p, int L, int S) {
    if (L <= 0 || L > p.rq || S <= 0) return 1;
    return min((S + p.split_len - 1) / p.split_len, p.max_splits);
}

// Keys of the last item, scaled by its query passes (q lengths past rq take
// several) and capped at INT_MAX; -1 for a sequence with no queries (nothing
// to do).
__device__ __forceinline__ int decode_last_work(const FaParams &p, int L, int S) {
    if (L <= 0) return -1;
    if (L > p.rq) {
        const long long w = static_cast<long long>(S) * ((L + 32 / p.G - 1) / (32 / p.G));
        return static_cast<int>(min(w, 0x7fffffffLL));
    }
    return S - (decode_items(p, L, S) - 1) * p.split_len;
}

// Workgroup i's work item in longest-first order, for batches of up to 64
// sequences: first the full split_len items of every sequence (all the same
// size), then each (sequence, kv head) last item, longest first (ties by
// sequence).  Without the ordering the full splits of long sequences are
// dispatched last and run in the tail (equal lengths with the same total keys
// took 183 us against 201 us for lengths spread over 512..8192).  Lane t of
// wave 0 reads sequence t's lengths and leaves the choice in LDS; returns
// false for workgroups past the last item.
__device__ bool decode_item(const FaParams &p, int i, int &b, int &kvh, int &split,
                            long long &q_off, int &L, int &S) {
    __shared__ long long pick_off;
    __shared__ int pick[4];  // sequence, item code, q length, kv length
    if (threadIdx.x < 64) {
        const int t = threadIdx.x;
        if (t == 0) pick[0] = -1;
        int f = 0, w = -2, Lt = 0, St = 0;  // lanes past the batch: w = -2
        long long ot = 0;
        if (t < p.batch) {
            Lt = q_len_of(p, t);
            St = kv_len(p, t);
            if (p.q_lens == nullptr) ot = p.cu_q[t];
            f = (decode_items(p, Lt, St) - 1) * p.Hkv;  // full items
            w = decode_last_work(p, Lt, St);
        }
        int x = f;  // inclusive prefix of the full items
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int v = __shfl_up(x, d, 64);
            if (t >= d) x += v;
        }
        if (p.q_lens != nullptr) {  // q offsets: exclusive prefix of the q lengths
            long long xq = Lt;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const long long vq = __shfl_up(xq, d, 64);
                if (t >= d) xq += vq;
            }
            ot = xq - Lt;
        }
        const int pre = x - f;
        if (t < p.batch && i >= pre && i < pre + f) {
            pick[0] = t;
            pick[1] = i - pre;
            pick[2] = Lt;
            pick[3] = St;
            pick_off = ot;
        }
        const int j = i - __shfl(x, 63, 64);
        if (j >= 0 && j < p.batch * p.Hkv) {
            // last items, longest first: the rank of sequence t, from scalar
            // broadcasts (v_readlane) of every lane's work; a batch whose
            // last items are all the same size keeps sequence order
            const int rank = j / p.Hkv;
            int r = 0;
            if (__all(t >= p.batch || w == __builtin_amdgcn_readfirstlane(w))) {
                r = t;
            } else {
#pragma unroll
                for (int v = 0; v < 64; ++v) {
                    const int wu = __builtin_amdgcn_readlane(w, v);
                    r += (wu > w || (wu == w && v < t)) ? 1 : 0;
                }
            }
            if (t < p.batch && r == rank) {
                pick[0] = t;
                pick[1] = -1 - (j % p.Hkv);
                pick[2] = Lt;
                pick[3] = St;
                pick_off = ot;
            }
        }
    }
    __syncthreads();
    b = pick[0];
    if (b < 0) return false;
    const int r = pick[1];
    L = pick[2];
    S = pick[3];
    q_off = pick_off;
    if (r >= 0) {
        kvh = r % p.Hkv;
        split = r / p.Hkv;
    } else {
        kvh = -1 - r;
        split = decode_items(p, L, S) - 1;
    }
    return true;
}

template <typename T, int D, int BSM>
__global__ void __launch_bounds__(256, D > 128 ? 1 : 2) fa_decode_kernel(FaParams p) {
    extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
    if (blockIdx.x == 0 && blockIdx.y == 0) zero_tail_rows(p, D);
    int b, kvh, split, L, S;
    long long q_off;
    if (p.batch <= 64 && !p.direct) {
        if (!decode_item(p, blockIdx.y * gridDim.x + blockIdx.x, b, kvh, split, q_off, L, S))
            return;
    } else {
        // Larger batches keep the grid's order, (sequence, kv head) by split:
        // with hundreds of items per CU the tail is short, and a scan over
        // every sequence in each workgroup would cost more than it saves.  So
        // do grids of no more workgroups than CUs, which all run at once (32 heads
        // over 8, us by the lookup / in grid order: 4 sequences of 255..1000 keys
        // 13.1 / 11.5, 8 of 258..500 17.3 / 15.3, 1 x 4096 13.1 / 12.5; at up to two
        // per CU 4 x 4095 20.8 / 20.1, but 8 of 258..1656 16.7 / 18.4).
        b = turned_place(blockIdx.x / p.Hkv, blockIdx.y, p.turn, p.batch);
        kvh = blockIdx.x % p.Hkv;
        split = blockIdx.y;
        seq_info(p, b, q_off, L);
        S = kv_len(p, b);
        if (split >= decode_items(p, L, S)) return;
    }
    if (L <= 0) return;
    if (L > p.rq) {
        if (split != 0) return;
        const int rq = 32 / p.G;
        for (int r0 = 0; r0 < L; r0 += rq) {
            decode_pass<T, D, BSM>(p, smem, b, kvh, q_off, L, S, 0, S, rq, r0);
            merge_waves<D>(smem, p.G * rq, [&](int c, int d, float acc, float, float l) {
                const int hl = c / rq, row = r0 + c % rq;
                if (row >= L) return;
                const int h = kvh * p.G + hl;
                p.o[((q_off + row) * p.H + h) * D + d] = Cvt<T>::from(l > 0.0f ? acc / l : 0.0f);
            });
            __syncthreads();  // the next pass refills the LDS
        }
        return;
    }
    const int kv_lo = split * p.split_len;
    const int kv_hi = split == decode_items(p, L, S) - 1 ? S : min(S, kv_lo + p.split_len);
    decode_pass<T, D, BSM>(p, smem, b, kvh, q_off, L, S, kv_lo, kv_hi, p.rq, 0);
    if (p.max_splits == 1) {
        // one split per sequence: the rows are final here, normalised with
        // the merge kernel's arithmetic (the reciprocal of l, then a product),
        // and no merge kernel runs
        merge_waves<D>(smem, p.ncols, [&](int c, int d, float acc, float, float l) {
            const int hl = c / p.rq, row = c % p.rq;
            if (hl >= p.G || row >= L) return;
            const float inv = l > 0.0f ? 1.0f / l : 0.0f;
            p.o[((q_off + row) * p.H + kvh * p.G + hl) * D + d] = Cvt<T>::from(inv * acc);
        });
        return;
    }
    const long long base = ((static_cast<long long>(b) * p.Hkv + kvh) * p.max_splits + split) *
                           p.ncols;
    merge_waves<D>(smem, p.ncols, [&](int c, int d, float acc, float M, float l) {
        p.ws_o[(base + c) * D + d] = acc;
        if (d == 0) {
            p.ws_ml[(base + c) * 2] = M;
            p.ws_ml[(base + c) * 2 + 1] = l;
        }
    });
}

// Merges the split partials of (b, kv head) into the output rows: a row of
// lanes, four dims each, takes every ways-th split of one column, kAhead loads
// at a time.  The first ones are asked for before the lengths are known (splits
// a sequence does not have are skipped afterwards), so with up to kAhead *
// ways splits the kernel is one trip to memory; the ways meet in LDS.  One
// workgroup per (b, kv head), with the weights staged first and one thread per
// element, took 4.4 us of 8 sequences of 255..4095 keys and 27 of 1 x 32768 by
// 1 kv head (8 heads, 64 splits; the call 43 us, now 18).
constexpr int kAhead = 4;

template <int D>
constexpr int combine_rows() {  // rows of lanes in a workgroup (a power of two)
    int n = 1;
    while (2 * n * (D / 4) <= 256) n *= 2;
    return n;
}

template <typename T, int D>
__global__ void __launch_bounds__(256) fa_decode_combine_kernel(FaParams p, int ways) {
    constexpr int ROWS = combine_rows<D>(), V = D / 4;
    // (a caller's workspace need not be aligned to 16 bytes)
    typedef float4_t __attribute__((aligned(4))) float4_u;
    typedef float2_t __attribute__((aligned(4))) float2_u;
    __shared__ __attribute__((aligned(16))) float4_t acc_of[ROWS * V];
    __shared__ float m_of[ROWS], l_of[ROWS];
    const int kvh = blockIdx.x % p.Hkv;
    const int b = blockIdx.x / p.Hkv;
    const int slot = threadIdx.x / V, e = threadIdx.x % V;
    const int way = slot % ways, c = blockIdx.y * (ROWS / ways) + slot / ways;
    const bool active = slot < ROWS && c < p.ncols;
    const long long base = (static_cast<long long>(b) * p.Hkv + kvh) * p.max_splits;
    const float *o_src = p.ws_o + (base * p.ncols + min(c, p.ncols - 1)) * D + 4 * e;
    const float *ml_src = p.ws_ml + (base * p.ncols + min(c, p.ncols - 1)) * 2;
    const long long step = static_cast<long long>(p.ncols);
    float4_t o[kAhead];
    float2_t ml[kAhead];
    const auto load = [&](int s0) {
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int sp = min(s0 + u * ways, p.max_splits - 1);
            ml[u] = *reinterpret_cast<const float2_u *>(ml_src + sp * step * 2);
            o[u] = *reinterpret_cast<const float4_u *>(o_src + sp * step * D);
        }
    };
    load(way);
    long long q_off;
    int L;
    seq_info(p, b, q_off, L);
    if (L <= 0 || L > p.rq) return;  // L > rq: written by fa_decode_kernel
    const int S = kv_len(p, b);
    const int nsplit = min(S <= 0 ? 1 : (S + p.split_len - 1) / p.split_len, p.max_splits);
    float M = 0.0f, l = 0.0f;  // the maxima are clamped at 0
    float4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int s0 = way; s0 < nsplit; s0 += kAhead * ways) {
        if (s0 != way) load(s0);
        float Mn = M;
#pragma unroll
        for (int u = 0; u < kAhead; ++u)
            if (s0 + u * ways < nsplit) Mn = fmaxf(Mn, ml[u].x);
        const float f = __builtin_amdgcn_exp2f(M - Mn);
        M = Mn;
        l *= f;
        acc *= f;
#pragma unroll
        for (int u = 0; u < kAhead; ++u)
            if (s0 + u * ways < nsplit) {
                const float g = __builtin_amdgcn_exp2f(ml[u].x - Mn);
                l += g * ml[u].y;
                acc += g * o[u];
            }
    }
    if (ways > 1) {
        if (slot < ROWS) {
            acc_of[threadIdx.x] = acc;
            if (e == 0) {
                m_of[slot] = M;
                l_of[slot] = l;
            }
        }
        __syncthreads();
        if (!active || way != 0) return;
        for (int w = 1; w < ways; ++w) M = fmaxf(M, m_of[slot + w]);
        l = 0.0f;
        acc = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
        for (int w = 0; w < ways; ++w) {
            const float f = __builtin_amdgcn_exp2f(m_of[slot + w] - M);
            l += f * l_of[slot + w];
            acc += f * acc_of[threadIdx.x + w * V];
        }
    }
    const int hl = c / p.rq, row = c % p.rq;
    if (!active || hl >= p.G || row >= L) return;
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    store_row4<T>(p.o + ((q_off + row) * p.H + kvh * p.G + hl) * D + 4 * e, acc.x * inv, acc.y * inv,
                  acc.z * inv, acc.w * inv);
}

// ------------------------------------------------------------------- host


Plan make_plan(int batch, int H, int Hkv, int q_hint, int k_hint) {
    Plan pl{};
    const int G = H / Hkv;
    pl.decode = q_hint >= 1 && G * q_hint <= 32;
    pl.rq = q_hint;
    pl.rk = k_hint;
    pl.ncols = G * q_hint;
    // Split the key range so that the grid has at least ~512 workgroups (one
    // per slot of the 256 CUs, two each), with splits as long as that allows:
    // from 2048 keys down to 512.  Long splits write and merge fewer
    // partials; at B=64, Hkv=8 and kv_len <= 8192, 2048-key splits ran in
    // 194 us against 217 us at 512.
    // Small grids go on down to one 128-key tile while all workgroups still
    // run at once: then the time is a workgroup's serial chain of tiles.  32
    // heads over 8, us at 512 / 256 / 128 keys: 1 x 600 17.0 / 12.6 / 10.9, 1 x
    // 4096 17.9 / 13.7 / 12.5, 4 of 255..1000 17.6 / 13.1 / 11.4; over 1 kv head 4
    // x 4095 18.2 / 14.1 / 12.3.  Past two workgroups per CU it turns: 4 x 4095
    // 21.1 / 20.8 / 27.1, 8 of 258..1656 18.2 / 16.7 / 23.2, 4 of 677..3209 18.4 /
    // 15.8 / 16.1.
    // Up to 512 keys are never split, so that such a call needs no scratch.
    const long long units = static_cast<long long>(batch) * Hkv;
    const auto groups = [&](int len) { return units * ((k_hint + len - 1) / len); };
    int split = 2048;
    while (split > 512 && groups(split) < 512) split >>= 1;
    if (k_hint > 512)
        while (split <= 512 && split > kDecTile && groups(split / 2) <= 512) split >>= 1;
    pl.split_len = split;
    pl.max_splits = k_hint <= 0 ? 1 : (k_hint + split - 1) / split;
    return pl;
}

size_t workspace_bytes(const Plan &pl, int batch, int Hkv, int D) {
    if (!pl.decode) return 0;
    const size_t per = static_cast<size_t>(batch) * Hkv * pl.max_splits * pl.ncols;
    return per * D * sizeof(float) + per * 2 * sizeof(float) + 256;
}

// Prefill over a grid of ceil(q_hint / QT) query tiles per (b, kv head, head
// group); the workgroups of tile 0 cover any tiles past them.
template <typename T, int D, int W, int HW, int QSUB, int BSM, int TILE>
tecoopsStatus_t launch_prefill(FaParams p, const Plan &pl, hipStream_t s) {
    constexpr int QT = 32 * QSUB * (W / HW);
    auto *kern = &fa_prefill_kernel<T, D, W, HW, QSUB, BSM, TILE>;
    const size_t lds = prefill_lds_bytes<D, TILE, W, HW, QSUB, BSM>();
    if (!tecoops::reserve_lds(reinterpret_cast<const void *>(kern), lds))
        return TECOOPS_STATUS_INTERNAL_ERROR;
    const int units = p.batch * p.Hkv * (p.G / HW);
    const int tiles = (pl.rq + QT - 1) / QT;
    p.turn = turn_shift(p.Hkv * (p.G / HW), p.batch, pl.rq, p.total_q);
    hipLaunchKernelGGL(kern, dim3(units, tiles), dim3(W * 64), lds, s, p);
    TECO_CHECK_LAUNCH("flash_attention prefill");
    return TECOOPS_STATUS_SUCCESS;
}

template <typename T, int D, int W, int QSUB, int BSM, int TILE = 64>
tecoopsStatus_t prefill_hw(const FaParams &p, const Plan &pl, hipStream_t s) {
    const int G = p.G;
    if (G % 4 == 0) return launch_prefill<T, D, W, 4, QSUB, BSM, TILE>(p, pl, s);
    if (G % 2 == 0) return launch_prefill<T, D, W, 2, QSUB, BSM, TILE>(p, pl, s);
    return launch_prefill<T, D, W, 1, QSUB, BSM, TILE>(p, pl, s);
}

// D = 128 prefill route for a query bound of at most 1024 rows: true takes
// the 12-wave kernel (96-row tiles, one workgroup per CU), false the 4-wave
// kernel over 32-row tiles (three per CU).  Over a long cached context the
// 12-wave kernel is ~10 % faster per row and key (each K/V tile serves
// three times the rows), but it pads rows to 96 and has a third of the
// workgroup slots.  So it is taken when the context is long (keys at least
// 4x the rows, or 2x and 2048 or more), its grid covers most CUs (160
// workgroups on 256 CUs), and it needs no more dispatch rounds (workgroups
// over slots, rounded up) than the 32-row kernel.  bf16 H32 Hkv8 causal
// block 16, µs 32-row / 12-wave (batch x query rows / keys):
//   taken: 64 x 64 / 4096 409 / 387, 64 x 96 / 4096 590 / 417, 16 x 256 /
//     4096 354 / 325, 8 x 512 / 4096 323 / 293, 16 x 512 / 2048 291 / 267,
//     8 x 1024 / 2048 246 / 219, 8 x 1024 / 4096 547 / 471, 2 x 1024 /
//     16384 (176 workgroups) 585 / 551, 32 x 256 / 1024 168 / 163, 12 x 700
//     / 4096 605 / 509, 40 x 160 / 4096 594 / 530
//   more rounds: 24 x 250 / 1000 (3 against 2) 120 / 135, 64 x 128 / 1024
//     196 / 222, 64 x 16 / 4096 205 / 358
//   short context: 32 x 256 / 512 88 / 99, 64 x 96 / 192 40 / 42, 64 x 256
//     / 256 105 / 118, 32 x 512 / 512 129 / 152, 16 x 1024 / 1024 191 / 190
//   under 160 workgroups: 4 x 256 / 16384 (96) 434 / 510, 16 x 64 / 16384
//     (128) 443 / 521, 3 x 1024 / 16384 (2 rounds against 1) 830 / 1118
//   where the rule misses: 48 x 200 / 2000 (5 rounds against 4) 482 / 454,
//     6 x 256 / 16384 (144 workgroups) 528 / 516, 16 x 512 / 1024 137 / 135
bool prefill_wide(const FaParams &p, const Plan &pl) {
    const long long q = pl.rq, k = pl.rk;
    if (k < 2 * q || (k < 4 * q && k < 2048)) return false;
    const int hw = p.G % 4 == 0 ? 4 : (p.G % 2 == 0 ? 2 : 1);
    const long long units = static_cast<long long>(p.batch) * p.Hkv * (p.G / hw);
    const long long n12 = units * ((q + 95) / 96), n4 = units * ((q + 31) / 32);
    const long long cus = tecoops::device_cus();
    if (n12 * 256 < 160 * cus) return false;
    return (n12 + cus - 1) / cus <= (n4 + 3 * cus - 1) / (3 * cus);
}

// Whether a prefill is worth splitting over its keys (fa_split.hip), and how;
// the loaders are those that run() picks for these block sizes.
// Without a split a query tile runs over all its keys in one workgroup, so the
// call takes the longest tile's time, or the chip's share of all keys if that
// is more; a split evens the two out for ~12 us of plan and merge.  Measured
// (32 heads of 128 over 8 kv heads, 16-token blocks; unsplit / split, us):
//   1 x 32 rows over 16384 keys 432 / 42, 1 x 256 431 / 94, 4 x 256 433 / 313,
//   4 x 16 over 4096 112 / 35, 16 x 16 113 / 81, 64 x 16 207 / 209, 2 x 1024
//   over 16384 535 / 537, 8 x 512 over 4096 290 / 308: pays where the longest
//   tile is 1.5 times the share and the overhead (twice with one query head
//   per kv head: its tiles are 384 rows).
//   Uneven batches (16..256 rows over 512..7936 cached keys each): 8 chunks 234
//   / 98, 16 172 / 109, 32 267 / 161, 64 556 / 396; the hints hold only the
//   longest, so the share is taken as about half of what they say.  Below some
//   1200 keys past it the gain is down to what the plan and merge take: 40 heads
//   over 8, 9 chunks of 5..21 rows over 919..1272 keys 47 / 56; 32 over 8, 4 of 95..460
//   over 481..520 27 / 34, 6 of 9..238 over 679..1454 49 / 45.
//   Where a cut in two would not fit the slots, contexts may yet be alike and
//   the plan then cuts nothing, for 12 us (10 chunks of 91..307 rows over
//   1954..3087 keys 104 / 116): only long contexts, for which that is little.
//   Fresh prompts (nothing cached) have their tiles' lengths spread evenly
//   and lose: 1 x 4096 157 / 180, 8 of 256..4096 95 / 108.
// The 12-wave kernel reads K and V least often, the 4-wave one (a third of the
// rows per tile) pads less: 16 x 16 over 4096 81 with 4 waves, 111 with 12;
// 4 x 256 over 16384 314 / 313; 32 of 64..1024 rows 638 / 580.
SplitArgs plan_split(const FaParams &p, const Plan &pl, int D) {
    SplitArgs a{0, 256, 0};
    if (pl.decode || (D != 64 && D != 96 && D != 128)) return a;
    if (p.lbs < 3 && (D != 128 || p.bs % 8 != 0)) return a;
    // (the plan's sums are 32-bit)
    if (p.batch > tecoops::fa::kSplitMaxBatch || p.kv_cap > (1 << 20) || p.total_q > (1 << 20)) return a;
    const double past = pl.rk - pl.rq;
    if (past <= 0) return a;
    const int hw = p.G % 4 == 0 ? 4 : (p.G % 2 == 0 ? 2 : 1);
    const int q12 = 32 * (12 / hw), q4 = 32 * (4 / hw);
    const double mean = std::max(1.0, static_cast<double>(p.total_q) / p.batch);
    a.wide = mean + 0.5 * q12 <= 1.2 * (mean + 0.5 * q4);
    const int slots = tecoops::device_cus() * (a.wide ? 1 : D == 128 ? 3 : 2);
    const int qt = a.wide ? q12 : q4;
    const double tiles = static_cast<double>(p.Hkv) * (p.G / hw) * p.batch * std::ceil(mean / qt);
    const double share = tiles * (p.causal ? past + 0.5 * (mean + qt) : pl.rk) / slots;
    const bool uneven = pl.rq >= 1.5 * mean;
    if (pl.rk >= (hw == 1 ? 2.0 : 1.5) * (share + 800.0) ||
        (uneven && pl.rk >= 0.44 * share + 1200.0 && (2 * tiles <= slots || pl.rk >= 6144)))
        a.slots = slots;
    return a;
}

template <typename T, int D>
tecoopsStatus_t run(hipStream_t s, const FaParams &p, const Plan &pl) {
    // Block-size mode (block_of): the uniform-page loaders take block sizes
    // that are multiples of 8 (their 4- and 8-row groups start at multiples
    // of 8, so none crosses a cache block), powers of two with a shift
    const int bsm = p.lbs >= 3 ? 1 : (p.bs % 8 == 0 ? 2 : 0);
    if (pl.decode) {
        const size_t lds = decode_lds_bytes<D>();
        // mode 2 only where a uniform-page loader exists (else mode 0)
        auto *kern = bsm == 1 ? &fa_decode_kernel<T, D, 1> : &fa_decode_kernel<T, D, 0>;
        if constexpr (D == 64 || D == 96 || D == 128)
            if (bsm == 2) kern = &fa_decode_kernel<T, D, 2>;
        if (!tecoops::reserve_lds(reinterpret_cast<const void *>(kern), lds)) return TECOOPS_STATUS_INTERNAL_ERROR;
        dim3 grid(p.batch * p.Hkv, pl.max_splits);
        hipLaunchKernelGGL(kern, grid, dim3(256), lds, s, p);
        TECO_CHECK_LAUNCH("flash_attention decode");
        if (pl.max_splits > 1) {
            // as many ways as leave each kAhead splits or fewer
            constexpr int rows = combine_rows<D>();
            int ways = 1;
            while (ways < rows && ways * kAhead < pl.max_splits) ways *= 2;
            hipLaunchKernelGGL((fa_decode_combine_kernel<T, D>),
                               dim3(p.batch * p.Hkv, tecoops::ceil_div(pl.ncols, rows / ways)), dim3(256),
                               0, s, p, ways);
            TECO_CHECK_LAUNCH("flash_attention combine");
        }
        return TECOOPS_STATUS_SUCCESS;
    }
    if constexpr (D == 128) {
        // the uniform-page loader.  Long query ranges: 12 waves (3 per SIMD)
        // over 96 query rows and 96-key tiles.  Up to 1024 query rows (short
        // prompts, chunks over a cached context): 4 waves over 32 rows and
        // 32-key tiles, three workgroups per CU, which wastes fewer masked
        // rows and hides each workgroup's start-up behind the others, unless
        // prefill_wide finds a long cached context and a full grid.  bf16
        // H32 Hkv8, µs 12-wave / 4-wave: 4 x 4096 643 / 689, 1 x 16384
        // 2162 / 2370.
        const bool wide = pl.rq > 1024 || prefill_wide(p, pl);
        if (bsm == 1) {
            if (!wide) return prefill_hw<T, D, 4, 1, 1, 32>(p, pl, s);
            return prefill_hw<T, D, 12, 1, 1, 96>(p, pl, s);
        }
        if (bsm == 2) {  // block 24, µs mode 0 / 2: B4 S4096 606 / 587, B16 S1024 244 / 208
            if (!wide) return prefill_hw<T, D, 4, 1, 2, 32>(p, pl, s);
            return prefill_hw<T, D, 12, 1, 2, 96>(p, pl, s);
        }
        // other block sizes (the generic loader): the 12-wave kernel above
        // 1024 query rows too.  Block 24, µs 4-wave 64-key / 12-wave: B4
        // S4096 771 / 610, B1 S16384 2868-2883 / 2264-2269 (up to 1024 rows
        // the 4-wave 32-key kernel with this loader lost: 64 x 16 rows over
        // 4096 keys 262 / 342 us)
        if (pl.rq > 1024) return prefill_hw<T, D, 12, 1, 0, 96>(p, pl, s);
    }
    if constexpr (D == 64) {
        // long query ranges: 12 waves over 192-key tiles (3 per SIMD, 136
        // VGPRs).  bf16 H32 Hkv8 causal, µs 4-wave 64-key / 12-wave: B4 S4096
        // 371-376 / 335, B1 S16384 1417-1421 / 1276, B2 S8192 718-733 / 654,
        // B8 S2048 197-201 / 190; 8 waves over 128 keys 362 / 1374 / 701 / 204
        // and 16 over 256 (128 VGPRs, spills) 342 / 1290 / 657 / 192.
        if (bsm == 1 && pl.rq > 1024) return prefill_hw<T, D, 12, 1, 1, 192>(p, pl, s);
        // other block sizes, generic loader: block 24, B4 S4096 433 -> 354 us
        if (pl.rq > 1024) return prefill_hw<T, D, 12, 1, 0, 192>(p, pl, s);
    }
    if constexpr (D == 96) {
        // long query ranges: 12 waves over 96-key tiles (142 VGPRs).  µs
        // 4-wave 64-key / 12-wave 96-key / 12-wave 192-key: B4 S4096 598 /
        // 472 / 486, B1 S16384 2196 / 1771 / 1828, B8 S2048 316 / 267 / 278
        if (bsm == 1 && pl.rq > 1024) return prefill_hw<T, D, 12, 1, 1, 96>(p, pl, s);
        // other block sizes, generic loader: block 24, B4 S4096 648 -> 494 us
        if (pl.rq > 1024) return prefill_hw<T, D, 12, 1, 0, 96>(p, pl, s);
    }
    if constexpr (D == 32) {
        // long query ranges: 8 waves over 128-key tiles.  µs 4-wave 64-key /
        // 12-wave 192-key / 8-wave 128-key: B4 S4096 256 / 245 / 233, B1
        // S16384 986 / 904 / 883, B8 S2048 139 / 142 / 126
        if (pl.rq > 1024)
            return bsm == 1 ? prefill_hw<T, D, 8, 1, 1, 128>(p, pl, s)
                            : prefill_hw<T, D, 8, 1, 0, 128>(p, pl, s);
    }
    if constexpr (D > 128) {
        // 8 waves (2 per SIMD, 234 / 252 VGPRs) over 64-key tiles instead of
        // 4 waves at one per SIMD.  µs, 4 / 8 waves: D = 192 B4 S4096 2078 /
        // 938, B16 S1024 631 / 311, 16 x 256 rows over 4096 keys 1081 / 488,
        // 64 x 16 over 4096 566 / 489; D = 160 1410 / 854, 443 / 284, 691 /
        // 458, and 378 / 477 at 64 x 16 over 4096, where 4 waves stay.
        if (D == 192 || pl.rq > 16)
            return bsm == 1 ? prefill_hw<T, D, 8, 1, 1, 64>(p, pl, s)
                            : prefill_hw<T, D, 8, 1, 0, 64>(p, pl, s);
    }
    return bsm == 1 ? prefill_hw<T, D, 4, 1, 1>(p, pl, s) : prefill_hw<T, D, 4, 1, 0>(p, pl, s);
}

// Head sizes the kernels are built for: the reference takes the head size as
// its K-dimension tile (BK = size_per_head, flash_attention.scpp:188, looped
// at :347-348) in 32-column slabs, bounded by its on-chip buffers.
constexpr int kHeadSizes[] = {32, 64, 96, 128, 160, 192};

bool head_size_supported(int D) {
    for (int d : kHeadSizes)
        if (d == D) return true;
    return false;
}

template <typename T>
tecoopsStatus_t run_d(hipStream_t s, const FaParams &p, const Plan &pl, int D) {
    switch (D) {
        case 32: return run<T, 32>(s, p, pl);
        case 64: return run<T, 64>(s, p, pl);
        case 96: return run<T, 96>(s, p, pl);
        case 128: return run<T, 128>(s, p, pl);
        case 160: return run<T, 160>(s, p, pl);
        case 192: return run<T, 192>(s, p, pl);
        default: return TECOOPS_STATUS_NOT_SUPPORTED;
    }
}

bool is_packed_rowmajor(const tecoopsTensorStruct *d) {
    int expect = 1;
    for (int i = d->nbDims - 1; i >= 0; --i) {
        if (d->dimA[i] > 1 && d->strideA[i] != expect) return false;
        expect *= d->dimA[i];
    }
    return true;
}


// Argument checks of reference flash_attention.cpp:44-69, extended to bf16 and
// to the shape facts the kernels rely on; fills everything but the split-KV
// workspace.  max_seqlen_q / max_seqlen_k are launch-shape hints only: any
// value is accepted (the reference never reads them).  The q hint is raised to
// the mean q length (sum(q) / batch from q's descriptor) and the k hint
// capped by the block-table width * block_size, or taken as that width when
// <= 0.  fixed_hints keeps both as given (a q hint <= 0 becoming the mean),
// for a caller workspace sized by tecoopsGetFlashAttentionWorkspaceSize.
tecoopsStatus_t fa_prepare(tecoopsHandle_t handle, int max_seqlen_q, int max_seqlen_k,
                           const int *q_seq_lens, const int *cu_seqlens_q, const int *kv_seq_lens,
                           const tecoopsTensorDescriptor_t btDesc, const void *blockTable,
                           const tecoopsTensorDescriptor_t qDesc, const void *qData,
                           const tecoopsTensorDescriptor_t kDesc, const void *kCache,
                           const tecoopsTensorDescriptor_t vDesc, const void *vCache,
                           const tecoopsTensorDescriptor_t oDesc, void *oData, float softmax_scale,
                           int causal, bool fixed_hints, FaCall &c) {
    if (handle == nullptr) return TECOOPS_STATUS_NOT_INITIALIZED;
    if (!btDesc || !qDesc || !kDesc || !vDesc || !oDesc) return TECOOPS_STATUS_BAD_PARAM;
    if (!blockTable || !qData || !kCache || !vCache || !oData || !kv_seq_lens)
        return TECOOPS_STATUS_BAD_PARAM;
    if (q_seq_lens == nullptr && cu_seqlens_q == nullptr) return TECOOPS_STATUS_BAD_PARAM;
    TECO_RETURN_IF(kDesc->dataType != vDesc->dataType, TECOOPS_STATUS_BAD_PARAM,
                   "k_cache data_type must be equal to v_cache data_type");
    TECO_RETURN_IF(!tecoops::is_16bit_float(kDesc->dataType), TECOOPS_STATUS_BAD_PARAM,
                   "k/v cache must be TECOOPS_DATA_HALF or TECOOPS_DATA_BFLOAT16");
    TECO_RETURN_IF(qDesc->dataType != kDesc->dataType || oDesc->dataType != kDesc->dataType,
                   TECOOPS_STATUS_BAD_PARAM, "q, k/v cache and output types must agree");
    TECO_RETURN_IF(kDesc->nbDims != 4 || vDesc->nbDims != 4 || qDesc->nbDims != 3 ||
                   oDesc->nbDims != 3 || btDesc->nbDims != 2,
                   TECOOPS_STATUS_BAD_PARAM, "flash_attention: unexpected tensor ranks");
    for (int i = 0; i < 4; ++i)
        TECO_RETURN_IF(kDesc->dimA[i] != vDesc->dimA[i], TECOOPS_STATUS_BAD_PARAM,
                       "shape of k v cache is not equal");
    for (int i = 0; i < 3; ++i)
        TECO_RETURN_IF(qDesc->dimA[i] != oDesc->dimA[i], TECOOPS_STATUS_BAD_PARAM,
                       "q and output shapes differ");
    const int total_q = qDesc->dimA[0], H = qDesc->dimA[1], D = qDesc->dimA[2];
    const int num_blocks = kDesc->dimA[0], Hkv = kDesc->dimA[1], bs = kDesc->dimA[2];
    const int batch = btDesc->dimA[0], bt_cols = btDesc->dimA[1];
    TECO_RETURN_IF(kDesc->dimA[3] != D, TECOOPS_STATUS_BAD_PARAM, "head_size mismatch");
    TECO_RETURN_IF(!head_size_supported(D), TECOOPS_STATUS_NOT_SUPPORTED,
                   "flash_attention: head_size %d not supported (32, 64, 96, 128, 160, 192)", D);
    TECO_RETURN_IF(H <= 0 || Hkv <= 0 || H % Hkv != 0, TECOOPS_STATUS_BAD_PARAM,
                   "num_heads must be a multiple of num_kv_heads");
    TECO_RETURN_IF(bs <= 0 || num_blocks <= 0 || batch <= 0 || total_q < 0 || bt_cols < 0,
                   TECOOPS_STATUS_BAD_PARAM, "empty cache or batch");
    TECO_RETURN_IF(fixed_hints && max_seqlen_k <= 0, TECOOPS_STATUS_BAD_PARAM,
                   "flash_attention: a caller workspace needs the max_seqlen_k it was sized for");
    TECO_RETURN_IF(!is_packed_rowmajor(qDesc) || !is_packed_rowmajor(oDesc) ||
                   !is_packed_rowmajor(kDesc) || !is_packed_rowmajor(vDesc) ||
                   btDesc->strideA[1] != 1,
                   TECOOPS_STATUS_NOT_SUPPORTED, "flash_attention: tensors must be row-major");
    for (const void *ptr : {qData, kCache, vCache, static_cast<const void *>(oData)})
        TECO_RETURN_IF(!tecoops::aligned(ptr, 16), TECOOPS_STATUS_BAD_PARAM,
                       "flash_attention: tensors must be 16-byte aligned");

    FaParams &p = c.p;
    p = FaParams{};
    p.q = static_cast<const uint16_t *>(qData);
    p.kc = static_cast<const uint16_t *>(kCache);
    p.vc = static_cast<const uint16_t *>(vCache);
    p.o = static_cast<uint16_t *>(oData);
    p.bt = static_cast<const int *>(blockTable);
    p.bt_stride = btDesc->strideA[0];
    p.q_lens = q_seq_lens;
    p.cu_q = cu_seqlens_q;
    p.kv_lens = kv_seq_lens;
    p.batch = batch;
    p.H = H;
    p.Hkv = Hkv;
    p.G = H / Hkv;
    p.bs = bs;
    p.lbs = (bs & (bs - 1)) == 0 ? __builtin_ctz(static_cast<unsigned>(bs)) : -1;
    p.num_blocks = num_blocks;
    const long long cap = static_cast<long long>(bt_cols) * bs;
    p.kv_cap = cap > 0x7fffffffLL ? 0x7fffffff : static_cast<int>(cap);
    p.page_stride = static_cast<long long>(Hkv) * bs * D;
    const float scale = softmax_scale > 0.0f ? softmax_scale : 1.0f / std::sqrt(static_cast<float>(D));
    p.scale_log2 = scale * 1.4426950408889634f;
    p.inv_scale_log2 = 1.0f / p.scale_log2;
    p.causal = causal != 0;

    // The q bound routes the call (decode or prefill) and sizes the prefill
    // grid.  It is raised to the mean q length, which the host knows: a bound
    // that is too small (the reference never reads it) would otherwise send a
    // prefill down the decode route, correct but many times slower.  A caller
    // workspace was sized for the bounds as given, so they are kept then.
    const int q_mean = std::max(1, (total_q + batch - 1) / batch);
    const int q_hint = fixed_hints ? (max_seqlen_q > 0 ? max_seqlen_q : q_mean)
                                    : std::max(max_seqlen_q, q_mean);
    int k_hint = max_seqlen_k;
    if (!fixed_hints) k_hint = max_seqlen_k > 0 ? std::min(max_seqlen_k, p.kv_cap) : p.kv_cap;
    c.pl = make_plan(batch, H, Hkv, q_hint, k_hint);
    p.total_q = total_q;
    if (c.pl.decode) {
        p.rq = c.pl.rq;
        p.ncols = c.pl.ncols;
        p.split_len = c.pl.split_len;
        p.max_splits = c.pl.max_splits;
        p.turn = turn_shift(p.Hkv, p.batch);
        p.direct = static_cast<long long>(p.batch) * p.Hkv * p.max_splits <= tecoops::device_cus();
    } else {
        p.rq = 0x7fffffff;
    }
    c.split = plan_split(p, c.pl, D);
    c.D = D;
    c.bf16 = kDesc->dataType == TECOOPS_DATA_BFLOAT16;
    return TECOOPS_STATUS_SUCCESS;
}

size_t fa_workspace_bytes(const FaCall &c) {
    return workspace_bytes(c.pl, c.p.batch, c.p.Hkv, c.D);
}

// Enqueues the call on stream s with its split-KV partials in ws (at least
// fa_workspace_bytes(c) bytes; a prefill that may split does so if ws, of
// split_bytes, is given).
tecoopsStatus_t fa_launch(hipStream_t s, FaCall &c, void *ws) {
    if (c.pl.decode) {
        const size_t per = static_cast<size_t>(c.p.batch) * c.p.Hkv * c.pl.max_splits * c.pl.ncols;
        c.p.ws_o = static_cast<float *>(ws);
        c.p.ws_ml = c.p.ws_o + per * c.D;
    }
    if (!c.pl.decode && c.split.slots > 0 && ws != nullptr) {
        c.p.ws_plan = ws;
        c.p.ws_o = reinterpret_cast<float *>(static_cast<char *>(ws) + tecoops::fa::kSplitPlanBytes);
        return tecoops::fa::launch_split(s, c.p, c.split, c.D, c.bf16);
    }
    using tecoops::dev::bf16;
    using tecoops::dev::f16;
    return c.bf16 ? run_d<bf16>(s, c.p, c.pl, c.D) : run_d<f16>(s, c.p, c.pl, c.D);
}

}  // namespace

namespace tecoops {
namespace fa {

tecoopsStatus_t prepare(tecoopsHandle_t handle, int max_seqlen_q, int max_seqlen_k,
                        const int *q_seq_lens, const int *cu_seqlens_q, const int *kv_seq_lens,
                        const tecoopsTensorDescriptor_t btDesc, const void *blockTable,
                        const tecoopsTensorDescriptor_t qDesc, const void *qData,
                        const tecoopsTensorDescriptor_t kDesc, const void *kCache,
                        const tecoopsTensorDescriptor_t vDesc, const void *vCache,
                        const tecoopsTensorDescriptor_t oDesc, void *oData, float softmax_scale,
                        int causal, bool fixed_hints, FaCall &c) {
    return fa_prepare(handle, max_seqlen_q, max_seqlen_k, q_seq_lens, cu_seqlens_q, kv_seq_lens,
                      btDesc, blockTable, qDesc, qData, kDesc, kCache, vDesc, vCache, oDesc, oData,
                      softmax_scale, causal, fixed_hints, c);
}

size_t workspace_bytes(const FaCall &c) { return fa_workspace_bytes(c); }

size_t workspace_bytes(int batch, int H, int Hkv, int D, int q_hint, int k_hint) {
    return ::workspace_bytes(make_plan(batch, H, Hkv, q_hint, k_hint), batch, Hkv, D);
}

tecoopsStatus_t launch(hipStream_t s, FaCall &c, void *ws) { return fa_launch(s, c, ws); }

}  // namespace fa
}  // namespace tecoops

extern "C" tecoopsStatus_t tecoopsGetFlashAttentionWorkspaceSize(int batch, int num_heads,
                                                                 int head_size, int max_seqlen_q,
                                                                 int max_seqlen_k, size_t *bytes) {
    if (bytes == nullptr || batch <= 0 || num_heads <= 0 || head_size <= 0 || max_seqlen_k <= 0)
        return TECOOPS_STATUS_BAD_PARAM;
    // Worst case over kv-head counts; max_seqlen_q <= 0 takes the longest q
    // length the decode route admits (32 / G rows).
    size_t worst = 0;
    for (int hkv = 1; hkv <= num_heads; ++hkv) {
        if (num_heads % hkv) continue;
        const int G = num_heads / hkv;
        const int q_hint = max_seqlen_q > 0 ? max_seqlen_q : std::max(1, 32 / G);
        const Plan pl = make_plan(batch, num_heads, hkv, q_hint, max_seqlen_k);
        const size_t b = workspace_bytes(pl, batch, hkv, head_size);
        if (b > worst) worst = b;
    }
    *bytes = worst;
    return TECOOPS_STATUS_SUCCESS;
}

extern "C" tecoopsStatus_t tecoopsFlashAttentionEx(
    tecoopsHandle_t handle, int max_seqlen_q, int max_seqlen_k, const int *q_seq_lens,
    const int *cu_seqlens_q, const int *kv_seq_lens, const tecoopsTensorDescriptor_t btDesc,
    const void *blockTable, const tecoopsTensorDescriptor_t qDesc, const void *qData,
    const tecoopsTensorDescriptor_t kDesc, const void *kCache,
    const tecoopsTensorDescriptor_t vDesc, const void *vCache,
    const tecoopsTensorDescriptor_t oDesc, void *oData, float softmax_scale, int causal,
    void *workspace) {
    FaCall c;
    tecoopsStatus_t st = fa_prepare(handle, max_seqlen_q, max_seqlen_k, q_seq_lens, cu_seqlens_q,
                                    kv_seq_lens, btDesc, blockTable, qDesc, qData, kDesc, kCache,
                                    vDesc, vCache, oDesc, oData, softmax_scale, causal,
                                    workspace != nullptr, c);
    if (st != TECOOPS_STATUS_SUCCESS) return st;
    // A caller's workspace is sized for the decode route.  A prefill is split
    // where the handle has scratch to spare (not under capture) and runs
    // unsplit, to the same values up to rounding, where it does not.
    void *ws = c.pl.decode ? workspace : nullptr;
    if (c.split.slots > 0 && workspace == nullptr)
        ws = tecoops::handle_scratch_if_any(handle, tecoops::fa::split_bytes(c.split, c.D));
    // With one split per sequence the decode kernel writes the output rows
    // itself and reads no partials: no scratch is needed then.
    if (c.pl.decode && c.pl.max_splits > 1 && ws == nullptr) {
        st = tecoops::handle_scratch(handle, fa_workspace_bytes(c), &ws);
        if (st != TECOOPS_STATUS_SUCCESS) return st;
    }
    return fa_launch(handle->stream, c, ws);
}

extern "C" tecoopsStatus_t tecoopsFlashAttention(
    tecoopsHandle_t handle, int max_seqlen_q, int max_seqlen_k, int max_block_num,
    const int *q_seq_lens, const int *kv_seq_lens, const tecoopsTensorDescriptor_t blockTableDesc,
    const void *blockTable, const tecoopsTensorDescriptor_t qDataDesc, const void *qData,
    const tecoopsTensorDescriptor_t kCacheDesc, const void *kCache,
    const tecoopsTensorDescriptor_t vCacheDesc, const void *vCache,
    const tecoopsTensorDescriptor_t oDataDesc, void *oData, void *workspace) {
    // The reference accepts workspace and never reads it
    // (flash_attention.cpp:110), and takes the block count from kCacheDesc:
    // both are ignored here too, so a caller's unrelated buffer is never
    // written.  The split-KV partials live in the handle's scratch.
    (void)max_block_num;
    (void)workspace;
    if (q_seq_lens == nullptr) return handle ? TECOOPS_STATUS_BAD_PARAM : TECOOPS_STATUS_NOT_INITIALIZED;
    return tecoopsFlashAttentionEx(handle, max_seqlen_q, max_seqlen_k, q_seq_lens, nullptr,
                                   kv_seq_lens, blockTableDesc, blockTable, qDataDesc, qData,
                                   kCacheDesc, kCache, vCacheDesc, vCache, oDataDesc, oData,
                                   -1.0f, 1, nullptr);
}

