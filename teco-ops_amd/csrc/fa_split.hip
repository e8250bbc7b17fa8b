// fa_split.hip — prefill over split keys: query tiles whose keys are cut into
// pieces of about equal work, one workgroup each.
//
// fa_prefill_kernel gives a query tile all its keys, so a batch with few query
// tiles and long or uneven contexts (chunks of a prompt over a cached context,
// a few prompts of different lengths) runs as long as its longest tile while
// most CUs are idle.  Here fa_split_plan_kernel reads the lengths on the
// device and picks a piece length; a tile with more keys than that is cut into
// pieces of it, whose unnormalised states (fp32) go to a workspace and are
// merged by fa_split_merge_kernel.  The plan, and with it the rounding of the
// result, depends on the lengths and the call's sizes alone.
//
// Bound like fa_prefill_kernel (a slot's serial loop over its keys); the plan
// takes ~6 us, the merge 5-14 (traced; 16 chunks as below 6.7 and 14.6).  16 chunks of 16..256 rows over 512..7936
// cached keys (32 heads of 128 over 8 kv heads): 172 us unsplit, 109 split; 1 x
// 32 rows over 16384 keys 432 / 42.  When a call is split: plan_split in
// flash_attention.hip.
#include <algorithm>

#include "fa_device.h"

namespace {

using tecoops::fa::kSplitMaxBatch;
using tecoops::fa::SplitArgs;

// Sum of ceil(j / k) for j = 1 .. m.
__device__ __forceinline__ int sum_ceil(int m, int k) {
    const int q = m / k, r = m - q * k;
    return k * (q * (q + 1) / 2) + r * (q + 1);
}

// The pieces of one sequence, in units of QT keys: query tile t of n sees
// min(a + t + 1, s) of them.
struct SeqPieces {
    int n, a, s;
    __device__ __forceinline__ int seen(int t) const { return min(a + t + 1, s); }
    // all tiles' units
    __device__ __forceinline__ long long units() const {
        const long long m = min(n, s - a);
        return m * a + m * (m + 1) / 2 + static_cast<long long>(n - m) * s;
    }
    __device__ __forceinline__ int pieces(int t, int k) const { return max(1, (seen(t) + k - 1) / k); }
    // pieces of tiles 0 .. n-1
    __device__ __forceinline__ int all(int k) const {
        const int m = min(n, s - a);
        return sum_ceil(a + m, k) - sum_ceil(a, k) + (n - m) * max(1, (s + k - 1) / k);
    }
    // tiles of a single piece (the first ones)
    __device__ __forceinline__ int single(int k) const { return s <= k ? n : min(max(k - a, 0), n); }
};

__device__ __forceinline__ SeqPieces seq_pieces(const FaParams &p, int b, int qt) {
    SeqPieces q{0, 0, 0};
    if (b >= p.batch) return q;  // no tiles
    const int L = p.q_lens != nullptr ? p.q_lens[b] : p.cu_q[b + 1] - p.cu_q[b];
    const int S = kv_len(p, b);
    q.n = max(0, (L + qt - 1) / qt);
    q.s = (S + qt - 1) / qt;
    q.a = p.causal ? min(q.s, (max(S - L, 0) + qt - 1) / qt) : q.s;
    return q;
}

// The plan, at the start of the workspace: units of QT keys per piece, and
// for each sequence in the order they run (and the end) what comes before it.
struct PlanOut {
    int k;
    int order[kSplitMaxBatch];       // sequences, longest first
    int pieces[kSplitMaxBatch + 1];  // pieces of one unit (kv head and head group)
    int cut[kSplitMaxBatch + 1];     // those of tiles cut in two or more
    int tiles[kSplitMaxBatch + 1];   // tiles cut in two or more
};
static_assert(sizeof(PlanOut) <= tecoops::fa::kSplitPlanBytes, "the plan's part of the workspace");

// One workgroup.  Candidate j (lane) cuts the longest tile into j + 1 pieces;
// its cost in keys is the longest piece when all pieces run at once, else
// their mean over the slots and a piece for the last round, and what the cut
// pieces' states and the merge take.  Only candidates whose pieces fit the
// workspace and the grid count; the uncut one always does.
constexpr float kPieceKeys = 384.0f;   // a piece's start and end
constexpr float kMergeKeys = 200.0f;   // the merge
// ... and per cut piece for its state (12 waves x 128 dims: 196 KiB written
// and read at ~5 TB/s, while a slot takes ~22 keys per us)
constexpr float kStateKeys = 1.73f / (12 * 128);
// A cut has to promise a tenth: for eight prompts of 256..4096 rows it promised
// less and took 135 us for 95; at a quarter, 16 chunks at 64 dims stay uncut
// (155 us for 88).
constexpr float kCutMargin = 1.1f;

__global__ void __launch_bounds__(256) fa_split_plan_kernel(FaParams p, SplitArgs a, int qt, int step,
                                                            int units, int wd) {
    __shared__ int part[4][64], cutp[4][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    PlanOut *out = reinterpret_cast<PlanOut *>(p.ws_plan);
    const SeqPieces mine = seq_pieces(p, lane, qt);  // sequence `lane`
    int m = mine.n > 0 ? mine.seen(mine.n - 1) : 0;
    long long total = mine.units();
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) {
        m = max(m, __shfl_xor(m, d, 64));
        total += __shfl_xor(total, d, 64);
    }
    // lane = candidate: units per piece, whole K/V tiles
    int k = (m + lane) / (lane + 1);
    k = max(max(k, (a.least + qt - 1) / qt), 1);
    k = (k + step - 1) / step * step;
    int all = 0, cut = 0;
    for (int b = wave; b < p.batch; b += 4) {
        SeqPieces q;
        q.n = __builtin_amdgcn_readlane(mine.n, b);
        q.a = __builtin_amdgcn_readlane(mine.a, b);
        q.s = __builtin_amdgcn_readlane(mine.s, b);
        const int x = q.all(k);
        all += x;
        cut += x - q.single(k);
    }
    part[wave][lane] = all;
    cutp[wave][lane] = cut;
    __syncthreads();
    if (wave != 0) return;
    all = part[0][lane] + part[1][lane] + part[2][lane] + part[3][lane];
    cut = cutp[0][lane] + cutp[1][lane] + cutp[2][lane] + cutp[3][lane];
    int tiles = mine.n;
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) tiles += __shfl_xor(tiles, d, 64);
    const float keys = static_cast<float>(k) * qt + kPieceKeys;
    const float pieces = static_cast<float>(all) * units;
    float cost = pieces <= a.slots ? keys
                                   : (static_cast<float>(total) * qt * units + pieces * kPieceKeys) / a.slots + keys;
    if (cut > 0) cost = kCutMargin * (cost + kMergeKeys + kStateKeys * wd * cut * units);
    if (lane > 0 && ((all - tiles) * units > a.slots || cut * units > 2 * a.slots)) cost = 3.0e38f;
    float best = cost;
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) best = fminf(best, __shfl_xor(best, d, 64));
    const unsigned long long who = __ballot(cost == best);
    k = __builtin_amdgcn_readlane(k, __builtin_ctzll(who));
    // the sequences by their longest tile, so that the last workgroups to start
    // are short ones (lane = sequence, then place)
    const int key = mine.n > 0 ? mine.seen(mine.n - 1) : -1;
    int rank = 0;
#pragma unroll
    for (int v = 0; v < 64; ++v) {
        const int other = __builtin_amdgcn_readlane(key, v);
        rank += other > key || (other == key && v < lane) ? 1 : 0;
    }
    const int seq = __builtin_amdgcn_ds_permute(rank << 2, lane);  // lane `rank` gets this lane's number
    const SeqPieces at = seq_pieces(p, seq, qt);
    // prefixes over the sequences in that order
    const int np = at.all(k), one = at.single(k);
    int x = np, y = np - one, z = at.n - one;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int vx = __shfl_up(x, d, 64), vy = __shfl_up(y, d, 64), vz = __shfl_up(z, d, 64);
        if (lane >= d) {
            x += vx;
            y += vy;
            z += vz;
        }
    }
    if (lane < p.batch) {
        out->order[lane] = seq;
        out->pieces[lane + 1] = x;
        out->cut[lane + 1] = y;
        out->tiles[lane + 1] = z;
    }
    if (lane == 0) {
        out->k = k;
        out->pieces[0] = out->cut[0] = out->tiles[0] = 0;
    }
}

// A workgroup's piece (or, for the merge, its tile of two pieces or more).
struct Piece {
    int b, t, u;   // sequence, query tile, unit (kv head and head group)
    int s, n;      // piece s of n
    int slot;      // workspace slot of piece 0 (pieces are `units` slots apart)
    int k;         // units of QT keys per piece of this tile
};

// The i-th piece (MERGE: the i-th tile of several pieces) in the order
// sequence, heaviest tile first, piece, unit; false past the last.  A tile's
// pieces are cut evenly (to whole K/V tiles, so the last may be empty): with
// full pieces and a remainder, long and short ones would alternate, and an
// XCD deals its workgroups to its shader engines in turn.
template <bool MERGE>
__device__ __forceinline__ bool pick_piece(const FaParams &p, int qt, int step, int units, int i,
                                           Piece &r) {
    const auto *pl = (const __attribute__((address_space(4))) PlanOut *)(p.ws_plan);
    const int at = i / units;
    r.u = i - at * units;
    const int k = pl->k;
    const auto before = [&](int b) { return MERGE ? pl->tiles[b] : pl->pieces[b]; };
    if (at >= before(p.batch)) return false;
    int lo = 0, hi = p.batch - 1;  // the last sequence with before(b) <= at
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (before(mid) <= at) lo = mid; else hi = mid - 1;
    }
    r.b = pl->order[lo];
    const int j = at - before(lo), first = pl->cut[lo];
    SeqPieces q = seq_pieces(p, r.b, qt);
    q.n = __builtin_amdgcn_readfirstlane(q.n);
    q.a = __builtin_amdgcn_readfirstlane(q.a);
    q.s = __builtin_amdgcn_readfirstlane(q.s);
    if constexpr (MERGE) {
        r.t = q.n - 1 - j;
        r.s = 0;
        r.n = q.pieces(r.t, k);
        SeqPieces upto = q;  // the pieces of the tiles after this one come first
        upto.n = r.t + 1;
        r.slot = (first + q.all(k) - upto.all(k)) * units + r.u;
        return true;
    }
    // tiles from the heaviest on, 64 at a time: the one that holds piece j
    const int lane = threadIdx.x & 63;
    int base = 0;  // pieces of the tiles before these
    for (int t1 = q.n - 1; t1 >= 0; t1 -= 64) {
        const int t = t1 - lane;
        const int np = t >= 0 ? q.pieces(t, k) : 0;
        int x = np;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int v = __shfl_up(x, d, 64);
            if (lane >= d) x += v;
        }
        const unsigned long long hit = __ballot(base + x > j);
        if (hit != 0) {
            const int l = __builtin_ctzll(hit);
            r.t = t1 - l;
            r.n = __builtin_amdgcn_readlane(np, l);
            const int start = base + __builtin_amdgcn_readlane(x, l) - r.n;
            r.s = j - start;
            r.slot = (first + start) * units + r.u;
            r.k = (q.seen(r.t) + r.n - 1) / r.n;
            r.k = (r.k + step - 1) / step * step;
            return true;
        }
        base += __builtin_amdgcn_readlane(x, 63);
    }
    return false;
}

template <int TILE, int QT>
constexpr int piece_step() {
    return TILE > QT ? TILE / QT : 1;
}

template <typename T, int D, int W, int HW, int BSM, int TILE>
__global__ void __launch_bounds__(W * 64, (W >= 12 || TILE == 32) ? 3 : 2)
fa_split_kernel(FaParams p) {
    constexpr int QT = 32 * (W / HW);
    static_assert(QT % TILE == 0 || TILE % QT == 0, "pieces are whole K/V tiles");
    extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
    if (blockIdx.x == 0) zero_tail_rows(p, D);
    const int ngroups = p.G / HW, units = p.Hkv * ngroups;
    Piece r;
    if (!pick_piece<false>(p, QT, piece_step<TILE, QT>(), units, blockIdx.x, r)) return;
    long long q_off;
    int L;
    seq_info(p, r.b, q_off, L);
    const int S = kv_len(p, r.b);
    const int kv_lo = r.s * r.k * QT;
    float *part = r.n > 1 ? p.ws_o + static_cast<long long>(r.slot + r.s * units) * (W * frag_floats<D>())
                          : nullptr;
    prefill_tile<T, D, W, HW, 1, BSM, TILE, true>(p, lds, r.b, r.u / ngroups, r.u % ngroups, q_off, L,
                                                  S, r.t * QT, kv_lo,
                                                  r.n > 1 ? kv_lo + r.k * QT : 0x7fffffff, part);
}

// Merges the pieces of a split tile: workgroup (tile, wave w of the tile's
// workgroups) the 32 rows x D values of one head.  A wave takes DBW blocks of
// 32 dims of every kMergeWays-th piece; the ways meet in LDS.  The pieces'
// states are read as they were written (1 KiB per instruction), the rows leave
// through LDS in 16-byte stores.  A tile of 64 pieces (32 rows over 16384
// keys): 67 us with one way, 17 with four.
constexpr int kMergeWays = 4;

template <int D>
constexpr int merge_blocks() {
    return D % 64 == 0 ? 2 : 1;
}
template <int D>
constexpr int merge_threads() {
    return 64 * kMergeWays * (D / 32 / merge_blocks<D>());
}

template <typename T, int D, int W, int HW>
__global__ void __launch_bounds__(merge_threads<D>()) fa_split_merge_kernel(FaParams p) {
    constexpr int QT = 32 * (W / HW), NT = merge_threads<D>(), ROW = D + 8;
    constexpr int DBW = merge_blocks<D>(), WPW = D / 32 / DBW;  // waves per way
    __shared__ __attribute__((aligned(16))) uint16_t rows[32 * ROW];
    __shared__ __attribute__((aligned(16))) float sums[kMergeWays - 1][D / 32][4 * 64 * 4];
    __shared__ float lsum[kMergeWays][32];
    const int ngroups = p.G / HW, units = p.Hkv * ngroups;
    Piece r;
    if (!pick_piece<true>(p, QT, 1, units, blockIdx.x, r)) return;
    long long q_off;
    int L;
    seq_info(p, r.b, q_off, L);
    const int w = blockIdx.y;
    const int h = (r.u / ngroups) * p.G + (r.u % ngroups) * HW + w % HW;
    const int row0 = r.t * QT + (w / HW) * 32;
    if (row0 >= L) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int db0 = wave % WPW * DBW, way = wave / WPW;
    const int g = lane >> 5, r32 = lane & 31;
    const long long pitch = static_cast<long long>(units) * W * frag_floats<D>();
    const float *f = p.ws_o + (static_cast<long long>(r.slot) * W + w) * frag_floats<D>();
    const float *ml = f + 32 * D + 2 * r32;
    float M = 0.0f;  // the running maxima are clamped at 0
#pragma unroll 8
    for (int s = 0; s < r.n; ++s) M = fmaxf(M, ml[s * pitch]);
    float l = 0.0f;
    float4_t o[4 * DBW];
#pragma unroll
    for (int u = 0; u < 4 * DBW; ++u) o[u] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 2
    for (int s = way; s < r.n; s += kMergeWays) {
        const float2_t v = *reinterpret_cast<const float2_t *>(ml + s * pitch);
        const float e = __builtin_amdgcn_exp2f(v.x - M);
        l += e * v.y;
#pragma unroll
        for (int u = 0; u < 4 * DBW; ++u)
            o[u] += e * *reinterpret_cast<const float4_t *>(f + s * pitch + ((db0 * 4 + u) * 64 + lane) * 4);
    }
    if (way > 0) {
#pragma unroll
        for (int u = 0; u < 4 * DBW; ++u)
            *reinterpret_cast<float4_t *>(&sums[way - 1][db0 + u / 4][(u % 4 * 64 + lane) * 4]) = o[u];
    }
    if (db0 == 0 && g == 0) lsum[way][r32] = l;
    __syncthreads();
    if (way == 0) {
        l = 0.0f;
#pragma unroll
        for (int v = 0; v < kMergeWays; ++v) l += lsum[v][r32];
        const float inv = l > 0.0f ? 1.0f / l : 0.0f;
#pragma unroll
        for (int u = 0; u < 4 * DBW; ++u) {
#pragma unroll
            for (int v = 0; v < kMergeWays - 1; ++v)
                o[u] += *reinterpret_cast<const float4_t *>(&sums[v][db0 + u / 4][(u % 4 * 64 + lane) * 4]);
            store_row4<T>(rows + r32 * ROW + 32 * (db0 + u / 4) + 8 * (u % 4) + 4 * g, o[u].x * inv,
                          o[u].y * inv, o[u].z * inv, o[u].w * inv);
        }
    }
    __syncthreads();
    for (int c = threadIdx.x; c < 32 * D / 8; c += NT) {
        const int rr = c / (D / 8), cc = c % (D / 8);
        if (row0 + rr < L)
            *reinterpret_cast<u32x4 *>(p.o + ((q_off + row0 + rr) * p.H + h) * D + cc * 8) =
                *reinterpret_cast<const u32x4 *>(rows + rr * ROW + cc * 8);
    }
}

// ------------------------------------------------------------------- host

template <typename T, int D, int W, int HW, int BSM, int TILE>
tecoopsStatus_t launch_hw(hipStream_t s, const FaParams &p, const SplitArgs &a) {
    constexpr int QT = 32 * (W / HW);
    auto *kern = &fa_split_kernel<T, D, W, HW, BSM, TILE>;
    const size_t lds = prefill_lds_bytes<D, TILE, W, HW, 1, BSM>();
    if (!tecoops::reserve_lds(reinterpret_cast<const void *>(kern), lds))
        return TECOOPS_STATUS_INTERNAL_ERROR;
    const int units = p.Hkv * (p.G / HW);
    // query tiles of any batch of these sizes, and the cuts (fewer than slots)
    const long long tiles = (p.total_q + QT - 1) / QT + p.batch;
    hipLaunchKernelGGL(fa_split_plan_kernel, dim3(1), dim3(256), 0, s, p, a, QT, piece_step<TILE, QT>(),
                       units, W * D);
    TECO_CHECK_LAUNCH("flash_attention split plan");
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(tiles * units + a.slots)), dim3(W * 64), lds, s,
                       p);
    TECO_CHECK_LAUNCH("flash_attention split prefill");
    hipLaunchKernelGGL((fa_split_merge_kernel<T, D, W, HW>),
                       dim3(static_cast<unsigned>(std::min<long long>(a.slots, tiles * units)), W),
                       dim3(merge_threads<D>()), 0, s, p);
    TECO_CHECK_LAUNCH("flash_attention split merge");
    return TECOOPS_STATUS_SUCCESS;
}

template <typename T, int D, int W, int BSM, int TILE>
tecoopsStatus_t launch_g(hipStream_t s, const FaParams &p, const SplitArgs &a) {
    if (p.G % 4 == 0) return launch_hw<T, D, W, 4, BSM, TILE>(s, p, a);
    if (p.G % 2 == 0) return launch_hw<T, D, W, 2, BSM, TILE>(s, p, a);
    return launch_hw<T, D, W, 1, BSM, TILE>(s, p, a);
}

template <typename T>
tecoopsStatus_t launch_d(hipStream_t s, const FaParams &p, const SplitArgs &a, int D) {
    if (D == 64) return a.wide ? launch_g<T, 64, 12, 1, 192>(s, p, a) : launch_g<T, 64, 4, 1, 64>(s, p, a);
    if (D == 96) return a.wide ? launch_g<T, 96, 12, 1, 96>(s, p, a) : launch_g<T, 96, 4, 1, 64>(s, p, a);
    if (p.lbs >= 3) return a.wide ? launch_g<T, 128, 12, 1, 96>(s, p, a) : launch_g<T, 128, 4, 1, 32>(s, p, a);
    return a.wide ? launch_g<T, 128, 12, 2, 96>(s, p, a) : launch_g<T, 128, 4, 2, 32>(s, p, a);
}

}  // namespace

namespace tecoops {
namespace fa {

size_t split_bytes(const SplitArgs &a, int D) {
    return kSplitPlanBytes +
           static_cast<size_t>(2) * a.slots * (a.wide ? 12 : 4) * (32 * D + 64) * sizeof(float);
}

tecoopsStatus_t launch_split(hipStream_t s, const FaParams &p, const SplitArgs &a, int D, bool is_bf16) {
    return is_bf16 ? launch_d<dev::bf16>(s, p, a, D) : launch_d<dev::f16>(s, p, a, D);
}

}  // namespace fa
}  // namespace tecoops
