// fa_device.h — device code shared by the flash-attention kernels
// (flash_attention.hip, fa_split.hip): K/V tile loaders, the attention of one
// wave over staged keys, and the prefill of one query tile.
#pragma once

#include <cmath>

#include "common.h"
#include "device.h"
#include "flash_attention.h"

namespace {

using namespace tecoops::dev;
using tecoops::fa::FaParams;

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef float float2_t __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

template <typename T> struct Mma;
template <> struct Mma<bf16> {
    static __device__ __forceinline__ f32x16_t run(const u32x4 &a, const u32x4 &b, f32x16_t c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                       __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t pack2(float a, float b) {
        float2_t v = {a, b};
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf162_t));
    }
};
template <> struct Mma<f16> {
    static __device__ __forceinline__ f32x16_t run(const u32x4 &a, const u32x4 &b, f32x16_t c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a),
                                                      __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t pack2(float a, float b) {
        float2_t v = {a, b};
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, half2_t));
    }
};

constexpr float kNegInf = -INFINITY;


// P values are computed against a running max that is only raised when a
// tile's max exceeds it by more than this (log2 domain), so that the O / l
// rescale runs rarely; P <= 2^kRescaleSlack stays exact in fp32 and keeps
// its relative precision in 16 bit.
constexpr float kRescaleSlack = 8.0f;

// Pad (elements) of a row-major V row in LDS: each 16-lane group of the PV
// product's transposing reads takes 4 key rows x 8 dwords, which a row pitch
// of 72 dwords puts on distinct banks (measured against pads of 8 and 32:
// prefill 547 vs 554 and 550 us at B4 x 4096).
constexpr int kVRowPad = 16;

// With q_lens the offset is the sum of the lengths before b, taken by the 64
// lanes of the wave in parallel (called by every lane of every wave).
__device__ __forceinline__ void seq_info(const FaParams &p, int b, long long &q_off, int &L) {
    if (p.q_lens == nullptr) {
        q_off = p.cu_q[b];
        L = p.cu_q[b + 1] - p.cu_q[b];
    } else {
        long long off = 0;
        for (int i = threadIdx.x & 63; i < b; i += 64) off += p.q_lens[i];
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) off += __shfl_xor(off, d, 64);
        q_off = off;
        L = p.q_lens[b];
    }
}

// kv length of sequence b.  The reference reads block_table[b][j / block_size]
// for every key j < kv_len from a row of block_table_dim entries
// (flash_attention.scpp:190, :206), so kv_len <= block_table_dim * block_size
// is its precondition; clamping to that keeps every block-table read inside
// the row.  A negative length counts as 0.
__device__ __forceinline__ int kv_len(const FaParams &p, int b) {
    return min(max(p.kv_lens[b], 0), p.kv_cap);
}

// Output rows past cu_seqlens_q[batch] belong to no sequence (padding of a
// captured graph, say).  With cumulative offsets they are written as zeros,
// as the reference torch wrapper zeroes its whole output before the call
// (api/torch_ext.cpp:128-132); the rows of the sequences are all written by
// the attention kernels, so only this tail needs it.  One workgroup, 16-byte
// stores; in the usual case the offsets cover every row and nothing is done.
__device__ __forceinline__ void zero_tail_rows(const FaParams &p, int D) {
    if (p.cu_q == nullptr) return;
    const long long end = max(p.cu_q[p.batch], 0);
    if (end >= p.total_q) return;
    const long long chunks = static_cast<long long>(p.H) * D / 8;  // per row
    u32x4 *o = reinterpret_cast<u32x4 *>(p.o);
    const u32x4 zero = {0u, 0u, 0u, 0u};
    for (long long c = end * chunks + threadIdx.x; c < p.total_q * chunks; c += blockDim.x) o[c] = zero;
}

// 16-byte K/V load; STREAM selects the non-temporal policy for data read once.
template <bool STREAM>
__device__ __forceinline__ u32x4 load16(const uint16_t *p) {
    if constexpr (STREAM)
        return __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(p));
    else
        return *reinterpret_cast<const u32x4 *>(p);
}

// Element offset of key row `kv` of the (sequence, kv head) whose block-table
// row is bt_row and whose head offset inside a block is head_off.  Rows at or
// beyond kv_limit, and rows whose page id is out of range, are redirected to
// a row that exists and reported through ok = false; the caller zeroes V for
// them and masks K.
// Block-size modes of the loaders (a template argument, so that the power
// of two case keeps its shift): 0 any block_size (one block-table lookup per
// key row), 1 a power of two >= 8, 2 another multiple of 8.  Cache block of
// key row kv: a shift in mode 1, a division otherwise.
template <int BSM>
__device__ __forceinline__ int block_of(const FaParams &p, int kv) {
    return BSM == 1 ? kv >> p.lbs : kv / p.bs;
}

template <int D, int BSM>
__device__ __forceinline__ long long row_offset(const FaParams &p, const int *bt_row,
                                                long long head_off, int kv, int kv_limit,
                                                bool &ok) {
    ok = kv < kv_limit;
    const int kvs = ok ? kv : 0;
    int blk, off;
    if (BSM == 1) {
        blk = kvs >> p.lbs;
        off = kvs & (p.bs - 1);
    } else {
        blk = kvs / p.bs;
        off = kvs - blk * p.bs;
    }
    int page = bt_row[blk];
    ok = ok && page >= 0 && page < p.num_blocks;
    page = ok ? page : 0;
    return static_cast<long long>(page) * p.page_stride + head_off + static_cast<long long>(off) * D;
}

// Cooperative global -> register -> LDS staging of one TILE-key K/V tile by NT
// threads, for any head size D that is a multiple of 32.  K is stored
// row-major [TILE][D + 8]; V transposed [D][TILE + 4].  The TILE * D/8
// 16-byte chunks of K are dealt to the threads in order (chunk tid + i*NT is
// row / column (tid + i*NT) / (D/8), % (D/8)); each thread also owns VPT
// (4-row x 8-column) blocks of V.
template <int D, int TILE, int NT, int BSM, bool STREAM = false>
struct TileLoader {
    static constexpr int KP = D + 8;
    static constexpr int VP = TILE + 4;
    static constexpr int VR = 0;
    static constexpr int VOFF = TILE * KP;  // V region of a tile buffer
    static constexpr bool DMA = false;
    static constexpr int STAGES = 2;  // tile buffers in LDS
    static constexpr int ELEMS = TILE * KP + D * VP;  // one K + V^T buffer
    static constexpr int CPR = D / 8;                  // 16-byte chunks per row
    static constexpr int KTASKS = TILE * CPR;
    static constexpr int KCH = (KTASKS + NT - 1) / NT;
    static constexpr int VTASKS = (TILE / 4) * CPR;
    static constexpr int VPT = (VTASKS + NT - 1) / NT;
    static_assert(D % 32 == 0 && TILE % 4 == 0, "whole 32-column slabs and 4-row V blocks");
    u32x4 k[KCH];
    u32x4 v[VPT][4];
    uint32_t vok;  // bit 4i+r: V row of v[i][r] is valid (below kv_limit, page in range)

    __device__ __forceinline__ void prefetch(const FaParams &, const int *, int, int) {}

    __device__ __forceinline__ void load(const FaParams &p, const int *bt_row, long long head_off,
                                         int j0, int kv_limit) {
        const int tid = threadIdx.x;
        // All page lookups first, then all K/V loads: a load whose address
        // waits on a block-table read interleaved with the K/V loads would
        // wait for every K/V load issued before it (loads complete in order),
        // one round trip per row.
        long long ko[KCH], vo[VPT][4];
#pragma unroll
        for (int i = 0; i < KCH; ++i) {
            const int task = tid + i * NT;
            if (KTASKS % NT != 0 && task >= KTASKS) continue;
            bool ok;
            ko[i] = row_offset<D, BSM>(p, bt_row, head_off, j0 + task / CPR, kv_limit, ok);
        }
        // Invalid V rows are zeroed in store(), so the wave does not wait for
        // the loads here.
        vok = 0;
#pragma unroll
        for (int i = 0; i < VPT; ++i) {
            const int task = tid + i * NT;
            if (VTASKS % NT != 0 && task >= VTASKS) continue;
            const int rg = task % (TILE / 4);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                bool ok;
                vo[i][r] = row_offset<D, BSM>(p, bt_row, head_off, j0 + 4 * rg + r, kv_limit, ok);
                vok |= (ok ? 1u : 0u) << (4 * i + r);
            }
        }
#pragma unroll
        for (int i = 0; i < KCH; ++i) {
            if (KTASKS % NT != 0 && tid + i * NT >= KTASKS) continue;
            k[i] = load16<STREAM>(p.kc + ko[i] + ((tid + i * NT) % CPR) * 8);
        }
#pragma unroll
        for (int i = 0; i < VPT; ++i) {
            const int task = tid + i * NT;
            if (VTASKS % NT != 0 && task >= VTASKS) continue;
            const int cg = task / (TILE / 4);
#pragma unroll
            for (int r = 0; r < 4; ++r) v[i][r] = load16<STREAM>(p.vc + vo[i][r] + cg * 8);
        }
    }

    __device__ __forceinline__ void store(uint16_t *buf) const {
        uint16_t *Ks = buf;
        uint16_t *Vt = buf + TILE * KP;
        const int tid = threadIdx.x;
#pragma unroll
        for (int i = 0; i < KCH; ++i) {
            const int task = tid + i * NT;
            if (KTASKS % NT != 0 && task >= KTASKS) continue;
            *reinterpret_cast<u32x4 *>(Ks + (task / CPR) * KP + (task % CPR) * 8) = k[i];
        }
#pragma unroll
        for (int i = 0; i < VPT; ++i) {
            const int task = tid + i * NT;
            if (VTASKS % NT != 0 && task >= VTASKS) continue;
            const int rg = task % (TILE / 4), cg = task / (TILE / 4);
            const u32x4 zero = {0u, 0u, 0u, 0u};
            const u32x4 a = (vok >> (4 * i)) & 1u ? v[i][0] : zero;
            const u32x4 b = (vok >> (4 * i + 1)) & 1u ? v[i][1] : zero;
            const u32x4 c = (vok >> (4 * i + 2)) & 1u ? v[i][2] : zero;
            const u32x4 d = (vok >> (4 * i + 3)) & 1u ? v[i][3] : zero;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                // columns d = 8cg + 2w (low halves) and 8cg + 2w + 1 (high halves)
                u32x2 lo2, hi2;
                lo2.x = __builtin_amdgcn_perm(b[w], a[w], 0x05040100u);
                lo2.y = __builtin_amdgcn_perm(d[w], c[w], 0x05040100u);
                hi2.x = __builtin_amdgcn_perm(b[w], a[w], 0x07060302u);
                hi2.y = __builtin_amdgcn_perm(d[w], c[w], 0x07060302u);
                *reinterpret_cast<u32x2 *>(Vt + (8 * cg + 2 * w) * VP + 4 * rg) = lo2;
                *reinterpret_cast<u32x2 *>(Vt + (8 * cg + 2 * w + 1) * VP + 4 * rg) = hi2;
            }
        }
    }
};

// Block id of the aligned row group (a multiple of 4 rows inside one cache
// block) starting at `row0` (wave-uniform), or 0 past kv_limit.  The block
// table is read-only for the launch: read through the constant address space,
// the wave-uniform entry is always a scalar load, so waiting for it never
// waits for the K/V vector loads in flight (a vector load here would, under
// s_waitcnt vmcnt).
template <int BSM>
__device__ __forceinline__ int uniform_group_page(const FaParams &p, const int *bt_row, int row0,
                                                  int kv_limit) {
    row0 = __builtin_amdgcn_readfirstlane(row0);
    const auto *bt4 = (const __attribute__((address_space(4))) int *)(bt_row);
    return row0 < kv_limit ? bt4[block_of<BSM>(p, row0)] : 0;
}

// Element offset of such a group's first row (page 0 when its id is out of
// range).
template <int D, int BSM>
__device__ __forceinline__ long long uniform_group_base(const FaParams &p, long long head_off,
                                                        int row0, int page) {
    if (page < 0 || page >= p.num_blocks) page = 0;
    return static_cast<long long>(page) * p.page_stride + head_off +
           static_cast<long long>(BSM == 1 ? row0 & (p.bs - 1)
                                            : row0 - block_of<BSM>(p, row0) * p.bs) * D;
}

// Loader for D = 128 and a block_size that is a multiple of 8.  Wave w stages rows
// [w*RW, (w+1)*RW) of the tile.  Each K load instruction covers 4 aligned rows
// (16 lanes x 16 bytes per row) and each V load instruction 8 aligned rows
// (lane l: rows 2*(l%4) + {0,1}, column block l/4), so the cache block
// holding an instruction's rows is the same for the whole wave: its id is a
// scalar, read from the block table one load() call ahead (prefetch), so the
// global loads never wait for it.  K and V are both stored row-major, [TILE]
// [D + 8] and [TILE][D + kVRowPad] (VP = 0, VR = row pitch tells wave_attend
// so): V is not transposed on the way in, the PV product reads it with
// transposing LDS reads.  load() must be
// called for consecutive tiles after one prefetch() of the first.
template <int TILE, int W, int BSM, bool STREAM = false>
struct PagedLoader128 {
    static constexpr int D = 128;
    static constexpr int KP = D + 8;
    static constexpr int VP = 0;
    static constexpr int VR = D + kVRowPad;
    static constexpr int VOFF = TILE * KP;
    static constexpr bool DMA = false;
    static constexpr int STAGES = 2;  // tile buffers in LDS
    static constexpr int ELEMS = TILE * (KP + VR);
    static constexpr int RW = TILE / W;     // rows per wave
    static constexpr int KI = RW / 4;       // K load instructions per wave
    static constexpr int VI = RW / 8;       // V load instruction pairs per wave
    static_assert(RW % 8 == 0, "each wave stages whole 8-row groups");
    u32x4 k[KI];
    u32x4 v[VI][2];
    uint32_t vok;     // bit 2i+j: V row of v[i][j] is below kv_limit
    int pg[KI + VI];  // cache block ids of the next load()'s row groups (uniform)

    static __device__ __forceinline__ int group_page(const FaParams &p, const int *bt_row,
                                                     int row0, int kv_limit) {
        return uniform_group_page<BSM>(p, bt_row, row0, kv_limit);
    }
    static __device__ __forceinline__ long long group_base(const FaParams &p, long long head_off,
                                                           int row0, int page) {
        return uniform_group_base<D, BSM>(p, head_off, row0, page);
    }

    __device__ __forceinline__ void prefetch(const FaParams &p, const int *bt_row, int j0,
                                             int kv_limit) {
        const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
        for (int i = 0; i < KI; ++i) pg[i] = group_page(p, bt_row, j0 + w * RW + 4 * i, kv_limit);
#pragma unroll
        for (int i = 0; i < VI; ++i)
            pg[KI + i] = group_page(p, bt_row, j0 + w * RW + 8 * i, kv_limit);
    }

    __device__ __forceinline__ void load(const FaParams &p, const int *bt_row, long long head_off,
                                         int j0, int kv_limit) {
        const int lane = threadIdx.x & 63;
        const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const int kr = lane >> 4, kc = lane & 15;          // K: row in group of 4, chunk
        const int vr = 2 * (lane & 3), vc = lane >> 2;     // V: row pair, column block
#pragma unroll
        for (int i = 0; i < KI; ++i) {
            const int row0 = j0 + w * RW + 4 * i;
            const long long base = group_base(p, head_off, row0, pg[i]);
            k[i] = load16<STREAM>(p.kc + base + kr * D + kc * 8);
        }
        // V rows at or past kv_limit are zeroed in store(), not here: a select
        // on the loaded value would make the wave wait for the load at once.
        vok = 0;
#pragma unroll
        for (int i = 0; i < VI; ++i) {
            const int row0 = j0 + w * RW + 8 * i;
            const long long base = group_base(p, head_off, row0, pg[KI + i]);
            const uint16_t *src = p.vc + base + vr * D + vc * 8;
            v[i][0] = load16<STREAM>(src);
            v[i][1] = load16<STREAM>(src + D);
            vok |= (row0 + vr < kv_limit ? 1u : 0u) << (2 * i);
            vok |= (row0 + vr + 1 < kv_limit ? 1u : 0u) << (2 * i + 1);
        }
        prefetch(p, bt_row, j0 + TILE, kv_limit);
    }

    __device__ __forceinline__ void store(uint16_t *buf) const {
        uint16_t *Ks = buf;
        uint16_t *Vs = buf + TILE * KP;
        const int lane = threadIdx.x & 63;
        const int w = threadIdx.x >> 6;
        const int kr = lane >> 4, kc = lane & 15;
        const int vr = 2 * (lane & 3), vc = lane >> 2;
#pragma unroll
        for (int i = 0; i < KI; ++i)
            *reinterpret_cast<u32x4 *>(Ks + (w * RW + 4 * i + kr) * KP + kc * 8) = k[i];
#pragma unroll
        for (int i = 0; i < VI; ++i) {
            const int r = w * RW + 8 * i + vr;
            const u32x4 zero = {0u, 0u, 0u, 0u};
            *reinterpret_cast<u32x4 *>(Vs + r * VR + vc * 8) = (vok >> (2 * i)) & 1u ? v[i][0] : zero;
            *reinterpret_cast<u32x4 *>(Vs + (r + 1) * VR + vc * 8) =
                (vok >> (2 * i + 1)) & 1u ? v[i][1] : zero;
        }
    }
};

// Bytes of one 4-row block of the prefill's D = 128 DMA tile layout: 4 key
// rows of 256 bytes stored chunk-major (16-byte chunk c of row j at 64c +
// 16j), then a 64-byte pad.  One global_load_lds_dwordx4 fills a block (lane
// l's 16 bytes land at 16l), the 128-bit K reads of 16 consecutive rows and
// the transposing V reads of each half-wave fall on distinct banks, and the
// fragment offsets stay additive (instruction offsets).
constexpr int kLdsBlockBytes = 1088;

// 16 zero bytes: the source of V rows past the end of a sequence.
__device__ __attribute__((aligned(16))) const uint32_t kZero16[4] = {0u, 0u, 0u, 0u};

// HBM -> LDS with no register staging: 16 bytes per lane into
// dst + 16 * lane (dst wave-uniform, in M0).  Inline assembly on purpose:
// through the builtin the compiler treats every transposing LDS read as
// possibly reading the copy's destination and waits for all copies in flight
// before each one, which serialises the next tile's copy with this tile's
// work.  Here the copies are ordered by wait_dma() and the workgroup barrier
// after it.  No other code of these kernels uses M0.
__device__ __forceinline__ void dma16(const void *src, void *dst) {
    const uint32_t lds = static_cast<uint32_t>(
        reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) void *)(dst)));
    asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds)
                 : "memory");
}

// Prefill loader for D = 128 and a block_size that is a multiple of 8: K and
// V go from the paged caches straight into LDS (global_load_lds_dwordx4), in
// the 4-row block layout above, so the tile costs no registers and no LDS
// stores.  Wave w stages rows [w*RW, (w+1)*RW) of the tile, 4 aligned rows
// per instruction (lane l: row l % 4, chunk l / 4), whose cache block is the
// same for the whole wave: its id is a scalar, read from the block table one
// load() ahead.  V rows at or past kv_limit are read from kZero16; K rows
// there are read from some cache row and masked in the softmax.  load()
// issues the copies into a tile buffer, wait_tiles() waits for them (the
// caller's barrier then publishes the tile).
template <int TILE, int W, int BSM>
struct PagedLoaderDma128 {
    static constexpr int D = 128;
    static constexpr bool DMA = true;
    static constexpr int KP = 0, VP = 0, VR = 0;      // the block layout
    static constexpr int VOFF = TILE / 4 * kLdsBlockBytes / 2;  // elements
    static constexpr int ELEMS = 2 * VOFF;
    static constexpr int RW = TILE / W;  // rows per wave
    static constexpr int KI = RW / 4;    // 4-row blocks per wave
    static constexpr int STAGES = 3;     // tile buffers: copies run two tiles ahead
    static constexpr int PER_TILE = 2 * KI;  // copy instructions per tile and lane
    static_assert(RW % 4 == 0, "each wave stages whole 4-row blocks");
    static_assert(PER_TILE < 16, "vmcnt immediate");
    int pg[KI];  // cache block ids of the next load()'s row groups (uniform)

    __device__ __forceinline__ void prefetch(const FaParams &p, const int *bt_row, int j0,
                                             int kv_limit) {
        const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
        for (int i = 0; i < KI; ++i)
            pg[i] = uniform_group_page<BSM>(p, bt_row, j0 + w * RW + 4 * i, kv_limit);
    }

    __device__ __forceinline__ void load(const FaParams &p, const int *bt_row, long long head_off,
                                         int j0, int kv_limit, uint16_t *dst) {
        const int lane = threadIdx.x & 63;
        const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const int r = lane & 3, c = lane >> 2;
        char *kd = reinterpret_cast<char *>(dst) + w * KI * kLdsBlockBytes;
#pragma unroll
        for (int i = 0; i < KI; ++i) {
            const int row0 = j0 + w * RW + 4 * i;
            const long long off =
                uniform_group_base<D, BSM>(p, head_off, row0, pg[i]) + r * D + c * 8;
            dma16(p.kc + off, kd + i * kLdsBlockBytes);
            dma16(row0 + r < kv_limit ? static_cast<const void *>(p.vc + off)
                                      : static_cast<const void *>(kZero16),
                  kd + 2 * VOFF + i * kLdsBlockBytes);
        }
        prefetch(p, bt_row, j0 + TILE, kv_limit);
    }

    // Waits until this wave has at most NEWER tiles' copies in flight, i.e.
    // the tile issued before them has landed (vector memory counter; no
    // other vector loads are in flight in the tile loop).
    template <int NEWER>
    static __device__ __forceinline__ void wait_tiles() {
        __builtin_amdgcn_s_waitcnt(0x0F70 | (NEWER * PER_TILE));
    }
};

// The same scheme for D = 64: each K load instruction covers 8 aligned rows
// (8 lanes x 16 bytes per row); each V instruction covers two 8-row groups,
// one per half-wave (lane l: rows 8*(l/32) + 2*(l%4) + {0,1}, column block
// (l/4)%8), whose cache blocks are looked up separately, so block sizes of 8
// work too.
template <int TILE, int W, int BSM, bool STREAM = false>
struct PagedLoader64 {
    static constexpr int D = 64;
    static constexpr int KP = D + 8;
    static constexpr int VP = TILE + 4;
    static constexpr int VR = 0;
    static constexpr int VOFF = TILE * KP;  // V region of a tile buffer
    static constexpr bool DMA = false;
    static constexpr int STAGES = 2;  // tile buffers in LDS
    static constexpr int ELEMS = TILE * KP + D * VP;
    static constexpr int RW = TILE / W;     // rows per wave
    static constexpr int KI = RW / 8;       // K load instructions per wave
    static constexpr int VI = RW / 16;      // V load instruction pairs per wave
    static_assert(RW % 16 == 0, "each wave stages whole 16-row groups");
    u32x4 k[KI];
    u32x4 v[VI][2];
    uint32_t vok;            // bit 2i+j: V row of v[i][j] is below kv_limit
    int pg[KI + 2 * VI];     // cache block ids of the next load()'s 8-row groups (uniform)

    __device__ __forceinline__ void prefetch(const FaParams &p, const int *bt_row, int j0,
                                             int kv_limit) {
        const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
        for (int i = 0; i < KI; ++i)
            pg[i] = uniform_group_page<BSM>(p, bt_row, j0 + w * RW + 8 * i, kv_limit);
#pragma unroll
        for (int i = 0; i < 2 * VI; ++i)
            pg[KI + i] = uniform_group_page<BSM>(p, bt_row, j0 + w * RW + 8 * i, kv_limit);
    }

    static __device__ __forceinline__ long long group_base(const FaParams &p, long long head_off,
                                                           int row0, int page) {
        if (page < 0 || page >= p.num_blocks) page = 0;
        return static_cast<long long>(page) * p.page_stride + head_off +
               static_cast<long long>(BSM == 1 ? row0 & (p.bs - 1)
                                                : row0 - block_of<BSM>(p, row0) * p.bs) * D;
    }

    __device__ __forceinline__ void load(const FaParams &p, const int *bt_row, long long head_off,
                                         int j0, int kv_limit) {
        const int lane = threadIdx.x & 63;
        const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const int kr = lane >> 3, kc = lane & 7;                            // K: row of 8, chunk
        const int vb = lane >> 5, vr = 2 * (lane & 3), vc = (lane >> 2) & 7;  // V: group, pair, block
#pragma unroll
        for (int i = 0; i < KI; ++i) {
            const int row0 = j0 + w * RW + 8 * i;
            k[i] = load16<STREAM>(p.kc + group_base(p, head_off, row0, pg[i]) + kr * D + kc * 8);
        }
        vok = 0;
#pragma unroll
        for (int i = 0; i < VI; ++i) {
            const int row0 = j0 + w * RW + 16 * i;
            const long long b0 = group_base(p, head_off, row0, pg[KI + 2 * i]);
            const long long b1 = group_base(p, head_off, row0 + 8, pg[KI + 2 * i + 1]);
            const uint16_t *src = p.vc + (vb ? b1 : b0) + vr * D + vc * 8;
            v[i][0] = load16<STREAM>(src);
            v[i][1] = load16<STREAM>(src + D);
            const int r = row0 + 8 * vb + vr;
            vok |= (r < kv_limit ? 1u : 0u) << (2 * i);
            vok |= (r + 1 < kv_limit ? 1u : 0u) << (2 * i + 1);
        }
        prefetch(p, bt_row, j0 + TILE, kv_limit);
    }

    __device__ __forceinline__ void store(uint16_t *buf) const {
        uint16_t *Ks = buf;
        uint16_t *Vt = buf + TILE * KP;
        const int lane = threadIdx.x & 63;
        const int w = threadIdx.x >> 6;
        const int kr = lane >> 3, kc = lane & 7;
        const int vb = lane >> 5, vr = 2 * (lane & 3), vc = (lane >> 2) & 7;
#pragma unroll
        for (int i = 0; i < KI; ++i)
            *reinterpret_cast<u32x4 *>(Ks + (w * RW + 8 * i + kr) * KP + kc * 8) = k[i];
#pragma unroll
        for (int i = 0; i < VI; ++i) {
            const int r = w * RW + 16 * i + 8 * vb + vr;
            const u32x4 zero = {0u, 0u, 0u, 0u};
            const u32x4 a = (vok >> (2 * i)) & 1u ? v[i][0] : zero;
            const u32x4 b = (vok >> (2 * i + 1)) & 1u ? v[i][1] : zero;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t lo = __builtin_amdgcn_perm(b[e], a[e], 0x05040100u);
                const uint32_t hi = __builtin_amdgcn_perm(b[e], a[e], 0x07060302u);
                *reinterpret_cast<uint32_t *>(Vt + (8 * vc + 2 * e) * VP + r) = lo;
                *reinterpret_cast<uint32_t *>(Vt + (8 * vc + 2 * e + 1) * VP + r) = hi;
            }
        }
    }
};

// The same scheme for D = 96 (12 chunks of 16 bytes per row): a K load
// instruction covers 4 aligned rows on lanes 0-47 and a V instruction 8
// aligned rows (lane l: rows 2*(l%4) + {0,1}, column block l/4) on lanes
// 0-47; lanes 48-63 repeat lane 47's load and store nothing.
template <int TILE, int W, int BSM, bool STREAM = false>
struct PagedLoader96 {
    static constexpr int D = 96;
    static constexpr int KP = D + 8;
    static constexpr int VP = TILE + 4;
    static constexpr int VR = 0;
    static constexpr int VOFF = TILE * KP;  // V region of a tile buffer
    static constexpr bool DMA = false;
    static constexpr int STAGES = 2;  // tile buffers in LDS
    static constexpr int ELEMS = TILE * KP + D * VP;
    static constexpr int RW = TILE / W;     // rows per wave
    static constexpr int KI = RW / 4;       // K load instructions per wave
    static constexpr int VI = RW / 8;       // V load instruction pairs per wave
    static_assert(RW % 8 == 0, "each wave stages whole 8-row groups");
    u32x4 k[KI];
    u32x4 v[VI][2];
    uint32_t vok;     // bit 2i+j: V row of v[i][j] is below kv_limit
    int pg[KI + VI];  // cache block ids of the next load()'s row groups (uniform)

    __device__ __forceinline__ void prefetch(const FaParams &p, const int *bt_row, int j0,
                                             int kv_limit) {
        const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
        for (int i = 0; i < KI; ++i)
            pg[i] = uniform_group_page<BSM>(p, bt_row, j0 + w * RW + 4 * i, kv_limit);
#pragma unroll
        for (int i = 0; i < VI; ++i)
            pg[KI + i] = uniform_group_page<BSM>(p, bt_row, j0 + w * RW + 8 * i, kv_limit);
    }

    static __device__ __forceinline__ long long group_base(const FaParams &p, long long head_off,
                                                           int row0, int page) {
        if (page < 0 || page >= p.num_blocks) page = 0;
        return static_cast<long long>(page) * p.page_stride + head_off +
               static_cast<long long>(BSM == 1 ? row0 & (p.bs - 1)
                                                : row0 - block_of<BSM>(p, row0) * p.bs) * D;
    }

    __device__ __forceinline__ void load(const FaParams &p, const int *bt_row, long long head_off,
                                         int j0, int kv_limit) {
        const int lane = min(static_cast<int>(threadIdx.x & 63), 47);
        const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const int kr = lane / 12, kc = lane % 12;          // K: row in group of 4, chunk
        const int vr = 2 * (lane & 3), vc = lane >> 2;     // V: row pair, column block
#pragma unroll
        for (int i = 0; i < KI; ++i) {
            const int row0 = j0 + w * RW + 4 * i;
            k[i] = load16<STREAM>(p.kc + group_base(p, head_off, row0, pg[i]) + kr * D + kc * 8);
        }
        vok = 0;
#pragma unroll
        for (int i = 0; i < VI; ++i) {
            const int row0 = j0 + w * RW + 8 * i;
            const uint16_t *src = p.vc + group_base(p, head_off, row0, pg[KI + i]) + vr * D + vc * 8;
            v[i][0] = load16<STREAM>(src);
            v[i][1] = load16<STREAM>(src + D);
            vok |= (row0 + vr < kv_limit ? 1u : 0u) << (2 * i);
            vok |= (row0 + vr + 1 < kv_limit ? 1u : 0u) << (2 * i + 1);
        }
        prefetch(p, bt_row, j0 + TILE, kv_limit);
    }

    __device__ __forceinline__ void store(uint16_t *buf) const {
        const int lane = threadIdx.x & 63;
        if (lane >= 48) return;
        uint16_t *Ks = buf;
        uint16_t *Vt = buf + TILE * KP;
        const int w = threadIdx.x >> 6;
        const int kr = lane / 12, kc = lane % 12;
        const int vr = 2 * (lane & 3), vc = lane >> 2;
#pragma unroll
        for (int i = 0; i < KI; ++i)
            *reinterpret_cast<u32x4 *>(Ks + (w * RW + 4 * i + kr) * KP + kc * 8) = k[i];
#pragma unroll
        for (int i = 0; i < VI; ++i) {
            const int r = w * RW + 8 * i + vr;
            const u32x4 zero = {0u, 0u, 0u, 0u};
            const u32x4 a = (vok >> (2 * i)) & 1u ? v[i][0] : zero;
            const u32x4 b = (vok >> (2 * i + 1)) & 1u ? v[i][1] : zero;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t lo = __builtin_amdgcn_perm(b[e], a[e], 0x05040100u);
                const uint32_t hi = __builtin_amdgcn_perm(b[e], a[e], 0x07060302u);
                *reinterpret_cast<uint32_t *>(Vt + (8 * vc + 2 * e) * VP + r) = lo;
                *reinterpret_cast<uint32_t *>(Vt + (8 * vc + 2 * e + 1) * VP + r) = hi;
            }
        }
    }
};

// Loader choice: the uniform-page loader when it applies, else TileLoader.
// STREAM marks K/V read once per launch (decode): non-temporal loads.
template <int D, int TILE, int W, int BSM, bool STREAM = false>
struct LoaderSel {
    using type = TileLoader<D, TILE, W * 64, BSM, STREAM>;
};
template <int TILE, int W, bool STREAM>
struct LoaderSel<128, TILE, W, 1, STREAM> {
    using type = PagedLoader128<TILE, W, 1, STREAM>;
};
template <int TILE, int W, bool STREAM>
struct LoaderSel<128, TILE, W, 2, STREAM> {
    using type = PagedLoader128<TILE, W, 2, STREAM>;
};
// prefill (K/V re-read from L2 by every query tile): LDS DMA, no registers
template <int TILE, int W>
struct LoaderSel<128, TILE, W, 1, false> {
    using type = PagedLoaderDma128<TILE, W, 1>;
};
template <int TILE, int W>
struct LoaderSel<128, TILE, W, 2, false> {
    using type = PagedLoaderDma128<TILE, W, 2>;
};
template <int TILE, int W, bool STREAM>
struct LoaderSel<64, TILE, W, 1, STREAM> {
    using type = PagedLoader64<TILE, W, 1, STREAM>;
};
template <int TILE, int W, bool STREAM>
struct LoaderSel<64, TILE, W, 2, STREAM> {
    using type = PagedLoader64<TILE, W, 2, STREAM>;
};
template <int TILE, int W, bool STREAM>
struct LoaderSel<96, TILE, W, 1, STREAM> {
    using type = PagedLoader96<TILE, W, 1, STREAM>;
};
template <int TILE, int W, bool STREAM>
struct LoaderSel<96, TILE, W, 2, STREAM> {
    using type = PagedLoader96<TILE, W, 2, STREAM>;
};

template <typename T> struct Ones2;
template <> struct Ones2<bf16> {
    static __device__ __forceinline__ float dot(uint32_t a, float c) {
        return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf162_t, a),
                                               __builtin_bit_cast(bf162_t, 0x3f803f80u), c, false);
    }
};
template <> struct Ones2<f16> {
    static __device__ __forceinline__ float dot(uint32_t a, float c) {
        return __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, a),
                                      __builtin_bit_cast(half2_t, 0x3c003c00u), c, false);
    }
};

// ds_read_b64_tr_b16: 8 bytes per lane, transposed within each 16-lane group
// (see the row-major V read in wave_attend).
__device__ __forceinline__ u32x2 tr_b16_b64(const uint16_t *p) {
    typedef short i16x4_t __attribute__((ext_vector_type(4)));
    const i16x4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) i16x4_t *)(p));
    return __builtin_bit_cast(u32x2, v);
}

// Max of one lane's 16 scores as a tree of three-input maxima (v_max3_f32):
// 8 instructions, 3 deep.
__device__ __forceinline__ float max16(const f32x16_t &s) {
    const auto m3 = [](float a, float b, float c) { return fmaxf(fmaxf(a, b), c); };
    const float a0 = m3(s[0], s[1], s[2]), a1 = m3(s[3], s[4], s[5]), a2 = m3(s[6], s[7], s[8]);
    const float a3 = m3(s[9], s[10], s[11]), a4 = m3(s[12], s[13], s[14]);
    return fmaxf(m3(a0, a1, a2), m3(a3, a4, s[15]));
}

// One wave's online-softmax attention over NKB 32-key blocks staged in LDS at
// rows [kv_row0, kv_row0 + 32*NKB).  Lane l owns query column (l % 32) of each
// of its QSUB column blocks.
//   qf:   Q^T B-operand fragments (8 x 16-bit per lane per 16-dim k-step)
//   oacc: O^T accumulators, element v of block db is d = 32db + 8(v/4) + 4(l/32) + v%4
//   m:    running max (log2 domain, >= 0), lsum: this half-wave's partial sum of P
//   lim:  key r (0-based in the staged rows, r = 32kb + 8(v/4) + 4(l/32) + v%4)
//         is visible when r - 4(l/32) < lim[qs]
template <typename T, int D, int KP, int VP, int VR, int NKB, int QSUB, bool MASK>
__device__ __forceinline__ void wave_attend(const uint16_t *Ks, const uint16_t *Vt, int kv_row0,
                                            const u32x4 (&qf)[QSUB][D / 16],
                                            f32x16_t (&oacc)[QSUB][D / 32], float (&m)[QSUB],
                                            float (&lsum)[QSUB], const int (&lim)[QSUB],
                                            float scale_log2, float inv_scale_log2,
                                            bool mask = MASK) {
    const float slack_raw = kRescaleSlack * inv_scale_log2;
    // row-major V (pitch VR): this lane's element offset for the transposing
    // reads, key 4g + s / 4 and head dim 16 (G % 2) + 4 (s % 4) of a 16-key,
    // 32-dim block (G = lane / 16, s = lane % 16)
    const int vlane = (4 * (threadIdx.x >> 5 & 1) + ((threadIdx.x & 15) >> 2)) * VR +
                      16 * (threadIdx.x >> 4 & 1) + 4 * (threadIdx.x & 3);
    const int lane = threadIdx.x & 63;
    const int g = lane >> 5, r32 = lane & 31;
    // the 4-row block layout (KP == 0), byte offsets of this lane: K row r32,
    // chunk g; V (transposing reads as above) key 4g + s / 4, head dims 16 (G
    // % 2) + 4 (s % 4) .. +3
    const int kblane = (r32 >> 2) * kLdsBlockBytes + 16 * (r32 & 3) + 64 * g;
    const int vblane = g * kLdsBlockBytes + 16 * ((lane & 15) >> 2) + 128 * (lane >> 4 & 1) +
                       64 * (lane >> 1 & 1) + 8 * (lane & 1);
    const char *Kb = reinterpret_cast<const char *>(Ks) + (kv_row0 >> 2) * kLdsBlockBytes;
    const char *Vb = reinterpret_cast<const char *>(Vt) + (kv_row0 >> 2) * kLdsBlockBytes;
    f32x16_t s[NKB][QSUB];
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int qs = 0; qs < QSUB; ++qs)
#pragma unroll
            for (int v = 0; v < 16; ++v) s[kb][qs][v] = 0.0f;
    // Issue priority by phase: the QK product highest, the PV product next,
    // the softmax lowest, so that when waves of a SIMD compete the ones with
    // matrix work issue first and the softmax fills the matrix core's gaps
    // (BASELINE prefill 513 -> 493 us; the same three levels with the softmax
    // at the PV level: 512, QK and PV equal: 505, PV raised alone: 502,
    // softmax raised: 532 us).
    __builtin_amdgcn_s_setprio(2);
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) {
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) {
            const u32x4 a =
                KP == 0 ? *reinterpret_cast<const u32x4 *>(Kb + kblane + 8 * kb * kLdsBlockBytes +
                                                           128 * ks)
                        : *reinterpret_cast<const u32x4 *>(
                              Ks + (kv_row0 + 32 * kb + r32) * KP + 16 * ks + 8 * g);
#pragma unroll
            for (int qs = 0; qs < QSUB; ++qs) s[kb][qs] = Mma<T>::run(a, qf[qs][ks], s[kb][qs]);
        }
    }
    __builtin_amdgcn_s_setprio(0);
#pragma unroll
    for (int qs = 0; qs < QSUB; ++qs) {
        // masked scores, then their max as a tree (short dependency chain)
        if (MASK && mask) {
#pragma unroll
            for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    float x = s[kb][qs][v];
                    if (!(32 * kb + 8 * (v >> 2) + (v & 3) < lim[qs])) x = kNegInf;
                    s[kb][qs][v] = x;
                }
        }
        // The rescale test runs on this half-wave's raw scores: every lane's
        // max of its 16 keys is within the slack exactly when every query
        // column's max over all 32 keys is, so the exchange with the other
        // half-wave and the scaling are only needed when the max is raised.
        // (The test's rounding can differ from that of the scaled max by an
        // ulp; either outcome is exact, see kRescaleSlack.)
        float mx = max16(s[0][qs]);
#pragma unroll
        for (int kb = 1; kb < NKB; ++kb) mx = fmaxf(mx, max16(s[kb][qs]));
        if (!__all(mx <= fmaf(m[qs], inv_scale_log2, slack_raw))) {
            mx = half_swap_max(mx) * scale_log2;
            const float m_new = fmaxf(m[qs], mx);  // m >= 0 keeps the reference clamp
            const float alpha = __builtin_amdgcn_exp2f(m[qs] - m_new);
            m[qs] = m_new;
            lsum[qs] *= alpha;
#pragma unroll
            for (int db = 0; db < D / 32; ++db)
#pragma unroll
                for (int v = 0; v < 16; ++v) oacc[qs][db][v] *= alpha;
        }
        const float mneg = -m[qs];
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
            for (int v = 0; v < 16; ++v)
                s[kb][qs][v] = __builtin_amdgcn_exp2f(fmaf(s[kb][qs][v], scale_log2, mneg));
    }
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int t = 0; t < 2 * NKB; ++t) {
        const int kb = t >> 1, o = 8 * (t & 1);
        u32x4 pf[QSUB];
#pragma unroll
        for (int qs = 0; qs < QSUB; ++qs) {
            pf[qs].x = Mma<T>::pack2(s[kb][qs][o + 0], s[kb][qs][o + 1]);
            pf[qs].y = Mma<T>::pack2(s[kb][qs][o + 2], s[kb][qs][o + 3]);
            pf[qs].z = Mma<T>::pack2(s[kb][qs][o + 4], s[kb][qs][o + 5]);
            pf[qs].w = Mma<T>::pack2(s[kb][qs][o + 6], s[kb][qs][o + 7]);
            float l = lsum[qs];
            l = Ones2<T>::dot(pf[qs].x, l);
            l = Ones2<T>::dot(pf[qs].y, l);
            l = Ones2<T>::dot(pf[qs].z, l);
            l = Ones2<T>::dot(pf[qs].w, l);
            lsum[qs] = l;
        }
#pragma unroll
        for (int db = 0; db < D / 32; ++db) {
            u32x4 a;
            if constexpr (KP == 0) {
                const char *vb = Vb + vblane + 4 * t * kLdsBlockBytes + 256 * db;
                const u32x2 lo2 = tr_b16_b64(reinterpret_cast<const uint16_t *>(vb));
                const u32x2 hi2 =
                    tr_b16_b64(reinterpret_cast<const uint16_t *>(vb + 2 * kLdsBlockBytes));
                a = u32x4{lo2.x, lo2.y, hi2.x, hi2.y};
            } else if constexpr (VR > 0) {
                // V row-major [key][VR]: each 16-lane group of a
                // ds_read_b64_tr_b16 hands lane i value i % 4 of the group's
                // lanes i / 4 + {0, 4, 8, 12}; lane s points at key s / 4 and
                // head dims 4 (s % 4) .. +3 of its group's 16, so lane i gets
                // head dim d0 + i of 4 consecutive keys (the A operand's k
                // order of the V^T layout below)
                const uint16_t *vb = Vt + (kv_row0 + 16 * t) * VR + 32 * db + vlane;
                const u32x2 lo2 = tr_b16_b64(vb);
                const u32x2 hi2 = tr_b16_b64(vb + 8 * VR);
                a = u32x4{lo2.x, lo2.y, hi2.x, hi2.y};
            } else {
                const uint16_t *vr = Vt + (32 * db + r32) * VP + kv_row0 + 16 * t + 4 * g;
                const u32x2 lo2 = *reinterpret_cast<const u32x2 *>(vr);
                const u32x2 hi2 = *reinterpret_cast<const u32x2 *>(vr + 8);
                a = u32x4{lo2.x, lo2.y, hi2.x, hi2.y};
            }
#pragma unroll
            for (int qs = 0; qs < QSUB; ++qs) oacc[qs][db] = Mma<T>::run(a, pf[qs], oacc[qs][db]);
        }
    }
}

template <typename T>
__device__ __forceinline__ void store_row4(uint16_t *dst, float a, float b, float c, float d) {
    uint2 w;
    w.x = Mma<T>::pack2(a, b);
    w.y = Mma<T>::pack2(c, d);
    *reinterpret_cast<uint2 *>(dst) = w;
}

// ---------------------------------------------------------------- prefill

// Elements of one staged K/V tile of TILE keys: K [TILE][D + 8] and V either
// transposed [D][TILE + 4] or row-major [TILE][D + kVRowPad], whichever the
// loader uses (the larger of the two).
template <int D, int TILE>
constexpr size_t kv_tile_elems() {
    constexpr size_t vt = static_cast<size_t>(D) * (TILE + 4),
                     vr = static_cast<size_t>(TILE) * (D + kVRowPad);
    return static_cast<size_t>(TILE) * (D + 8) + (vt > vr ? vt : vr);
}

// Padded LDS row of the staged O rows of a prefill workgroup (HW heads x D
// values): the pad spreads the 8-byte fragment writes of consecutive rows
// over the banks.
template <int D, int HW>
constexpr int o_row() {
    return HW * D + 8;
}

// LDS of a prefill workgroup: the loader's K/V tile buffers, which the
// staged O rows ([32*QSUB*(W/HW)][o_row]) reuse at the end of the tile.
template <int D, int TILE, int W, int HW, int QSUB, int BSM>
constexpr size_t prefill_lds_bytes() {
    using Loader = typename LoaderSel<D, TILE, W, BSM>::type;
    constexpr size_t kv = static_cast<size_t>(Loader::STAGES) * Loader::ELEMS;
    constexpr size_t o = static_cast<size_t>(32 * QSUB * (W / HW)) * o_row<D, HW>();
    return sizeof(uint16_t) * (kv > o ? kv : o);
}

// One query tile [q0, q0 + QT) of workgroup (b, kv head kvh, head group hg):
// the body of fa_prefill_kernel.  Ends with a barrier, so the LDS tile
// buffers can be refilled by the next call.
// SPLIT: over the keys [kv_lo, kv_hi) only (kv_lo a multiple of TILE, kv_hi
// one too or past the last visible key); with `part` the state goes there
// unnormalised instead of to the output rows, a fragment of frag_floats<D>()
// per wave and 32-row block: O as the accumulators lie (16 bytes per lane and
// instruction), then (max, sum) of each row.
template <int D>
constexpr int frag_floats() {
    return 32 * D + 64;
}

template <typename T, int D, int W, int HW, int QSUB, int BSM, int TILE, bool SPLIT = false>
__device__ __forceinline__ void prefill_tile(const FaParams &p, uint16_t *lds, int b, int kvh,
                                             int hg, long long q_off, int L, int S, int q0,
                                             int kv_lo = 0, int kv_hi = 0x7fffffff,
                                             float *part = nullptr) {
    constexpr int NKB = TILE % 64 == 0 ? 2 : 1;
    constexpr int KB = 32 * NKB;
    using Loader = typename LoaderSel<D, TILE, W, BSM>::type;
    constexpr int KP = Loader::KP, VP = Loader::VP, VR = Loader::VR;
    constexpr int WROWS = 32 * QSUB;
    constexpr int QT = WROWS * (W / HW);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int g = lane >> 5, r32 = lane & 31;
    const int h = kvh * p.G + hg * HW + (wave % HW);
    const int qw0 = q0 + (wave / HW) * WROWS;
    const int q_start = p.causal ? max(S - L, 0) : 0;
    int kv_end = p.causal ? min(S, q_start + min(q0 + QT, L)) : S;
    int wave_kv_end =
        __builtin_amdgcn_readfirstlane(p.causal ? min(S, q_start + min(qw0 + WROWS, L)) : S);
    if constexpr (SPLIT) {
        kv_end = min(kv_end, kv_hi);
        wave_kv_end = min(wave_kv_end, kv_hi);
    }
    const int wave_min_vis = __builtin_amdgcn_readfirstlane(p.causal ? min(S, q_start + qw0 + 1) : S);
    const int *bt_row = p.bt + b * p.bt_stride;
    const long long head_off = static_cast<long long>(kvh) * p.bs * D;

    u32x4 qf[QSUB][D / 16];
    int vis[QSUB];
#pragma unroll
    for (int qs = 0; qs < QSUB; ++qs) {
        const int row = qw0 + 32 * qs + r32;
        const uint16_t *src = p.q + ((q_off + min(row, L - 1)) * p.H + h) * D;
#pragma unroll
        for (int ks = 0; ks < D / 16; ++ks) {
            const u32x4 x = *reinterpret_cast<const u32x4 *>(src + 16 * ks + 8 * g);
            const u32x4 zero = {0u, 0u, 0u, 0u};
            qf[qs][ks] = row < L ? x : zero;
        }
        vis[qs] = p.causal ? min(S, q_start + row + 1) : S;
    }

    float m[QSUB], lsum[QSUB];
    f32x16_t oacc[QSUB][D / 32];
#pragma unroll
    for (int qs = 0; qs < QSUB; ++qs) {
        m[qs] = 0.0f;
        lsum[qs] = 0.0f;
#pragma unroll
        for (int db = 0; db < D / 32; ++db)
#pragma unroll
            for (int v = 0; v < 16; ++v) oacc[qs][db][v] = 0.0f;
    }

    Loader ld;
    const int ntiles = (kv_end + TILE - 1) / TILE;
    const int it0 = SPLIT ? kv_lo / TILE : 0;
    // Tile t lives in LDS buffer t % NS.  A DMA loader copies straight into
    // the buffer (NS = 3: tile t + 2 is copied while tile t is attended), the
    // others stage tile t + 1 in registers and store it after tile t (NS = 2).
    constexpr int NS = Loader::STAGES;
    // (the offset goes through readfirstlane so that it stays one scalar:
    // otherwise the compiler precomputes lane addresses for every buffer)
    auto buf = [&](int t) { return lds + __builtin_amdgcn_readfirstlane((t % NS) * Loader::ELEMS); };
    auto load = [&](int t) {
        if constexpr (Loader::DMA)
            ld.load(p, bt_row, head_off, t * TILE, S, buf(t));
        else
            ld.load(p, bt_row, head_off, t * TILE, S);
    };
    // tile t is in LDS for this wave (the barrier after it publishes it)
    auto land = [&](int t) {
        if constexpr (Loader::DMA) {
            if (NS > 2 && t + 1 < ntiles)
                Loader::template wait_tiles<1>();
            else
                Loader::template wait_tiles<0>();
        } else {
            ld.store(buf(t));
        }
    };
    if (ntiles > it0) {
        ld.prefetch(p, bt_row, it0 * TILE, S);
        load(it0);
        if constexpr (NS > 2)
            if (ntiles > it0 + 1) load(it0 + 1);
        land(it0);
    }
    __syncthreads();
    for (int it = it0; it < ntiles; ++it) {
        const uint16_t *cur = buf(it);
        if (it + NS - 1 < ntiles) load(it + NS - 1);
#pragma unroll
        for (int hb = 0; hb < TILE / KB; ++hb) {
            const int j0 = it * TILE + KB * hb;
            if (j0 < wave_kv_end) {
                int lim[QSUB];
#pragma unroll
                for (int qs = 0; qs < QSUB; ++qs) lim[qs] = vis[qs] - j0 - 4 * g;
                // one copy of the block code; the mask is a uniform branch
                wave_attend<T, D, KP, VP, VR, NKB, QSUB, true>(cur, cur + Loader::VOFF, KB * hb, qf, oacc, m,
                                                           lsum, lim, p.scale_log2,
                                                           p.inv_scale_log2, j0 + KB > wave_min_vis);
            }
        }
        if (it + 1 < ntiles) land(it + 1);
        __syncthreads();
    }

    if constexpr (SPLIT) {
        if (part != nullptr) {
#pragma unroll
            for (int qs = 0; qs < QSUB; ++qs) {
                float *f = part + (wave * QSUB + qs) * frag_floats<D>();
                const float lt = half_swap_sum(lsum[qs]);
#pragma unroll
                for (int db = 0; db < D / 32; ++db)
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        *reinterpret_cast<float4_t *>(f + ((db * 4 + u) * 64 + lane) * 4) =
                            float4_t{oacc[qs][db][4 * u], oacc[qs][db][4 * u + 1],
                                     oacc[qs][db][4 * u + 2], oacc[qs][db][4 * u + 3]};
                if (g == 0)
                    *reinterpret_cast<float2_t *>(f + 32 * D + 2 * r32) = float2_t{m[qs], lt};
            }
            return;
        }
    }

    // O leaves through LDS, a row (HW heads x D values) at a time, 16 bytes
    // per lane: the O^T fragments would be stored 8 bytes per lane over 32
    // rows per instruction (prefill B = 64 x 256 rows: 155 -> 108 us, the
    // BASELINE prefill 1.5 % faster).  The tile loop ended with a barrier, so
    // the K/V buffers are free.
    constexpr int OROW = o_row<D, HW>();
    constexpr int RCH = HW * D / 8;  // 16-byte chunks per row
    constexpr int NOC = (QT * RCH + W * 64 - 1) / (W * 64);
    static_assert(NS * Loader::ELEMS * sizeof(uint16_t) <= prefill_lds_bytes<D, TILE, W, HW, QSUB, BSM>() &&
                      QT * OROW * sizeof(uint16_t) <= prefill_lds_bytes<D, TILE, W, HW, QSUB, BSM>(),
                  "K/V tiles and staged O rows fit the workgroup's LDS");
#pragma unroll
    for (int qs = 0; qs < QSUB; ++qs) {
        const float lt = half_swap_sum(lsum[qs]);
        const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
        uint16_t *dst = lds + ((wave / HW) * WROWS + 32 * qs + r32) * OROW + (wave % HW) * D;
#pragma unroll
        for (int db = 0; db < D / 32; ++db)
#pragma unroll
            for (int u = 0; u < 4; ++u)
                store_row4<T>(dst + 32 * db + 8 * u + 4 * g, oacc[qs][db][4 * u] * inv,
                              oacc[qs][db][4 * u + 1] * inv, oacc[qs][db][4 * u + 2] * inv,
                              oacc[qs][db][4 * u + 3] * inv);
    }
    __syncthreads();
    uint16_t *o_rows = p.o + (q_off * p.H + kvh * p.G + hg * HW) * D;
#pragma unroll
    for (int j = 0; j < NOC; ++j) {
        const int c = static_cast<int>(threadIdx.x) + j * W * 64;
        const int rr = c / RCH;
        if (c < QT * RCH && q0 + rr < L)
            *reinterpret_cast<u32x4 *>(o_rows + static_cast<long long>(q0 + rr) * p.H * D +
                                       (c - rr * RCH) * 8) =
                *reinterpret_cast<const u32x4 *>(lds + rr * OROW + (c - rr * RCH) * 8);
    }
    __syncthreads();  // the next tile of the same workgroup refills the LDS
}

}  // namespace
