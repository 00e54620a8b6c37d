// Wide column steps: the kernels of a prefill over hundreds to thousands of columns per layer.
//
// A 64-column pass reads every weight once per 64 tokens and pays nine dependent launches per layer for them; what
// bounded it was the activations, which every row block reads from L2 again.  Here a layer's products run as tiled
// matrix products over all columns at once, and the attention as one pass over the keys per block of query rows.
//   k_gemm_wide   y[m][n] = sum_k x[m][k] W[n][k] over packed weight tiles (block dequantisation as in sp_gemv.h)
//   k_rope_wide   rotation; K and V of the new columns into a contiguous staging area (and their ring slots when no
//                 slot still visible to a column of the call is overwritten)
//   k_attn_mq<.., STAGED>, k_attn_combine (sp_attn.h): attention of the new columns over ring keys and staged keys
//   k_ring_commit staged K and V into the ring, for calls longer than the ring has room for
// Every value is formed with the operations, and in the order, of the step over at most 64 columns that the same
// columns would take chunk by chunk (sp_engine::step): a prompt gives the same bits, and so the same greedy ids, however
// it is passed in.  Each kernel says below what that fixes.
// Replaces the K/V-batch command buffer of the reference's prefill (native/vulkan_decode/qwen_vk.cpp:415-437) and the
// multi-token case of Qwen2Engine.forward (seedplane/qwen_engine.py:105-144).
#pragma once
#include "sp_attn.h"
#include "sp_device.h"
#include "sp_gemv.h"

namespace wide {

// ------------------------------------------------------------------------------------------------ LDS copies
// One global-to-LDS copy per lane: lane i's 16 (4) bytes at base + off land at LDS byte address lds + 16 i (4 i).  Inline
// asm so that the compiler does not track the copies: it would make every LDS read wait for all of them, and the
// main loop keeps the next stage's copies in flight while it reads the current one.  They complete in order with the
// wave's other vector memory operations; copies_wait counts them.  M0 (the LDS address) is used by nothing else here; a
// scalar write of M0 needs one wait state before a copy reads it, which the compiler does not add inside inline asm.
__device__ __forceinline__ void copy16(const void *base, uint32_t off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds) : "memory");
}
__device__ __forceinline__ void copy4(const void *base, uint32_t off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(off), "s"(base), "s"(lds) : "memory");
}
template <int N>
__device__ __forceinline__ void copies_wait() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
__device__ __forceinline__ void barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// ------------------------------------------------------------------------------------------------ matrix product
// Block tile: BM = 16 MTW WM columns x BN = 16 RW WN weight rows, WM x WN waves, each wave MTW x RW 16 x 16 outputs.
// A stage holds KB 32-wide k-blocks (TPS weight k-tiles): the activations as MFMA fragments (1 KiB per 16 columns x 32 k,
// the layout the producing kernels write, so a stage is copied in whole KiB), the packed weight tiles and their scales.
template <int FMT, int MTW, int RW, int WM, int WN, bool LO>
struct Tile {
    static constexpr int NW = WM * WN, BMT = MTW * WM, BNG = RW * WN;      // waves, column tiles, row groups
    static constexpr int TPS = FMT == 1 ? 2 : 1;                           // weight k-tiles per stage
    static constexpr int KB = FMT == 3 ? 4 : 2;                            // 32-wide k-blocks per stage
    static constexpr int KBT = KB / TPS;                                   // ... and per weight k-tile
    static constexpr int A_KIB = KB * BMT * (LO ? 2 : 1), W_KIB = BNG * TPS;
    static constexpr int S_BYTES = FMT == 1 ? 0 : (FMT == 2 ? BNG * 64 : BNG * 256);
    static constexpr int A_PER = A_KIB / NW, W_PER = W_KIB / NW;           // copies per wave and stage
    static constexpr int S_PIECES = S_BYTES / 256;                         // side copies (256 bytes each) of a stage
    static constexpr int S_PER = FMT == 1 ? 0 : 1;
    static constexpr int COPIES = A_PER + W_PER + S_PER;
    static constexpr int STAGE = (A_KIB + W_KIB) * 1024 + S_BYTES;
    // stages in LDS: 3, or 2 where that lets a CU hold a second block (fp16 128 x 128 tiles, whose stage is 32 KiB:
    // Qwen2-0.5B gate_up over 1152 columns 48.1 -> 40.3 us; their 64 x 64 tiles lose with 2: 31 -> 53 us)
    static constexpr int NS = (FMT == 1 && MTW * WM >= 8 && !LO) || 3 * STAGE > 160 * 1024 ? 2 : 3;
    static constexpr int SMEM = NS * STAGE;
    static_assert(A_KIB % NW == 0 && W_KIB % NW == 0, "every wave copies the same number of KiB");
    static_assert(W_PER % TPS == 0, "a wave's weight copies run through the stage's k-tiles in turn");
    static_assert(FMT == 1 || (S_PIECES >= 1 && S_PIECES <= NW), "one side copy per wave");
    static_assert(SMEM <= 160 * 1024, "the stages fit a CU's LDS");
};

// The order in which k_gemv adds the k-tiles of one output: the k-slices of `per` tiles in turn; in a slice its waves in
// turn; of a wave the tiles w, w + nw, ... of the slice.  A walk visits the tiles of [first, last) in that order.
struct Walk {
    int kt, w, lo, hi;     // the tile, its wave, its slice's tiles [lo, hi)
    __device__ __forceinline__ void start(int first, int last, int per) {
        kt = lo = first;
        w = 0;
        hi = min(last, first + per);
    }
    __device__ __forceinline__ bool wave_ends(int nw) const { return kt + nw >= hi; }
    __device__ __forceinline__ bool slice_ends(int nw) const { return wave_ends(nw) && (w + 1 >= nw || lo + w + 1 >= hi); }
    __device__ __forceinline__ void next(int last, int per, int nw) {
        const bool ws = wave_ends(nw), ss = slice_ends(nw);
        if (ss) { lo = hi; hi = min(last, hi + per); w = 0; kt = lo; }
        else if (ws) { ++w; kt = lo + w; }
        else kt += nw;
    }
};

struct GemmArgs {
    const uint8_t *w;
    const f16 *sz;
    int nkt, nrg;          // k-tiles per row group, row groups
    int n_real;            // real output rows (EPI_SILU: intermediate size)
    const f16 *x, *xlo;    // fragment-major activations and (LO) their remainders
    int mtp;               // column tiles of the layout
    int m;                 // columns
    float *out_f32;        // EPI_STORE / EPI_RESID [m][ldo]; EPI_PART: slice s at out_f32 + s * pstride
    f16 *out_f16;          // EPI_SILU, fragment-major with mtp column tiles
    int ldo;
    const float *bias;
    int epi;
    int mblocks, nblocks;  // grid tiles; gridDim.x = mblocks * nblocks
    int per, nw;           // the order of the sums (Walk): k-tiles per slice, waves of a slice
    size_t pstride;
};

// gridDim.y == 1: the block forms every slice; gridDim.y > 1: slice blockIdx.y, whose sum goes to the partial buffer.
// acc is one wave's sum of k_gemv, tot the slice's (the waves' sums in wave order), and with SUM (several slices in one
// block) grand the sums of the slices in slice order on top of the residual, as the consumer of k_gemv's slices adds
// them.  A sum that starts at +0 never becomes -0, so starting tot and grand from 0 changes no bit.
// Bound by the vector instructions of the block scales (four multiply-adds per MFMA for int8, eight for int4) and, with
// these sums, two more per output and wave of the order: Qwen2-1.5B int8 gate_up over 2048 columns 186 us (0.61 PFLOP/s;
// 176 with one sum per output, whose bits are no step's), Qwen2-0.5B fp16 gate_up over 980 columns 36 (33).
template <int FMT, int MTW, int RW, int WM, int WN, bool PAIR, bool LO, bool SUM>
__global__ void __launch_bounds__(64 * WM * WN) k_gemm_wide(GemmArgs a) {
    using T = Tile<FMT, MTW, RW, WM, WN, LO>;
    static_assert(!PAIR || RW % 2 == 0, "a wave holds the gate and the up row groups of its outputs");
    static_assert(!PAIR || !SUM, "the SwiGLU pair is never split");
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int wm = wv % WM, wn = wv / WM;
    // Consecutive block ids go to the 8 XCDs in turn; each XCD takes a contiguous range of tiles, ordered so that
    // blocks sharing weight rows (all column tiles of one row tile) run on one XCD at the same time.
    int tile;
    {
        const int total = a.mblocks * a.nblocks, q = total >> 3, rem = total & 7, xcd = blockIdx.x & 7;
        tile = xcd * q + min(xcd, rem) + (blockIdx.x >> 3);
    }
    const int nb = tile / a.mblocks, mb = tile - nb * a.mblocks;
    const int mt0 = mb * T::BMT, rg0 = nb * T::BNG;
    // the block's k-tiles
    const int first = gridDim.y > 1 ? blockIdx.y * a.per : 0;
    const int last = gridDim.y > 1 ? min(a.nkt, first + a.per) : a.nkt;
    const int n_kt = last - first, n_st = (n_kt + T::TPS - 1) / T::TPS;

    // ---- this wave's copies: scalar addresses of k-tile 0.  Column tiles and row groups past the matrix re-read the
    // last one (their outputs are not stored).
    const uint8_t *ab[T::A_PER], *wb[T::W_PER];
    uint32_t al[T::A_PER], wl[T::W_PER];
    bool a1[T::A_PER];                                      // the copy belongs to the stage's second k-tile
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(size_t)((__attribute__((address_space(3))) unsigned char *)smem));
#pragma unroll
    for (int i = 0; i < T::A_PER; ++i) {
        const int blk = wv * T::A_PER + i;                  // [hi / lo][k-block][column tile]
        const int half = blk / (T::KB * T::BMT), b2 = blk - half * (T::KB * T::BMT);
        const int kb = b2 / T::BMT, mt = min(mt0 + b2 - kb * T::BMT, a.mtp - 1);
        const f16 *src = LO && half ? a.xlo : a.x;
        a1[i] = kb >= T::KBT;
        ab[i] = (const uint8_t *)(src + ((size_t)(kb % T::KBT) * a.mtp + mt) * 512);
        al[i] = lds0 + blk * 1024;
    }
#pragma unroll
    for (int i = 0; i < T::W_PER; ++i) {
        const int blk = wv * T::W_PER + i;                  // [row group][k-tile of the stage]
        const int rg = min(rg0 + blk / T::TPS, a.nrg - 1);
        wb[i] = a.w + (size_t)rg * a.nkt * TILE_BYTES;
        wl[i] = lds0 + (T::A_KIB + blk) * 1024;
    }
    const uint8_t *sb = nullptr;
    uint32_t soff = 0, sl = 0;
    if constexpr (FMT != 1) {
        const int piece = wv % T::S_PIECES;
        sl = lds0 + (T::A_KIB + T::W_KIB) * 1024 + piece * 256;
        if constexpr (FMT == 2) {                           // 4 row groups: 16 rows x 2 scales each
            const int rg = min(rg0 + piece * 4 + g, a.nrg - 1);
            sb = (const uint8_t *)a.sz;
            soff = (uint32_t)rg * a.nkt * 64 + r * 4;
        } else {                                            // one row group: 16 rows x 4 (scale, zero)
            const int rg = min(rg0 + piece, a.nrg - 1);
            sb = (const uint8_t *)a.sz + (size_t)rg * a.nkt * 256;
            soff = lane * 4;
        }
    }
    const uint32_t lo16 = lane * 16;
    const size_t astep = (size_t)T::KBT * a.mtp * 1024;     // bytes of activations per k-tile
    Walk in;
    in.start(first, last, a.per);
    // copies of the next TPS tiles of the walk (past its end: the last tile again, which is not used)
    auto issue = [&](int slot) {
        const uint32_t d = slot * T::STAGE;
        int kt[T::TPS];
#pragma unroll
        for (int i = 0; i < T::TPS; ++i) {
            kt[i] = min(in.kt, last - 1);
            in.next(last, a.per, a.nw);
        }
#pragma unroll
        for (int i = 0; i < T::W_PER; ++i) copy16(wb[i] + (size_t)kt[i % T::TPS] * TILE_BYTES, lo16, wl[i] + d);
        if constexpr (FMT != 1) copy4(sb + (size_t)kt[0] * (FMT == 2 ? 64 : 256), soff, sl + d);
        const size_t a0 = kt[0] * astep, a2 = kt[T::TPS - 1] * astep;
#pragma unroll
        for (int i = 0; i < T::A_PER; ++i) copy16(ab[i] + (a1[i] ? a2 : a0), lo16, al[i] + d);
    };

    const f32x4 zero4 = (f32x4){0.f, 0.f, 0.f, 0.f};
    f32x4 acc[RW][MTW], tot[RW][MTW], grand[SUM ? RW : 1][SUM ? MTW : 1];
#pragma unroll
    for (int i = 0; i < RW; ++i)
#pragma unroll
        for (int j = 0; j < MTW; ++j) {
            acc[i][j] = tot[i][j] = zero4;
            if constexpr (SUM) {
                grand[i][j] = zero4;
                const int n = (rg0 + wn * RW + i) * 16 + r, mbase = (mt0 + wm * MTW + j) * 16 + 4 * g;
                if (a.epi == EPI_RESID && n < a.n_real) {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (mbase + e < a.m) grand[i][j][e] = a.out_f32[(size_t)(mbase + e) * a.ldo + n];
                }
            }
        }
    const f16x8 ones8 = (f16x8){1, 1, 1, 1, 1, 1, 1, 1};

#pragma unroll
    for (int p = 0; p < T::NS - 1; ++p)
        if (p < n_st) issue(p);
    Walk at;
    at.start(first, last, a.per);
    int left = n_kt;
    // after the products of one k-tile: the ends of its wave's and its slice's sums
    auto tile_done = [&]() {
        if (at.wave_ends(a.nw)) {
#pragma unroll
            for (int i = 0; i < RW; ++i)
#pragma unroll
                for (int j = 0; j < MTW; ++j) { tot[i][j] += acc[i][j]; acc[i][j] = zero4; }
            if constexpr (SUM) {
                if (at.slice_ends(a.nw)) {
#pragma unroll
                    for (int i = 0; i < RW; ++i)
#pragma unroll
                        for (int j = 0; j < MTW; ++j) { grand[i][j] += tot[i][j]; tot[i][j] = zero4; }
                }
            }
        }
        at.next(last, a.per, a.nw);
        --left;
    };
    int slot = 0, fill = T::NS - 1;
    for (int t = 0; t < n_st; ++t) {
        // stage t has landed (this wave's copies, then every wave's); the slot of stage t - 1 is free for t + NS - 1
        if (t + T::NS - 1 <= n_st) copies_wait<(T::NS - 2) * T::COPIES>();
        else copies_wait<0>();
        barrier();
        if (t + T::NS - 1 < n_st) issue(fill);
        fill = fill + 1 == T::NS ? 0 : fill + 1;
        const unsigned char *st = smem + slot * T::STAGE;
        slot = slot + 1 == T::NS ? 0 : slot + 1;
        const unsigned char *wst = st + T::A_KIB * 1024, *sst = wst + T::W_KIB * 1024;

        u32x4 wt[RW];
        uint32_t s8[RW];
        u32x4 s4[RW];
        if constexpr (FMT != 1) {
#pragma unroll
            for (int i = 0; i < RW; ++i) {
                const int rg = wn * RW + i;
                wt[i] = *(const u32x4 *)(wst + rg * 1024 + lane * 16);
                if constexpr (FMT == 2) s8[i] = *(const uint32_t *)(sst + (rg * 16 + r) * 4);
                else s4[i] = *(const u32x4 *)(sst + rg * 256 + r * 16);
            }
        }
#pragma unroll
        for (int kb = 0; kb < T::KB; ++kb) {
            if (FMT == 1 && kb > 0 && left <= 0) break;     // a second k-tile past the walk's end
            f16x8 xa[MTW], xl[LO ? MTW : 1];
#pragma unroll
            for (int j = 0; j < MTW; ++j) {
                xa[j] = *(const f16x8 *)(st + ((kb * T::BMT + wm * MTW + j) * 1024) + lane * 16);
                if constexpr (LO)
                    xl[j] = *(const f16x8 *)(st + (((T::KB + kb) * T::BMT + wm * MTW + j) * 1024) + lane * 16);
            }
            if constexpr (FMT == 1) {
#pragma unroll
                for (int i = 0; i < RW; ++i) {
                    const f16x8 b = *(const f16x8 *)(wst + ((wn * RW + i) * T::TPS + kb) * 1024 + lane * 16);
#pragma unroll
                    for (int j = 0; j < MTW; ++j) {
                        acc[i][j] = mfma16(xa[j], b, acc[i][j]);
                        if constexpr (LO) acc[i][j] = mfma16(xl[j], b, acc[i][j]);
                    }
                }
                tile_done();
            } else {
                f32x4 xs[MTW];
                if constexpr (FMT == 3) {
#pragma unroll
                    for (int j = 0; j < MTW; ++j) {
                        xs[j] = mfma16(xa[j], ones8, zero4);
                        if constexpr (LO) xs[j] = mfma16(xl[j], ones8, xs[j]);
                    }
                }
#pragma unroll
                for (int i = 0; i < RW; ++i) {
                    const f16x8 b = unpack_step<FMT>(wt[i], kb);
                    f32x4 dd[MTW];
#pragma unroll
                    for (int j = 0; j < MTW; ++j) {
                        dd[j] = mfma16(xa[j], b, zero4);
                        if constexpr (LO) dd[j] = mfma16(xl[j], b, dd[j]);
                    }
                    if constexpr (FMT == 2) {
                        const float scale = (float)__builtin_bit_cast(f16, (uint16_t)(kb == 0 ? (s8[i] & 0xffffu) : (s8[i] >> 16)));
#pragma unroll
                        for (int j = 0; j < MTW; ++j) acc[i][j] += scale * dd[j];
                    } else {
                        const uint32_t d = kb == 0 ? s4[i].x : kb == 1 ? s4[i].y : kb == 2 ? s4[i].z : s4[i].w;
                        const float scale = (float)__builtin_bit_cast(f16, (uint16_t)(d & 0xffffu));
                        const float zero = (float)__builtin_bit_cast(f16, (uint16_t)(d >> 16));
#pragma unroll
                        for (int j = 0; j < MTW; ++j) acc[i][j] += scale * (dd[j] - zero * xs[j]);
                    }
                }
            }
        }
        if constexpr (FMT != 1) tile_done();
    }

    // ---- outputs: lane holds D[column 16 mt + 4 g + j][row 16 rg + r]
#pragma unroll
    for (int jt = 0; jt < MTW; ++jt) {
        const int mbase = (mt0 + wm * MTW + jt) * 16 + 4 * g;
        if constexpr (PAIR) {
#pragma unroll
            for (int i = 0; i < RW; i += 2) {
                const int n = ((rg0 + wn * RW + i) >> 1) * 16 + r;
                if (n >= a.n_real) continue;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (mbase + j < a.m) {
                        f16 hi, lo;
                        split_f16(silu_f(tot[i][jt][j]) * tot[i + 1][jt][j], hi, lo);
                        a.out_f16[act_off(mbase + j, n, a.n_real, a.mtp)] = hi;
                    }
            }
        } else {
#pragma unroll
            for (int i = 0; i < RW; ++i) {
                const int n = (rg0 + wn * RW + i) * 16 + r;
                if (n >= a.n_real) continue;
                float *o = a.out_f32 + (a.epi == EPI_PART ? (size_t)blockIdx.y * a.pstride : 0) + (size_t)mbase * a.ldo + n;
                const float bn = a.epi == EPI_STORE && a.bias ? a.bias[n] : 0.f;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (mbase + j < a.m) {
                        float v = tot[i][jt][j];
                        if constexpr (SUM) v = grand[i][jt][j];
                        else if (a.epi == EPI_RESID) v = o[(size_t)j * a.ldo] + v;
                        if (a.epi == EPI_STORE) v += bn;
                        o[(size_t)j * a.ldo] = v;
                    }
            }
        }
    }
}

// ------------------------------------------------------------------------------------------------ rotation, K/V
struct RopeWideArgs {
    RopeArgs r;             // r.kc / r.vc: the ring
    f16 *kn, *vn;           // staging [kv_head][cap][HD], row = column of the call
    int cap, to_ring;
};
// One block per column: rotates its queries and keys, stages K and V, and stores them to the column's ring slot when
// to_ring (no column of the call still sees what the slot held).
__global__ void __launch_bounds__(256) k_rope_wide(RopeWideArgs w) {
    const RopeArgs &a = w.r;
    const int b = blockIdx.x, half = a.HD >> 1;
    const sp_token t = a.toks[b];
    for (int idx = threadIdx.x; idx < (a.NH + a.NKV) * half; idx += 256) {
        const int head = idx / half, i = idx - head * half;
        const float2 cs = a.rtab[(size_t)b * half + i];
        const float x1 = qkv_value<0>(a, b, head * a.HD + i), x2 = qkv_value<0>(a, b, head * a.HD + i + half);
        float o1, o2;
        rope_pair(x1, x2, cs.x, cs.y, o1, o2);
        if (head < a.NH) {
            float *q = a.q + (size_t)b * a.NH * a.HD + head * a.HD;
            q[i] = o1; q[i + half] = o2;
        } else {
            const int kvh = head - a.NH;
            f16 *k = w.kn + ((size_t)kvh * w.cap + b) * a.HD;
            k[i] = (f16)o1; k[i + half] = (f16)o2;
            if (w.to_ring) {
                f16 *kr = a.kc + (((size_t)t.seq * a.NKV + kvh) * a.n_slots + t.slot) * a.HD;
                kr[i] = (f16)o1; kr[i + half] = (f16)o2;
            }
        }
    }
    const int v0 = (a.NH + a.NKV) * a.HD;
    for (int idx = threadIdx.x; idx < a.NKV * a.HD; idx += 256) {
        const int kvh = idx / a.HD, d = idx - kvh * a.HD;
        const f16 v = (f16)qkv_value<0>(a, b, v0 + idx);
        w.vn[((size_t)kvh * w.cap + b) * a.HD + d] = v;
        if (w.to_ring) a.vc[(((size_t)t.seq * a.NKV + kvh) * a.n_slots + t.slot) * a.HD + d] = v;
    }
}

// Staged K and V of every column that the ring still holds after the call (the last n_slots positions of its run).
__global__ void __launch_bounds__(256) k_ring_commit(const f16 *kn, const f16 *vn, f16 *kc, f16 *vc, const sp_token *toks,
                                                     const int *keep, int NKV, int HD, int n_slots, int cap) {
    const int b = blockIdx.x;
    if (!keep[b]) return;
    const sp_token t = toks[b];
    const int per = HD / 8;
    for (int i = threadIdx.x; i < NKV * per; i += 256) {
        const int kvh = i / per, c = (i - kvh * per) * 8;
        const size_t so = ((size_t)kvh * cap + b) * HD + c, dO = (((size_t)t.seq * NKV + kvh) * n_slots + t.slot) * HD + c;
        *(f16x8 *)(kc + dO) = *(const f16x8 *)(kn + so);
        *(f16x8 *)(vc + dO) = *(const f16x8 *)(vn + so);
    }
}

// --------------------------------------------------------------------------------------------------------- RMSNorm
// k_rmsnorm's work for the columns of a wide pass: x += the NP pending slices (in slice order, written back), then the
// normalised row as fp16 (and its remainders) in fragment order.  Four columns per block, two waves each: a lane
// holds octets of eight consecutive elements (16-byte loads, one 16-byte store per octet) and the four columns' stores
// of an octet are 64 contiguous bytes.  One block of 1024 threads per column stored 2 bytes per lane, in pieces of 16 bytes
// whose neighbours came from other blocks on other XCDs, and two such blocks fill a CU.  2048 columns of 1536: 11.5 -> 6.6
// us without pending slices, 18.8 -> 13.6 with two (63 MB: 4.6 TB/s); 16 ragged 0.5B prompts and a step 1278 -> 1206 us.
// H: a multiple of 8, at most 8 * 128 * 4.
// The sum of squares is k_rmsnorm's, bit for bit: its thread t squares elements t, t + 1024, .. in turn, its waves add
// their 64 threads by wave_sum_dpp, and the 16 wave sums are added in order.  Lane L of a column here holds the elements
// of threads 8 L .. 8 L + 7 (octets L, L + 128, ..), so eight lanes are one of those waves.
constexpr int NORM_COLS = 4, NORM_LANES = 128, NORM_MAX_H = 8 * NORM_LANES * 4;
static_assert(NORM_THREADS == 8 * NORM_LANES && NORM_PER_THREAD * NORM_THREADS == NORM_MAX_H,
              "k_rmsnorm's assignment of elements");

template <int NP, int NO>
__device__ __forceinline__ void norm_wide_body(float *x, int n, const float *part, size_t pstride, const float *w, int H,
                                               float eps, f16 *out, f16 *out_lo, int mtp) {
    constexpr int WAVES = NORM_LANES / 8;
    __shared__ float red[NORM_COLS][WAVES];
    const int t = threadIdx.x, lane = t & (NORM_LANES - 1), b = blockIdx.x * NORM_COLS + t / NORM_LANES;
    const int bc = min(b, n - 1), no = H >> 3;
    float *xr = x + (size_t)bc * H;
    f32x4 v[NO][2], wk[NO][2];
#pragma unroll
    for (int i = 0; i < NO; ++i) {
        const int k = 8 * min(lane + i * NORM_LANES, no - 1);      // octets past H re-read the last one
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            v[i][h] = *(const f32x4 *)(xr + k + 4 * h);
            wk[i][h] = *(const f32x4 *)(w + k + 4 * h);
        }
#pragma unroll
        for (int s = 0; s < NP; ++s)
#pragma unroll
            for (int h = 0; h < 2; ++h) v[i][h] += *(const f32x4 *)(part + s * pstride + (size_t)bc * H + k + 4 * h);
    }
    float s[8];
    {
#pragma clang fp contract(off)
#pragma unroll
        for (int e = 0; e < 8; ++e) s[e] = 0.f;
#pragma unroll
        for (int i = 0; i < NO; ++i) {
            const bool in = lane + i * NORM_LANES < no;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float u = in ? v[i][e >> 2][e & 3] : 0.f;
                s[e] += u * u;
            }
        }
    }
    // row16_sum over the lane's eight threads and its neighbour's, then the four rows of the wave
    float ss = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
    ss += dpp_mov<0xB1>(ss, 0.f);      // lane ^ 1
    ss += dpp_mov<0x4E>(ss, 0.f);      // lane ^ 2
    ss += dpp_mov<0x141>(ss, 0.f);     // the other four lanes of eight
    const int c = t / NORM_LANES;
    if ((t & 7) == 0) red[c][lane >> 3] = ss;
    __syncthreads();
    float tot = 0.f;
#pragma unroll
    for (int j = 0; j < WAVES; ++j) tot += red[c][j];
    const float rs = 1.0f / sqrtf(tot / (float)H + eps);
    if (b >= n) return;
#pragma unroll
    for (int i = 0; i < NO; ++i) {
        const int o = lane + i * NORM_LANES;
        if (o >= no) continue;
        f16x8 hi, lo;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            f16 a, r;
            split_f16((v[i][e >> 2][e & 3] * rs) * wk[i][e >> 2][e & 3], a, r);
            hi[e] = a;
            lo[e] = r;
        }
        const size_t at = act_off(b, 8 * o, H, mtp);
        *(f16x8 *)(out + at) = hi;
        if (out_lo) *(f16x8 *)(out_lo + at) = lo;
        if constexpr (NP > 0) {
            *(f32x4 *)(xr + 8 * o) = v[i][0];
            *(f32x4 *)(xr + 8 * o + 4) = v[i][1];
        }
    }
}
template <int NP>
__global__ void __launch_bounds__(NORM_COLS * NORM_LANES) k_norm_wide(float *x, int n, const float *part, size_t pstride,
                                                                      const float *w, int H, float eps, f16 *out,
                                                                      f16 *out_lo, int mtp) {
    if (H <= 8 * NORM_LANES) norm_wide_body<NP, 1>(x, n, part, pstride, w, H, eps, out, out_lo, mtp);
    else if (H <= 16 * NORM_LANES) norm_wide_body<NP, 2>(x, n, part, pstride, w, H, eps, out, out_lo, mtp);
    else norm_wide_body<NP, 4>(x, n, part, pstride, w, H, eps, out, out_lo, mtp);
}

// ------------------------------------------------------------------------------------------------ rows for the head
// x_out[i] = x[cols[i]] (fp32 rows of H) and attn_out's column i = attn's column cols[i] (fragment-major, K values): the
// columns whose logits are wanted, after the last layer's attention.
__global__ void __launch_bounds__(256) k_gather_cols(const float *x, const f16 *attn, const int *cols, int H, int K, int mtp,
                                                     float *x_out, f16 *attn_out, int mtp_out) {
    const int i = blockIdx.x, c = cols[i];
    for (int k = threadIdx.x; k < H; k += 256) x_out[(size_t)i * H + k] = x[(size_t)c * H + k];
    for (int k = 8 * threadIdx.x; k < K; k += 8 * 256)
        *(f16x8 *)(attn_out + act_off(i, k, 0, mtp_out)) = *(const f16x8 *)(attn + act_off(c, k, 0, mtp));
}

}  // namespace wide
