// Wide column steps: the kernels of a prefill over hundreds to thousands of columns per layer.
//
// A 64-column pass reads every weight once per 64 tokens and pays nine dependent launches per layer for them; what
// bounded it was the activations, which every row block reads from L2 again.  Here a layer's products run as tiled
// matrix products over all columns at once, and the attention as one pass over the keys per block of query rows.
//   k_gemm_wide   y[m][n] = sum_k x[m][k] W[n][k] over packed weight tiles (block dequantisation as in sp_gemv.h)
//   k_rope_wide   rotation; K and V of the new columns into a contiguous staging area (and their ring slots when no
//                 slot still visible to a column of the call is overwritten)
//   k_attn_wide   causal / windowed attention of the new columns over ring keys and staged keys, online softmax
//   k_ring_commit staged K and V into the ring, for calls longer than the ring has room for
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
// A stage holds KB 32-wide k-blocks: the activations as MFMA fragments (1 KiB per 16 columns x 32 k, the layout the
// producing kernels write, so a stage is copied in whole KiB), the packed weight tiles and their scales.
template <int FMT, int MTW, int RW, int WM, int WN, bool LO>
struct Tile {
    static constexpr int NW = WM * WN, BMT = MTW * WM, BNG = RW * WN;      // waves, column tiles, row groups
    static constexpr int TPS = FMT == 1 ? 2 : 1;                           // weight k-tiles per stage
    static constexpr int KB = FMT == 3 ? 4 : 2;                            // 32-wide k-blocks per stage
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
    static_assert(FMT == 1 || (S_PIECES >= 1 && S_PIECES <= NW), "one side copy per wave");
    static_assert(SMEM <= 160 * 1024, "the stages fit a CU's LDS");
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
    int mblocks, nblocks;  // grid tiles; gridDim.x = mblocks * nblocks, gridDim.y = k-slices
    int kslice;            // stages per slice
    int nst;               // stages of the whole K
    size_t pstride;
};

template <int FMT, int MTW, int RW, int WM, int WN, bool PAIR, bool LO>
__global__ void __launch_bounds__(64 * WM * WN) k_gemm_wide(GemmArgs a) {
    using T = Tile<FMT, MTW, RW, WM, WN, LO>;
    static_assert(!PAIR || RW % 2 == 0, "a wave holds the gate and the up row groups of its outputs");
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
    const int s0 = blockIdx.y * a.kslice, s1 = min(a.nst, s0 + a.kslice);

    // ---- this wave's copies: scalar base addresses, advanced by a constant per stage.  Column tiles and row groups
    // past the matrix re-read the last one (their outputs are not stored).
    const uint8_t *ab[T::A_PER], *wb[T::W_PER];
    uint32_t al[T::A_PER], wl[T::W_PER];
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(size_t)((__attribute__((address_space(3))) unsigned char *)smem));
#pragma unroll
    for (int i = 0; i < T::A_PER; ++i) {
        const int blk = wv * T::A_PER + i;                  // [hi / lo][k-block][column tile]
        const int half = blk / (T::KB * T::BMT), b2 = blk - half * (T::KB * T::BMT);
        const int kb = b2 / T::BMT, mt = min(mt0 + b2 - kb * T::BMT, a.mtp - 1);
        const f16 *src = LO && half ? a.xlo : a.x;
        ab[i] = (const uint8_t *)(src + ((size_t)(s0 * T::KB + kb) * a.mtp + mt) * 512);
        al[i] = lds0 + blk * 1024;
    }
#pragma unroll
    for (int i = 0; i < T::W_PER; ++i) {
        const int blk = wv * T::W_PER + i;                  // [row group][k-tile of the stage]
        const int rg = min(rg0 + blk / T::TPS, a.nrg - 1);
        wb[i] = a.w + ((size_t)rg * a.nkt + s0 * T::TPS + blk % T::TPS) * TILE_BYTES;
        wl[i] = lds0 + (T::A_KIB + blk) * 1024;
    }
    const uint8_t *sb = nullptr;
    uint32_t soff = 0, sl = 0;
    if constexpr (FMT != 1) {
        const int piece = wv % T::S_PIECES;
        sl = lds0 + (T::A_KIB + T::W_KIB) * 1024 + piece * 256;
        if constexpr (FMT == 2) {                           // 4 row groups: 16 rows x 2 scales each
            const int rg = min(rg0 + piece * 4 + g, a.nrg - 1);
            sb = (const uint8_t *)a.sz + (size_t)s0 * 64;
            soff = (uint32_t)rg * a.nkt * 64 + r * 4;
        } else {                                            // one row group: 16 rows x 4 (scale, zero)
            const int rg = min(rg0 + piece, a.nrg - 1);
            sb = (const uint8_t *)a.sz + ((size_t)rg * a.nkt + s0) * 256;
            soff = lane * 4;
        }
    }
    const uint32_t lo16 = lane * 16;
    const size_t astep = (size_t)T::KB * a.mtp * 1024;
    auto issue = [&](int slot) {
        const uint32_t d = slot * T::STAGE;
#pragma unroll
        for (int i = 0; i < T::W_PER; ++i) { copy16(wb[i], lo16, wl[i] + d); wb[i] += T::TPS * TILE_BYTES; }
        if constexpr (FMT != 1) { copy4(sb, soff, sl + d); sb += FMT == 2 ? 64 : 256; }
#pragma unroll
        for (int i = 0; i < T::A_PER; ++i) { copy16(ab[i], lo16, al[i] + d); ab[i] += astep; }
    };

    f32x4 acc[RW][MTW];
#pragma unroll
    for (int i = 0; i < RW; ++i)
#pragma unroll
        for (int j = 0; j < MTW; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const f16x8 ones8 = (f16x8){1, 1, 1, 1, 1, 1, 1, 1};

    const int n_st = s1 - s0;
#pragma unroll
    for (int p = 0; p < T::NS - 1; ++p)
        if (p < n_st) issue(p);
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
            } else {
                f32x4 xs[MTW];
                if constexpr (FMT == 3) {
#pragma unroll
                    for (int j = 0; j < MTW; ++j) {
                        xs[j] = mfma16(xa[j], ones8, (f32x4){0.f, 0.f, 0.f, 0.f});
                        if constexpr (LO) xs[j] = mfma16(xl[j], ones8, xs[j]);
                    }
                }
#pragma unroll
                for (int i = 0; i < RW; ++i) {
                    const f16x8 b = unpack_step<FMT>(wt[i], kb);
                    f32x4 dd[MTW];
#pragma unroll
                    for (int j = 0; j < MTW; ++j) {
                        dd[j] = mfma16(xa[j], b, (f32x4){0.f, 0.f, 0.f, 0.f});
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
                    if (mbase + j < a.m)
                        a.out_f16[act_off(mbase + j, n, a.n_real, a.mtp)] = (f16)(silu_f(acc[i][jt][j]) * acc[i + 1][jt][j]);
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
                        const float v = acc[i][jt][j] + bn;
                        o[(size_t)j * a.ldo] = a.epi == EPI_RESID ? o[(size_t)j * a.ldo] + v : v;
                    }
            }
        }
    }
}

// ------------------------------------------------------------------------------------------------ rotation, K/V
// A run: consecutive columns of one sequence at consecutive positions.
struct Run {
    int first_col, ncols, seq, p0;      // p0: cache position of the first column
};
// Query rows of one attention block: rows [row0, row0 + rows) of run `run` (row = column in the run * G + head in the group)
struct Item {
    int run, row0;
};

struct RopeWideArgs {
    RopeArgs r;             // r.kc / r.vc: the ring
    f16 *kn, *vn;           // staging [kv_head][cap][HD], row = column of the call
    int cap, to_ring;
};
// One block per column: rotates its queries and keys, stages K and V, and stores them to the column's ring slot when
// to_ring (no column of the call still sees what the slot held).
template <int NP>
__global__ void __launch_bounds__(256) k_rope_wide(RopeWideArgs w) {
    const RopeArgs &a = w.r;
    const int b = blockIdx.x, half = a.HD >> 1;
    const sp_token t = a.toks[b];
    for (int idx = threadIdx.x; idx < (a.NH + a.NKV) * half; idx += 256) {
        const int head = idx / half, i = idx - head * half;
        const float2 cs = a.rtab[(size_t)b * half + i];
        const float x1 = qkv_value<NP>(a, b, head * a.HD + i), x2 = qkv_value<NP>(a, b, head * a.HD + i + half);
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
        const f16 v = (f16)qkv_value<NP>(a, b, v0 + idx);
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

// ------------------------------------------------------------------------------------------------ attention
struct AttnWideArgs {
    const float *q;         // [columns][NH * HD]
    const f16 *kc, *vc;     // ring
    const f16 *kn, *vn;     // staging
    const sp_token *toks;
    const Run *runs;
    const Item *items;
    int NH, NKV, n_slots, cap, mtp;
    float scale;
    f16 *out;               // fragment-major [NH * HD]
};

// One block per (item, kv head): 64 RT query rows, RT tiles of 16 per wave, over the keys that any of its columns
// sees, 64 at a time: K row-major and V as transposed key pairs in LDS (the conflict-free layout of k_attn_mq), the
// next 64 keys' loads in flight meanwhile.  Scores take the queries as fp16 value + remainder (two MFMAs per step);
// the running maximum, sum and output are fp32.  Keys at or past the run's first position come from the staging
// area, earlier ones from the ring.  Bound by the vector instructions of a chunk's serial chain (load, stage, scores,
// softmax, P V), not by its matrix work (2048 columns, window 1024, 12 + 2 heads of 128: 14.5 GFLOP with the remainders
// in 55 us; 65 us with an address per key and a guarded natural exponential per score).
template <int HD, int G, int RT>
__global__ void __launch_bounds__(256) k_attn_wide(AttnWideArgs a) {
    constexpr int CH = 64, KP = HD + 8, VP = CH + 8, NST = CH / 16, NS2 = CH / 32, ST = HD / 32, CPR = HD / 8;
    constexpr int KPER = CH * CPR / 256, VPER = CH / 2 * CPR / 256;
    constexpr float LOG2E = 1.44269504088896340736f;     // scores in units of log 2: the weights are exp2 of differences
    __shared__ __align__(16) f16 k_s[CH][KP];
    __shared__ __align__(16) f16 vt_s[HD][VP];
    __shared__ __align__(16) f16 p_s[4][16][VP];
    const Item it = a.items[blockIdx.x];
    const Run run = a.runs[it.run];
    const int kvh = blockIdx.y, R = run.ncols * G;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, r16 = lane & 15, g4 = lane >> 4;
    const int c_first = it.row0 / G, c_last = min(it.row0 + 64 * RT - 1, R - 1) / G;
    const int lo = a.toks[run.first_col + c_first].ctx_lo, hi = run.p0 + c_last;
    // every row of the block sees keys [lo_all, hi_all]: chunks inside need no mask
    const int lo_all = a.toks[run.first_col + c_last].ctx_lo, hi_all = run.p0 + c_first;
    const size_t ring = ((size_t)run.seq * a.NKV + kvh) * a.n_slots, stage = (size_t)kvh * a.cap + run.first_col;

    // The thread's pieces of a chunk: K piece i is key (tid + 256 i) / CPR, V item i the key pair (tid + 256 i) % (CH / 2).
    // A chunk that lies in one piece of memory (all of it staged, or in the ring without a wrap: nearly every chunk) is
    // loaded from one base address; the others (across the first new position, the ring's end or the last key) find
    // each key's row by itself.
    f16x8 kf[KPER], vf[VPER][2];
    auto load = [&](int k0) {
        const int slot0 = k0 % a.n_slots;            // slot of key k0
        const bool staged = k0 >= run.p0;
        if (k0 + CH - 1 <= hi && (staged || (k0 + CH <= run.p0 && slot0 + CH <= a.n_slots))) {
            const size_t base = (staged ? stage + (k0 - run.p0) : ring + slot0) * HD;
            const f16 *kb = (staged ? a.kn : a.kc) + base, *vb = (staged ? a.vn : a.vc) + base;
#pragma unroll
            for (int i = 0; i < KPER; ++i) kf[i] = *(const f16x8 *)(kb + (tid + 256 * i) * 8);
#pragma unroll
            for (int i = 0; i < VPER; ++i) {
                const int idx = tid + 256 * i, kp2 = idx % (CH / 2), ch = idx / (CH / 2);
#pragma unroll
                for (int h = 0; h < 2; ++h) vf[i][h] = *(const f16x8 *)(vb + (2 * kp2 + h) * HD + ch * 8);
            }
            return;
        }
        auto row = [&](int j, bool &st) -> size_t {  // key k0 + j (clamped to the block's last key)
            const int p = min(k0 + j, hi);
            int s = slot0 + (p - k0);
            s = s >= a.n_slots ? s - a.n_slots : s;
            s = a.n_slots >= CH ? s : p % a.n_slots;
            st = p >= run.p0;
            return (st ? stage + (p - run.p0) : ring + s) * HD;
        };
#pragma unroll
        for (int i = 0; i < KPER; ++i) {
            const int idx = tid + 256 * i, j = idx / CPR, ch = idx - j * CPR;
            bool st;
            const size_t o = row(j, st);
            kf[i] = *(const f16x8 *)((st ? a.kn : a.kc) + o + ch * 8);
        }
#pragma unroll
        for (int i = 0; i < VPER; ++i) {
            const int idx = tid + 256 * i, kp2 = idx % (CH / 2), ch = idx / (CH / 2);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                bool st;
                const size_t o = row(2 * kp2 + h, st);
                vf[i][h] = *(const f16x8 *)((st ? a.vn : a.vc) + o + ch * 8);
            }
        }
    };
    load(lo);

    // query fragments of the wave's rows (value and remainder); rows past R are zero
    f16x8 qa[RT][ST], ql[RT][ST];
    int rlo[RT][4], rhi[RT][4];                      // visible range of the lane's output rows 4 g4 + j
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const int t0 = it.row0 + (wv * RT + rt) * 16;
        const int row = t0 + r16, rowc = min(row, R - 1), col = rowc / G, h = rowc - col * G;
        const float *qp = a.q + (size_t)(run.first_col + col) * a.NH * HD + (kvh * G + h) * HD + 8 * g4;
        const float qs = row < R ? a.scale * LOG2E : 0.f;
#pragma unroll
        for (int s = 0; s < ST; ++s) {
            const f32x4 x0 = *(const f32x4 *)(qp + 32 * s), x1 = *(const f32x4 *)(qp + 32 * s + 4);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                f16 vh, vl;
                split_f16((e < 4 ? x0[e & 3] : x1[e & 3]) * qs, vh, vl);
                qa[rt][s][e] = vh;
                ql[rt][s][e] = vl;
            }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int c = min(t0 + 4 * g4 + j, R - 1) / G;
            rlo[rt][j] = a.toks[run.first_col + c].ctx_lo;
            rhi[rt][j] = run.p0 + c;
        }
    }
    float mrow[RT][4], lrow[RT][4];
    f32x4 o[RT][HD / 16];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
        for (int j = 0; j < 4; ++j) { mrow[rt][j] = -INFINITY; lrow[rt][j] = 0.f; }
#pragma unroll
        for (int dt = 0; dt < HD / 16; ++dt) o[rt][dt] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }

    for (int k0 = lo; k0 <= hi; k0 += CH) {
        __syncthreads();                             // the previous keys have been read
#pragma unroll
        for (int i = 0; i < KPER; ++i) {
            const int idx = tid + 256 * i, j = idx / CPR, ch = idx - j * CPR;
            *(f16x8 *)&k_s[j][ch * 8] = kf[i];
        }
#pragma unroll
        for (int i = 0; i < VPER; ++i) {
            const int idx = tid + 256 * i, kp2 = idx % (CH / 2), ch = idx / (CH / 2);
#pragma unroll
            for (int e = 0; e < 8; ++e) *(f16x2 *)&vt_s[ch * 8 + e][2 * kp2] = (f16x2){vf[i][0][e], vf[i][1][e]};
        }
        __syncthreads();
        if (k0 + CH <= hi) load(k0 + CH);
        const bool whole = k0 >= lo_all && k0 + CH - 1 <= hi_all;

        f32x4 sc[RT][NST];
#pragma unroll
        for (int st = 0; st < NST; ++st) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) sc[rt][st] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < ST; ++s) {
                const f16x8 kb = *(const f16x8 *)&k_s[16 * st + r16][32 * s + 8 * g4];
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
                    sc[rt][st] = mfma16(qa[rt][s], kb, sc[rt][st]);
                    sc[rt][st] = mfma16(ql[rt][s], kb, sc[rt][st]);
                }
            }
        }
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            if (!whole) {
#pragma unroll
                for (int st = 0; st < NST; ++st) {
                    const int p = k0 + 16 * st + r16;
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        sc[rt][st][j] = ((p >= rlo[rt][j]) & (p <= rhi[rt][j])) ? sc[rt][st][j] : -INFINITY;
                }
            }
            float corr[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float mx = mrow[rt][j];
#pragma unroll
                for (int st = 0; st < NST; ++st) mx = fmaxf(mx, sc[rt][st][j]);
                mx = row16_max(mx);
                // a row without a visible key so far has mx = -inf and takes 0 as its reference: its weights are 0
                const float ref = mx == -INFINITY ? 0.f : mx;
                corr[j] = __builtin_amdgcn_exp2f(mrow[rt][j] - ref);
                float ls = 0.f;
#pragma unroll
                for (int st = 0; st < NST; ++st) {
                    const float e = __builtin_amdgcn_exp2f(sc[rt][st][j] - ref);
                    p_s[wv][4 * g4 + j][16 * st + r16] = (f16)e;
                    ls += e;
                }
                lrow[rt][j] = lrow[rt][j] * corr[j] + row16_sum(ls);
                mrow[rt][j] = mx;
            }
            __builtin_amdgcn_wave_barrier();
            f16x8 pa[NS2];
#pragma unroll
            for (int s2 = 0; s2 < NS2; ++s2) pa[s2] = *(const f16x8 *)&p_s[wv][r16][32 * s2 + 8 * g4];
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int dt = 0; dt < HD / 16; ++dt) {
#pragma unroll
                for (int j = 0; j < 4; ++j) o[rt][dt][j] *= corr[j];
#pragma unroll
                for (int s2 = 0; s2 < NS2; ++s2)
                    o[rt][dt] = mfma16(pa[s2], *(const f16x8 *)&vt_s[16 * dt + r16][32 * s2 + 8 * g4], o[rt][dt]);
            }
        }
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int row = it.row0 + (wv * RT + rt) * 16 + 4 * g4 + j;
            if (row >= R) continue;
            const int col = row / G, h = row - col * G;
            const float il = 1.f / lrow[rt][j];
#pragma unroll
            for (int dt = 0; dt < HD / 16; ++dt)
                a.out[act_off(run.first_col + col, (kvh * G + h) * HD + 16 * dt + r16, 0, a.mtp)] = (f16)(o[rt][dt][j] * il);
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
constexpr int NORM_COLS = 4, NORM_LANES = 128, NORM_MAX_H = 8 * NORM_LANES * 4;

template <int NP, int NO>
__device__ __forceinline__ void norm_wide_body(float *x, int n, const float *part, size_t pstride, const float *w, int H,
                                               float eps, f16 *out, f16 *out_lo, int mtp) {
    __shared__ float red[2 * NORM_COLS];
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
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NO; ++i) {
        const bool in = lane + i * NORM_LANES < no;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const f32x4 u = v[i][h];
            const float q = (u[0] * u[0] + u[1] * u[1]) + (u[2] * u[2] + u[3] * u[3]);
            ss += in ? q : 0.f;
        }
    }
    ss = wave_sum(ss);
    if ((t & 63) == 0) red[t >> 6] = ss;
    __syncthreads();
    const int c = t / NORM_LANES;
    const float rs = 1.0f / sqrtf((red[2 * c] + red[2 * c + 1]) / (float)H + eps);
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
// out[i] = x[cols[i]]: the residual rows whose logits are wanted
__global__ void __launch_bounds__(256) k_gather_rows(const float *x, const int *cols, int H, float *out) {
    const float *src = x + (size_t)cols[blockIdx.x] * H;
    for (int k = threadIdx.x; k < H; k += 256) out[(size_t)blockIdx.x * H + k] = src[k];
}

}  // namespace wide
