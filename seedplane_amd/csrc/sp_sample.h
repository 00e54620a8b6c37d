// Seeded sampling and speculative acceptance on the GPU, in float64.
//
// Every distribution is softmax(logits / T) over a full fp32 logits row, computed in fp64 with one fixed summation
// order so the CPU oracle can restate it: the row is cut into SMP_THREADS contiguous chunks of
// C = ceil(V / SMP_THREADS) entries; each chunk is summed sequentially in index order, and the chunk sums are added
// sequentially in chunk order.  Inverse-CDF draws use the same chunks: target = u * Z, the chunk whose prefix range
// holds the target is found from the sequential chunk prefixes, then scanned sequentially.
//
// Acceptance (speculative sampling with a residual, Leviathan et al. 2023 / Chen et al. 2023, extended to a tree
// of drafts as in SpecInfer, Miao et al. 2023): at a node, its trials -- the child each draft branch through the
// node drew, in branch (= draw) order, repeats kept in place -- are tried in turn; a child x is accepted iff
// u < p(x) / q(x) with p the target's current distribution and q the drafter's distribution at that node; each
// rejection replaces p by the residual norm(max(p - q, 0)).  If every child is rejected, the next token is drawn from the residual; if the
// accepted node has no children, a bonus token is drawn from the target's distribution there.  Uniforms are
// consumed in that order, one per trial and one for the final draw.
#pragma once
#include "sp_device.h"

constexpr int SMP_THREADS = 1024;      // chunks per row

// Seeded draws on many blocks per row, three launches, in the summation order stated at the top of this file:
//   k_smp_max   SMX_BLOCKS blocks per draw: partial maxima of the row (a maximum is exact in any order);
//   k_smp_sum   SMP_THREADS / SMS_CPB blocks per draw: the row maximum m from the partial maxima, then the sums of
//               SMS_CPB chunks: the block's threads compute the weights exp((l_i - m) / T) of a window of entries into
//               LDS, and one thread per chunk adds its chunk's entries of the window in index order, carrying the
//               chunk's running sum from window to window (the same additions as one thread summing its chunk);
//   k_smp_draw  one block per draw: thread 0 adds the chunk sums in chunk order (the total and the exclusive
//               prefixes), the chunk holding target = u * total is found, and its entries are scanned in index order
//               (weights computed by the block a window at a time, running sum by thread 0).
// Every total, prefix and comparison is that order's, so a sequential evaluation reproduces every draw bit for bit;
// the fallbacks: a chunk with no running sum above the target gives its last positive-weight index, no positive
// weight where the target fell gives the last positive-weight index of the row (0 if none).
// Scratch per draw: SMX_BLOCKS floats and SMP_THREADS doubles.
constexpr int SMX_BLOCKS = 64, SMS_CPB = 8, SMS_T = 256, SMS_WIN = 2048;

__device__ __forceinline__ double smp_weight(const float *l, int i, float m, double invT) {
    return exp(((double)l[i] - (double)m) * invT);
}

__device__ __forceinline__ float smp_row_max(const float *pmax) {
    float m = pmax[0];
    for (int j = 1; j < SMX_BLOCKS; ++j) m = fmaxf(m, pmax[j]);
    return m;
}

__global__ void __launch_bounds__(SMS_T) k_smp_max(const float *logits, int V, int ld, const int *rows, float *pmax) {
    __shared__ float red[SMS_T / 64];
    const int s = blockIdx.y, bk = blockIdx.x;
    const float *l = logits + (size_t)rows[s] * ld;
    const int per = (V + SMX_BLOCKS - 1) / SMX_BLOCKS;
    const int lo = bk * per, hi = min(V, lo + per);
    float m = -INFINITY;
    for (int i = lo + (int)threadIdx.x; i < hi; i += SMS_T) m = fmaxf(m, l[i]);
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        float t = red[0];
        for (int j = 1; j < SMS_T / 64; ++j) t = fmaxf(t, red[j]);
        pmax[s * SMX_BLOCKS + bk] = t;
    }
}

__global__ void __launch_bounds__(SMS_T) k_smp_sum(const float *logits, int V, int ld, const int *rows, double invT,
                                                    const float *pmax, double *csum) {
    __shared__ double w[SMS_WIN];
    const int s = blockIdx.y;
    const float *l = logits + (size_t)rows[s] * ld;
    const float m = smp_row_max(pmax + s * SMX_BLOCKS);
    const int C = (V + SMP_THREADS - 1) / SMP_THREADS;
    const int c0 = blockIdx.x * SMS_CPB;
    const int lo = min(V, c0 * C), hi = min(V, (c0 + SMS_CPB) * C);
    const int t = threadIdx.x;
    // thread t < SMS_CPB owns chunk c0 + t: entries [clo, chi)
    const int clo = min(V, (c0 + t) * C), chi = min(V, (c0 + t + 1) * C);
    double acc = 0.0;
    for (int wlo = lo; wlo < hi; wlo += SMS_WIN) {
        const int whi = min(hi, wlo + SMS_WIN);
        for (int i = wlo + t; i < whi; i += SMS_T) w[i - wlo] = smp_weight(l, i, m, invT);
        __syncthreads();
        if (t < SMS_CPB) {
            const int a = max(clo, wlo), e = min(chi, whi);
            for (int i = a; i < e; ++i) acc += w[i - wlo];
        }
        __syncthreads();
    }
    if (t < SMS_CPB) csum[(size_t)s * SMP_THREADS + c0 + t] = acc;
}

__global__ void __launch_bounds__(SMS_T) k_smp_draw(const float *logits, int V, int ld, const int *rows,
                                                     const double *u, double invT, const float *pmax,
                                                     const double *csum, int *out) {
    __shared__ double pre[SMP_THREADS + 1];
    __shared__ double w[SMS_WIN + 16];
    __shared__ int sel, found;
    __shared__ int last[SMS_T / 64];
    const int s = blockIdx.x, t = threadIdx.x;
    const float *l = logits + (size_t)rows[s] * ld;
    const float m = smp_row_max(pmax + s * SMX_BLOCKS);
    const int C = (V + SMP_THREADS - 1) / SMP_THREADS;
    for (int j = t; j < SMP_THREADS; j += SMS_T) pre[j] = csum[(size_t)s * SMP_THREADS + j];
    if (t == 0) { sel = -1; found = -1; }
    __syncthreads();
    if (t == 0) {
        // the sums in chunk order; each batch of 32 is read into registers first, so the reads do not wait on the
        // prefixes written before them
        double p = 0.0;
        for (int j0 = 0; j0 < SMP_THREADS; j0 += 32) {
            double c[32];
#pragma unroll
            for (int k = 0; k < 32; ++k) c[k] = pre[j0 + k];
#pragma unroll
            for (int k = 0; k < 32; ++k) {
                pre[j0 + k] = p;
                p += c[k];
            }
        }
        pre[SMP_THREADS] = p;
    }
    __syncthreads();
    const double target = u[s] * pre[SMP_THREADS];
    for (int j = t; j < SMP_THREADS; j += SMS_T)
        if (target >= pre[j] && (j + 1 == SMP_THREADS || target < pre[j + 1])) sel = j;
    __syncthreads();
    if (sel >= 0) {
        // scan chunk sel from zero against target - prefix: the first index whose running sum exceeds it, else the
        // chunk's last positive-weight index
        const int clo = min(V, sel * C), chi = min(V, sel * C + C);
        const double tl = target - pre[sel];
        double acc = 0.0;
        int pick = -1, lastpos = -1;
        for (int wlo = clo; wlo < chi; wlo += SMS_WIN) {
            const int whi = min(chi, wlo + SMS_WIN);
            for (int i = wlo + t; i < whi; i += SMS_T) w[i - wlo] = smp_weight(l, i, m, invT);
            __syncthreads();
            if (t == 0 && pick < 0) {
                // in index order, 16 weights read ahead at a time (what lies past the window is read, never used)
                for (int i0 = wlo; i0 < whi && pick < 0; i0 += 16) {
                    double c[16];
#pragma unroll
                    for (int k = 0; k < 16; ++k) c[k] = w[i0 - wlo + k];
#pragma unroll
                    for (int k = 0; k < 16; ++k) {
                        const int i = i0 + k;
                        if (pick < 0 && i < whi) {
                            if (c[k] > 0.0) lastpos = i;
                            acc += c[k];
                            if (acc > tl) pick = i;
                        }
                    }
                }
                found = pick;
            }
            __syncthreads();
            if (found >= 0) break;
        }
        if (t == 0 && pick < 0) found = lastpos;
        __syncthreads();
    }
    if (found < 0) {
        // no positive weight where the target fell: the last positive-weight index of the row (0 if none)
        int best = 0;
        for (int i = t; i < V; i += SMS_T)
            if (smp_weight(l, i, m, invT) > 0.0) best = max(best, i);
        for (int o = 32; o > 0; o >>= 1) best = max(best, __shfl_xor(best, o, SP_WAVE));
        if ((t & 63) == 0) last[t >> 6] = best;
        __syncthreads();
        if (t == 0) {
            int b = last[0];
            for (int j = 1; j < SMS_T / 64; ++j) b = max(b, last[j]);
            found = b;
        }
        __syncthreads();
    }
    if (t == 0) out[s] = found;
}

// One level of a drafter's proposal on the device (one block, thread b = branch b < nb; tokens [levels][nb]): the
// branch's canonical branch at `level` -- the first branch whose tokens at levels 0..level equal its own, so every
// branch through a tree node draws from that node's one row -- then, for the level's columns, column b's tree mask
// (the canonical node of its branch at every earlier level, node index level' * nb + canonical, and the column
// itself) and the row its next token is drawn from (its canonical column).
__global__ void k_draft_link(const int *tokens, int nb, int level, int *canon, unsigned long long *masks, int *rows) {
    const int b = threadIdx.x;
    if (b >= nb) return;
    int c = b;
    for (int o = 0; o < b; ++o) {
        bool same = true;
        for (int lv = 0; lv <= level; ++lv) same = same && tokens[lv * nb + o] == tokens[lv * nb + b];
        if (same) { c = o; break; }
    }
    canon[level * nb + b] = c;
    unsigned long long m = 1ull << (level * nb + b);
    for (int lv = 0; lv < level; ++lv) m |= 1ull << (lv * nb + canon[lv * nb + b]);
    masks[b] = m;
    rows[b] = c;
}

// ---------------------------------------------------------------------------------------------------------------
// Tree acceptance on ACC_NB co-resident blocks (a plain launch: 64 blocks of 256 threads are all resident on the
// 256-CU chip once the stream's previous kernel has finished, and every exchange wait is bounded, so a block that
// never arrives ends the launch with an error instead of a hang; a cooperative launch enqueued behind a running
// kernel slowed that kernel by ~10 %).  The vocabulary is cut into ACC_NB x ACC_T contiguous chunks of
// C = ceil(V / (ACC_NB * ACC_T)) entries; thread t of block b owns chunk b * ACC_T + t and keeps its logits' weights
// in registers.  Sums are taken sequentially inside a chunk, then over the ACC_T chunk sums of a block (butterfly in
// each wave, wave sums in order: the block partial), then sequentially over the ACC_NB block partials.  Block partials are all-gathered through
// tagged 64-bit words (32-bit payload + 32-bit tag, single-copy atomic; relaxed agent-scope atomics, no fences), so
// every block holds every partial and takes every accept / reject decision itself.
//
// Normalisers in one exchange per node: block b finds its maximum m_b, its entries' local weights
// e_i = exp((l_i - m_b) * (1/T)) (all zero if m_b = -inf) and their sum s_b, and the exchange hands every block every
// (m_b, s_b).  With M = max m_b and f_b = exp((m_b - M) * (1/T)): Z = sum over b of s_b * f_b in block order, the
// probability of entry i of block b is p_i = e_i * (f_b / Z), and a bonus draw takes the weights e_i * f_b with block
// partials s_b * f_b.
//
// Residual after j >= 1 rejections at a node: r_j = max(p - c_j q, 0) / S_j with c_1 = 1, S_j = sum of the numerator,
// c_{j+1} = c_j + S_j -- algebraically the same as replacing p by norm(max(p - q, 0)) after each rejection, but each
// rejection costs one reduction instead of a rewrite of the distribution.  All arithmetic is float64 with explicit
// single roundings (no contraction): d_i = p_i - c * q_i.
constexpr int ACC_NB = 64, ACC_T = 256, ACC_PER = 16;
constexpr int ACC_XW = 6;   // exchange words per block: two doubles (two words each) and two floats
// Tree inputs staged in LDS by every block at the start (one round of independent loads, also from pinned host
// memory): up to ACC_MAX_NODES nodes, ACC_MAX_TRIALS trials and the first ACC_U_LDS uniforms (later ones are read
// where they lie).
constexpr int ACC_MAX_NODES = 64, ACC_MAX_TRIALS = 1024, ACC_U_LDS = 256;

struct AcceptArgs {
    const float *p_logits;   // target logits [nodes][ld]
    const float *q_logits;   // drafter logits [nodes][ld] (rows of nodes with trials)
    int V, ld;
    const int *token;        // [nodes] token of node i (node 0 = root)
    const int *trial_start;  // [nodes] first entry of node i's trials
    const int *n_trials;     // [nodes]
    const int *trials;       // child node index of each trial
    const double *u;         // uniforms, consumed in order
    int n_u;
    double invT;
    unsigned long long *xbuf;   // exchange words [4][ACC_NB][ACC_XW]
    unsigned *err;           // tag_base | 1 if an exchange timed out, tag_base | 2 for a malformed tree (words of
                             // earlier launches carry other tags, so the word is never cleared)
    unsigned tag_base;       // distinct per launch (low 12 bits are the exchange counter)
    int n_nodes, n_trials_total;
    int *out;                // [0] k, [1..k] accepted node ids, [max_depth+1] final token, [max_depth+2] uniforms used,
                             // [max_depth+3] bonus flag
    int max_depth;
    int *host;               // may be NULL: pinned host block written directly: [0] the err word, [1] block 0's
                             // completion tag, [2] the drawing block's tag, [ACC_HOST_OUT ..] a copy of out
    const int *q_row;        // may be NULL: node i's drafter row is q_row[i] (< n_q_rows) instead of i
    int n_q_rows;
};
constexpr int ACC_HOST_OUT = 16;

struct AccShared {
    double tsum[ACC_T];      // thread chunk sums
    double bpart0[ACC_NB], bpart1[ACC_NB];
    float bmax0[ACC_NB], bmax1[ACC_NB];
    double fac0[ACC_NB], fac1[ACC_NB];
    float fred[ACC_T / 64], fred2[ACC_T / 64];
    double tl;
    int found;
    int ok;
};

__device__ __forceinline__ double d_w(float l, float m, double invT) {
    return exp(__dmul_rn(__dsub_rn((double)l, (double)m), invT));
}

// Whether a block of this launch has reported a failure.
__device__ __forceinline__ bool acc_failed(const AcceptArgs &a) {
    const unsigned e = __hip_atomic_load(a.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return (e & ~0xfffu) == a.tag_base && (e & 0xfffu) != 0;
}

// All-gather of two doubles (and, with W = ACC_XW, two floats) per block into sh.bpart0 / bpart1 (bmax0 / bmax1).
// Returns false on timeout (every block then stops).
template <int W>
__device__ bool acc_exchange(const AcceptArgs &a, unsigned &ex, double v0, double v1, float f0, float f1,
                             AccShared &sh) {
    static_assert(W == 4 || W == ACC_XW, "two doubles, or two doubles and two floats");
    const unsigned tag = a.tag_base | (ex & 0xfffu);
    unsigned long long *slot = a.xbuf + (size_t)(ex & 3u) * ACC_NB * ACC_XW;
    ++ex;
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned long long b0 = __double_as_longlong(v0), b1 = __double_as_longlong(v1);
        const unsigned long long t = (unsigned long long)tag << 32;
        unsigned long long *w = slot + blockIdx.x * ACC_XW;
        __hip_atomic_store(w + 0, t | (b0 & 0xffffffffull), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(w + 1, t | (b0 >> 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(w + 2, t | (b1 & 0xffffffffull), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(w + 3, t | (b1 >> 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (W == ACC_XW) {
            __hip_atomic_store(w + 4, t | __float_as_uint(f0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(w + 5, t | __float_as_uint(f1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    if (threadIdx.x == 0) sh.ok = 1;
    __syncthreads();
    if (threadIdx.x < ACC_NB) {
        unsigned long long *w = slot + threadIdx.x * ACC_XW;
        unsigned long long x[W];
        long spins = 0;
        for (;;) {
            bool all = true;
#pragma unroll
            for (int i = 0; i < W; ++i) x[i] = __hip_atomic_load(w + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (int i = 0; i < W; ++i) all = all && (unsigned)(x[i] >> 32) == tag;
            if (all) break;
            if (++spins > (1l << 22) || acc_failed(a)) {
                __hip_atomic_store(a.err, a.tag_base | 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                sh.ok = 0;
                break;
            }
        }
        sh.bpart0[threadIdx.x] = __longlong_as_double((long long)((x[0] & 0xffffffffull) | (x[1] << 32)));
        sh.bpart1[threadIdx.x] = __longlong_as_double((long long)((x[2] & 0xffffffffull) | (x[3] << 32)));
        if (W == ACC_XW) {
            sh.bmax0[threadIdx.x] = __uint_as_float((unsigned)x[W == ACC_XW ? 4 : 0]);
            sh.bmax1[threadIdx.x] = __uint_as_float((unsigned)x[W == ACC_XW ? 5 : 0]);
        }
    }
    __syncthreads();
    return sh.ok != 0;
}

// Wave sum of doubles by the butterfly that adds lane l ^ o for o = 32, 16, .. 1 (every lane ends with the same bits),
// on register moves instead of LDS-routed shuffles.  The half-wave and row swaps hand every lane both values of its
// pair; within a row of 16 a rotation by 8 is lane ^ 8, and after that step lanes l and l ^ 8 hold the same bits, so a
// rotation by 4 stands for lane ^ 4.
template <int CTRL>
__device__ __forceinline__ double acc_dpp(double v) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, 0xF, 0xF, false);
    const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, 0xF, 0xF, false);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ double acc_wave_sum(double v) {
    auto both = [&](bool half) {
        const unsigned long long b = (unsigned long long)__double_as_longlong(v);
        const unsigned lo = (unsigned)b, hi = (unsigned)(b >> 32);
        const u32x2 l = half ? __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(lo, lo, false, false))
                             : __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(lo, lo, false, false));
        const u32x2 h = half ? __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(hi, hi, false, false))
                             : __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(hi, hi, false, false));
        v = __longlong_as_double((long long)(((unsigned long long)h[0] << 32) | l[0])) +
            __longlong_as_double((long long)(((unsigned long long)h[1] << 32) | l[1]));
    };
    both(true);                     // lane ^ 32
    both(false);                    // lane ^ 16
    v += acc_dpp<0x128>(v);         // row_ror:8
    v += acc_dpp<0x124>(v);         // row_ror:4
    v += acc_dpp<0x4E>(v);          // quad_perm [2,3,0,1]
    v += acc_dpp<0xB1>(v);          // quad_perm [1,0,3,2]
    return v;
}

// Block sum of the ACC_T thread chunk sums: butterfly inside each wave, then the ACC_T / 64 wave sums in wave order.
// Also leaves the thread sums in sh.tsum for a draw.
__device__ double acc_block_sum(double mine, AccShared &sh) {
    __shared__ double wsum[ACC_T / 64];
    __syncthreads();
    sh.tsum[threadIdx.x] = mine;
    const double v = acc_wave_sum(mine);
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = 0.0;
#pragma unroll
    for (int j = 0; j < ACC_T / 64; ++j) t += wsum[j];
    return t;
}

// Block sums / maxima of two values at once (one barrier round for both); no thread sums are kept.
__device__ void acc_block_sum2(double &a, double &b, AccShared &sh) {
    __shared__ double w2[2][ACC_T / 64];
    a = acc_wave_sum(a);
    b = acc_wave_sum(b);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) { w2[0][threadIdx.x >> 6] = a; w2[1][threadIdx.x >> 6] = b; }
    __syncthreads();
    a = 0.0; b = 0.0;
#pragma unroll
    for (int j = 0; j < ACC_T / 64; ++j) { a += w2[0][j]; b += w2[1][j]; }
}

__device__ void acc_block_max2(float &a, float &b, AccShared &sh) {
    a = wave_max_dpp(a);
    b = wave_max_dpp(b);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) { sh.fred[threadIdx.x >> 6] = a; sh.fred2[threadIdx.x >> 6] = b; }
    __syncthreads();
    a = sh.fred[0]; b = sh.fred2[0];
    for (int j = 1; j < ACC_T / 64; ++j) { a = fmaxf(a, sh.fred[j]); b = fmaxf(b, sh.fred2[j]); }
}

// Position of `target` in the running sum of v[0..N), in that order: the first t with target < v[0] + ... + v[t] (any
// comparison order finds the same one, the sums never fall), or, when no sum exceeds it, the last positive entry;
// `before` receives the running sum before it.  The values are read ACC_SCAN at a time, so a batch costs one LDS round
// trip and its dependent additions instead of a round trip and a branch per entry.  The walk is a serial chain (loads,
// exponentials, block sums, one exchange per node and rejection, the draw's scans); with these scans, the sums on
// register moves and a node's trials evaluated side by side, a call over an 8 x 4 tree and 151936 entries went from
// 77.7 to 62.0 us.
constexpr int ACC_SCAN = 16;
template <int N>
__device__ __forceinline__ int acc_find(const double *v, double target, double &before) {
    double run = 0.0;
    for (int b = 0; b < N; b += ACC_SCAN) {
        double x[ACC_SCAN], sum[ACC_SCAN];
#pragma unroll
        for (int i = 0; i < ACC_SCAN; ++i) x[i] = v[b + i];
        sum[0] = run + x[0];
#pragma unroll
        for (int i = 1; i < ACC_SCAN; ++i) sum[i] = sum[i - 1] + x[i];
        if (target < sum[ACC_SCAN - 1]) {
            int at = b + ACC_SCAN - 1;
            before = sum[ACC_SCAN - 2];
#pragma unroll
            for (int i = ACC_SCAN - 2; i >= 0; --i)
                if (target < sum[i]) { at = b + i; before = i > 0 ? sum[i > 0 ? i - 1 : 0] : run; }
            return at;
        }
        run = sum[ACC_SCAN - 1];
    }
    int last = 0;
    double q = 0.0;
    before = 0.0;
    for (int t = 0; t < N; ++t) {
        if (v[t] > 0.0) { last = t; before = q; }
        q += v[t];
    }
    return last;
}
// Sum of the ACC_NB block partials in block order.
__device__ __forceinline__ double acc_sum_blocks(const double *bp) {
    double t = 0.0;
#pragma unroll
    for (int b = 0; b < ACC_NB; b += ACC_SCAN) {
        double x[ACC_SCAN];
#pragma unroll
        for (int i = 0; i < ACC_SCAN; ++i) x[i] = bp[b + i];
#pragma unroll
        for (int i = 0; i < ACC_SCAN; ++i) t += x[i];
    }
    return t;
}
// Inverse-CDF draw over the distributed weights w[] (this thread's chunk; thread chunk sums in sh.tsum, block
// partials in bp).  Three levels, each "first entry whose running sum exceeds the target, else the last positive
// entry": block (every block, redundantly), thread (thread 0 of the owning block), element (the owning thread).
// If no weight is positive at all the token is 0.  Returns the token in the owning block, -1 in the others.
template <int CP>
__device__ int acc_draw(const double *w, int lo, int n, double u, const double *bp, AccShared &sh) {
    const double target = __dmul_rn(u, acc_sum_blocks(bp));
    double Pown;
    const int owner = acc_find<ACC_NB>(bp, target, Pown);
    if ((int)blockIdx.x != owner) return -1;
    const double tb = __dsub_rn(target, Pown);
    __syncthreads();
    if (threadIdx.x == 0) {
        double qsel;
        sh.found = acc_find<ACC_T>(sh.tsum, tb, qsel);
        sh.tl = __dsub_rn(tb, qsel);
    }
    __syncthreads();
    const int tsel = sh.found;
    __syncthreads();
    if ((int)threadIdx.x == tsel) {
        const double tl = sh.tl;
        double acc = 0.0;
        int pick = -1, lastpos = -1;
        for (int i = 0; i < CP; ++i) {
            if (i < n) {
                if (w[i] > 0.0) lastpos = lo + i;
                acc += w[i];
                if (acc > tl) { pick = lo + i; break; }
            }
        }
        if (pick < 0) pick = lastpos >= 0 ? lastpos : lo;
        sh.found = pick;
    }
    __syncthreads();
    return sh.found;
}

// Stops every block identically (the condition depends only on the inputs) and reports a malformed tree.
__device__ __forceinline__ bool acc_bad(const AcceptArgs &a) {
    if (blockIdx.x == 0 && threadIdx.x == 0)
        __hip_atomic_store(a.err, a.tag_base | 2u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return false;
}

__device__ __forceinline__ void acc_put(const AcceptArgs &a, int i, int v) {
    a.out[i] = v;
    if (a.host) a.host[ACC_HOST_OUT + i] = v;
}

// CP >= C: the entries per thread as a compile-time count, so every per-entry loop is straight-line code whose loads
// and exponentials are independent (entries past the thread's n are read from a clamped index and masked).
template <int CP>
__global__ void __launch_bounds__(ACC_T) k_accept_tree(AcceptArgs a) {
    // p - c q products and differences are rounded separately, as the definition writes them (hipcc would otherwise
    // contract them into fused multiply-adds; __dmul_rn / __dsub_rn are plain operators in HIP)
#pragma clang fp contract(off)
    __shared__ AccShared sh;
    __shared__ int s_token[ACC_MAX_NODES], s_tstart[ACC_MAX_NODES], s_ntr[ACC_MAX_NODES], s_trials[ACC_MAX_TRIALS];
    __shared__ int s_qrow[ACC_MAX_NODES];
    __shared__ double s_u[ACC_U_LDS];
    const int C = (a.V + ACC_NB * ACC_T - 1) / (ACC_NB * ACC_T);
    const int lo = (blockIdx.x * ACC_T + threadIdx.x) * C;
    const int n = max(0, min(C, a.V - lo));
    // the tree and the uniforms into LDS (independent loads, all in flight together)
    for (int i = threadIdx.x; i < a.n_nodes; i += ACC_T) {
        s_token[i] = a.token[i];
        s_tstart[i] = a.trial_start[i];
        s_ntr[i] = a.n_trials[i];
        s_qrow[i] = a.q_row ? a.q_row[i] : i;
    }
    for (int i = threadIdx.x; i < a.n_trials_total; i += ACC_T) s_trials[i] = a.trials[i];
    for (int i = threadIdx.x; i < min(a.n_u, ACC_U_LDS); i += ACC_T) s_u[i] = a.u[i];
    __syncthreads();
    auto uni = [&](int i) { return i < a.n_u ? (i < ACC_U_LDS ? s_u[i] : a.u[i]) : 0.5; };
    double wp[CP], w[CP];
    unsigned ex = 0;
    int cur = 0, k = 0, ui = 0, final_tok = -1, bonus = 0;
    bool alive = true;
    for (;;) {
        const float *pl = a.p_logits + (size_t)cur * a.ld;
        const int nt = s_ntr[cur];
        const int t0 = s_tstart[cur];
        if (nt < 0 || t0 < 0 || t0 > a.n_trials_total - nt) { alive = acc_bad(a); break; }
        for (int j = t0; j < t0 + nt && alive; ++j) {
            const int child = s_trials[j];
            if (child <= 0 || child >= a.n_nodes || s_token[child] < 0 || s_token[child] >= a.V) alive = acc_bad(a);
        }
        const int qr = s_qrow[cur];
        if (nt > 0 && a.q_row && (qr < 0 || qr >= a.n_q_rows)) alive = acc_bad(a);
        if (!alive) break;
        const bool draw_bonus = nt == 0 || k >= a.max_depth;
        const float *ql = a.q_logits + (size_t)(nt > 0 ? qr : 0) * a.ld;
        // the trials' logits, lane j holding trial t0 + j (the tree was validated above; lanes past the node's trials
        // repeat the last one, trials past a wave's 64 lanes are loaded when their turn comes)
        const int lane = threadIdx.x & 63;
        const int xl = nt > 0 ? s_token[s_trials[t0 + min(lane, nt - 1)]] : 0;
        const float lpl = pl[xl], lql = ql[xl];
        // ---- the node's logits (one batch of loads, clamped indices), this block's maxima, its local weights
        // e_i = exp((l_i - m_b) / T) (zero in a block without a finite logit) and their block sums s_b; one exchange
        // of (s_b, m_b) for p and q
        float lp[CP], lq[CP];
#pragma unroll
        for (int i = 0; i < CP; ++i) {
            const int kk = min(lo + i, a.V - 1);
            lp[i] = pl[kk];
            lq[i] = ql[kk];
        }
        float mp = -INFINITY, mq = -INFINITY;
#pragma unroll
        for (int i = 0; i < CP; ++i) {
            if (i < n) { mp = fmaxf(mp, lp[i]); mq = fmaxf(mq, lq[i]); }
        }
        if (draw_bonus) mq = -INFINITY;
        acc_block_max2(mp, mq, sh);
        const bool livep = mp > -INFINITY, liveq = mq > -INFINITY;
        double ep[CP], eq[CP];
#pragma unroll
        for (int i = 0; i < CP; ++i) ep[i] = livep ? d_w(lp[i], mp, a.invT) : 0.0;
        if (!draw_bonus) {
#pragma unroll
            for (int i = 0; i < CP; ++i) eq[i] = liveq ? d_w(lq[i], mq, a.invT) : 0.0;
        }
        double sp = 0.0, sq = 0.0;
#pragma unroll
        for (int i = 0; i < CP; ++i) {
            if (i < n) {
                sp += ep[i];
                if (!draw_bonus) sq += eq[i];
            }
        }
        acc_block_sum2(sp, sq, sh);
        if (!(alive = acc_exchange<ACC_XW>(a, ex, sp, sq, mp, mq, sh))) break;
        // factors f_b = exp((m_b - M) / T) of the global maxima and the block partials s_b * f_b (wave 0, lane b for
        // block b: the maxima are a reduction over its lanes)
        static_assert(ACC_NB == SP_WAVE, "one lane per block");
        if (threadIdx.x < ACC_NB) {
            const int b = threadIdx.x;
            const float Mp = wave_max_dpp(sh.bmax0[b]), Mq = wave_max_dpp(sh.bmax1[b]);
            const double fp = d_w(sh.bmax0[b], Mp, a.invT);
            sh.fac0[b] = fp;
            sh.bpart0[b] = __dmul_rn(sh.bpart0[b], fp);
            if (!draw_bonus) {
                const double fq = d_w(sh.bmax1[b], Mq, a.invT);
                sh.fac1[b] = fq;
                sh.bpart1[b] = __dmul_rn(sh.bpart1[b], fq);
            }
        }
        __syncthreads();
        if (draw_bonus) {
            // weights e_i * f_b; thread chunk sums into sh.tsum, block partials s_b * f_b in sh.bpart0
            const double f = sh.fac0[blockIdx.x];
            sp = 0.0;
#pragma unroll
            for (int i = 0; i < CP; ++i) {
                wp[i] = i < n ? __dmul_rn(ep[i], f) : 0.0;
                if (i < n) sp += wp[i];
            }
            (void)acc_block_sum(sp, sh);
            final_tok = acc_draw<CP>(wp, lo, n, uni(ui), sh.bpart0, sh);
            ++ui;
            bonus = 1;
            break;
        }
        const double Zp = acc_sum_blocks(sh.bpart0), Zq = acc_sum_blocks(sh.bpart1);
        // ---- trials in draw order, with p_i = e_i * (f_b / Zp) and q_i likewise (formed only after a rejection)
        const double gp = __ddiv_rn(sh.fac0[blockIdx.x], Zp), gq = __ddiv_rn(sh.fac1[blockIdx.x], Zq);
        const int span = ACC_T * C;     // entries per block
        int accepted = -1, J = 0;
        double c = 0.0, S = 0.0;
        // p(x) and q(x) of a trial; the node's trials are evaluated side by side, one per lane, and read by lane below
        auto at_token = [&](int x, float lpx, float lqx, double &px, double &qx) {
            const int bx = x / span;
            const float mpx = sh.bmax0[bx], mqx = sh.bmax1[bx];
            px = mpx > -INFINITY ? __dmul_rn(d_w(lpx, mpx, a.invT), __ddiv_rn(sh.fac0[bx], Zp)) : 0.0;
            qx = mqx > -INFINITY ? __dmul_rn(d_w(lqx, mqx, a.invT), __ddiv_rn(sh.fac1[bx], Zq)) : 0.0;
        };
        double pxl, qxl;
        at_token(xl, lpl, lql, pxl, qxl);
        auto from_lane = [](double v, int l) {
            const unsigned long long b = (unsigned long long)__double_as_longlong(v);
            const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, l);
            const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), l);
            return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
        };
        for (int j = t0; j < t0 + nt; ++j) {
            const int child = s_trials[j];
            double px0, qx;
            if (j - t0 < SP_WAVE) {
                px0 = from_lane(pxl, __builtin_amdgcn_readfirstlane(j - t0));
                qx = from_lane(qxl, __builtin_amdgcn_readfirstlane(j - t0));
            } else {
                const int x = s_token[child];
                at_token(x, pl[x], ql[x], px0, qx);
            }
            double px = px0;
            if (J > 0) {
                const double dx = __dsub_rn(px0, __dmul_rn(c, qx));
                px = dx > 0.0 ? __ddiv_rn(dx, S) : 0.0;
            }
            const double uu = uni(ui);
            ++ui;
            if (uu < __ddiv_rn(px, qx)) { accepted = child; break; }
            // rejection: next residual numerator max(p - c q, 0) with c = 1 (first) or c + S
            c = J == 0 ? 1.0 : c + S;
            ++J;
            double sr = 0.0;
#pragma unroll
            for (int i = 0; i < CP; ++i) {
                const double d = __dsub_rn(__dmul_rn(ep[i], gp), __dmul_rn(c, __dmul_rn(eq[i], gq)));
                w[i] = (i < n && d > 0.0) ? d : 0.0;
            }
#pragma unroll
            for (int i = 0; i < CP; ++i)
                if (i < n) sr += w[i];
            // leaves this residual's thread chunk sums in sh.tsum for a possible final draw
            const double bsr = acc_block_sum(sr, sh);
            if (!(alive = acc_exchange<4>(a, ex, bsr, 0.0, 0.f, 0.f, sh))) break;
            S = acc_sum_blocks(sh.bpart0);
        }
        if (!alive) break;
        if (accepted >= 0) {
            if (blockIdx.x == 0 && threadIdx.x == 0) acc_put(a, 1 + k, accepted);
            ++k;
            cur = accepted;
            continue;
        }
        // every trial rejected: draw from the last residual (weights w, block partials in sh.bpart0)
        final_tok = acc_draw<CP>(w, lo, n, uni(ui), sh.bpart0, sh);
        ++ui;
        break;
    }
    if (alive && threadIdx.x == 0) {
        if (blockIdx.x == 0) {          // every block took the same decisions; block 0 reports them
            acc_put(a, 0, k);
            for (int i = 1 + k; i <= a.max_depth; ++i) acc_put(a, i, -1);   // unused path entries
            acc_put(a, a.max_depth + 2, ui);
            acc_put(a, a.max_depth + 3, bonus);
        }
        if (final_tok >= 0) acc_put(a, a.max_depth + 1, final_tok);   // only the block owning the draw has it
    }
    // host read-back without a copy or a stream synchronisation: each writer's entries reach host memory before its
    // tag (system-scope fence); the host waits for block 0's tag and, unless the err word reports a failure, for the
    // drawing block's
    if (threadIdx.x == 0 && a.host) {
        if (alive && final_tok >= 0) {
            __threadfence_system();
            __hip_atomic_store(a.host + 2, (int)a.tag_base, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        if (blockIdx.x == 0) {
            a.host[0] = (int)__hip_atomic_load(a.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __threadfence_system();
            __hip_atomic_store(a.host + 1, (int)a.tag_base, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------
// Filtered sampling: temperature, top-k and top-p (nucleus) exactly as Qwen2Engine.sample defines them
// (qwen_engine.py:146-156; native Sampler::distribution, sampler.hpp:22-57), many blocks of FS_THREADS per draw.
//   z_i   = fp32(l_i / T);  the order is z descending, ties by ascending index (the native sampler's comparator);
//   top-k (0 < k < V): keep z_i >= the k-th largest z (ties at the cutoff kept);
//   mass  m_i = floor(exp(z_i - z_max) * 2^40) as a 64-bit integer (fp64 exp; z_max = the row maximum, so m <= 2^40
//         and a row sum stays below 2^58): sums are exact and independent of order, so the kernel needs no fixed
//         summation tree; the 2^-40 quantum is far below any probability the cut or the draw can resolve;
//   top-p (p < 1): with F the total mass of the kept tokens, keep the sorted prefix whose exclusive cumulative mass
//         is <= floor(p * F) (first index whose inclusive mass exceeds that, and everything before it);
//   draw: target = floor(u * K) (clamped below K) over the kept mass K; the token is the first in sorted order whose
//         inclusive cumulative mass exceeds the target (inverse CDF, Sampler::draw, sampler.hpp:93-97).
// Selections in sorted order sort lists of at most FS_THREADS entries only.  The 32-bit order key is split 12 + 10 + 10 bits: a histogram of the top 12
// bits over the row (counts for the k-th largest, 64-bit masses for a cumulative target; 4096 bins in LDS per block,
// added into the row's global histogram with integer atomics) names the bin that holds the token looked for, the
// entries of that bin are gathered into a list, and two 10-bit levels over the list end at one key, whose tokens (equal
// masses) are ordered by index.
//
// Launches (each covers a row with one block per FM_SPAN entries, so all passes over a row run on the whole chip):
//   k_fm_top      row maximum; with top-k the count histogram
//   top-k up to FM_SMALL_K:  k_fm_gather collects every entry of the boundary bin and above (the k kept tokens are among
//                 them) and k_fm_finish does the rest on the list, one block per row
//   otherwise:    [k_fm_gather: the boundary bin of top-k], k_fm_mass: mass histogram of the kept entries,
//                 [k_fm_gather: the bin of the top-p cut], k_fm_gather: the bin of the draw, k_fm_finish
// A radix level of 8 bits used to be one launch over whole rows (9 to 14 launches).  16 rows of 151936 logits, device time
// per call, before and now: top-k 50 + top-p 0.9 87 -> 26 us, top-p 0.9 95 -> 69, temperature only 65 -> 44.
// A list that would hold more than FM_CAP entries (a row whose logits are mostly equal) is not used: the block that
// needs it scans the row instead.
constexpr int FS_THREADS = 1024;

__device__ __forceinline__ uint32_t fs_key(float z) {      // monotone: larger z, larger key
    const uint32_t b = __float_as_uint(z);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float fs_unkey(uint32_t k) {
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}
__device__ __forceinline__ unsigned long long fs_mass(float z, float zmax) {
    return (unsigned long long)(exp((double)z - (double)zmax) * 1099511627776.0);    // 2^40
}

constexpr int FM_U = 8;                            // entries per thread and pass
constexpr int FM_SPAN = FS_THREADS * FM_U;         // entries of a row per block
constexpr int FM_ROWS = 256;                       // rows per launch sequence (the scratch holds this many)
constexpr int FM_B0 = 4096, FM_B1 = 1024;          // bins of the first level (key >> 20) and of the two below
constexpr int FM_CAP = 8192;                       // entries a list holds
// top-k up to this runs on one list: with at most 1024 kept tokens the boundary bin and those above it (an eighth of an
// octave of z each) hold a few thousand entries at most for ordinary logits
constexpr int FM_SMALL_K = 1024;
struct FmPair { uint32_t key; int idx; };
// Per-row scratch.  kmax, n and the histograms are zero between calls: the finishing kernel clears what the call used, and
// the host clears everything after a call whose launches did not all go through.
struct FmState {
    unsigned long long mass[FM_B0];
    unsigned int cnt[FM_B0];
    unsigned int kmax;
    unsigned int n[3];                             // entries of lists 0 (top-k), 1 (top-p), 2 (draw)
    unsigned int kbin, krem, kmin;                 // top-k: boundary bin, tokens to take from it; smallest kept key
    unsigned int tbin, dbin;                       // bins of the top-p cut and of the draw
    unsigned long long tabove, dabove, tgt;        // mass before those bins, and the draw's target
};
struct FmArgs {
    const float *logits;
    int V, ld;
    const int *rows;
    const double *u;
    float T;
    int top_k;                                     // 0: no top-k
    double top_p;                                  // < 1: top-p
    int *out;
    FmState *st;                                   // [FM_ROWS]
    FmPair *list;                                  // [3][FM_ROWS][FM_CAP]
};

struct FmScan {                                    // LDS of the block-wide choices
    unsigned long long wave[FS_THREADS / 64];
    unsigned long long above;
    unsigned int bin;
};
// Inclusive prefix sums over the 64 lanes of a wave.
template <typename I>
__device__ __forceinline__ I fs_wave_scan(I v) {
    const int lane = threadIdx.x & 63;
    for (int o = 1; o < 64; o <<= 1) {
        const I t = __shfl_up(v, o);
        if (lane >= o) v += t;
    }
    return v;
}
// The block's sum of v and, in excl, the sum over the earlier threads.
__device__ __forceinline__ unsigned long long fm_block_scan(unsigned long long v, unsigned long long &excl, FmScan &sc) {
    const int w = threadIdx.x >> 6;
    const unsigned long long incl = fs_wave_scan<unsigned long long>(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 63) sc.wave[w] = incl;
    __syncthreads();
    unsigned long long before = 0, total = 0;
    for (int i = 0; i < FS_THREADS / 64; ++i) {
        const unsigned long long t = sc.wave[i];
        before += i < w ? t : 0ull;
        total += t;
    }
    excl = before + incl - v;
    return total;
}
// Choice over NB bins in descending order (thread t holds bins NB - 1 - t PB - j): the first bin at which `above` plus
// the bins before it and the bin itself exceeds `target` (for counts: reaches target + 1); every thread gets the bin
// and the sum before it.  No such bin (a degenerate row): bin 0.
template <int NB, typename H>
__device__ __forceinline__ unsigned int fm_choose(const H *h, unsigned long long above, unsigned long long target,
                                                  unsigned long long &above_out, FmScan &sc) {
    constexpr int PB = NB / FS_THREADS;
    unsigned long long v[PB], ls = 0, excl;
#pragma unroll
    for (int j = 0; j < PB; ++j) {
        v[j] = h[NB - 1 - (int)threadIdx.x * PB - j];
        ls += v[j];
    }
    const unsigned long long total = fm_block_scan(ls, excl, sc);
    if (threadIdx.x == 0) { sc.bin = 0; sc.above = above + total; }
    __syncthreads();
    if (above + excl <= target && above + excl + ls > target) {
        unsigned long long a = above + excl;
        int bin = NB - 1 - (int)threadIdx.x * PB;
#pragma unroll
        for (int j = 0; j < PB - 1; ++j)
            if (a + v[j] <= target && bin == NB - 1 - (int)threadIdx.x * PB - j) { a += v[j]; --bin; }
        sc.bin = (unsigned)bin;
        sc.above = a;
    }
    __syncthreads();
    above_out = sc.above;
    const unsigned int bin = sc.bin;
    __syncthreads();
    return bin;
}
template <typename H>
__device__ __forceinline__ unsigned long long fm_total(const H *h, FmScan &sc) {
    unsigned long long s = 0, e;
    for (int b = threadIdx.x; b < FM_B0; b += FS_THREADS) s += h[b];
    return fm_block_scan(s, e, sc);
}

// Wave sum of 64-bit integers on register moves (the exchanges of acc_wave_sum; integer sums need no order).
__device__ __forceinline__ unsigned long long fm_wave_sum(unsigned long long v) {
    auto swap = [&](bool half) {
        const unsigned lo = (unsigned)v, hi = (unsigned)(v >> 32);
        const u32x2 l = half ? __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(lo, lo, false, false))
                             : __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(lo, lo, false, false));
        const u32x2 h = half ? __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(hi, hi, false, false))
                             : __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(hi, hi, false, false));
        v = (((unsigned long long)h[0] << 32) | l[0]) + (((unsigned long long)h[1] << 32) | l[1]);
    };
    swap(true);
    swap(false);
    auto turn = [&](auto ctrl) {
        v += (unsigned long long)__double_as_longlong(acc_dpp<decltype(ctrl)::value>(__longlong_as_double((long long)v)));
    };
    turn(std::integral_constant<int, 0x128>());
    turn(std::integral_constant<int, 0x124>());
    turn(std::integral_constant<int, 0x4E>());
    turn(std::integral_constant<int, 0xB1>());
    return v;
}
// Histogram add of a mass with the lanes that share the first active lane's bin combined: most keys of a row share
// their top bits, and 64 lanes adding to one LDS word serialise.  Integer sums: the result is order-independent.
__device__ __forceinline__ void fm_add(unsigned long long *h, bool act, int bin, unsigned long long v) {
    const int lane = threadIdx.x & 63;
    const unsigned long long pend = __ballot(act);
    if (pend == 0) return;
    const int leader = __ffsll((long long)pend) - 1;
    const bool mine = act && bin == __builtin_amdgcn_readlane(bin, leader);
    const unsigned long long s = fm_wave_sum(mine ? v : 0ull);
    if (lane == leader) atomicAdd(&h[bin], s);
    else if (act && !mine) atomicAdd(&h[bin], v);
}

// fm_add of one count per active lane: the leader's bin gets the number of lanes that share it from the ballot.
template <typename H>
__device__ __forceinline__ void fm_count(H *h, bool act, int bin) {
    const unsigned long long pend = __ballot(act);
    if (pend == 0) return;
    const int leader = __ffsll((long long)pend) - 1;
    const bool mine = act && bin == __builtin_amdgcn_readlane(bin, leader);
    const unsigned long long same = __ballot(mine);
    if ((int)(threadIdx.x & 63) == leader) atomicAdd(&h[bin], (H)__popcll(same));
    else if (act && !mine) atomicAdd(&h[bin], (H)1);
}

// The entries a level looks at: a list in LDS, or (list too long) the whole row.
struct FmSource {
    bool listed;
    int n;
    const FmPair *pairs;
    const float *row;
    float T;
    // fn(active, key, index) for every entry, by all threads together
    template <typename F>
    __device__ __forceinline__ void each(F &&fn) const {
        for (int i0 = 0; i0 < n; i0 += FS_THREADS) {
            const int i = i0 + threadIdx.x;
            const bool in = i < n;
            uint32_t key = 0;
            int idx = 0;
            if (in && listed) { key = pairs[i].key; idx = pairs[i].idx; }
            if (in && !listed) { key = fs_key(__fdiv_rn(row[i], T)); idx = i; }
            fn(in, key, idx);
        }
    }
};
// List `which` of row r into LDS, or the row when the list overflowed.
__device__ __forceinline__ FmSource fm_source(const FmArgs &a, int r, int which, const float *row, FmPair *lds) {
    const unsigned int n = a.st[r].n[which];
    FmSource s{n <= (unsigned)FM_CAP, n <= (unsigned)FM_CAP ? (int)n : a.V, lds, row, a.T};
    if (s.listed) {
        const FmPair *src = a.list + ((size_t)which * FM_ROWS + r) * FM_CAP;
        for (int i = threadIdx.x; i < s.n; i += FS_THREADS) lds[i] = src[i];
    }
    __syncthreads();
    return s;
}
// The key that holds `target` among the entries of bin `bin` (first level) with key >= kmin, and the mass (COUNT: the
// number of entries) before it in sorted order.
template <bool COUNT>
__device__ __forceinline__ uint32_t fm_descend(const FmSource &src, uint32_t bin, uint32_t kmin, float zmax,
                                               unsigned long long above, unsigned long long target,
                                               unsigned long long &above_out, unsigned long long *h, FmScan &sc) {
    uint32_t prefix = bin;
#pragma unroll
    for (int level = 0; level < 2; ++level) {
        const int hi = level == 0 ? 20 : 10, lo = hi - 10;
        for (int b = threadIdx.x; b < FM_B1; b += FS_THREADS) h[b] = 0ull;
        __syncthreads();
        src.each([&](bool in, uint32_t key, int) {
            const bool act = in && (key >> hi) == prefix && key >= kmin;
            const int b = (key >> lo) & (FM_B1 - 1);
            if constexpr (COUNT) fm_count(h, act, b);
            else fm_add(h, act, b, act ? fs_mass(fs_unkey(key), zmax) : 0ull);
        });
        __syncthreads();
        prefix = (prefix << 10) | fm_choose<FM_B1>(h, above, target, above, sc);
    }
    above_out = above;
    return prefix;
}

__global__ void __launch_bounds__(FS_THREADS) k_fm_top(FmArgs a) {
    __shared__ unsigned int red[FS_THREADS / 64];
    __shared__ unsigned int h[FM_B0];
    const int r = blockIdx.y, i0 = blockIdx.x * FM_SPAN;
    const float *row = a.logits + (size_t)a.rows[r] * a.ld;
    float lv[FM_U];
#pragma unroll
    for (int u = 0; u < FM_U; ++u) lv[u] = row[min(i0 + u * FS_THREADS + (int)threadIdx.x, a.V - 1)];
    if (a.top_k) {
        for (int b = threadIdx.x; b < FM_B0; b += FS_THREADS) h[b] = 0u;
        __syncthreads();
    }
    uint32_t k = 0;
#pragma unroll
    for (int u = 0; u < FM_U; ++u) {
        const uint32_t key = fs_key(__fdiv_rn(lv[u], a.T));
        const bool in = i0 + u * FS_THREADS + (int)threadIdx.x < a.V;
        k = max(k, key);                           // an entry past the row repeats the last one
        if (a.top_k) fm_count(h, in, key >> 20);
    }
    for (int o = 32; o > 0; o >>= 1) k = max(k, (uint32_t)__shfl_xor((int)k, o));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = k;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < FS_THREADS / 64; ++i) k = max(k, red[i]);
        atomicMax(&a.st[r].kmax, k);
    }
    if (a.top_k)
        for (int b = threadIdx.x; b < FM_B0; b += FS_THREADS)
            if (h[b]) atomicAdd(&a.st[r].cnt[b], h[b]);
}

// Smallest key kept by top-k: the krem-th largest of the boundary bin.
__device__ __forceinline__ uint32_t fm_kmin(const FmArgs &a, int r, const FmSource &src, unsigned long long *h, FmScan &sc) {
    unsigned long long above;
    return fm_descend<true>(src, a.st[r].kbin, 0u, 0.f, 0ull, (unsigned long long)a.st[r].krem - 1, above, h, sc);
}

// Mass histogram of the kept entries (after top-k: those of at least kmin, found from list 0 by every block).
template <bool TOPK>
__global__ void __launch_bounds__(FS_THREADS) k_fm_mass(FmArgs a) {
    __shared__ unsigned long long m0[FM_B0];
    __shared__ unsigned long long h[TOPK ? FM_B1 : 1];
    __shared__ FmPair lds[TOPK ? FM_CAP : 1];
    __shared__ FmScan sc;
    const int r = blockIdx.y, i0 = blockIdx.x * FM_SPAN;
    FmState &S = a.st[r];
    const float *row = a.logits + (size_t)a.rows[r] * a.ld;
    float lv[FM_U];
#pragma unroll
    for (int u = 0; u < FM_U; ++u) lv[u] = row[min(i0 + u * FS_THREADS + (int)threadIdx.x, a.V - 1)];
    for (int b = threadIdx.x; b < FM_B0; b += FS_THREADS) m0[b] = 0ull;
    uint32_t kmin = 0;
    if constexpr (TOPK) {
        const FmSource src = fm_source(a, r, 0, row, lds);
        kmin = fm_kmin(a, r, src, h, sc);
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) S.kmin = kmin;
    __syncthreads();
    const float zmax = fs_unkey(S.kmax);
#pragma unroll
    for (int u = 0; u < FM_U; ++u) {
        const float z = __fdiv_rn(lv[u], a.T);
        const uint32_t key = fs_key(z);
        const bool in = i0 + u * FS_THREADS + (int)threadIdx.x < a.V && key >= kmin;
        const unsigned long long m = in ? fs_mass(z, zmax) : 0ull;
        fm_add(m0, m != 0ull, key >> 20, m);
    }
    __syncthreads();
    for (int b = threadIdx.x; b < FM_B0; b += FS_THREADS)
        if (m0[b]) atomicAdd(&S.mass[b], m0[b]);
}

// What the top-p cut keeps: floor(top_p F) of the kept mass F is the target of the cut.
__device__ __forceinline__ bool fm_cut(const FmArgs &a, unsigned long long F, unsigned long long &tp) {
    tp = (unsigned long long)(a.top_p * (double)F);
    return a.top_p < 1.0 && tp < F;
}
__device__ __forceinline__ unsigned long long fm_target(const FmArgs &a, int r, unsigned long long K) {
    unsigned long long t = (unsigned long long)(a.u[r] * (double)K);
    return t >= K ? K - 1 : t;
}
// The kept mass after the cut: the tokens before the cut's key and those of the key up to the cut.
__device__ __forceinline__ unsigned long long fm_kept(uint32_t key, float zmax, unsigned long long above,
                                                      unsigned long long tp) {
    const unsigned long long m = fs_mass(fs_unkey(key), zmax);
    return above + ((m > 0 ? (tp - above) / m : 0) + 1) * m;
}

// Collects entries of a row into a list.  MODE 0: the boundary bin of top-k and every bin above it; 1: the boundary bin
// alone; 2: the bin of the top-p cut; 3: the bin of the draw (with top-p: after the cut, resolved from list 1).
template <int MODE>
__global__ void __launch_bounds__(FS_THREADS) k_fm_gather(FmArgs a) {
    constexpr int WHICH = MODE <= 1 ? 0 : MODE - 1;
    __shared__ unsigned long long h[MODE == 3 ? FM_B1 : 1];
    __shared__ FmPair lds[MODE == 3 ? FM_CAP : 1];
    __shared__ FmScan sc;
    __shared__ unsigned int base;
    const int r = blockIdx.y, i0 = blockIdx.x * FM_SPAN;
    FmState &S = a.st[r];
    const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
    const float *row = a.logits + (size_t)a.rows[r] * a.ld;
    float lv[FM_U];
#pragma unroll
    for (int u = 0; u < FM_U; ++u) lv[u] = row[min(i0 + u * FS_THREADS + (int)threadIdx.x, a.V - 1)];
    unsigned long long above;
    uint32_t bin, kmin = 0;
    if constexpr (MODE <= 1) {
        bin = fm_choose<FM_B0>(S.cnt, 0ull, (unsigned long long)a.top_k - 1, above, sc);
        if (lead) { S.kbin = bin; S.krem = (unsigned)a.top_k - (unsigned)above; }
    } else {
        kmin = S.kmin;
        const unsigned long long F = fm_total(S.mass, sc);
        unsigned long long tp;
        const bool cut = fm_cut(a, F, tp);
        if constexpr (MODE == 2) {
            if (!cut) return;
            bin = fm_choose<FM_B0>(S.mass, 0ull, tp, above, sc);
            if (lead) { S.tbin = bin; S.tabove = above; }
        } else {
            unsigned long long K = F;
            if (cut) {
                const float zmax = fs_unkey(S.kmax);
                const FmSource src = fm_source(a, r, 1, row, lds);
                const uint32_t key = fm_descend<false>(src, S.tbin, kmin, zmax, S.tabove, tp, above, h, sc);
                K = fm_kept(key, zmax, above, tp);
            }
            const unsigned long long tgt = fm_target(a, r, K);
            bin = fm_choose<FM_B0>(S.mass, 0ull, tgt, above, sc);
            if (lead) { S.dbin = bin; S.dabove = above; S.tgt = tgt; }
        }
    }
    uint32_t key[FM_U];
    unsigned int mine = 0;
#pragma unroll
    for (int u = 0; u < FM_U; ++u) {
        key[u] = fs_key(__fdiv_rn(lv[u], a.T));
        const bool in = i0 + u * FS_THREADS + (int)threadIdx.x < a.V;
        const bool take = in && (MODE == 0 ? (key[u] >> 20) >= bin : (key[u] >> 20) == bin && key[u] >= kmin);
        mine |= (unsigned)take << u;
    }
    unsigned long long excl;
    const unsigned int total = (unsigned)fm_block_scan((unsigned long long)__popc(mine), excl, sc);
    if (threadIdx.x == 0) base = total ? atomicAdd(&S.n[WHICH], total) : 0u;
    __syncthreads();
    FmPair *list = a.list + ((size_t)WHICH * FM_ROWS + r) * FM_CAP;
    unsigned int at = base + (unsigned)excl;
#pragma unroll
    for (int u = 0; u < FM_U; ++u)
        if ((mine >> u) & 1u) {
            if (at < (unsigned)FM_CAP) list[at] = FmPair{key[u], i0 + u * FS_THREADS + (int)threadIdx.x};
            ++at;
        }
}

// Index of the rank-th token (index order) whose key equals `key` (a block-wide scan over contiguous chunks), -1 when
// there is none.
__device__ int fs_index_of(const float *row, int V, float T, uint32_t key, unsigned long long rank, FmScan &sc) {
    const int C = (V + FS_THREADS - 1) / FS_THREADS, lo = min(V, (int)threadIdx.x * C), hi = min(V, lo + C);
    unsigned int cnt = 0;
    for (int i = lo; i < hi; ++i) cnt += fs_key(__fdiv_rn(row[i], T)) == key;
    unsigned long long before;
    (void)fm_block_scan(cnt, before, sc);
    __shared__ int found;
    if (threadIdx.x == 0) found = -1;
    __syncthreads();
    if (rank >= before && rank < before + cnt) {
        unsigned long long r = rank - before;
        for (int i = lo; i < hi; ++i)
            if (fs_key(__fdiv_rn(row[i], T)) == key) {
                if (r == 0) { found = i; break; }
                --r;
            }
    }
    __syncthreads();
    return found;
}

// A list of at most one entry per thread, sorted (z descending, ties by ascending index), and everything after the
// gather on the sorted masses' prefix sums: the top-k cut is entry top_k - 1's key, the top-p cut and the draw are the
// first entries whose inclusive mass exceeds their targets.  Bitonic over (key, ~index); exchanges inside a wave are
// shuffles, the others go through LDS.  16 rows of top-k 50 (lists of a few hundred entries): k_fm_finish 23 -> 9.4 us
// against the histogram descents below.
__device__ int fm_small_list(const FmArgs &a, int r, const FmSource &src, float zmax, unsigned long long *h, FmScan &sc) {
    const int t = threadIdx.x;
    unsigned long long v = 0ull;
    if (t < src.n) v = ((unsigned long long)src.pairs[t].key << 32) | (uint32_t)~src.pairs[t].idx;
    for (int k = 2; k < 2 * src.n && k <= FS_THREADS; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1) {
            unsigned long long o;
            if (j < SP_WAVE) {
                o = __shfl_xor(v, j);
            } else {
                __syncthreads();
                h[t] = v;
                __syncthreads();
                o = h[t ^ j];
            }
            const bool larger = ((t & k) == 0) == ((t & j) == 0);       // this thread keeps the larger of the pair
            v = (o > v) == larger ? o : v;
        }
    __shared__ unsigned long long pick;        // K, then the drawn entry
    __syncthreads();
    h[t] = v;
    if (t == 0) pick = 0ull;
    __syncthreads();
    const uint32_t kmin = (uint32_t)(h[min(a.top_k, src.n) - 1] >> 32), key = (uint32_t)(v >> 32);
    const unsigned long long m = t < src.n && key >= kmin ? fs_mass(fs_unkey(key), zmax) : 0ull;
    unsigned long long excl, tp;
    unsigned long long K = fm_block_scan(m, excl, sc);
    if (fm_cut(a, K, tp)) {
        if (excl <= tp && excl + m > tp) pick = excl + m;
        __syncthreads();
        K = pick;
        __syncthreads();
    }
    const unsigned long long tgt = fm_target(a, r, K);
    if (t == 0) pick = 0xffffffff00000000ull;  // no entry (a degenerate row): -1
    __syncthreads();
    if (excl <= tgt && excl + m > tgt) pick = v;
    __syncthreads();
    return (int)~(uint32_t)pick;
}

// The drawn token by histogram descents.  SMALL: everything after the gather of MODE 0, on list 0 (m0: a first-level
// mass histogram); else: the draw, on list 2.
template <bool SMALL>
__device__ int fm_descents(const FmArgs &a, int r, const FmSource &src, const float *row, float zmax, unsigned long long *m0,
                           unsigned long long *h, FmScan &sc) {
    const FmState &S = a.st[r];
    __shared__ unsigned int first;
    unsigned long long above, tgt;
    uint32_t key;
    if constexpr (SMALL) {
        const uint32_t kmin = fm_kmin(a, r, src, h, sc);
        for (int b = threadIdx.x; b < FM_B0; b += FS_THREADS) m0[b] = 0ull;
        __syncthreads();
        src.each([&](bool in, uint32_t k, int) {
            const unsigned long long m = in && k >= kmin ? fs_mass(fs_unkey(k), zmax) : 0ull;
            fm_add(m0, m != 0ull, k >> 20, m);
        });
        __syncthreads();
        unsigned long long K = fm_total(m0, sc), tp;
        if (fm_cut(a, K, tp)) {
            const uint32_t bin = fm_choose<FM_B0>(m0, 0ull, tp, above, sc);
            key = fm_descend<false>(src, bin, kmin, zmax, above, tp, above, h, sc);
            K = fm_kept(key, zmax, above, tp);
        }
        tgt = fm_target(a, r, K);
        const uint32_t bin = fm_choose<FM_B0>(m0, 0ull, tgt, above, sc);
        key = fm_descend<false>(src, bin, kmin, zmax, above, tgt, above, h, sc);
    } else {
        tgt = S.tgt;
        key = fm_descend<false>(src, S.dbin, S.kmin, zmax, S.dabove, tgt, above, h, sc);
    }
    const unsigned long long m = fs_mass(fs_unkey(key), zmax);
    const unsigned long long rank = m > 0 ? (tgt - above) / m : 0;
    if (rank > 0) return fs_index_of(row, a.V, a.T, key, rank, sc);
    // always, unless the drawn z value is shared by several tokens: the group's smallest index
    if (threadIdx.x == 0) first = 0xffffffffu;
    __syncthreads();
    src.each([&](bool in, uint32_t k, int idx) {
        if (in && k == key) atomicMin(&first, (unsigned)idx);
    });
    __syncthreads();
    return (int)first;
}

// The drawn token, then the row's scratch is cleared for the next call.
template <bool SMALL>
__global__ void __launch_bounds__(FS_THREADS) k_fm_finish(FmArgs a) {
    __shared__ unsigned long long m0[SMALL ? FM_B0 : 1];
    __shared__ unsigned long long h[FM_B1];
    __shared__ FmPair lds[FM_CAP];
    __shared__ FmScan sc;
    const int r = blockIdx.x;
    FmState &S = a.st[r];
    const float *row = a.logits + (size_t)a.rows[r] * a.ld;
    const float zmax = fs_unkey(S.kmax);
    const FmSource src = fm_source(a, r, SMALL ? 0 : 2, row, lds);
    int tok;
    if (SMALL && src.listed && src.n >= 1 && src.n <= FS_THREADS) tok = fm_small_list(a, r, src, zmax, h, sc);
    else tok = fm_descents<SMALL>(a, r, src, row, zmax, m0, h, sc);
    if (threadIdx.x == 0) {
        a.out[r] = tok;
        S.kmax = 0u;
        S.n[0] = S.n[1] = S.n[2] = 0u;
    }
    for (int b = threadIdx.x; b < FM_B0; b += FS_THREADS) {
        if (a.top_k) S.cnt[b] = 0u;
        if (!SMALL) S.mass[b] = 0ull;
    }
}
