// Gemma-4 text-encoder attention (Sources/LTXModules/GemmaTextEncoder.swift:158-239, mask
// :288-321) for gfx950: head dims 256 / 512, 16 query heads over 8 or 1 KV heads, causal +
// sliding-window + left-padding mask, scale 1.0, 1024 tokens per prompt.
//
// Three launches (the first is the whole prologue, its q/k rows and its v blocks side by side):
//   gemma_prep_kernel   one wave per (batch row, token, head) row of q or k: the per-head
//                       RMS norm (fp32, (mean + eps)^-0.5, times the weight), rotate_half
//                       RoPE with the fp32 tables, q scaled by scale*log2(e). Rounding points:
//                       the reference's norm returns the input dtype (GemmaTextEncoder.swift
//                       :114), so its normed q and k are bf16, and its fp32 RoPE leaves both
//                       fp32. Here q and k are normed and rotated in fp32 without that
//                       rounding and rounded once, after the rotation, to fp16 (11
//                       significant bits, against bf16's 8): q' [B][Hq][T][D] and k' are the
//                       fp16 operands of the products, far inside fp16's range: the RMS norm
//                       bounds a channel, and the rotation a channel pair, by sqrt(D) times
//                       the weight (times log2(e) for q'). The single rounding, finer than the
//                       reference's, brings the result nearer the exact one than the
//                       reference's own arithmetic (its rounded normed q alone moves the
//                       1024-token layers' max-abs error to about 2e-2).
//                       k' is stored in MFMA operand order: per (batch row, KV head, 32-key
//                       block) D/16 units of 1 KB, lane r + 32g of unit c holding channels
//                       16c + 8g .. +7 of key r.
//   (same launch)       v with the weightless per-head norm, in fp16, transposed through an
//                       LDS tile of one 32-key block into operand order: per key half hf and
//                       32-channel block cb one 1 KB unit, lane r + 32g holding channel
//                       32cb + r at keys 16hf + 4g + {0..3, 8..11}. Keys past T are zeros in both layouts, and
//                       a key block's k' and v'^T are each one contiguous run of units.
//   gemma_attn*_kernel  128 queries of a head per workgroup (64 at D = 512 for short prompts), a
//                       wave 256 channels of them; the key blocks of the workgroup's range are
//                       copied HBM -> LDS by the buffer-load-to-LDS path and read from LDS by
//                       every wave. Per key block: S^T = K.Q'^T in fp16 products (at D = 512 the
//                       two halves' partial sums are exchanged through LDS and added), the mask,
//                       exp2 with each row's max fixed at its first block with an allowed key,
//                       and O^T += V^T.P^T with v' and P in fp16 (the reference's weights are
//                       fp32; with the max fixed a weight stays below 2^kGemmaBound). A block
//                       whose weights would pass 2^kGemmaBound sends the workgroup to an exact
//                       pass over its range (D 256: online max with rescaling; D 512: with the
//                       maxima that the first pass saw). O is written in fp32, the dtype the
//                       reference's explicit path returns.
//   gemma_combine_kernel  the long query blocks' keys run as ranges (the host's plan) on
//                       separate workgroups, each writing unnormalised O and (max, sum); the
//                       merge rescales and adds them.
#include <type_traits>

#include "lds_copy.hpp"
#include "mfma_s.hpp"

namespace ltx {
namespace {

// ---- prologue ------------------------------------------------------------------------------
// q/k rows: workgroup wg of the rows' part of the launch.
// Rows per wave of the q/k part: a wave takes kPrepPasses passes of 64 / (D / 8) rows and
// issues every pass's loads (the row, its table rows) before the first use, so the launch's
// waves each wait for one round trip instead of one per row (one row per wave and pass took
// the 1024-token prologue 18-21 us, most of it waiting).
constexpr int kPrepPasses = 4;   // 8 measured slower (23.6 / 19.8 against 16.5 / 16.3 us)

template <int D>
__device__ __forceinline__ void gemma_prep_rows(const GemmaPrepParams &p, int wg) {
    // 8 channels per lane: a row of D = 512 takes a wave, a row of D = 256 half a wave
    constexpr int E = 8;
    constexpr int LPR = D / E;                      // lanes per row: 64 or 32
    constexpr int RPW = 64 / LPR;                   // rows per wave and pass
    constexpr int NP = kPrepPasses;
    const int lane = threadIdx.x & (LPR - 1);       // lane within the row
    // (row indices in 32 bits: the launch refuses 2^31 rows or more)
    const uint32_t heads = p.Hq + p.Hkv;            // q heads, then k heads, per token
    const uint32_t total = (uint32_t)p.B * p.T * heads;
    // the wave's rows: RPW * NP consecutive rows, pass j taking rows base + RPW*j + (0..RPW-1)
    const uint32_t base = ((uint32_t)wg * 4 + (threadIdx.x >> 6)) * (RPW * NP) +
                          ((threadIdx.x & 63) / LPR);
    const int col = (lane & (LPR / 2 - 1)) * E;     // table column of the lane's channels
    u32x4 raw[NP];
    f32x4 cs[NP][2], sn[NP][2];
    int hrs[NP], ts[NP], bs[NP];
#pragma unroll
    for (int j = 0; j < NP; ++j) {
        const uint32_t row = base + RPW * j;
        const uint32_t bt = row / heads;
        hrs[j] = (int)(row - bt * heads);
        bs[j] = (int)(bt / (uint32_t)p.T);
        ts[j] = (int)(bt - (uint32_t)bs[j] * p.T);
    }
#pragma unroll
    for (int j = 0; j < NP; ++j) {
        if (base + RPW * j >= total) continue;
        const int hr = hrs[j], t = ts[j], b = bs[j];
        const bf16 *src = hr < p.Hq
            ? (const bf16 *)p.q + (int64_t)b * p.q_bs + (int64_t)t * p.q_rs + (int64_t)hr * D
            : (const bf16 *)p.k + (int64_t)b * p.k_bs + (int64_t)t * p.k_rs +
                  (int64_t)(hr - p.Hq) * D;
        raw[j] = ldg16(src + lane * E);
        const float *c = p.cos + (int64_t)t * (D / 2) + col;
        const float *sv = p.sin + (int64_t)t * (D / 2) + col;
        cs[j][0] = *(const f32x4 *)c;
        cs[j][1] = *(const f32x4 *)(c + 4);
        sn[j][0] = *(const f32x4 *)sv;
        sn[j][1] = *(const f32x4 *)(sv + 4);
    }
    float wq[E], wk[E];
    unpack8(ldg16((const bf16 *)p.q_w + lane * E), wq);
    unpack8(ldg16((const bf16 *)p.k_w + lane * E), wk);
    const bool first = lane < LPR / 2;
#pragma unroll
    for (int j = 0; j < NP; ++j) {
        if (base + RPW * j >= total) continue;
        const int hr = hrs[j], t = ts[j], b = bs[j];
        const int kind = hr < p.Hq ? 0 : 1;         // q, k
        const int h = kind == 0 ? hr : hr - p.Hq;
        float x[E];
        unpack8(raw[j], x);
        // the reductions and the partner exchange stay within the row's lanes (offsets < LPR)
        float ss = 0.f;
#pragma unroll
        for (int e = 0; e < E; ++e) ss += x[e] * x[e];
        ss = lane_sum<LPR>(ss);
        const float rs = 1.0f / sqrtf(ss / (float)D + p.eps);
#pragma unroll
        for (int e = 0; e < E; ++e) x[e] = (x[e] * rs) * (kind == 0 ? wq[e] : wk[e]);
        // rotate_half pairs channel c with c +- D/2: lane l holds channels E*l ..; its partner
        // is lane l ^ LPR/2. Table column of channel c is c mod D/2.
        const float f = kind == 0 ? p.q_factor : 1.0f;
        float y[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const float other = LPR == 64 ? xlane32(x[e]) : xlane16(x[e]);
            const float c = cs[j][e >> 2][e & 3], s = sn[j][e >> 2][e & 3];
            // first half: x1 c - x2 s; second half: x2 c + x1 s
            y[e] = (first ? x[e] * c - other * s : x[e] * c + other * s) * f;
        }
        // q' and k' as fp16 (11 significant bits, rounded once, to nearest)
        if (kind == 1) {
            // k' in operand order: 32-key block t/32, 16-channel chunk c, lane (t%32) + 32g
            // holds channels 16c + 8g .. +7 of key t
            const int ch = lane * E, c = ch >> 4, g = (ch >> 3) & 1;
            const int nkb = (p.T + 31) / 32;
            const int64_t off =
                ((((int64_t)b * p.Hkv + h) * nkb + (t >> 5)) * (D / 16) + c) * 512 +
                ((t & 31) + 32 * g) * 8 + (ch & 7);
            *(u32x4 *)((_Float16 *)p.kp + off) = pack8_f16(y);
        } else {
            const int64_t off = (((int64_t)b * p.Hq + h) * p.T + t) * D + lane * E;
            *(u32x4 *)((_Float16 *)p.qp + off) = pack8_f16(y);
        }
    }
}

// v: the weightless per-head norm, stored transposed in operand order. One workgroup per
// (batch row, KV head, 32-key block): each wave loads its 8 token rows at once, normalises
// them into an LDS tile, then the tile leaves as the block's P.V operand units. Workgroup wg
// of the v part of the launch.
template <int D>
__device__ __forceinline__ void gemma_vt_block(const GemmaPrepParams &p, int wg,
                                               _Float16 (&tile)[32][D + 8]) {
    constexpr int E = D / 64;
    constexpr int TT = 32;                          // tokens per workgroup: one key block
    constexpr int RW = TT / 4;                      // rows per wave
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int nkb = (p.T + TT - 1) / TT;
    const int kb = wg % nkb, t0 = kb * TT;
    const int bh = wg / nkb;
    const int h = bh % p.Hkv, b = bh / p.Hkv;
    // every row's load issued before the first use: a row past T loads row T - 1 and is
    // zeroed afterwards (a branch around each load would make each wait for the one before)
    float x[RW][E];
    typedef __attribute__((ext_vector_type(E / 2))) uint32_t uvec;
    uvec raw[RW];
#pragma unroll
    for (int j = 0; j < RW; ++j) {
        const int t = min(t0 + wave * RW + j, p.T - 1);
        raw[j] = *(const uvec *)((const bf16 *)p.v + (int64_t)b * p.v_bs + (int64_t)t * p.v_rs +
                                 (int64_t)h * D + lane * E);
    }
#pragma unroll
    for (int j = 0; j < RW; ++j) {
        const bool in = t0 + wave * RW + j < p.T;
#pragma unroll
        for (int e = 0; e < E; e += 2) {
            x[j][e] = in ? bf_lo(raw[j][e / 2]) : 0.f;
            x[j][e + 1] = in ? bf_hi(raw[j][e / 2]) : 0.f;
        }
    }
#pragma unroll
    for (int j = 0; j < RW; ++j) {
        float ss = 0.f;
#pragma unroll
        for (int e = 0; e < E; ++e) ss += x[j][e] * x[j][e];
        ss = lane_sum<64>(ss);
        const float rs = 1.0f / sqrtf(ss / (float)D + p.eps);
#pragma unroll
        for (int e = 0; e < E; ++e) tile[wave * RW + j][lane * E + e] = (_Float16)(x[j][e] * rs);
    }
    __syncthreads();
    // Operand units of the block: per key half hf and 32-channel block cb one 1 KB unit whose
    // lane r + 32g holds channel 32cb + r at keys 32kb + 16hf + 4g + {0..3, 8..11}. Keys past T
    // are written as zeros (their weights are 0, and 0 * 0 keeps the products finite); the
    // last block's k' rows past T are zeroed too.
    _Float16 *vbase = (_Float16 *)p.vt + (((int64_t)b * p.Hkv + h) * nkb + kb) * (D * 32);
    for (int u = threadIdx.x; u < 2 * (D / 32) * 64; u += 256) {
        const int l = u & 63, rest = u >> 6;
        const int cb = rest % (D / 32), hf = rest / (D / 32);
        const int r = l & 31, g = l >> 5;
        float f[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int tl = 16 * hf + 4 * g + (e & 3) + 8 * (e >> 2);
            f[e] = t0 + tl < p.T ? (float)tile[tl][32 * cb + r] : 0.f;
        }
        *(u32x4 *)(vbase + ((int64_t)hf * (D / 32) + cb) * 512 + l * 8) = pack8_f16(f);
    }
    if ((p.T & 31) && kb == nkb - 1) {
        _Float16 *kbase = (_Float16 *)p.kp + (((int64_t)b * p.Hkv + h) * nkb + kb) * (D * 32);
        for (int u = threadIdx.x; u < (D / 16) * 64; u += 256) {
            const int l = u & 63;
            if (t0 + (l & 31) >= p.T) *(u32x4 *)(kbase + u * 8) = u32x4{0, 0, 0, 0};
        }
    }
}

// The prologue as one launch: the q/k rows' workgroups, then the v blocks' (they write
// disjoint parts of k': rows below T, and the zeroed rows past T of the last block). (The v
// blocks first measured 1.5 us faster at D = 512, with 32 of them, and 1.6 us slower at
// D = 256, with 256.)
template <int D>
__global__ __launch_bounds__(256) void gemma_prep_kernel(const GemmaPrepParams p, int row_wgs) {
    __shared__ __attribute__((aligned(16))) _Float16 tile[32][D + 8];
    const int wg = blockIdx.x;
    if (wg < row_wgs) gemma_prep_rows<D>(p, wg);
    else gemma_vt_block<D>(p, wg - row_wgs, tile);
}
// ---- attention -----------------------------------------------------------------------------
// A workgroup runs 128 queries of one head over a range of 32-key blocks, whose K' and V'^T
// operand units (D/16 and 2 * D/32 units of 1 KB, contiguous per block in the prologue's layout)
// are copied HBM -> LDS by the buffer-load-to-LDS path. A wave works on 256 channels: Q' and K' in
// kNCW 16-channel chunks, V'^T and O in kNDW 32-channel blocks.
constexpr int kGemmaQueries = 128;
constexpr int kNCW = 256 / 16, kNDW = 256 / 32;
constexpr int kGemmaShortQueries = 64;           // of the kernel for short prompts (gemma_short)

// Key blocks of the query block [q0, q0 + nq): causal / window / padding bounds; a block with
// rows inside the left padding (their rows have no allowed key) runs over all keys, those rows
// unmasked.
struct KeyBlocks {
    int lo, hi;
};
__device__ __forceinline__ KeyBlocks gemma_key_blocks(const GemmaAttnParams &p, int q0, int nq,
                                                      int fv) {
    return KeyBlocks{gemma_key_lo(q0, fv, p.window), gemma_key_hi(p.T, q0, nq, fv)};
}

// The fast pass keeps each row's max from its first block with an allowed key; a later block
// whose weights would pass 2^kGemmaBound (log2 units over that max) sends the workgroup to
// the exact pass.
constexpr float kGemmaBound = 15.0f;   // the fp16 weights stay below 65504

// Partial rows before query block qblk's within its head: the key ranges of the earlier query
// blocks that split (more than one range). Spread over the wave: lane j counts block j (j + 64,
// ...), and four ballots add the counts (at most kGemmaMaxChunks = 8: four bits), so the wave
// spends a few vector instructions instead of a scalar loop over every earlier block, which the
// CU's one scalar unit would run for each of its waves in turn. Every lane must be active; the
// result is uniform.
__device__ __forceinline__ int gemma_part_offset(int T, int window, int chunk, int qwg, int fv,
                                                 int qblk) {
    const int lane = (int)threadIdx.x & 63;
    int off = 0;
    for (int j0 = 0; j0 < qblk; j0 += 64) {
        const int j = j0 + lane;
        int n = j < qblk ? gemma_ranges(T, window, chunk, j * qwg, qwg, fv) : 0;
        if (n < 2) n = 0;
#pragma unroll
        for (int bit = 0; bit < 4; ++bit) off += __popcll(__ballot((n >> bit) & 1)) << bit;
    }
    return off;
}

// The work of a workgroup: grid layer `chunk` holds every query block's chunk-th key range;
// within a layer the heaviest (latest) query blocks come first, each across all (batch row, head)
// pairs, so the workgroups that the dispatcher deals to the 8 XCDs in turn carry equal work.
struct GemmaItem {
    int chunk, nch;              // key range, of how many of its query block (chunk >= nch: none)
    int qblk, q0, h, b, kvh, fv;
    int kb_lo, kb_hi;            // its key blocks
};
__device__ __forceinline__ GemmaItem gemma_item(const GemmaAttnParams &p, int qwg) {
    GemmaItem w;
    const int nqb = (p.T + qwg - 1) / qwg, nbh = p.B * p.Hq, per_layer = nbh * nqb;
    w.chunk = (int)blockIdx.x / per_layer;
    const int rem = (int)blockIdx.x - w.chunk * per_layer;
    w.qblk = nqb - 1 - rem / nbh;
    const int bh = rem % nbh;
    w.h = bh % p.Hq;
    w.b = bh / p.Hq;
    w.kvh = w.h / (p.Hq / p.Hkv);
    w.q0 = w.qblk * qwg;
    w.fv = p.first_valid[w.b];
    const KeyBlocks kr = gemma_key_blocks(p, w.q0, qwg, w.fv);
    w.nch = gemma_ranges(p.T, p.window, p.chunk, w.q0, qwg, w.fv);
    w.kb_lo = kr.lo + w.chunk * p.chunk;
    w.kb_hi = min(w.kb_lo + p.chunk - 1, kr.hi);
    return w;
}

// The row's allowed keys as one range [k_lo, k_hi]: all keys for a row inside the left padding,
// else causal (k <= q), past the padding (k >= fv) and inside the window (q - k < window); k_hi <=
// T - 1 also masks the keys past T of the last block.
__device__ __forceinline__ void gemma_allowed(const GemmaAttnParams &p, int fv, int q, int &k_lo,
                                              int &k_hi) {
    const bool free_row = q < fv;
    k_lo = free_row ? 0 : max(fv, p.window > 0 ? q - p.window + 1 : 0);
    k_hi = free_row ? p.T - 1 : min(q, p.T - 1);
}

// Mask S of key block kb (key 32 kb + 8 (i >> 2) + 4 g + (i & 3) in s[i]) and return the row's
// max. A block inside every row's allowed range of the wave (most blocks of a causal or windowed
// range) needs no mask: its five instructions per weight were a tenth of the block's.
__device__ __forceinline__ float gemma_mask_max(f32x16 &s, int kb, int k_lo, int k_hi, int g) {
    float mx = -INFINITY;
    if (__builtin_amdgcn_ballot_w64(k_lo > 32 * kb || 32 * kb + 31 > k_hi) == 0) {
#pragma unroll
        for (int e = 0; e < 16; ++e) mx = fmaxf(mx, s[e]);
    } else {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int k = 32 * kb + 8 * (e >> 2) + 4 * g + (e & 3);
            s[e] = ((k >= k_lo) & (k <= k_hi)) ? s[e] : -INFINITY;
            mx = fmaxf(mx, s[e]);
        }
    }
    return fmaxf(mx, xlane32(mx));
}

// fp32 weights against the row's max, their fp32 sum over this lane's keys (returned), and P in
// fp16 for P.V (11 significant bits; the reference's explicit path multiplies fp32 weights); a row
// with no allowed key so far has none.
__device__ __forceinline__ float gemma_weights(const f32x16 &s, float m, u32x4 (&wh)[2]) {
    float ts = 0.f;
    if (m == -INFINITY) {
        wh[0] = wh[1] = u32x4{0, 0, 0, 0};
    } else {
#pragma unroll
        for (int hf = 0; hf < 2; ++hf)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float x0 = __builtin_amdgcn_exp2f(s[8 * hf + 2 * e] - m);
                const float x1 = __builtin_amdgcn_exp2f(s[8 * hf + 2 * e + 1] - m);
                ts += x0 + x1;
                wh[hf][e] = pack_f16x2(x0, x1);
            }
    }
    return ts;
}

// Resource over the head's Q' rows from row `row` on (rows past T read as zeros).
template <int D>
__device__ __forceinline__ u32x4 gemma_q_rsrc(const GemmaAttnParams &p, const GemmaItem &w, int row) {
    return rsrc_words((const _Float16 *)p.qp + (((int64_t)w.b * p.Hq + w.h) * p.T + row) * D,
                      (int64_t)max(0, p.T - row) * (D * 2));
}

// One lane's copies of 32 * N rows of Q' (128 channels from byte `col` of the row) into N * 8 KB
// of LDS: rows of 256 bytes, 16-byte units XOR-swizzled by row. Read by the lanes themselves, 32
// rows per load, a workgroup's Q' held the address unit for 4 us; so the rows arrive as runs of
// 256 bytes. Rows past the resource arrive as zeros.
template <int D, int N>
__device__ __forceinline__ void gemma_copy_q(const u32x4 &rq, char *area, int lane, int col) {
#pragma unroll
    for (int j = 0; j < 8 * N; ++j) {
        const int row = 4 * j + (lane >> 4);
        copy_plus(rq, (uint32_t)(uintptr_t)(lds_void *)(area + j * 1024),
                  row * (D * 2) + 16 * ((lane & 15) ^ (row & 15)), col);
    }
}
__device__ __forceinline__ f16x8 gemma_q_opnd(const char *area, int row, int c, int g) {
    return *(const __attribute__((address_space(3))) f16x8 *)(
        (lds_void *)(area + row * 256 + 16 * ((2 * c + g) ^ (row & 15))));
}

// 32 rows x 128 channels of O^T accumulators (times `scale`) to rows of fp32 at `dst`, the first
// `rows` of them, through the wave's own 16 KB of LDS (units swizzled by row): they leave as runs of
// 512 bytes, where the lanes that hold them would store 32 rows per instruction.
__device__ __forceinline__ void gemma_store_rows(char *area, const f32x16 (&o)[4], float scale, int r,
                                                 int g, float *dst, int64_t stride, int rows) {
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
            f32x4 w;
#pragma unroll
            for (int e = 0; e < 4; ++e) w[e] = o[db][4 * i4 + e] * scale;
            *(f32x4 *)(area + r * 512 + 16 * ((8 * db + 2 * i4 + g) ^ r)) = w;
        }
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const int row = 2 * j + g;
        const f32x4 w = *(const f32x4 *)(area + row * 512 + 16 * (r ^ row));
        if (row < rows) *(f32x4 *)(dst + row * stride + 4 * r) = w;
    }
}

// Where a range's rows go from row `row0` of its query block on: the output, or the partials.
struct GemmaRows {
    float *o;                    // head's first channel
    int64_t stride;
    int rows;                    // rows that exist
    float *ml;                   // partial (max, sum) or null
};
__device__ __forceinline__ GemmaRows gemma_rows(const GemmaAttnParams &p, const GemmaItem &w, int D,
                                                int row0) {
    constexpr int qwg = kGemmaQueries;
    GemmaRows x;
    if (w.nch > 1) {
        const int64_t row = p.part_row0[w.b] +
                            ((int64_t)w.h * p.part_chunks[w.b] +
                             gemma_part_offset(p.T, p.window, p.chunk, qwg, w.fv, w.qblk) + w.chunk) *
                                qwg + row0;
        x = GemmaRows{p.part_o + row * D, D, qwg, p.part_ml + row * 2};
    } else {
        const int q = w.q0 + row0;
        x = GemmaRows{p.out + (int64_t)w.b * p.o_bs + (int64_t)q * p.o_rs + (int64_t)w.h * D, p.o_rs,
                      p.T - q, nullptr};
    }
    return x;
}

// D = 256: eight waves (two per SIMD, at most 256 registers each); a wave owns 32 queries over
// the whole head, and a query group's two waves the even and the odd key blocks of the range,
// merging at its end. A step is a pair of key blocks (64 KB of K' and V'^T), copied into one of
// two stages while the other is read; one barrier per step. Two waves per SIMD overlap: alone, a
// wave's chain S -> softmax -> P.V leaves the matrix cores idle most of the time (four waves of
// up to 512 registers took 1.8 us per 128 queries and key block, these 0.73 us, 1.46 us a step
// against 1.0 us of products per SIMD). No unit is full: over 2 x 2048 tokens, window 1024 (87 us) the
// matrix cores are busy 32% of the time, LDS (256 KB of operand reads and 64 KB of copies a step)
// 20%, the address unit's queue is full 14%; waves wait for data or the barrier 32% and to issue 37%
// of theirs, with two of them per SIMD to cover it. (Two sets of waves in opposite phases, one forming S while the other ran
// softmax and P.V, with two barriers a step, measured 0.88 us.)
__global__ __attribute__((amdgpu_flat_work_group_size(512, 512), amdgpu_waves_per_eu(2, 2)))
void gemma_attn256_kernel(const GemmaAttnParams p) {
    constexpr int D = 256, QWG = kGemmaQueries, NCW = kNCW, NDW = kNDW;
    constexpr int KBYTES = D * 32 * 2, BLOCK = 2 * KBYTES, STEP = 2 * BLOCK;
    constexpr int COPIES = BLOCK / 1024 / 8;         // 1 KB copies per wave per key block
    __shared__ __attribute__((aligned(16))) char smem[2 * STEP];
    __shared__ __attribute__((aligned(16))) float xs[8 * 64 * 2];   // (max, sum) of every lane

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, g = lane >> 5;
    // query group and key blocks' parity (waves w and w + 4, on one SIMD, are a group's two)
    const int grp = wave & 3, par = wave >> 2;
    const GemmaItem wi = gemma_item(p, QWG);
    if (wi.chunk >= wi.nch) return;                  // this block has fewer key ranges
    const int T = p.T, kb_lo = wi.kb_lo, nblk = wi.kb_hi - wi.kb_lo + 1;
    // steps of the range; of this wave (the last may hold no odd block)
    const int nstep = (nblk + 1) / 2, mysteps = (nblk - par + 1) / 2;

    // ---- copies of key blocks into the stages ---------------------------------------------
    const int nkb_all = (T + 31) / 32;
    const int64_t head_off = ((int64_t)wi.b * p.Hkv + wi.kvh) * nkb_all * (D * 32);   // elements
    const u32x4 rk = rsrc_words((const _Float16 *)p.kp + head_off, (int64_t)nkb_all * KBYTES);
    const u32x4 rv = rsrc_words((const _Float16 *)p.vt + head_off, (int64_t)nkb_all * KBYTES);
    auto copy_step = [&](int i) __attribute__((always_inline)) {   // i-th step of the range
        char *dst = smem + (i & 1) * STEP;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            if (k > 0 && i * 2 + k >= nblk) continue;        // (read by no wave)
            const int kb = kb_lo + i * 2 + k;
#pragma unroll
            for (int j = 0; j < COPIES; ++j) {
                const int u = wave * COPIES + j;             // 1 KB unit of the block: K' then V'^T
                const bool isk = u < KBYTES / 1024;
                const int uu = isk ? u : u - KBYTES / 1024;
                copy_plus(isk ? rk : rv,
                          (uint32_t)(uintptr_t)(lds_void *)(dst + k * BLOCK + u * 1024), lane * 16,
                          kb * KBYTES + uu * 1024);
            }
        }
    };
    // The first step's copies go out before the Q' loads, so the two latencies overlap.
    copy_step(0);

    // ---- Q' of this wave: query q0 + 32 grp + r, channels 16 c + 8 g .. +7 -----------------
    // (through the second stage, 128 channels at a time in the wave's own 8 KB)
    const int q = wi.q0 + 32 * grp + r;              // this lane's query row
    f16x8 qh[NCW];
    {
        const u32x4 rq = gemma_q_rsrc<D>(p, wi, wi.q0 + 32 * grp);
        char *area = smem + STEP + wave * 8192;
#pragma unroll
        for (int ps = 0; ps < 2; ++ps) {
            gemma_copy_q<D, 1>(rq, area, lane, 256 * ps);
            wait_copies();
#pragma unroll
            for (int c = 0; c < NCW / 2; ++c)
                qh[ps * (NCW / 2) + c] = gemma_q_opnd(area, r, c, g);
            // (in registers before the next pass's copies)
#pragma unroll
            for (int c = 0; c < NCW / 2; ++c) asm volatile("" : "+v"(qh[ps * (NCW / 2) + c]));
        }
    }
    int k_lo, k_hi;
    gemma_allowed(p, wi.fv, q, k_lo, k_hi);

    f32x16 o[NDW];
    float m, l;
    bool overflow = false;                           // some row's weights passed the bound

    // One pass over the range's key blocks. SAFE: the exact online softmax (O and l rescaled
    // when a row's max grows); otherwise each row's max is fixed at the wave's first block with
    // an allowed key. `first`: the first step's copies are already on their way.
    auto run = [&](auto safe, bool first) __attribute__((always_inline)) {
        constexpr bool SAFE = decltype(safe)::value;
#pragma unroll
        for (int db = 0; db < NDW; ++db) o[db] = splat16(0.f);
        m = -INFINITY;
        l = 0.f;
        if (!first) copy_step(0);
        for (int i = 0; i < mysteps; ++i) {
            // step i's copies have landed for this wave; after the barrier for every wave, and
            // the stage of step i - 1 is free
            wait_copies();
            __syncthreads();
            if (i + 1 < nstep) copy_step(i + 1);
            const char *Ks = smem + (i & 1) * STEP + par * BLOCK;
            const char *Vs = Ks + KBYTES;
            const int kb = kb_lo + i * 2 + par;
            auto opnd = [&](const char *base, int unit) __attribute__((always_inline)) {
                return *(const __attribute__((address_space(3))) f16x8 *)(
                    (lds_void *)(base + unit * 1024 + lane * 16));
            };
            // S^T: one chain (a product whose SrcC is the previous result issues without waiting
            // for it)
            constexpr int kAhead = 3;                // operands read ahead of their product
            f32x16 s = splat16(0.f);
            f16x8 ka[NCW];
#pragma unroll
            for (int c = 0; c < kAhead; ++c) ka[c] = opnd(Ks, c);
#pragma unroll
            for (int c = 0; c < NCW; ++c) {
                if (c + kAhead < NCW) ka[c + kAhead] = opnd(Ks, c + kAhead);
                s = mfma32(ka[c], qh[c], s);
                __builtin_amdgcn_sched_barrier(0);
            }
            // V'^T operands (unit hf * NDW + db), the first kAhead read now: they do not depend on
            // the softmax below, which hides their LDS round trip
            f16x8 va[2 * NDW];
#pragma unroll
            for (int j = 0; j < kAhead; ++j) va[j] = opnd(Vs, j);
            const float mx = gemma_mask_max(s, kb, k_lo, k_hi, g);
            if constexpr (SAFE) {
                if (__builtin_amdgcn_ballot_w64(mx > m) != 0) {
                    const float mn = fmaxf(m, mx);
                    const float alpha = mn > m ? __builtin_amdgcn_exp2f(m - mn) : 1.0f;  // 0 from -inf
#pragma unroll
                    for (int db = 0; db < NDW; ++db) o[db] *= splat16(alpha);
                    l *= alpha;
                    m = mn;
                }
            } else {
                if (m == -INFINITY) m = mx;              // the row's first allowed keys
                overflow |= mx > m + kGemmaBound;
            }
            u32x4 wh[2];
            l += gemma_weights(s, m, wh);
            // O^T += V^T.P^T; consecutive products update different accumulators (a key half over
            // all channel blocks)
#pragma unroll
            for (int j = 0; j < 2 * NDW; ++j) {
                if (j + kAhead < 2 * NDW) va[j + kAhead] = opnd(Vs, j + kAhead);
                o[j % NDW] = mfma32(va[j], __builtin_bit_cast(f16x8, wh[j / NDW]), o[j % NDW]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (mysteps < nstep) {
            wait_copies();
            __syncthreads();
        }
    };
    run(std::false_type{}, true);
    // the exact pass, for the whole workgroup, when any row outgrew its fixed max
    if (__syncthreads_or(overflow)) run(std::true_type{}, false);

    // ---- the even and odd key blocks' sums meet -------------------------------------------
    // A group's two waves pass each other half of their O through the (free) stages: wave `par`
    // keeps channel blocks 4 par .. 4 par + 3, both rescaled to the larger max.
    float lt = l + xlane32(l);
    f32x16 out[4];
    __syncthreads();                                 // every wave is past its last step
    {
        float *mine = (float *)(smem + wave * 16384) + lane * 4;
        const float *other = (const float *)(smem + (wave ^ 4) * 16384) + lane * 4;
        auto merge = [&](auto P) __attribute__((always_inline)) {
            constexpr int keep = decltype(P)::value * 4, pass = 4 - keep;
#pragma unroll
            for (int db = 0; db < 4; ++db)
#pragma unroll
                for (int i4 = 0; i4 < 4; ++i4) {
                    f32x4 w;
#pragma unroll
                    for (int e = 0; e < 4; ++e) w[e] = o[pass + db][4 * i4 + e];
                    *(f32x4 *)(mine + (db * 4 + i4) * 256) = w;
                }
            *(f32x2 *)(xs + (wave * 64 + lane) * 2) = f32x2{m, lt};
            __syncthreads();
            const f32x2 ml = *(const f32x2 *)(xs + ((wave ^ 4) * 64 + lane) * 2);
            const float mx = fmaxf(m, ml[0]);
            // (a wave in which the row allows no key has max -inf and adds nothing)
            const float f0 = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mx);
            const float f1 = ml[0] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ml[0] - mx);
            m = mx;
            lt = f0 * lt + f1 * ml[1];
#pragma unroll
            for (int db = 0; db < 4; ++db)
#pragma unroll
                for (int i4 = 0; i4 < 4; ++i4) {
                    const f32x4 w = *(const f32x4 *)(other + (db * 4 + i4) * 256);
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        out[db][4 * i4 + e] = f0 * o[keep + db][4 * i4 + e] + f1 * w[e];
                }
        };
        if (par) merge(std::integral_constant<int, 1>{});
        else merge(std::integral_constant<int, 0>{});
    }

    // ---- epilogue: O / l in fp32 (the reference's dtype here), or a range's partials ------
    // (the lane's row again from its LDS offset, which the loops keep: carried through them, it
    // and what hangs on it would spill)
    int lane_again = lane * 16;
    asm volatile("" : "+v"(lane_again));
    const int er = (lane_again >> 4) & 31, eg = lane_again >> 9;
    const GemmaRows to = gemma_rows(p, wi, D, 32 * grp);
    if (to.ml && par == 0 && eg == 0) *(f32x2 *)(to.ml + er * 2) = f32x2{m, lt};
    __syncthreads();                                 // the merge's halves are read
    gemma_store_rows(smem + wave * 16384, out, to.ml ? 1.0f : 1.0f / lt, er, eg,
                     to.o + 128 * par, to.stride, to.rows);
}

// D = 512: four waves (one per SIMD, up to 512 registers); a wave owns 64 queries over half of
// the head, its mate the other half, so that each LDS operand read feeds two products (eight
// waves of 32 queries x 256 channels read 256 KB per key block: calls of 2 x 1224 and 2 x 1472
// causal tokens took 120 and 138 us where this kernel took 109 and 129; it now takes 103 and 125,
// the kernel with 64 queries per workgroup 185 and 241; at 2 x 2048 the matrix cores are busy 41% of
// 163 us). The mates split the softmax: each
// completes S and forms P for 32 of the 64 queries, its own (local group 0; the mate's are group
// 1), so a step passes S partials one way and P the other. Software pipeline: step i issues the
// 32 products of S(i + 1) one at a time with a slice of the softmax of S(i) after each, then
// P(i).V; K' runs one block ahead of V'^T, two stages of each. Two barriers a step: the first
// publishes S(i)'s partials and the landed copies, the second P(i).
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256), amdgpu_waves_per_eu(1, 1)))
void gemma_attn512_kernel(const GemmaAttnParams p) {
    constexpr int D = 512, QWG = kGemmaQueries, NCW = kNCW, NDW = kNDW;
    constexpr int KBYTES = D * 32 * 2;               // K' (or V'^T) of one key block
    constexpr int COPIES = KBYTES / 1024 / 4;        // 1 KB copies per wave of either
    __shared__ __attribute__((aligned(16))) char sK[2 * KBYTES];
    __shared__ __attribute__((aligned(16))) char sV[2 * KBYTES];
    __shared__ __attribute__((aligned(16))) float xsS[4 * 64 * 16];  // S for the mate [4][4][64][4]
    __shared__ __attribute__((aligned(16))) uint32_t xsP[4 * 64 * 8];  // P for the mate [4][2][64][4]
    __shared__ __attribute__((aligned(16))) float xml[4 * 64 * 2];   // (max, sum) of every lane

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, g = lane >> 5;
    const int grp = wave >> 1, half = wave & 1, mate = wave ^ 1;
    const GemmaItem wi = gemma_item(p, QWG);
    if (wi.chunk >= wi.nch) return;                  // this block has fewer key ranges
    const int T = p.T, kb_lo = wi.kb_lo, nblk = wi.kb_hi - wi.kb_lo + 1;
    const int row0 = 64 * grp;                       // the wave's queries within the block

    const int nkb_all = (T + 31) / 32;
    const int64_t head_off = ((int64_t)wi.b * p.Hkv + wi.kvh) * nkb_all * (D * 32);   // elements
    const u32x4 rk = rsrc_words((const _Float16 *)p.kp + head_off, (int64_t)nkb_all * KBYTES);
    const u32x4 rv = rsrc_words((const _Float16 *)p.vt + head_off, (int64_t)nkb_all * KBYTES);
    auto copy1 = [&](const u32x4 &rs, char *stages, int i, int j) __attribute__((always_inline)) {
        const int u = wave * COPIES + j;
        copy_plus(rs, (uint32_t)(uintptr_t)(lds_void *)(stages + (i & 1) * KBYTES + u * 1024),
                  lane * 16, (kb_lo + i) * KBYTES + u * 1024);
    };
    auto copy = [&](const u32x4 &rs, char *stages, int i) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < COPIES; ++j) copy1(rs, stages, i, j);
    };
    // ---- Q' of this wave: local group n's query q0 + row0 + 32 (half ^ n) + r, channels
    // 256 half + 16 c + 8 g .. +7 (through the V'^T stages, 128 channels at a time in the wave's
    // own 16 KB; K'(0) and K'(1) follow the first half's copies)
    f16x8 qh[2][NCW];
    {
        const u32x4 rq = gemma_q_rsrc<D>(p, wi, wi.q0 + row0);
        char *area = sV + wave * 16384;
#pragma unroll
        for (int ps = 0; ps < 2; ++ps) {
            gemma_copy_q<D, 2>(rq, area, lane, 512 * half + 256 * ps);
            if (ps == 0) {
                copy(rk, sK, 0);
                copy(rk, sK, 1);                     // (zeros past the last key block)
                wait_copies_but<2 * COPIES>();
            } else {
                wait_copies();
            }
#pragma unroll
            for (int n = 0; n < 2; ++n)
#pragma unroll
                for (int c = 0; c < NCW / 2; ++c)
                    qh[n][ps * (NCW / 2) + c] = gemma_q_opnd(area, 32 * (half ^ n) + r, c, g);
#pragma unroll
            for (int n = 0; n < 2; ++n)
#pragma unroll
                for (int c = 0; c < NCW / 2; ++c)
                    asm volatile("" : "+v"(qh[n][ps * (NCW / 2) + c]));
        }
    }
    const int q = wi.q0 + row0 + 32 * half + r;      // this lane's row of its own 32 queries
    int k_lo, k_hi;
    gemma_allowed(p, wi.fv, q, k_lo, k_hi);
    __syncthreads();                                 // the V'^T stages are read; K'(0), K'(1) are in
    copy(rv, sV, 0);

    f32x16 o[NDW][2];
    float m, l;
    float top = -INFINITY;                           // the largest S of this lane's keys
    f32x16 sc[2];                                    // partial S of the next step's block
    auto opnd = [&](const char *base, int unit) __attribute__((always_inline)) {
        return *(const __attribute__((address_space(3))) f16x8 *)(
            (lds_void *)(base + unit * 1024 + lane * 16));
    };
    constexpr int kAhead = 4;                        // operands read ahead of their products
    // Partial S of block i over this wave's channels, slice(k) after product k of 32.
    auto s_block = [&](int i, auto slice) __attribute__((always_inline)) {
        const char *Ks = sK + (i & 1) * KBYTES;
        f16x8 ka[NCW];
        f32x16 sn[2];
#pragma unroll
        for (int c = 0; c < kAhead; ++c) ka[c] = opnd(Ks, half * NCW + c);
#pragma unroll
        for (int c = 0; c < NCW; ++c) {
            if (c + kAhead < NCW) ka[c + kAhead] = opnd(Ks, half * NCW + c + kAhead);
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                if (c == 0) sn[n] = mfma_s_zero(ka[c], qh[n][c]);
                else mfma_s_next_v(sn[n], ka[c], qh[n][c]);
                slice(2 * c + n);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        s_ready(sn[0], sn[1]);
        sc[0] = sn[0];
        sc[1] = sn[1];
    };
    // The mate's queries' partial S goes to the mate.
    auto pass_s = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4)
            *(f32x4 *)(xsS + ((wave * 4 + i4) * 64 + lane) * 4) =
                f32x4{sc[1][4 * i4], sc[1][4 * i4 + 1], sc[1][4 * i4 + 2], sc[1][4 * i4 + 3]};
    };

    // A pass over the range's key blocks, each row's max fixed at its first block with an allowed
    // key; when any row outgrows it, a second pass with the rows' maxima, which the first has seen.
    m = -INFINITY;
    auto run = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int db = 0; db < NDW; ++db) o[db][0] = o[db][1] = splat16(0.f);
        l = 0.f;
        s_block(0, [](int) {});
        pass_s();
        for (int i = 0; i < nblk; ++i) {
            // This wave's share of K'(i + 1) has landed (V'^T(i)'s, issued after it, may not
            // have); then everyone's has, S(i)'s partials are in and K' stage i is free.
            wait_copies_but<COPIES>();
            __syncthreads();
            const int kb = kb_lo + i;
            f32x4 x[4];
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4) x[i4] = *(const f32x4 *)(xsS + ((mate * 4 + i4) * 64 + lane) * 4);
            f32x16 s = sc[0];
            u32x4 wh[2];
            // K'(i + 2) is copied between the products of S(i + 1), V'^T(i + 1) between those of
            // P(i).V: issued together they queue, 40 to 60 cycles each (1024 padded tokens: 103
            // -> 97 us a call). Past the range they read an empty resource, so that the waits' counts hold.
            u32x4 rkn = rk, rvn = rv;
            if (i + 2 >= nblk) rkn[2] = 0;
            if (i + 1 >= nblk) rvn[2] = 0;
            const bool more = i + 1 < nblk;
            // A block inside every row's allowed range of the wave, whose rows all have a max:
            // its softmax runs between the products of S(i + 1).
            if (more &&
                __builtin_amdgcn_ballot_w64(k_lo > 32 * kb || 32 * kb + 31 > k_hi || m == -INFINITY) == 0) {
                float ts = 0.f, mx = -INFINITY, ex[16];
                s_block(i + 1, [&](int k) __attribute__((always_inline)) {
                    if ((k & 3) == 3) copy1(rkn, sK, i + 2, k >> 2);
                    // slices 2..5 complete S, 6..9 its max, 10..25 take a weight each, and every
                    // other of 13..27 sums and packs two
                    if (k >= 2 && k < 6)
                        for (int e = 0; e < 4; ++e) s[4 * (k - 2) + e] += x[k - 2][e];
                    if (k >= 6 && k < 10)
                        for (int e = 0; e < 4; ++e) mx = fmaxf(mx, s[4 * (k - 6) + e]);
                    if (k >= 10 && k < 26) ex[k - 10] = __builtin_amdgcn_exp2f(s[k - 10] - m);
                    if (k >= 13 && k < 29 && (k & 1)) {
                        const int e = k - 13;
                        ts += ex[e] + ex[e + 1];
                        wh[e >> 3][(e >> 1) & 3] = pack_f16x2(ex[e], ex[e + 1]);
                    }
                });
                top = fmaxf(top, mx);
                l += ts;
            } else {
                copy(rkn, sK, i + 2);
#pragma unroll
                for (int e = 0; e < 16; ++e) s[e] += x[e >> 2][e & 3];
                const float mx = gemma_mask_max(s, kb, k_lo, k_hi, g);
                if (m == -INFINITY) m = mx;          // the row's first allowed keys
                top = fmaxf(top, mx);
                l += gemma_weights(s, m, wh);
                if (more) s_block(i + 1, [](int) {});
            }
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) *(u32x4 *)(xsP + ((wave * 2 + hf) * 64 + lane) * 4) = wh[hf];
            const char *Vs = sV + (i & 1) * KBYTES;
            auto v_opnd = [&](int j) __attribute__((always_inline)) {
                return opnd(Vs, (j / NDW) * (D / 32) + half * NDW + j % NDW);
            };
            f16x8 va[2 * NDW];
            wait_copies_but<COPIES>();
            __syncthreads();     // P(i) and V'^T(i) are in; S(i)'s partials are read
            if (more) pass_s();
            u32x4 wo[2];
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) wo[hf] = *(const u32x4 *)(xsP + ((mate * 2 + hf) * 64 + lane) * 4);
#pragma unroll
            for (int j = 0; j < kAhead; ++j) va[j] = v_opnd(j);
#pragma unroll
            for (int j = 0; j < 2 * NDW; ++j) {
                if (j + kAhead < 2 * NDW) va[j + kAhead] = v_opnd(j + kAhead);
                o[j % NDW][0] = mfma32(va[j], __builtin_bit_cast(f16x8, wh[j / NDW]), o[j % NDW][0]);
                o[j % NDW][1] = mfma32(va[j], __builtin_bit_cast(f16x8, wo[j / NDW]), o[j % NDW][1]);
                if (j & 1) copy1(rvn, sV, i + 1, j >> 1);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        wait_copies();
    };
    run();
    // (each lane holds half of the row's keys)
    top = fmaxf(top, xlane32(top));
    if (__syncthreads_or(top > m + kGemmaBound)) {
        m = top;
        copy(rk, sK, 0);
        if (nblk > 1) copy(rk, sK, 1);
        copy(rv, sV, 0);
        wait_copies();
        __syncthreads();
        run();
    }

    // ---- epilogue: O / l in fp32 (the reference's dtype here), or a range's partials ------
    // (the lane's row again from its LDS offset, as in the D 256 kernel)
    int lane_again = lane * 16;
    asm volatile("" : "+v"(lane_again));
    const int er = (lane_again >> 4) & 31, eg = lane_again >> 9, el = lane_again >> 4;
    const float lt = l + xlane32(l);
    *(f32x2 *)(xml + (wave * 64 + el) * 2) = f32x2{m, lt};
    __syncthreads();                                 // (also: every wave is past its last V'^T)
    char *area = (wave < 2 ? sK : sV) + (wave & 1) * 16384;
    const GemmaRows to = gemma_rows(p, wi, D, row0);
    if (to.ml && eg == 0) *(f32x2 *)(to.ml + (32 * half + er) * 2) = f32x2{m, lt};
#pragma unroll
    for (int n = 0; n < 2; ++n) {
        const int first = 32 * (half ^ n);           // of the group's 32 queries, within the 64
        asm volatile("" ::: "memory");               // (the sum from LDS when it is needed)
        const float sum = xml[((n == 0 ? wave : mate) * 64 + el) * 2 + 1];
        const float scale = to.ml ? 1.0f : 1.0f / sum;
#pragma unroll
        for (int d0 = 0; d0 < NDW; d0 += 4) {
            f32x16 out[4];
#pragma unroll
            for (int db = 0; db < 4; ++db) {
                // (whole in its registers until here: taken apart earlier, it was moved around)
                asm volatile("" : "+a"(o[d0 + db][n]));
                out[db] = o[d0 + db][n];
            }
            gemma_store_rows(area, out, scale, er, eg, to.o + first * to.stride + 256 * half + 32 * d0,
                             to.stride, to.rows - first);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// D = 512, short prompts: 64 queries per workgroup, a wave 32 of them over half of the head (its
// partner wave the other half), one key block at a time, no key ranges. Twice as many
// workgroups, each with half of the 128-query kernel's start and epilogue, which bound a prompt of
// a few blocks: 72 / 144 / 256 / 384 / 512 tokens 18.5 / 22.4 / 31.7 / 40.2 / 49.9 us a call against
// 23.0 / 25.7 / 35.2 / 42.5 / 51.4. Past 512 tokens a plan may have key ranges, which only the other
// kernel has.
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256), amdgpu_waves_per_eu(1, 1)))
void gemma_attn512_short_kernel(const GemmaAttnParams p) {
    constexpr int D = 512, QWG = kGemmaShortQueries, NCW = kNCW, NDW = kNDW;
    constexpr int KBYTES = D * 32 * 2, BLOCK = 2 * KBYTES, COPIES = BLOCK / 1024 / 4;
    __shared__ __attribute__((aligned(16))) char smem[2 * BLOCK];
    __shared__ __attribute__((aligned(16))) float xs[4 * 64 * 16];   // partial S [4][4][64][4]

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, g = lane >> 5;
    const int grp = wave >> 1, half = wave & 1;
    const GemmaItem wi = gemma_item(p, QWG);
    const int T = p.T, kb_lo = wi.kb_lo, nblk = wi.kb_hi - wi.kb_lo + 1;
    const int nkb_all = (T + 31) / 32;
    const int64_t head_off = ((int64_t)wi.b * p.Hkv + wi.kvh) * nkb_all * (D * 32);   // elements
    const u32x4 rk = rsrc_words((const _Float16 *)p.kp + head_off, (int64_t)nkb_all * KBYTES);
    const u32x4 rv = rsrc_words((const _Float16 *)p.vt + head_off, (int64_t)nkb_all * KBYTES);
    auto copy_block = [&](int i) __attribute__((always_inline)) {   // i-th block of the range
        char *dst = smem + (i & 1) * BLOCK;
#pragma unroll
        for (int j = 0; j < COPIES; ++j) {
            const int u = wave * COPIES + j;         // 1 KB unit of the block: K' then V'^T
            const bool isk = wave < 2;
            copy_plus(isk ? rk : rv, (uint32_t)(uintptr_t)(lds_void *)(dst + u * 1024), lane * 16,
                      (kb_lo + i) * KBYTES + (isk ? u : u - KBYTES / 1024) * 1024);
        }
    };
    copy_block(0);

    // Q' of this wave (through the wave's own 16 KB of the second stage)
    f16x8 qh[NCW];
    {
        const u32x4 rq = gemma_q_rsrc<D>(p, wi, wi.q0 + 32 * grp);
        char *area = smem + BLOCK + wave * 16384;
#pragma unroll
        for (int ps = 0; ps < 2; ++ps)
            gemma_copy_q<D, 1>(rq, area + ps * 8192, lane, 512 * half + 256 * ps);
        wait_copies();
#pragma unroll
        for (int c = 0; c < NCW; ++c)
            qh[c] = gemma_q_opnd(area + (c / 8) * 8192, r, c % 8, g);
        // Q' is only an MFMA operand: home it in AGPRs, leaving the VGPRs to S, P and operands
#pragma unroll
        for (int c = 0; c < NCW; ++c) asm volatile("" : "+a"(qh[c]));
    }
    const int q = wi.q0 + 32 * grp + r;              // this lane's query row
    int k_lo, k_hi;
    gemma_allowed(p, wi.fv, q, k_lo, k_hi);

    f32x16 o[NDW];
    float m = -INFINITY, l;
    float top = -INFINITY;                           // the row's largest S
    const f32x16 zero = splat16(0.f);                // the S chains' first SrcC
    auto opnd = [&](const char *base, int unit) __attribute__((always_inline)) {
        return *(const __attribute__((address_space(3))) f16x8 *)(
            (lds_void *)(base + unit * 1024 + lane * 16));
    };
    // Block i: landed and published, the next block's copies issued; S of this wave's rows, the
    // partner's half of the channels added.
    auto s_block = [&](int i) __attribute__((always_inline)) {
        wait_copies();
        __syncthreads();
        if (i + 1 < nblk) copy_block(i + 1);
        const char *Ks = smem + (i & 1) * BLOCK;
        f32x16 s;
#pragma unroll
        for (int c = 0; c < NCW; ++c) {
            const f16x8 a = opnd(Ks, half * NCW + c);
            if (c == 0) s = mfma_s_first(a, qh[0], zero);
            else mfma_s_next(s, a, qh[c]);
        }
        s_ready(s, zero);
        // (a wave's 16-byte accesses are lane-contiguous, free of bank conflicts)
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4)
            *(f32x4 *)(xs + ((wave * 4 + i4) * 64 + lane) * 4) =
                f32x4{s[4 * i4], s[4 * i4 + 1], s[4 * i4 + 2], s[4 * i4 + 3]};
        __syncthreads();
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
            const f32x4 x = *(const f32x4 *)(xs + (((wave ^ 1) * 4 + i4) * 64 + lane) * 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) s[4 * i4 + e] += x[e];
        }
        return s;
    };
    // Passes as in the 128-query kernel.
    auto run = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int db = 0; db < NDW; ++db) o[db] = splat16(0.f);
        l = 0.f;
        for (int i = 0; i < nblk; ++i) {
            f32x16 s = s_block(i);
            const char *Vs = smem + (i & 1) * BLOCK + KBYTES;
            auto v_opnd = [&](int hf, int db) __attribute__((always_inline)) {
                return opnd(Vs, hf * (D / 32) + half * NDW + db);
            };
            // the first key half's operands: their LDS round trip passes behind the softmax
            f16x8 va0[NDW], va1[NDW];
#pragma unroll
            for (int db = 0; db < NDW; ++db) va0[db] = v_opnd(0, db);
            const float mx = gemma_mask_max(s, kb_lo + i, k_lo, k_hi, g);
            if (m == -INFINITY) m = mx;              // the row's first allowed keys
            top = fmaxf(top, mx);
            u32x4 wh[2];
            l += gemma_weights(s, m, wh);
#pragma unroll
            for (int db = 0; db < NDW; ++db) {
                va1[db] = v_opnd(1, db);
                o[db] = mfma32(va0[db], __builtin_bit_cast(f16x8, wh[0]), o[db]);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int db = 0; db < NDW; ++db)
                o[db] = mfma32(va1[db], __builtin_bit_cast(f16x8, wh[1]), o[db]);
        }
    };
    run();
    if (__syncthreads_or(top > m + kGemmaBound)) {
        m = top;
        copy_block(0);
        run();
    }

    const float lt = l + xlane32(l);
    __syncthreads();                                 // every wave is past its last V'^T
    const GemmaRows to = gemma_rows(p, wi, D, 32 * grp);
#pragma unroll
    for (int d0 = 0; d0 < NDW; d0 += 4) {
        f32x16 out[4];
#pragma unroll
        for (int db = 0; db < 4; ++db) {
            asm volatile("" : "+a"(o[d0 + db]));
            out[db] = o[d0 + db];
        }
        gemma_store_rows(smem + (2 * wave + d0 / 4) * 16384, out, 1.0f / lt, r, g,
                         to.o + 256 * half + 32 * d0, to.stride, to.rows);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// Merge of a query block's key ranges: O = sum_c 2^(m_c - M) O_c / sum_c 2^(m_c - M) l_c over
// its ranges c (M the largest max; a range in which a row allows no key has m = -inf and adds
// nothing), written in fp32. A thread per 4 channels of kCombineRows rows (RPW rows apart);
// the workgroup's rows all belong to one query block (blocks with one range wrote their
// output themselves). The loads of a pass -- N ranges of `rows` rows, about 48 registers --
// are all issued before the first use: the merge is a chain of dependent loads otherwise, and
// several rows per thread keep the workgroups few enough that the launch runs in one round.
constexpr int kCombineRows = 4;

template <int D, int N>
__device__ __forceinline__ void gemma_merge_rows(const GemmaAttnParams &p, int64_t row0, int ch,
                                                 int q, float *out) {
    constexpr int QWG = kGemmaQueries;
    constexpr int RPW = 256 / (D / 4);
    constexpr int PASS = N <= 2 ? kCombineRows : N <= 4 ? kCombineRows / 2 : 1;
#pragma unroll
    for (int g0 = 0; g0 < kCombineRows; g0 += PASS) {
        f32x2 ml[PASS][N];
        f32x4 oc[PASS][N];
#pragma unroll
        for (int r = 0; r < PASS; ++r)
#pragma unroll
            for (int c = 0; c < N; ++c) {
                const int64_t row = row0 + (int64_t)(g0 + r) * RPW + (int64_t)c * QWG;
                ml[r][c] = *(const f32x2 *)(p.part_ml + row * 2);
                oc[r][c] = *(const f32x4 *)(p.part_o + row * D + ch);
            }
#pragma unroll
        for (int r = 0; r < PASS; ++r) {
            if (q + (g0 + r) * RPW >= p.T) continue;   // rows past T: partials, no output
            float mx = -INFINITY;
#pragma unroll
            for (int c = 0; c < N; ++c) mx = fmaxf(mx, ml[r][c][0]);
            float lsum = 0.f;
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < N; ++c) {
                const float m = ml[r][c][0];
                const float wgt = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mx);
                lsum += wgt * ml[r][c][1];
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[e] += wgt * oc[r][c][e];
            }
            const float inv = 1.0f / lsum;
            f32x4 w;
#pragma unroll
            for (int e = 0; e < 4; ++e) w[e] = acc[e] * inv;
            *(f32x4 *)(out + (int64_t)(g0 + r) * RPW * p.o_rs) = w;
        }
    }
}

template <int D>
__global__ __launch_bounds__(256) void gemma_combine_kernel(const GemmaAttnParams p) {
    constexpr int QWG = kGemmaQueries;
    constexpr int U = D / 4;                        // threads per row
    constexpr int RPW = 256 / U;                    // rows per pass of the workgroup
    constexpr int WG_PER_QB = QWG / (RPW * kCombineRows);
    static_assert(WG_PER_QB * RPW * kCombineRows == QWG, "a query block's rows split evenly");
    const int nqb = (p.T + QWG - 1) / QWG;
    const int blk = (int)blockIdx.x / WG_PER_QB;    // (batch row, head, query block)
    const int qblk = blk % nqb;
    const int bh = blk / nqb;
    const int h = bh % p.Hq, b = bh / p.Hq;
    const int q0 = qblk * QWG;
    const int nch = gemma_ranges(p.T, p.window, p.chunk, q0, QWG, p.first_valid[b]);
    if (nch <= 1) return;
    const int off = gemma_part_offset(p.T, p.window, p.chunk, QWG, p.first_valid[b], qblk);
    const int rr = ((int)blockIdx.x % WG_PER_QB) * RPW * kCombineRows + (int)threadIdx.x / U;
    const int c4 = (int)threadIdx.x % U;
    const int q = q0 + rr;
    const int64_t row0 = p.part_row0[b] + ((int64_t)h * p.part_chunks[b] + off) * QWG + rr;
    // partial rows past T exist (a range writes all its block's rows) and are read, not merged
    float *out = p.out + (int64_t)b * p.o_bs + (int64_t)q * p.o_rs + (int64_t)h * D + 4 * c4;
    static_assert(kGemmaMaxChunks == 8, "one case per range count");
    switch (nch) {
    case 2: gemma_merge_rows<D, 2>(p, row0, 4 * c4, q, out); break;
    case 3: gemma_merge_rows<D, 3>(p, row0, 4 * c4, q, out); break;
    case 4: gemma_merge_rows<D, 4>(p, row0, 4 * c4, q, out); break;
    case 5: gemma_merge_rows<D, 5>(p, row0, 4 * c4, q, out); break;
    case 6: gemma_merge_rows<D, 6>(p, row0, 4 * c4, q, out); break;
    case 7: gemma_merge_rows<D, 7>(p, row0, 4 * c4, q, out); break;
    default: gemma_merge_rows<D, 8>(p, row0, 4 * c4, q, out); break;
    }
}

}  // namespace

int launch_gemma_prep(const GemmaPrepParams &p, int D, void *stream) {
    // rows per workgroup: four waves of kPrepPasses passes of one (D = 512) or two (D = 256)
    // rows
    const int64_t rows = (int64_t)p.B * p.T * (p.Hq + p.Hkv);
    if (rows > 0x7fffffff) return (int)hipErrorInvalidValue;   // 32-bit row indices
    const int64_t rows_wg = (D == 512 ? 4 : 8) * kPrepPasses;
    const int64_t row_wgs = (rows + rows_wg - 1) / rows_wg;
    const int64_t v_wgs = (int64_t)p.B * p.Hkv * ((p.T + 31) / 32);
    if (row_wgs + v_wgs > 0x7fffffff) return (int)hipErrorInvalidValue;
    const dim3 grid((unsigned)(row_wgs + v_wgs)), block(256);
    hipStream_t st = (hipStream_t)stream;
    if (D == 512) hipLaunchKernelGGL(gemma_prep_kernel<512>, grid, block, 0, st, p, (int)row_wgs);
    else hipLaunchKernelGGL(gemma_prep_kernel<256>, grid, block, 0, st, p, (int)row_wgs);
    return (int)hipGetLastError();
}

int launch_gemma_attn(const GemmaAttnParams &p, int D, void *stream) {
    const int64_t per_layer = (int64_t)p.B * p.Hq * ((p.T + kGemmaQueries - 1) / kGemmaQueries);
    const dim3 grid((unsigned)(per_layer * p.nch_max));
    hipStream_t st = (hipStream_t)stream;
    if (gemma_short(D, p.T, p.nch_max))
        hipLaunchKernelGGL(gemma_attn512_short_kernel,
                           dim3((unsigned)((int64_t)p.B * p.Hq *
                                           ((p.T + kGemmaShortQueries - 1) / kGemmaShortQueries))),
                           dim3(256), 0, st, p);
    else if (D == 512) hipLaunchKernelGGL(gemma_attn512_kernel, grid, dim3(256), 0, st, p);
    else hipLaunchKernelGGL(gemma_attn256_kernel, grid, dim3(512), 0, st, p);
    if (p.nch_max > 1) {
        const dim3 cgrid((unsigned)(per_layer * kGemmaQueries / (256 / (D / 4) * kCombineRows)));
        if (D == 512) hipLaunchKernelGGL(gemma_combine_kernel<512>, cgrid, dim3(256), 0, st, p);
        else hipLaunchKernelGGL(gemma_combine_kernel<256>, cgrid, dim3(256), 0, st, p);
    }
    return (int)hipGetLastError();
}

int gemma_queries_per_workgroup() { return kGemmaQueries; }

}  // namespace ltx
