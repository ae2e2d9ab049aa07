// Projection GEMM for calls whose 256 x 256 tiles do not fill the CUs (the audio stream's and
// the text's projections, the gate logits): y = x . w^T (+ bias) in smaller tiles, each
// workgroup's waves splitting the reduction between them instead of the tile.
//
// linear_gemm.hip cuts such a call's tiles into k ranges whose 256 KiB fp32 partials go
// through memory to a second launch. Here a workgroup owns a 32*MB x 32*NB tile over all of K,
// and each of its waves the whole tile over its own 16 of every 64*KG channels: per wave and
// step MB + NB operand reads feed MB*NB products, so a 128 x 128 tile reads LDS as rarely per
// product as the 256 x 256 kernel does (waves that split the tile would read it twice as often
// and be bound by it). The waves' fp32 accumulators meet in LDS once, at the end.
//
// Staging follows linear_gemm.hip: tiles HBM -> LDS by the buffer-load-to-LDS path, rows of 64
// elements with XOR-swizzled 16-byte units, rows past M (N) read as zeros. A ring of NS
// steps; after step s's barrier every wave has step s in registers, so its stage takes the
// copies of step s + NS at once and NS - 1 steps stay in flight (the calls are short: what
// they wait for is latency). Steps past the end copy from an empty resource (zeros, no
// memory access), so the counts every wait relies on hold to the end.
//
// Rounding is linear_gemm.hip's: the fp32 sum to bf16, then the bias in fp32 and bf16 again.
// The statistic (sums of squares over 256 columns) spans several column tiles: each writes
// its columns' sums to the workspace and linear_stat_kernel adds a block's in order.
#include <type_traits>

#include "lds_copy.hpp"

namespace ltx {
namespace {

typedef __attribute__((address_space(3))) float lds_float;
typedef __attribute__((address_space(3))) f32x4 lds_f32x4;
typedef __attribute__((address_space(3))) char lds_char;

template <int MB, int NB, int KG>
struct KsTile {
    static constexpr int TM = 32 * MB, TN = 32 * NB;
    static constexpr int WAVES = 4 * KG;
    static constexpr int ROWS = TM + TN;               // x rows, then w rows, of a 64-wide step
    static constexpr int SUB = ROWS * 128;             // bytes of one 64-wide step
    static constexpr int STAGE = KG * SUB;             // bytes of a step (64 * KG channels)
    static constexpr int XC = TM / 32, WC = TN / 32;   // 1 KB copies per wave per step
    static constexpr int CPS = XC + WC;
    static constexpr int FIT = 160 * 1024 / STAGE;
    static constexpr int NS = FIT < 6 ? FIT : 6;       // stages of the ring
    // The accumulators' exchange: per wave and 32 x 32 block four planes of 64 lanes x 16
    // bytes, padded so that four planes' equal rows fall in distinct banks.
    static constexpr int PLANE = 1024 + 64, BLOCK = 4 * PLANE;
    static constexpr int BLOCKS = MB * NB;
    static constexpr int RB = BLOCKS * WAVES * BLOCK <= 150 * 1024 ? BLOCKS : BLOCKS / 2;
    static constexpr int RED = NB * TM * 4;            // row sums of squares per column block
    static constexpr int XCHG = RB * WAVES * BLOCK;
    static constexpr int BYTES = NS * STAGE > XCHG + RED ? NS * STAGE : XCHG + RED;
    static_assert(NS >= 3 && (NS - 1) * CPS < 64, "vmcnt range");
    static_assert(BYTES <= 160 * 1024, "LDS of one workgroup");
};

// GROUP: several projections (one is spared the look-up, about 1 us of a call's start).
template <int MB, int NB, int KG, bool GROUP>
__global__ __attribute__((amdgpu_flat_work_group_size(256 * KG, 256 * KG),
                          amdgpu_waves_per_eu(KG, KG)))
void linear_ks_kernel(const LinearGroup grp) {
    int which = 0;
    if constexpr (GROUP) {
#pragma unroll
        for (int i = 1; i < kLinearGroup; ++i) which += (int)blockIdx.x >= grp.first[i] ? 1 : 0;
    }
    const LinearParams &p = grp.p[which];
    const int wg = GROUP ? (int)blockIdx.x - grp.first[which] : (int)blockIdx.x;
    using T = KsTile<MB, NB, KG>;
    constexpr int TM = T::TM, TN = T::TN, NS = T::NS, CPS = T::CPS, WAVES = T::WAVES;
    __shared__ __attribute__((aligned(16))) char smem[T::BYTES];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, g = lane >> 5;
    const int sub = wave >> 2, ch = wave & 3;          // this wave's 64 and 16 of a step
    const int nsteps = p.K / 64;

    // Tile: groups of 8 row tiles walked column by column, each XCD a contiguous range of that
    // order, so the workgroups of one XCD share their x and w rows in its L2.
    int tm, tn;
    {
        const int t = xcd_major(wg, GROUP ? p.tiles_m * p.tiles_n : (int)gridDim.x);
        constexpr int GRP = 8;
        const int group = t / (GRP * p.tiles_n), first = group * GRP;
        const int rows = min(GRP, p.tiles_m - first), within = t - group * GRP * p.tiles_n;
        tm = first + within % rows;
        tn = within / rows;
    }
    const int m0 = tm * TM, n0 = tn * TN;
    const int xrow = (int)(p.x_rs * 2), wrow = (int)(p.w_rs * 2);
    const char *X0 = (const char *)p.x + (int64_t)m0 * xrow;
    const char *W0 = (const char *)p.w + (int64_t)n0 * wrow;
    const int64_t xbytes = (int64_t)min(TM, p.M - m0) * xrow;
    const int64_t wbytes = (int64_t)min(TN, p.N - n0) * wrow;

    // Copies: a wave stages its share of its own 64-wide part, XC copies of x rows (8 rows
    // each), then WC of w rows. The resources' bases move with the step (64 * KG channels).
    constexpr int XC = T::XC, WC = T::WC;
    int src[CPS];
#pragma unroll
    for (int j = 0; j < CPS; ++j) {
        const int row = 8 * (j < XC ? ch * XC + j : ch * WC + j - XC) + (lane >> 3);
        src[j] = row * (j < XC ? xrow : wrow) + 16 * ((lane & 7) ^ ((row >> 1) & 7));
    }
    const int lds0 = sub * T::SUB, ldx = lds0 + ch * XC * 1024, ldw = lds0 + TM * 128 + ch * WC * 1024;
    u32x4 rx = rsrc_words(X0 + sub * 128, sub < nsteps ? xbytes : 0);
    u32x4 rw = rsrc_words(W0 + sub * 128, sub < nsteps ? wbytes : 0);
    int left = nsteps - sub;                           // 64-wide steps from the resources' on
    auto copy = [&](int stage, int j) __attribute__((always_inline)) {
        copy_all(j < XC ? rx : rw,
                 (uint32_t)(uintptr_t)((lds_char *)smem + stage * T::STAGE +
                                       (j < XC ? ldx + j * 1024 : ldw + (j - XC) * 1024)),
                 src[j]);
    };
    auto advance = [&]() __attribute__((always_inline)) {
        left -= KG;
        const uint64_t ax = (((uint64_t)rx[1] << 32) | rx[0]) + 128 * KG;
        const uint64_t aw = (((uint64_t)rw[1] << 32) | rw[0]) + 128 * KG;
        rx[0] = (uint32_t)ax; rx[1] = (uint32_t)(ax >> 32);
        rw[0] = (uint32_t)aw; rw[1] = (uint32_t)(aw >> 32);
        if (left <= 0) rx[2] = rw[2] = 0;
    };
    // This wave's operand of stage rows row0 .. +31: lane (r, g) reads unit 2*ch + g.
    auto frag = [&](int stage, int row0) __attribute__((always_inline)) {
        const int row = row0 + r;
        return *(const __attribute__((address_space(3))) bf16x8 *)(
            (lds_char *)smem + stage * T::STAGE + sub * T::SUB + row * 128 +
            16 * ((2 * ch + g) ^ ((row >> 1) & 7)));
    };

    f32x16 acc[NB][MB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[nb][mb] = splat16(0.f);
    bf16x8 a[2][NB], b[2][MB];

    const int nit = (nsteps + KG - 1) / KG;
#pragma unroll
    for (int i = 0; i < NS; ++i) {
#pragma unroll
        for (int j = 0; j < CPS; ++j) copy(i, j);
        advance();
    }
    wait_copies_but<(NS - 1) * CPS>();
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NB; ++i) a[0][i] = frag(0, TM + 32 * i);
#pragma unroll
    for (int i = 0; i < MB; ++i) b[0][i] = frag(0, 32 * i);

    // A step whose operands are in a[P], b[P], from stage st. The barrier certifies that the
    // next step's copies landed and that every wave holds this step's operands. The copies and the
    // next operands' reads are spread over the products.
    auto step = [&](auto P, int st) __attribute__((always_inline)) {
        constexpr int cur = decltype(P)::value;
        const int st1 = st + 1 == NS ? 0 : st + 1;
        __builtin_amdgcn_sched_barrier(0);
        wait_copies_but<(NS - 2) * CPS>();
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        constexpr int PROD = MB * NB, RD = MB + NB;
        int rd = 0, cp = 0;
#pragma unroll
        for (int pr = 0; pr < PROD; ++pr) {
            // operand pr' of the next step in the order a[0], b[0], a[1], ...; the share of
            // this product of the step's reads, then of its copies
#pragma unroll
            for (; rd < (pr + 1) * RD / PROD; ++rd) {
                const int i = rd >> 1;
                if (MB == NB ? (rd & 1) == 0 : rd < NB) a[cur ^ 1][MB == NB ? i : rd] = frag(st1, TM + 32 * (MB == NB ? i : rd));
                else b[cur ^ 1][MB == NB ? i : rd - NB] = frag(st1, 32 * (MB == NB ? i : rd - NB));
            }
            acc[pr / MB][pr % MB] = mfma32(a[cur][pr / MB], b[cur][pr % MB], acc[pr / MB][pr % MB]);
#pragma unroll
            for (; cp < (pr + 1) * CPS / PROD; ++cp) copy(st, cp);
            __builtin_amdgcn_sched_barrier(0);
        }
        advance();
    };
    int st = 0, it = 0;
    auto next = [&]() __attribute__((always_inline)) { st = st + 1 == NS ? 0 : st + 1; };
    for (; it + 1 < nit; it += 2) {
        step(std::integral_constant<int, 0>{}, st);
        next();
        step(std::integral_constant<int, 1>{}, st);
        next();
    }
    if (it < nit) step(std::integral_constant<int, 0>{}, st);
    wait_copies();

    // ---- the waves' sums meet, and the tile leaves ----------------------------------------
    // A round stores RB blocks of every wave; then 16-row halves of the blocks are dealt to
    // the waves: lane (row 16*half + lane/4, column unit lane%4) adds the waves' eight columns
    // in wave order and holds 16 contiguous bytes of y.
    lds_char *X = (lds_char *)smem;
    lds_float *red = (lds_float *)(X + T::XCHG);
    const int q4 = lane & 3;
#pragma unroll
    for (int r0 = 0; r0 < T::BLOCKS; r0 += T::RB) {
        __syncthreads();                               // the ring (or the last round) is read
#pragma unroll
        for (int k = 0; k < T::RB; ++k) {
            const f32x16 &c = acc[(r0 + k) / MB][(r0 + k) % MB];
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4)
                *(lds_f32x4 *)(X + (wave * T::RB + k) * T::BLOCK + i4 * T::PLANE + lane * 16) =
                    f32x4{c[4 * i4], c[4 * i4 + 1], c[4 * i4 + 2], c[4 * i4 + 3]};
        }
        __syncthreads();
        for (int u = wave; u < 2 * T::RB; u += WAVES) {
            const int k = u >> 1, nb = (r0 + k) / MB, mb = (r0 + k) % MB;
            const int row = 16 * (u & 1) + (lane >> 2);
            f32x4 lo = {0.f, 0.f, 0.f, 0.f}, hi = lo;
#pragma unroll
            for (int w = 0; w < WAVES; ++w) {
                const lds_char *s = X + (w * T::RB + k) * T::BLOCK + q4 * T::PLANE + row * 16;
                const f32x4 l = *(const lds_f32x4 *)s, h = *(const lds_f32x4 *)(s + 512);
                if (w == 0) { lo = l; hi = h; }
                else { lo += l; hi += h; }
            }
            const int m = m0 + 32 * mb + row, n = n0 + 32 * nb + 8 * q4;
            u32x4 v = {pack_bf2(lo[0], lo[1]), pack_bf2(lo[2], lo[3]), pack_bf2(hi[0], hi[1]),
                       pack_bf2(hi[2], hi[3])};
            if (p.bias && n < p.N) {
                // (8-byte aligned; N is a multiple of 8: the unit is inside or outside)
                const u32x2 b0 = *(const u32x2 *)((const bf16 *)p.bias + n);
                const u32x2 b1 = *(const u32x2 *)((const bf16 *)p.bias + n + 4);
                const u32x4 bv = {b0[0], b0[1], b1[0], b1[1]};
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    v[e] = pack_bf2(bf_lo(v[e]) + bf_lo(bv[e]), bf_hi(v[e]) + bf_hi(bv[e]));
            }
            if (m < p.M && n < p.N) {
                // y is 8-byte aligned, with rows a multiple of 8 bytes apart
                typedef u32x4 u32x4_a8 __attribute__((aligned(8)));
                *(u32x4_a8 *)((bf16 *)p.y + (int64_t)m * p.y_rs + n) = v;
            }
            if (p.sumsq) {
                float sum = 0.f;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    sum += bf_lo(v[e]) * bf_lo(v[e]);
                    sum += bf_hi(v[e]) * bf_hi(v[e]);
                }
                sum += __shfl_xor(sum, 1, 64);
                sum += __shfl_xor(sum, 2, 64);
                if (q4 == 0) red[nb * TM + 32 * mb + row] = sum;
            }
        }
    }
    if (!p.sumsq) return;
    __syncthreads();
    if (tid < TM && m0 + tid < p.M) {
        float sum = red[tid];
#pragma unroll
        for (int nb = 1; nb < NB; ++nb) sum += red[nb * TM + tid];
        // the only column tile holds the block's sum; else linear_stat_kernel adds the tiles'
        float *dst = p.tiles_n == 1 ? p.sumsq + (int64_t)(m0 + tid) * p.ss_rs
                                    : p.part + (int64_t)(m0 + tid) * p.tiles_n + tn;
        *dst = sum;
    }
}

// Sums of squares over 256 columns from those of the column tiles (`per` tiles each, added in
// order). One thread per (row, block).
__global__ __launch_bounds__(256) void linear_stat_kernel(const LinearGroup grp, int per) {
    int which = 0;
#pragma unroll
    for (int i = 1; i < kLinearGroup; ++i) which += (int)blockIdx.x >= grp.stat_first[i] ? 1 : 0;
    const LinearParams &p = grp.p[which];
    const int blocks = (p.N + 255) / 256;
    const int64_t i = (int64_t)((int)blockIdx.x - grp.stat_first[which]) * 256 + threadIdx.x;
    if (i >= (int64_t)p.M * blocks) return;
    const int m = (int)(i / blocks), j = (int)(i % blocks);
    const float *src = p.part + (int64_t)m * p.tiles_n;
    float sum = 0.f;
    for (int t = j * per; t < min((j + 1) * per, p.tiles_n); ++t) sum += src[t];
    p.sumsq[(int64_t)m * p.ss_rs + j] = sum;
}

template <int MB, int NB, int KG>
int launch_ks(const LinearParams *p, int n, hipStream_t st) {
    using T = KsTile<MB, NB, KG>;
    LinearGroup grp{};
    grp.n = n;
    int64_t grid = 0, stat = 0;
    for (int i = 0; i < kLinearGroup; ++i) {
        grp.first[i] = (int32_t)grid;
        grp.stat_first[i] = (int32_t)stat;
        if (i >= n) continue;                        // (past the grid: chosen by no workgroup)
        LinearParams &q = grp.p[i] = p[i];
        q.tiles_m = (q.M + T::TM - 1) / T::TM;
        q.tiles_n = (q.N + T::TN - 1) / T::TN;
        grid += (int64_t)q.tiles_m * q.tiles_n;
        if (q.sumsq && q.tiles_n > 1) stat += ((int64_t)q.M * ((q.N + 255) / 256) + 255) / 256;
        if (grid > 0x7fffffff || stat > 0x7fffffff) return (int)hipErrorInvalidValue;
    }
    grp.first[kLinearGroup] = (int32_t)grid;
    grp.stat_first[kLinearGroup] = (int32_t)stat;
    const dim3 g((unsigned)grid), b(256 * KG);
    if (n > 1) hipLaunchKernelGGL((linear_ks_kernel<MB, NB, KG, true>), g, b, 0, st, grp);
    else hipLaunchKernelGGL((linear_ks_kernel<MB, NB, KG, false>), g, b, 0, st, grp);
    if (stat > 0)
        hipLaunchKernelGGL(linear_stat_kernel, dim3((unsigned)stat), dim3(256), 0, st, grp, 256 / T::TN);
    return (int)hipGetLastError();
}

}  // namespace

int launch_linear_ks(const LinearParams *p, int n, int tile, void *stream) {
    hipStream_t st = (hipStream_t)stream;
    switch (tile) {
    case kLinearKs128: return launch_ks<4, 4, 1>(p, n, st);
    case kLinearKs64: return launch_ks<2, 2, 2>(p, n, st);
    case kLinearKs64x32: return launch_ks<2, 1, 2>(p, n, st);
    case kLinearKs32: return launch_ks<1, 1, 2>(p, n, st);
    }
    return (int)hipErrorInvalidValue;
}

}  // namespace ltx
