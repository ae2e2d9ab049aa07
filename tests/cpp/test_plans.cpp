// Plans and routes of the C ABI on the host: ltx_attn_abi.cpp compiled into this program with
// launchers that record what they are given (nothing is launched, no HIP library is linked).
//
// Gemma: for a sweep of prompt lengths, head dims, windows, paddings and batches, every query
// block's ranges cover its key blocks, at most kGemmaMaxChunks of them, and the partials they
// write lie inside the workspace that the call asked for, apart from one another.
//
// Projections: which kernel a call takes, and the group call's contract: everything is checked
// before anything is launched, at most kLinearGroup small independent projections of one workspace
// in one launch, with their column sums apart inside it, everything else one by one in order.
#include <cstdio>
#include <cstdint>
#include <string>
#include <vector>

#include "../../ltx-2.5-swift_amd/csrc/ltx_attn_abi.cpp"

static int failures = 0, checks = 0;
static std::string where;
#define EXPECT(cond)                                                                         \
    do {                                                                                     \
        ++checks;                                                                            \
        if (!(cond) && ++failures <= 20)                                                     \
            std::printf("FAIL line %d [%s]: %s\n", __LINE__, where.c_str(), #cond);          \
    } while (0)

// ---- the HIP runtime and the launchers ------------------------------------------------------
static int g_cus = 256;                  // CUs of "the device"
static ltx::GemmaAttnParams g_gemma;
static int g_gemma_launches = 0;
struct LinearLaunch {
    std::vector<ltx::LinearParams> p;    // one, or a group's
    int tile;                            // of linear_ks.hip, or 0 for linear_gemm.hip
};
static std::vector<LinearLaunch> g_linear;

extern "C" {
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = g_cus; return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return ""; }
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *, int) { return hipErrorInvalidDevice; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
}
namespace ltx {
int launch_fmha(const FmhaParams &, int, int, void *) { return 0; }
int launch_fmha_short(const FmhaParams &, int, void *) { return 0; }
int launch_fmha_splitk(const FmhaParams &, int, void *) { return 0; }
int launch_prep(const PrepParams &, int, void *) { return 0; }
int launch_prep2(const PrepParams &, const PrepParams &, int, void *) { return 0; }
int launch_combine(const CombineParams &, int, void *) { return 0; }
int launch_passthrough(const PassParams &, int, void *) { return 0; }
int launch_linear(const LinearParams &p, void *) {
    g_linear.push_back({{p}, 0});
    return 0;
}
int launch_linear_ks(const LinearParams *p, int n, int tile, void *) {
    g_linear.push_back({std::vector<LinearParams>(p, p + n), tile});
    return 0;
}
int64_t linear_part_bytes(int64_t tiles, int splits) { return tiles * splits * (256 << 10); }
int launch_gemma_prep(const GemmaPrepParams &, int, void *) { return 0; }
int launch_gemma_attn(const GemmaAttnParams &p, int, void *) {
    g_gemma = p;
    ++g_gemma_launches;
    return 0;
}
int gemma_queries_per_workgroup() { return 128; }
}  // namespace ltx

// A distinct address per buffer, never read.
static void *fake(uintptr_t i) { return reinterpret_cast<void *>((uintptr_t)0x7f0000000000ull + (i << 36)); }

// ---- Gemma ------------------------------------------------------------------------------------
struct GemmaCall {
    ltx_gemma_attn_args a{};
    int32_t fv[ltx::kMaxBatch] = {};
    GemmaCall(int B, int T, int D, int window, std::vector<int> first) {
        a.B = B; a.T = T; a.D = D; a.Hq = 16; a.Hkv = D == 512 ? 1 : 8;
        a.q = fake(1); a.k = fake(2); a.v = fake(3);
        a.q_rs = (int64_t)a.Hq * D; a.k_rs = a.v_rs = (int64_t)a.Hkv * D;
        a.q_bs = T * a.q_rs; a.k_bs = a.v_bs = T * a.k_rs;
        a.q_norm_w = fake(4); a.k_norm_w = fake(5);
        a.eps = 1e-6f; a.scale = 1.0f;
        a.cos = (const float *)fake(6); a.sin = (const float *)fake(7);
        a.window = window;
        for (int b = 0; b < B; ++b) fv[b] = first[b];
        a.first_valid = fv;
        a.out = (float *)fake(8);
        a.o_rs = a.q_rs; a.o_bs = a.q_bs;
        a.workspace = fake(9);
        where = "B" + std::to_string(B) + " T" + std::to_string(T) + " D" + std::to_string(D) +
                " window " + std::to_string(window) + " first valid " + std::to_string(first[0]);
    }
};

// The recorded launch against the arguments: ranges and partials.
static void check_gemma_launch(const GemmaCall &c) {
    const ltx::GemmaAttnParams &p = g_gemma;
    const int qwg = 128, nkb = (c.a.T + 31) / 32;
    EXPECT(p.chunk >= 1 && p.nch_max >= 1 && p.nch_max <= ltx::kGemmaMaxChunks);
    EXPECT(p.chunk * p.nch_max >= nkb);
    // the kernel without key ranges only where no query block has a second one; a plan that splits
    // a short prompt goes to the kernel that has them
    EXPECT(!ltx::gemma_short(c.a.D, c.a.T, 2));
    if (ltx::gemma_short(c.a.D, c.a.T, p.nch_max)) {
        EXPECT(c.a.D == 512 && c.a.T <= 512);
        for (int b = 0; b < c.a.B; ++b) EXPECT(p.part_chunks[b] == 0 && p.chunk >= nkb);
    } else {
        EXPECT(c.a.D != 512 || c.a.T > 512);
    }
    const char *end = (const char *)c.a.workspace + c.a.workspace_bytes;
    int64_t row = 0;                         // where the batch rows' partials may start
    for (int b = 0; b < c.a.B; ++b) {
        int64_t ranges = 0;
        for (int q0 = 0; q0 < c.a.T; q0 += qwg) {
            const int len = ltx::gemma_key_hi(c.a.T, q0, qwg, c.fv[b]) -
                            ltx::gemma_key_lo(q0, c.fv[b], c.a.window) + 1;
            const int n = ltx::gemma_ranges(c.a.T, c.a.window, p.chunk, q0, qwg, c.fv[b]);
            EXPECT(len >= 1 && n == (len + p.chunk - 1) / p.chunk && n <= p.nch_max);
            if (n > 1) ranges += n;
        }
        EXPECT(p.part_chunks[b] == ranges);
        EXPECT(p.part_row0[b] >= row);
        row = p.part_row0[b] + c.a.Hq * ranges * qwg;
        if (ranges) {
            const char *o = (const char *)p.part_o, *ml = (const char *)p.part_ml;
            EXPECT(o >= (const char *)p.vt + 2 * (size_t)c.a.B * c.a.Hkv * nkb * 32 * c.a.D);
            EXPECT(o + row * c.a.D * 4 <= ml);
            EXPECT(ml + row * 2 * 4 <= end);
        }
    }
}

template <class F>
static void gemma_sweep(F each) {
    std::vector<int> lengths;
    for (int T = 4; T <= 1700; T += 4) lengths.push_back(T);
    for (int T : {2044, 2048, 3000, 4096, 4160, 8192}) lengths.push_back(T);
    for (int D : {256, 512})
        for (int T : lengths)
            for (int window : {0, 1, 17, 512, 1024})
                for (int pad : {0, 1, T / 3, T - T / 8, T - 1, T}) {
                    each(1, T, D, window, std::vector<int>{pad});
                    if (T % 100 < 4) each(2, T, D, window, std::vector<int>{pad, T / 2});
                }
}

// A prompt that fills its tokens with padding but for the last `real` runs as two ranges of half of
// its key blocks, whatever their number: 16 heads x 8 query blocks are half of the CUs.
static void test_gemma_padded_prompts_split() {
    for (int real = 1; real <= 400; ++real) {
        GemmaCall c(1, 1024, 512, 0, {1024 - real});
        c.a.workspace_bytes = ltx_gemma_attn_workspace_bytes(&c.a);
        EXPECT(ltx_gemma_attn_fwd(&c.a, nullptr) == LTX_ATTN_OK);
        EXPECT(g_gemma.nch_max == 2 && g_gemma.chunk == 16);
        // the size asked for before: accepted, with the ranges that it holds
        const size_t before = 2 * 1024 * 512 * (16 + 1 + 1) +
            (512 * 4 + 2 * 4) * (size_t)gemma_ranges_of(&c.a, 64, 16, nullptr, nullptr).rows;
        EXPECT(before <= c.a.workspace_bytes);
        c.a.workspace_bytes = before;
        EXPECT(ltx_gemma_attn_fwd(&c.a, nullptr) == LTX_ATTN_OK);
        check_gemma_launch(c);
    }
}

// The calls of the GPU tests that mean to merge ranges (test_gpu_gemma.py) do.
static void test_gemma_ranges_of_few_heads() {
    struct Case { int B, T, D, window, Hq; std::vector<int> pad; int ranges; };
    for (const Case &k : {Case{2, 2052, 512, 0, 2, {1026, 100}, 5}, Case{1, 2052, 512, 0, 2, {0}, 5},
                          Case{2, 3076, 256, 1500, 1, {1538, 100}, 6},
                          Case{1, 8324, 256, 3000, 1, {100}, 6}}) {
        GemmaCall c(k.B, k.T, k.D, k.window, k.pad);
        c.a.Hq = k.Hq; c.a.Hkv = 1;
        c.a.q_rs = c.a.o_rs = k.Hq * k.D; c.a.k_rs = c.a.v_rs = k.D;
        c.a.q_bs = c.a.o_bs = k.T * c.a.q_rs; c.a.k_bs = c.a.v_bs = k.T * c.a.k_rs;
        c.a.workspace_bytes = ltx_gemma_attn_workspace_bytes(&c.a);
        EXPECT(c.a.workspace_bytes <= (size_t)256 << 20);
        EXPECT(ltx_gemma_attn_fwd(&c.a, nullptr) == LTX_ATTN_OK && g_gemma.nch_max == k.ranges);
        EXPECT(k.B == 1 || g_gemma.part_chunks[0] != g_gemma.part_chunks[1]);
        check_gemma_launch(c);
    }
}

// On a part with other CUs a call runs the ranges that suit them, where its workspace holds them.
static void test_gemma_plan_for_other_parts() {
    GemmaCall c(1, 1024, 512, 0, {0});       // 128 query blocks: half of 256 CUs, all of 128
    c.a.workspace_bytes = ltx_gemma_attn_workspace_bytes(&c.a);
    EXPECT(ltx_gemma_attn_fwd(&c.a, nullptr) == LTX_ATTN_OK && g_gemma.nch_max == 2);
    const size_t need = c.a.workspace_bytes;
    for (int cus : {32, 64, 80, 128, 304}) {
        g_cus = cus;
        g_device_cus[0] = 0;                 // (kept from the first query)
        where = std::to_string(cus) + " CUs";
        EXPECT(ltx_gemma_attn_workspace_bytes(&c.a) == need);
        EXPECT(ltx_gemma_attn_fwd(&c.a, nullptr) == LTX_ATTN_OK);
        EXPECT(g_gemma.nch_max == (cus < 128 ? 1 : 2));
        check_gemma_launch(c);
        gemma_sweep([](int B, int T, int D, int window, std::vector<int> pad) {
            GemmaCall d(B, T, D, window, pad);
            d.a.workspace_bytes = ltx_gemma_attn_workspace_bytes(&d.a);
            EXPECT(ltx_gemma_attn_fwd(&d.a, nullptr) == LTX_ATTN_OK);
            check_gemma_launch(d);
        });
    }
    g_cus = 256;
    g_device_cus[0] = 0;
}

static void test_gemma_partials_fit() {
    gemma_sweep([](int B, int T, int D, int window, std::vector<int> pad) {
        GemmaCall c(B, T, D, window, pad);
        c.a.workspace_bytes = ltx_gemma_attn_workspace_bytes(&c.a);
        EXPECT(c.a.workspace_bytes > 0);
        EXPECT(ltx_gemma_attn_fwd(&c.a, nullptr) == LTX_ATTN_OK);
        check_gemma_launch(c);
        c.a.workspace_bytes -= 1;
        const int before = g_gemma_launches;
        if (ltx_gemma_attn_fwd(&c.a, nullptr) == LTX_ATTN_OK) check_gemma_launch(c);
        else EXPECT(g_gemma_launches == before);
    });
}

// ---- projections ------------------------------------------------------------------------------
static ltx_linear_args linear(int id, int M, int N, int K, bool sumsq, size_t ws = 64 << 20) {
    ltx_linear_args a{};
    a.M = M; a.N = N; a.K = K;
    a.x = fake(20 + 8 * id); a.w = fake(21 + 8 * id); a.bias = fake(22 + 8 * id); a.y = fake(23 + 8 * id);
    a.x_rs = a.w_rs = K; a.y_rs = N;
    if (sumsq) {
        a.sumsq = (float *)fake(24 + 8 * id);
        a.sumsq_rs = ltx_linear_sumsq_blocks(N);
    }
    a.workspace = ws ? fake(9) : nullptr;
    a.workspace_bytes = ws;
    return a;
}

// The route of a call: a tile of linear_ks.hip, or linear_gemm.hip's whole tiles, tail ranges behind
// whole rounds, or ranges alone.
enum Route { kWhole, kTail, kRanges, kKs };
static Route route(const ltx_linear_args &a) {
    g_linear.clear();
    where = std::to_string(a.M) + " x " + std::to_string(a.N) + " x " + std::to_string(a.K);
    EXPECT(ltx_linear(&a, nullptr) == LTX_ATTN_OK && g_linear.size() == 1);
    const ltx::LinearParams &p = g_linear[0].p[0];
    return g_linear[0].tile ? kKs : p.splits <= 1 ? kWhole : p.n_full > 0 ? kTail : kRanges;
}

static void test_linear_routes() {
    auto at = [](int M, int N, int K, int groups = 0, size_t ws = 64 << 20) {
        ltx_linear_args a = linear(0, M, N, K, true, ws);
        a.resident_groups = groups;
        return route(a);
    };
    // what the GPU tests of each route call (test_gpu_linear.py)
    EXPECT(at(12480, 4096, 4096) == kTail);
    EXPECT(at(3000, 1024, 512, 32) == kTail);
    EXPECT(at(300, 12288, 4096) == kRanges);
    EXPECT(at(512, 12288, 4096) == kRanges);
    EXPECT(at(700, 1000, 4096, 150) == kRanges);
    EXPECT(at(700, 6144, 4096) == kRanges);
    for (auto s : {std::pair<int, int>{13, 2048}, {12480, 32}, {200, 4096}, {1024, 4096}})
        EXPECT(at(s.first, s.second, 2048) == kKs);
    EXPECT(at(3120, 4096, 4096) == kWhole);
    EXPECT(at(12480, 32, 4096, 0, 0) == kWhole);          // no workspace: whole tiles
    EXPECT(at(12480, 32, 4096, 0, 1 << 20) == kWhole);    // nor with less than the ranges' partials
    // another part's plan where the workspace holds it
    g_cus = 128;
    g_device_cus[0] = 0;                     // (kept from the first query)
    EXPECT(at(12480, 4096, 4096) == kTail && g_linear[0].p[0].n_full == 768);
    g_cus = 256;
    g_device_cus[0] = 0;
}

static void test_linear_group() {
    using Calls = std::vector<ltx_linear_args>;
    auto run = [](const Calls &c) {
        g_linear.clear();
        return ltx_linear_group(c.data(), (int32_t)c.size(), nullptr);
    };
    auto module = [](size_t ws = 64 << 20) {
        return Calls{linear(0, 126, 2048, 2048, false, ws), linear(1, 126, 32, 2048, false, ws),
                     linear(2, 126, 2048, 2048, true, ws), linear(3, 126, 2048, 2048, true, ws)};
    };
    where = "group";
    EXPECT(ltx_linear_group(nullptr, 0, nullptr) == LTX_ATTN_OK);
    EXPECT(ltx_linear_group(nullptr, 2, nullptr) == LTX_ATTN_EINVAL);
    EXPECT(ltx_linear_group(nullptr, -1, nullptr) == LTX_ATTN_EINVAL);

    // one launch, in the caller's order, the column sums apart and inside the workspace
    Calls c = module();
    EXPECT(run(c) == LTX_ATTN_OK && g_linear.size() == 1 && g_linear[0].p.size() == 4);
    const char *ws = (const char *)c[0].workspace, *used = ws;
    for (size_t i = 0; i < c.size() && i < g_linear[0].p.size(); ++i) {
        const ltx::LinearParams &p = g_linear[0].p[i];
        EXPECT(p.y == c[i].y && p.sumsq == c[i].sumsq);
        if (!p.sumsq) continue;
        EXPECT((const char *)p.part >= used && ((uintptr_t)p.part & 255) == 0);
        used = (const char *)p.part + (size_t)p.M * ((p.N + 31) / 32) * 4;   // the narrowest tiles
        EXPECT(used <= ws + c[i].workspace_bytes);
    }
    // a bad call in any place: nothing is launched
    for (size_t bad = 0; bad < 6; ++bad) {
        c = module();
        c.push_back(linear(4, 40, 64, 256, false));
        c.push_back(linear(5, 40, 64, 256, false));
        c[bad].K = 96;
        EXPECT(run(c) != LTX_ATTN_OK && g_linear.empty());
    }
    // one by one, in order: more than a launch takes, an empty or a large one among them, other
    // workspaces
    auto in_order = [&](const Calls &calls, size_t launches) {
        EXPECT(run(calls) == LTX_ATTN_OK && g_linear.size() == launches);
        size_t at = 0;
        for (const LinearLaunch &l : g_linear) {
            EXPECT(l.p.size() == 1);
            while (at < calls.size() && calls[at].M == 0) ++at;
            EXPECT(at < calls.size() && l.p[0].y == calls[at].y);
            ++at;
        }
    };
    c = module();
    c.push_back(linear(4, 126, 2048, 2048, false));
    in_order(c, 5);
    c = module();
    c[1].M = 0;
    in_order(c, 3);
    c = module();
    c[0] = linear(0, 12480, 4096, 4096, false);
    in_order(c, 4);
    c = module();
    c[3].workspace = fake(10);
    in_order(c, 4);
    c = module(0);
    in_order(c, 4);
    // less than a call's ranges would need: it keeps whole tiles, so the others run by themselves too.
    // (A workspace that holds the ranges of each call, 8 bytes and more per element of its y, holds
    // the column sums of four, an eighth of a byte each.)
    c = module();
    c[3].workspace_bytes = 1 << 20;
    in_order(c, 4);
    // one by one: a call that reads or writes what another one writes, its workspace included
    auto apart = [&](auto change) {
        Calls d = module();
        change(d);
        in_order(d, d.size());
    };
    apart([](Calls &d) { d[2].x = d[0].y; });
    apart([](Calls &d) { d[0].x = d[2].y; });
    apart([](Calls &d) { d[2].w = d[0].y; });
    apart([](Calls &d) { d[1].bias = d[0].y; });
    apart([](Calls &d) { d[3].y = (char *)d[2].y + 126 * 2048 * 2 - 8; });
    apart([](Calls &d) { d[3].sumsq = d[2].sumsq; });
    apart([](Calls &d) { d[3].sumsq = (float *)d[0].y; });
    apart([](Calls &d) { d[3].bias = (char *)d[3].workspace + (1 << 20); });
    // y slices interleaved in one buffer: their spans meet, so they run one by one
    apart([](Calls &d) {
        for (int i : {0, 2, 3}) { d[i].y = (char *)fake(23) + 4096 * i; d[i].y_rs = 4 * 2048; }
    });
}

int main() {
    test_gemma_partials_fit();
    test_gemma_padded_prompts_split();
    test_gemma_ranges_of_few_heads();
    test_gemma_plan_for_other_parts();
    test_linear_routes();
    test_linear_group();
    std::printf("%d checks, %d failure(s)\n", checks, failures);
    return failures != 0;
}
