// Tile and split selection of the tiled linear layers (kernels: linear_gemm_kernels.hpp), and their
// f32 instantiations.
#include "linear_gemm_kernels.hpp"

#include <algorithm>

namespace llaisys::kernels {

namespace {

constexpr int kCUs = 256;
constexpr size_t kPartBytes = size_t(48) << 20; // most partial sums a launch keeps

// A launch: the tile (16-bit types), its extent, k per stage, and the split of K.
struct Plan {
    GemmTile tile;
    int bw, bx, ks;
    int splits, per;
};

size_t ceilDiv(size_t a, size_t b) { return (a + b - 1) / b; }

void setSplits(Plan &p, const LinearCall &c, size_t want) {
    const size_t nk = ceilDiv(c.K, p.ks), n = std::max<size_t>(1, std::min(want, nk));
    p.per = int(ceilDiv(nk, n));
    p.splits = int(ceilDiv(nk, p.per));
}

// setSplits for the 16-bit tiles, of stages of 64 k: the dense 192 x 256 tile takes the same ranges of K
// in stages of 32
void splitStages(Plan &p, const LinearCall &c, size_t want) {
    setSplits(p, c, want);
    if (p.tile == GemmTile::k192x256 && !c.scale) p.ks = 32, p.per *= 2;
}

// Splits that bring the blocks to `blocks`, each with at least `least` stages.  The outputs N are
// counted once with swiglu too, so that it sums as the two separate linears do.
void fillSplits(Plan &p, const LinearCall &c, size_t blocks, size_t least) {
    const size_t tiles = ceilDiv(c.N, p.bw) * ceilDiv(c.rows, p.bx);
    const size_t cap = kPartBytes / (c.rows * 2 * c.N * sizeof(float));
    setSplits(p, c, std::min({blocks / tiles, ceilDiv(c.K, p.ks) / least, cap}));
}

// f32: tiles of 64 weight rows x 32 or 64 rows, 64 k per stage shared by two (64 rows) or four waves
// per tile quarter, split until every CU has a block.  Bound by the f32 MFMA rate (154 TFLOP/s on
// a large product, 93 reached here at 128 rows): one decoder layer of 128 tokens (hidden 1536,
// intermediate 8960) 30.2 ms with one thread per output -> 0.187 ms.  Against tiles of 128 rows, whose
// blocks number 3.3 per CU at two together: gate / up + swiglu 97 -> 77 us, down 48 -> 39 us, 1536 ->
// 1536 23 -> 13.4 us.
Plan planF32(const LinearCall &c) {
    Plan p{GemmTile::k64x64, 64, c.rows <= 32 ? 32 : 64, 64, 1, 0};
    fillSplits(p, c, kCUs, 3);
    // unsplit with up to 8 blocks per CU: half as many weight rows per block, for a finer last round
    // (128 rows, 1536 -> 2 x 8960: 2.2 blocks per CU 94 us, 4.4 of half the size 77 us)
    const size_t tiles = ceilDiv(c.swiglu ? 2 * c.N : c.N, 64) * ceilDiv(c.rows, p.bx);
    if (p.splits == 1 && tiles <= 8 * kCUs) p.bw = 32;
    return p;
}

// Measured time of a 64-k stage of a tile, in ns, with 1, 2 or 3 of its blocks on a CU (`most`:
// how many run together; more run after one another).  From full launches over 96 to 4000 rows of
// 1536 -> 2 x 8960, 8960 -> 1536 and 1536 -> 1536; the small tiles wait for their loads when
// alone, the large ones run at 750 to 870 TFLOP/s.
struct TileTime {
    GemmTile tile;
    int bw, bx, most;
    int ns[3];
};
constexpr TileTime kDense[] = {
    {GemmTile::k64x64, 64, 64, 3, {360, 450, 640}},      {GemmTile::k128x64, 128, 64, 3, {580, 700, 1100}},
    {GemmTile::k128x128, 128, 128, 2, {800, 1300}},      {GemmTile::k192x128, 192, 128, 1, {950}},
    {GemmTile::k192x256, 192, 256, 1, {1700}},
};
constexpr TileTime kCodes[] = {
    {GemmTile::k64x64, 64, 64, 3, {450, 650, 770}},      {GemmTile::k128x64, 128, 64, 3, {650, 800, 1130}},
    {GemmTile::k128x128, 128, 128, 3, {900, 1400, 1950}}, {GemmTile::k192x128, 192, 128, 1, {1150}},
    {GemmTile::k256x128, 256, 128, 2, {1350, 2450}},     {GemmTile::k192x256, 192, 256, 1, {1900}},
};

// Expected ns of a launch over `n` weight rows split `splits` times
double launchTime(const TileTime &t, const LinearCall &c, size_t n, size_t splits) {
    const size_t on_cu = ceilDiv(ceilDiv(n, t.bw) * ceilDiv(c.rows, t.bx) * splits, kCUs);
    const double stage = double(on_cu / t.most) * t.ns[t.most - 1] + (on_cu % t.most ? t.ns[on_cu % t.most - 1] : 0);
    double ns = double(ceilDiv(ceilDiv(c.K, 64), splits)) * stage;
    // the partial sums written and read (about 5 TB/s), and one more launch
    if (splits > 1) ns += 3500 + 8.0 * double(splits * c.rows * n) / 5000;
    return ns;
}

// 16-bit types.  Up to 64 rows are bound by the weight's bytes in flight: 64 x 64 tiles with 128 k
// per stage, split until every CU has a block (37 rows, bf16: 1536 -> 2 x 8960 with swiglu 38 us in
// three launches -> 14.6 us, 8960 -> 1536 83 -> 12.1 us; W8A16 16.3 and 12.3 us).  More rows: the
// tile and split with the least expected time.  The split is that of the dense tiles for N outputs
// whatever the weight's type and whether swiglu follows, so that W8A16 with unit scales, and gate
// and up computed apart, sum in the same order.
Plan plan16(const LinearCall &c) {
    Plan p{GemmTile::k64x64Deep, 64, 64, 128, 1, 0};
    if (c.rows <= 64) {
        fillSplits(p, c, kCUs, 2);
        return p;
    }
    const size_t nk = ceilDiv(c.K, 64), cap = kPartBytes / (c.rows * 2 * c.N * sizeof(float));
    size_t splits = 1;
    double best = 1e30;
    for (const TileTime &t : kDense)
        for (size_t n = 1; n <= 16 && (n == 1 || (n <= cap && n <= nk / 4)); ++n) {
            const double ns = launchTime(t, c, c.N, n);
            if (ns < best) best = ns, splits = n;
        }
    best = 1e30;
    const size_t nw = c.swiglu ? 2 * c.N : c.N;
    const auto pick = [&](const TileTime &t) {
        const double ns = launchTime(t, c, nw, splits);
        if (ns < best) {
            best = ns;
            p = Plan{t.tile, t.bw, t.bx, 64, 1, 0};
        }
    };
    if (c.scale)
        for (const TileTime &t : kCodes) pick(t);
    else
        for (const TileTime &t : kDense) pick(t);
    splitStages(p, c, splits);
    return p;
}

Plan planOf(const LinearCall &c) { return c.dt == LLAISYS_DTYPE_F32 ? planF32(c) : plan16(c); }

// The partial sums of 2 N outputs with and without swiglu: where the scratch is short, gate / up in
// one launch and its halves apart go without a split alike.
size_t planBytes(const Plan &p, const LinearCall &c) {
    return p.splits > 1 ? size_t(p.splits) * c.rows * 2 * c.N * sizeof(float) : 0;
}

template <bool kSw>
void launchF32(const Plan &p, const GemmArgs &a, hipStream_t s) {
    if (p.bx == 32 && p.bw == 32)
        launchTile<F32, false, kSw, 32, 32, 1, 1, 4, 64, 3>(a, s);
    else if (p.bx == 32)
        launchTile<F32, false, kSw, 64, 32, 2, 1, 4, 64, 2>(a, s);
    else if (p.bw == 32)
        launchTile<F32, false, kSw, 32, 64, 1, 2, 2, 64, 2>(a, s);
    else
        launchTile<F32, false, kSw, 64, 64, 2, 2, 2, 64, 2>(a, s);
    if (a.part) launchReduce<F32, false, kSw>(a, s);
}

} // namespace

bool gemmTakes(const LinearCall &c) {
    const auto al = [](const void *p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    if (c.K == 0 || !al(c.x) || !al(c.w)) return false;
    if (c.dt == LLAISYS_DTYPE_F32) return !c.scale && c.rows > 1 && c.K % 4 == 0;
    return c.rows > 16 && c.K % (c.scale ? 16 : 8) == 0;
}

size_t gemmWorkspaceBytes(const LinearCall &c) { return planBytes(planOf(c), c); }

namespace {
void launchPlan(const Plan &p, const LinearCall &c, void *ws, hipStream_t s) {
    const size_t es = c.dt == LLAISYS_DTYPE_F32 ? 4 : 2;
    GemmArgs a{};
    a.out = c.out;
    a.x = c.x;
    a.w = c.w;
    a.scale = c.scale;
    a.bias = c.bias;
    a.part = p.splits > 1 ? static_cast<float *>(ws) : nullptr;
    a.M = int(c.rows);
    a.N = int(c.N);
    a.Nw = int(c.swiglu ? 2 * c.N : c.N);
    a.K = int(c.K);
    a.splits = p.splits;
    a.per = p.per;
    a.vec = c.N % 4 == 0 && reinterpret_cast<uintptr_t>(c.out) % (4 * es) == 0;
    if (c.dt == LLAISYS_DTYPE_BF16)
        gemmBf16(p.tile, a, c.swiglu, s);
    else if (c.dt == LLAISYS_DTYPE_F16)
        gemmF16(p.tile, a, c.swiglu, s);
    else
        c.swiglu ? launchF32<true>(p, a, s) : launchF32<false>(p, a, s);
}
} // namespace

void gemm(const LinearCall &c, void *ws, size_t ws_bytes, hipStream_t s) {
    if (c.rows == 0 || c.N == 0) return;
    Plan p = planOf(c);
    if (planBytes(p, c) > ws_bytes) setSplits(p, c, 1);
    launchPlan(p, c, ws, s);
}

extern "C" int llaisysTestLinearPlan(size_t rows, size_t K, size_t N, int int8, int swiglu, int dt, int plan[4]) {
    static const float one = 1.0f;
    const Plan p = planOf({nullptr, nullptr, nullptr, int8 ? &one : nullptr, nullptr, rows, K, N, swiglu != 0, llaisysDataType_t(dt)});
    plan[0] = int(p.tile);
    plan[1] = p.splits;
    plan[2] = p.per;
    plan[3] = p.ks;
    return 0;
}

extern "C" int llaisysTestLinearTile(void *out, const void *x, const void *w, const float *scale, const void *bias, size_t rows,
                                     size_t K, size_t N, int swiglu, int dt, int tile, size_t splits, void *ws, size_t ws_bytes) {
    const LinearCall c{out, x, w, scale, bias, rows, K, N, swiglu != 0, llaisysDataType_t(dt)};
    if (dt == LLAISYS_DTYPE_F32 || !gemmTakes(c) || splits == 0) return 0;
    Plan p{GemmTile(tile), 0, 0, 0, 1, 0};
    if (p.tile == GemmTile::k64x64Deep) p.ks = 128;
    if (scale)
        for (const TileTime &t : kCodes) p.ks = t.tile == p.tile ? 64 : p.ks;
    else
        for (const TileTime &t : kDense) p.ks = t.tile == p.tile ? 64 : p.ks;
    if (p.ks == 0) return 0;
    splitStages(p, c, splits);
    if (planBytes(p, c) > ws_bytes) return 0;
    launchPlan(p, c, ws, nullptr);
    return hipGetLastError() == hipSuccess && hipDeviceSynchronize() == hipSuccess ? p.splits : 0;
}

} // namespace llaisys::kernels
