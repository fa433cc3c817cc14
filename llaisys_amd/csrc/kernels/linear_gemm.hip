// Tiled linear layers for gfx950: several rows of activations against a weight, on MFMA.
//
// Semantics: reference src/ops/linear/cpu/linear_cpu.cpp:11-41 (dense) and the W8A16 rule of
// linear.hip; the sums run in f32 in the order of the tiles' k, split sums added in split order.
//
// Design.  A block owns a tile of BW weight rows x BX activation rows and one of `splits` ranges
// of K.  Per stage of 128 (or 256) bytes of a row, both operands move HBM -> LDS with
// global_load_lds_dwordx4 (1 KB per instruction, no register staging) through a ring of S
// stages, so S - 1 stages are in flight while the MFMAs run on one.  The load fills LDS
// contiguously, so rows cannot be padded: the lane that fills slot c of row r fetches chunk
// c ^ swz(r), and the operand reads apply the same XOR (no bank conflicts).  The MFMA computes
// out^T = w x^T, so a lane ends with 4 consecutive channels of one row.  INT8 codes stay codes
// in LDS and become exact bf16 / f16 values in registers.  f32 runs on v_mfma_f32_32x32x2_f32
// (f32 products and sums, 154 TFLOP/s on this card) with the same tiles: a 16-byte chunk is 4 k.
// When the tiles alone leave CUs idle, K is split over blocks; the partial sums go to the
// workspace in f32 and linearReduce adds them in split order, so results do not depend on
// which block ends first.
#include "common.hpp"
#include "launch.hpp"
#include "linear_common.hpp"
#include "linear_gemm.hpp"

#include <algorithm>
#include <type_traits>

namespace llaisys::kernels {

namespace {

using namespace lin;
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kXcds = 8; // accelerator complex dies, each with its own L2

struct GemmArgs {
    void *out;
    const void *x;
    const void *w;
    const float *scale;
    const void *bias;
    float *part;     // [splits][M][Nw] partial sums, or null: this launch writes out
    int M, N, Nw, K; // N outputs per row, Nw weight rows (2 N with swiglu)
    int splits, per; // K stages per split
    int vec;         // 4 consecutive outputs of a row are one aligned store
};

// A chunk of K past the row end is read from here: zeros add nothing to a sum.
__device__ const uint32_t kZeroChunk[4] = {0u, 0u, 0u, 0u};

// Slot XOR of row r when a row is C chunks of 16 bytes: 16 consecutive rows reading one logical
// chunk touch all 16 chunk positions of 256 bytes of LDS.
template <int C>
__device__ __forceinline__ int swz(int r) {
    return (r / (16 / C)) & (C - 1);
}

// D[m = 8 (i / 4) + 4 (l / 32) + i % 4][n = l % 32] += A[m = l % 32][..] B[..][n = l % 32] over
// one 16-byte chunk per lane: 16 k for the 16-bit types (8 per half wave), 8 k for f32 (4
// instructions of 2 k).
template <typename T>
__device__ __forceinline__ f32x16 mfmaChunk(const v4u &a, const v4u &b, f32x16 c) {
    if constexpr (std::is_same_v<T, BF16>) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    } else if constexpr (std::is_same_v<T, F16>) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            c = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a[e]), __uint_as_float(b[e]), c, 0, 0, 0);
        return c;
    }
}

// 4 consecutive channels n .. n + 3 of row m (all past N dropped)
template <typename T>
__device__ __forceinline__ void store4(void *out, int m, int n, int N, bool vec, const float (&v)[4]) {
    if (vec && n + 3 < N) {
        if constexpr (std::is_same_v<T, F32>) {
            *reinterpret_cast<v4u *>(static_cast<float *>(out) + size_t(m) * N + n) = Fmt<F32>::pack(v);
        } else {
            using C = std::conditional_t<std::is_same_v<T, BF16>, Bf16Cvt, F16Cvt>;
            const v2u p = {C::narrow(v[0]) | (C::narrow(v[1]) << 16), C::narrow(v[2]) | (C::narrow(v[3]) << 16)};
            *reinterpret_cast<v2u *>(static_cast<uint16_t *>(out) + size_t(m) * N + n) = p;
        }
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (n + e < N) Fmt<T>::put(out, size_t(m) * N + n + e, v[e]);
    }
}

// The finished sum of weight row n: scaled (INT8) and biased as linear_cpu.cpp:36-38
template <typename T, bool kInt8>
__device__ __forceinline__ float finish(const GemmArgs &a, float sum, int n) {
    if constexpr (kInt8) sum = a.scale[n] * sum;
    return a.bias ? sum + Fmt<T>::get(a.bias, n) : sum;
}

template <typename T, bool kInt8, bool kSw, int BW, int BX, int NWW, int NWX, int KS, int S>
__global__ void __launch_bounds__(NWW *NWX * 64)
    linearTile(GemmArgs a) {
    constexpr int kE = Fmt<T>::kBytes;
    constexpr int NWV = NWW * NWX;
    constexpr int WW = BW / NWW, WX = BX / NWX, TW = WW / 32, TX = WX / 32;
    constexpr int WB = KS * (kInt8 ? 1 : kE), XB = KS * kE; // bytes of a row per stage
    constexpr int WC = WB / 16, XC = XB / 16;               // chunks of a row per stage
    constexpr int kStageB = BW * WB + BX * XB;
    constexpr int WI = BW * WB / 1024, XI = BX * XB / 1024, kLoads = (WI + XI) / NWV;
    static_assert((WI + XI) % NWV == 0 && kLoads * (S - 2) < 64 && TW >= 1 && TX >= 1, "load split");
    static_assert(!kSw || TW % 2 == 0, "gate and up rows of a channel belong to one wave");
    __shared__ __align__(16) char lds[S * kStageB];
    const int tid = int(threadIdx.x), lane = tid % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    // Blocks go to the XCDs round-robin: give each XCD a contiguous range of tiles, row tiles
    // fastest, so that a weight tile stays in one L2 while the row tiles pass over it.
    const int nb = int(gridDim.x), b = int(blockIdx.x), xcd = b % kXcds;
    int v = xcd * (nb / kXcds) + min(xcd, nb % kXcds) + b / kXcds;
    const int nbx = (a.M + BX - 1) / BX;
    const int bx = v % nbx;
    v /= nbx;
    const int sp = v % a.splits, bw = v / a.splits;
    const int w0 = bw * BW, x0 = bx * BX;
    const int ww0 = (wave % NWW) * WW, wx0 = (wave / NWW) * WX;
    const int nk_all = (a.K + KS - 1) / KS;
    const int kt0 = sp * a.per, nk = min(nk_all - kt0, a.per);

    // weight row of tile row tr; with swiglu a wave's first half are gate rows, its second half
    // the up rows of the same channels
    const auto wrow = [&](int tr) {
        if constexpr (kSw) {
            const int in = tr % WW, ch = w0 / 2 + tr / WW * (WW / 2) + in % (WW / 2);
            return min(ch, a.N - 1) + (in < WW / 2 ? 0 : a.N);
        } else {
            return min(w0 + tr, a.N - 1);
        }
    };
    const char *src[kLoads];
    int left[kLoads]; // chunks of the row from the lane's first one on
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const int q = wave * kLoads + i;
        if (q < WI) {
            const int tr = q * (64 / WC) + lane / WC, c = (lane % WC) ^ swz<WC>(tr);
            src[i] = static_cast<const char *>(a.w) + size_t(wrow(tr)) * a.K * (kInt8 ? 1 : kE) + size_t(kt0) * WB + 16 * c;
            left[i] = a.K * (kInt8 ? 1 : kE) / 16 - kt0 * WC - c;
        } else {
            const int tr = (q - WI) * (64 / XC) + lane / XC, c = (lane % XC) ^ swz<XC>(tr);
            src[i] = static_cast<const char *>(a.x) + size_t(min(x0 + tr, a.M - 1)) * a.K * kE + size_t(kt0) * XB + 16 * c;
            left[i] = a.K * kE / 16 - kt0 * XC - c;
        }
    }
    const bool tail = a.K % KS != 0 && kt0 + nk == nk_all; // the last stage reaches past the rows
    const auto issue = [&](int kt) {
        char *dst = lds + (kt % S) * kStageB;
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const int q = wave * kLoads + i;
            const char *p = src[i] + size_t(kt) * (q < WI ? WB : XB);
            if (tail && kt == nk - 1 && kt * (q < WI ? WC : XC) >= left[i]) p = reinterpret_cast<const char *>(kZeroChunk);
            __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1))) *)(p),
                                             (void __attribute__((address_space(3))) *)(dst + q * 1024), 16, 0, 0);
        }
    };
    f32x16 acc[TW][TX];
#pragma unroll
    for (int i = 0; i < TW; ++i)
#pragma unroll
        for (int j = 0; j < TX; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
    const int r32 = lane % 32, h2 = lane / 32;
    // the lane's row base of each operand tile and its swizzle (32 i does not change the XOR)
    const int wsz = swz<WC>(ww0 + r32), xsz = swz<XC>(wx0 + r32);
    const int wbase = (ww0 + r32) * WB, xbase = BW * WB + (wx0 + r32) * XB;
#pragma unroll
    for (int st = 0; st < S - 1; ++st)
        if (st < nk) issue(st);
    for (int kt = 0; kt < nk; ++kt) {
        // this wave's loads of stage kt have landed (the stages after it may be in flight)
        if (kt + S - 2 < nk)
            waitVmcnt<kLoads * (S - 2)>();
        else
            waitVmcnt<0>();
        ldsBarrier(); // every wave's have; stage kt - 1 is no longer read
        if (kt + S - 1 < nk) issue(kt + S - 1);
        const char *tile = lds + (kt % S) * kStageB;
        // k order of a stage: 16-bit types, step st and half h: chunk 4 (st / 2) + 2 h + st % 2, so
        // that the 16 codes of an INT8 chunk serve two steps; f32: chunk 2 st + h
        constexpr int kSteps = XC / 2;
        if constexpr (kInt8) {
#pragma unroll
            for (int p = 0; p < kSteps / 2; ++p) {
                v4u ca[TW];
#pragma unroll
                for (int i = 0; i < TW; ++i)
                    ca[i] = *reinterpret_cast<const v4u *>(tile + wbase + 32 * i * WB + 16 * ((2 * p + h2) ^ wsz));
#pragma unroll
                for (int s2 = 0; s2 < 2; ++s2) {
                    v4u fb[TX];
#pragma unroll
                    for (int j = 0; j < TX; ++j)
                        fb[j] = *reinterpret_cast<const v4u *>(tile + xbase + 32 * j * XB + 16 * ((4 * p + 2 * h2 + s2) ^ xsz));
#pragma unroll
                    for (int i = 0; i < TW; ++i) {
                        const v4u fa = codesToT<T>(s2 ? v2u{ca[i].z, ca[i].w} : v2u{ca[i].x, ca[i].y});
#pragma unroll
                        for (int j = 0; j < TX; ++j) acc[i][j] = mfmaChunk<T>(fa, fb[j], acc[i][j]);
                    }
                }
            }
        } else {
#pragma unroll
            for (int st = 0; st < kSteps; ++st) {
                const int c = kE == 2 ? 4 * (st / 2) + 2 * h2 + st % 2 : 2 * st + h2;
                v4u fa[TW], fb[TX];
#pragma unroll
                for (int i = 0; i < TW; ++i) fa[i] = *reinterpret_cast<const v4u *>(tile + wbase + 32 * i * WB + 16 * (c ^ wsz));
#pragma unroll
                for (int j = 0; j < TX; ++j) fb[j] = *reinterpret_cast<const v4u *>(tile + xbase + 32 * j * XB + 16 * (c ^ xsz));
#pragma unroll
                for (int i = 0; i < TW; ++i)
#pragma unroll
                    for (int j = 0; j < TX; ++j) acc[i][j] = mfmaChunk<T>(fa[i], fb[j], acc[i][j]);
            }
        }
    }
    // D[8 q + 4 h + e][r32] of 32 x 32 tile (i, j): weight row 32 i + 8 q + 4 h + e of the wave's
    // rows, activation row 32 j + r32
    if (a.part) {
        float *part = a.part + size_t(sp) * a.M * a.Nw;
#pragma unroll
        for (int i = 0; i < TW; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                int n = w0 + ww0 + 32 * i + 8 * q + 4 * h2, top = a.N; // partial column and its end
                if constexpr (kSw) {
                    n = w0 / 2 + ww0 / 2 + 32 * (i % (TW / 2)) + 8 * q + 4 * h2 + (i < TW / 2 ? 0 : a.N);
                    top = i < TW / 2 ? a.N : a.Nw;
                }
#pragma unroll
                for (int j = 0; j < TX; ++j) {
                    const int m = x0 + wx0 + 32 * j + r32;
                    if (m >= a.M) continue;
                    float *p = part + size_t(m) * a.Nw + n;
                    if (a.N % 4 == 0 && n + 3 < top) {
                        *reinterpret_cast<f32x4 *>(p) = f32x4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (n + e < top) p[e] = acc[i][j][4 * q + e];
                    }
                }
            }
        return;
    }
    constexpr int TO = kSw ? TW / 2 : TW;
#pragma unroll
    for (int i = 0; i < TO; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int n = (kSw ? w0 / 2 + ww0 / 2 : w0 + ww0) + 32 * i + 8 * q + 4 * h2;
#pragma unroll
            for (int j = 0; j < TX; ++j) {
                const int m = x0 + wx0 + 32 * j + r32;
                if (m >= a.M) continue;
                float o[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int ne = min(n + e, a.N - 1);
                    o[e] = finish<T, kInt8>(a, acc[i][j][4 * q + e], ne);
                    if constexpr (kSw)
                        o[e] = SwigluOp::apply(Fmt<T>::round(o[e]), Fmt<T>::round(finish<T, kInt8>(a, acc[i + TO][j][4 * q + e], ne + a.N)));
                }
                store4<T>(a.out, m, n, a.N, a.vec, o);
            }
        }
}

// Sum of the splits' partials in split order, then what the tile kernel's epilogue does.  One
// thread per VEC consecutive outputs of a row.
template <typename T, bool kInt8, bool kSw, int VEC>
__global__ void __launch_bounds__(256)
    linearReduce(GemmArgs a) {
    const int per_row = (a.N + VEC - 1) / VEC;
    const size_t idx = size_t(blockIdx.x) * 256 + threadIdx.x;
    if (idx >= size_t(a.M) * per_row) return;
    const int m = int(idx / per_row), n = int(idx % per_row) * VEC;
    const size_t plane = size_t(a.M) * a.Nw;
    float o[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int h = 0; h < (kSw ? 2 : 1); ++h) {
        const float *p = a.part + size_t(m) * a.Nw + n + h * a.N;
        float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        constexpr int U = 8; // partials in flight
        for (int c = 0; c < a.splits; c += U) {
            f32x4 t[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const float *pu = p + size_t(min(c + u, a.splits - 1)) * plane;
                if constexpr (VEC == 4)
                    t[u] = *reinterpret_cast<const f32x4 *>(pu);
                else
                    t[u][0] = pu[0];
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (c + u < a.splits)
#pragma unroll
                    for (int e = 0; e < VEC; ++e) s[e] += t[u][e];
        }
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            const float y = finish<T, kInt8>(a, s[e], n + e + h * a.N);
            o[e] = h ? SwigluOp::apply(Fmt<T>::round(o[e]), Fmt<T>::round(y)) : y;
        }
    }
    if constexpr (VEC == 4)
        store4<T>(a.out, m, n, a.N, a.vec, o);
    else
        Fmt<T>::put(a.out, size_t(m) * a.N + n, o[0]);
}

// ---- launch ---------------------------------------------------------------------------------

// A tile shape and how often K is split over it.
struct Plan {
    int bw, bx, ks; // weight rows, activation rows, k per stage
    int splits, per;
};

constexpr size_t kPartBytes = size_t(48) << 20; // most partial sums a launch keeps

// K is split until about `blocks` blocks are in flight, each with at least `least` stages.  The
// outputs N are counted once with swiglu too, so that it sums as the two separate linears do.
void splitK(Plan &p, const LinearCall &c, int blocks, int least) {
    const size_t tiles = ((c.N + p.bw - 1) / p.bw) * ((c.rows + p.bx - 1) / p.bx);
    const int nk = int((c.K + p.ks - 1) / p.ks);
    const size_t cap = kPartBytes / (c.rows * 2 * c.N * sizeof(float));
    int n = int(std::min<size_t>({size_t(blocks) / std::max<size_t>(tiles, 1), size_t(nk / least), cap}));
    n = std::max(n, 1);
    p.per = (nk + n - 1) / n;
    p.splits = (nk + p.per - 1) / p.per;
}

// f32: 64 weight rows, the fewest row tiles that hold the rows.  Bound by the f32 MFMA rate (154
// TFLOP/s measured on a large product): one decoder layer of 128 tokens (hidden 1536, intermediate
// 8960) 30.2 ms with one thread per output -> 0.223 ms, gate / up + swiglu 89.6 us, down 43.4 us.
Plan planOf(const LinearCall &c) {
    Plan p{64, 64, 32, 1, 0};
    p.bx = c.rows <= 32 ? 32 : c.rows <= 64 ? 64 : 128;
    splitK(p, c, 512, 4);
    return p;
}

size_t planBytes(const Plan &p, const LinearCall &c) {
    return p.splits > 1 ? size_t(p.splits) * c.rows * (c.swiglu ? 2 * c.N : c.N) * sizeof(float) : 0;
}

template <typename T, bool kInt8, bool kSw, int BW, int BX, int NWW, int NWX, int KS, int S>
void launchTile(const GemmArgs &a, hipStream_t s) {
    const unsigned tiles = unsigned((a.Nw + BW - 1) / BW) * unsigned((a.M + BX - 1) / BX);
    linearTile<T, kInt8, kSw, BW, BX, NWW, NWX, KS, S><<<tiles * unsigned(a.splits), NWW * NWX * kWave, 0, s>>>(a);
}

template <typename T, bool kInt8, bool kSw>
void launchReduce(const GemmArgs &a, hipStream_t s) {
    const bool v4 = a.N % 4 == 0;
    const size_t n = size_t(a.M) * (v4 ? a.N / 4 : a.N);
    const unsigned blocks = unsigned((n + 255) / 256);
    if (v4)
        linearReduce<T, kInt8, kSw, 4><<<blocks, 256, 0, s>>>(a);
    else
        linearReduce<T, kInt8, kSw, 1><<<blocks, 256, 0, s>>>(a);
}

template <typename T, bool kInt8, bool kSw>
void launchPlan(const Plan &p, const GemmArgs &a, hipStream_t s) {
    if (p.bx == 32)
        launchTile<T, kInt8, kSw, 64, 32, 1, 1, 32, 4>(a, s);
    else if (p.bx == 64)
        launchTile<T, kInt8, kSw, 64, 64, 1, 2, 32, 3>(a, s);
    else
        launchTile<T, kInt8, kSw, 64, 128, 1, 4, 32, 3>(a, s);
    if (a.part) launchReduce<T, kInt8, kSw>(a, s);
}

} // namespace

bool gemmTakes(const LinearCall &c) {
    const auto al = [](const void *p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    return c.dt == LLAISYS_DTYPE_F32 && !c.scale && c.rows > 1 && c.K > 0 && c.K % 4 == 0 && al(c.x) && al(c.w);
}

size_t gemmWorkspaceBytes(const LinearCall &c) { return planBytes(planOf(c), c); }

void gemm(const LinearCall &c, void *ws, size_t ws_bytes, hipStream_t s) {
    if (c.rows == 0 || c.N == 0) return;
    Plan p = planOf(c);
    if (planBytes(p, c) > ws_bytes) {
        p.splits = 1;
        p.per = int((c.K + p.ks - 1) / p.ks);
    }
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
    if (c.swiglu)
        launchPlan<F32, false, true>(p, a, s);
    else
        launchPlan<F32, false, false>(p, a, s);
}

} // namespace llaisys::kernels
