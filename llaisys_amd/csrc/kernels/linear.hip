// Linear layers for gfx950: the reference's dense linear and W8A16 over INT8 weights.
//
// Semantics: reference src/ops/linear/cpu/linear_cpu.cpp:11-41 -- out[m][n] =
// T(sum_k x[m][k] * w[n][k] + bias[n]) with an f32 sum, x [rows, K], w [N, K].  W8A16 (no
// reference kernel): w is INT8 codes [N, K] with one f32 scale per output channel n, and
// out[m][n] = T(scale[n] * sum_k x[m][k] * code[n][k] + bias[n]).  The MFMA path sums the
// exact products of bf16 / f16 operands (INT8 codes are exact in both) in f32; the order of
// the sum differs from the reference's left-to-right loop, which the tests bound by the f32
// accumulation error.
//
// Design, by row count M (the launcher at the end picks the kernel):
//  - M = 1 (decode), linearGemvRow: HBM-bound on the weights, one wave per output channel
//    (4 for the INT8 lm_head) with its whole weight row requested up front in 1 KB load
//    instructions, x in LDS or L1 / L2, f32 FMAs, a butterfly.  linearGemv (the same sum,
//    no LDS) takes rows too long for that and M = 2 (INT8 weights with N >= 4096 and M = 2
//    go to linearSkinny instead).
//  - M <= 16, linearSkinny: HBM-bound; a block owns 16 channels, its waves split K, load
//    weight rows row-contiguously and transpose them through a per-wave LDS tile into
//    v_mfma_f32_16x16x32 operands; partials summed in LDS in wave order.
//  - more rows (prefill): linear_gemm.hip, MFMA tiles.
//  - f32: linearGemvRow / linearGemv for one row, linear_gemm.hip for more (K % 4 == 0).
//  - anything else (unaligned rows, K not a multiple of a 16-byte chunk, f32 against INT8
//    weights): linearScalar, one thread per output with the reference's sequential sum.
// INT8 codes enter every MFMA as exact bf16 / f16 values and the per-channel scale multiplies
// the f32 sum once.
#include "common.hpp"
#include "launch.hpp"
#include "linear_common.hpp"
#include "linear_gemm.hpp"
#include "rowplan.hpp"

#include <algorithm>
#include <type_traits>

namespace llaisys::kernels {

namespace {

using namespace lin;

struct LinearArgs {
    void *out;
    const void *x;
    const void *w;       // elements of T, or INT8 codes
    const float *scale;  // INT8 only
    const void *bias;    // T, or null
    int M, N, K;
    bool swiglu; // (linearSkinny) w, scale and bias have 2 N rows, the gate's first
};

// Few rows (M <= 16, decode): HBM-bound on the weights; the skinny MFMA loop of
// linear_common.hpp over one set of 16 channels, x rows >= M entering as zeros.  The waves'
// 16 x 16 partials are summed in LDS in wave order.  With kSw a block takes the 16 gate rows and the
// 16 up rows of its channels and finishes with swiglu of the two, rounded to T as the separate
// op would read them (each set sums as its own launch does: the same bits).  A launch costs about
// 2.4 us beside its bytes: 5 rows, 1536 -> 2 x 8960, bf16, 2 x 6.9 us and a swiglu launch -> one launch; the layer of 5 tokens
// 63.9 -> 59.0 us.
template <typename T, bool kInt8, bool kSw>
__global__ void __launch_bounds__(1024)
    linearSkinny(LinearArgs a) {
    constexpr int R = kSw ? 2 : 1;
    // dynamic LDS, sized by the launch: nw transpose tiles, then nw partial tiles
    extern __shared__ __align__(16) char smem[];
    const int nw = int(blockDim.x) / kWave;
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / kWave);
    const int lane = int(threadIdx.x) % kWave;
    const int r16 = lane % 16, g4 = lane / 16;
    const int n0 = int(blockIdx.x) * 16;
    char *tile = smem + size_t(wave) * R * 16 * skinnyPitch(kInt8);
    float(*red)[R][256] = reinterpret_cast<float(*)[R][256]>(smem + nw * R * 16 * skinnyPitch(kInt8));
    const char *xrow = static_cast<const char *>(a.x) + size_t(min(r16, a.M - 1)) * a.K * 2;
    const bool xlane = r16 < a.M;
    const v4u z4 = {0u, 0u, 0u, 0u};
    const auto xop = [&](int k) {
        const v4u v = *reinterpret_cast<const v4u *>(xrow + size_t(k < a.K ? k : 0) * 2);
        return xlane && k < a.K ? v : z4;
    };
    f32x4 acc[R];
    int rows0[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        acc[r] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        rows0[r] = n0 + r * a.N;
    }
    skinnyGroups<T, kInt8, R>(acc, static_cast<const char *>(a.w), rows0, R * a.N, a.K, tile, wave, nw, lane, xop);
    // D[m = 4 g + e][n = r16]
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int e = 0; e < 4; ++e) red[wave][r][(4 * g4 + e) * 16 + r16] = acc[r][e];
    __syncthreads();
    for (int t = int(threadIdx.x); t < 16 * a.M; t += int(blockDim.x)) {
        const int m = t / 16, n = n0 + t % 16;
        if (n < a.N) {
            float y[R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                float s = 0.0f;
                for (int w = 0; w < nw; ++w) s += red[w][r][t];
                if constexpr (kInt8) s = a.scale[n + r * a.N] * s;
                if (a.bias) s = s + Fmt<T>::get(a.bias, n + r * a.N);
                y[r] = s;
            }
            if constexpr (kSw) y[0] = SwigluOp::apply(Fmt<T>::round(y[0]), Fmt<T>::round(y[1]));
            Fmt<T>::put(a.out, size_t(m) * a.N + n, y[0]);
        }
    }
}

// One or two rows (decode): each wave owns one output channel and streams its weight row,
// 16 bytes per lane per load (1 KB contiguous per instruction, the pattern that streams HBM
// fastest), with FMAs in f32 against the matching x chunks (cache hits) and a DPP /
// permlane butterfly over the lane partials at the end.  No LDS and no cross-block
// synchronisation, so N output channels give N waves however small N is.
template <typename T, bool kInt8, int M>
__global__ void __launch_bounds__(256)
    linearGemv(LinearArgs a) {
    using F = Fmt<T>;
    constexpr int E = kInt8 ? 16 : F::kVec;  // weight elements per 16-byte chunk
    constexpr int XH = E / F::kVec;          // 16-byte chunks of x beside it
    constexpr int U = 4;                     // chunks in flight per lane
    const int lane = int(threadIdx.x) % kWave;
    const int n = int(blockIdx.x) * 4 + int(threadIdx.x) / kWave; // wave-uniform
    if (n >= a.N) return;
    const int nc = a.K / E; // K % E == 0
    const char *wrow = static_cast<const char *>(a.w) + size_t(n) * a.K * (kInt8 ? 1 : F::kBytes);
    const char *xb = static_cast<const char *>(a.x);
    float acc[M];
#pragma unroll
    for (int m = 0; m < M; ++m) acc[m] = 0.0f;
    for (int c0 = lane; c0 < nc; c0 += kWave * U) {
        // all loads first (a chunk past the row end reads chunk 0 and is masked below)
        v4u wv[U], xv[U][M][XH];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int c = c0 + kWave * u < nc ? c0 + kWave * u : 0;
            wv[u] = *reinterpret_cast<const v4u *>(wrow + size_t(c) * 16);
#pragma unroll
            for (int m = 0; m < M; ++m)
#pragma unroll
                for (int h = 0; h < XH; ++h)
                    xv[u][m][h] = load16<T>(xb, size_t(m) * a.K + size_t(c) * E + F::kVec * h);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (c0 + kWave * u >= nc) continue;
            float wf[E];
            if constexpr (kInt8) {
                const uint32_t ww[4] = {wv[u].x, wv[u].y, wv[u].z, wv[u].w};
#pragma unroll
                for (int e = 0; e < E; ++e) wf[e] = float(int8_t(ww[e / 4] >> (8 * (e % 4))));
            } else {
                Fmt<T>::unpack(wv[u], wf);
            }
#pragma unroll
            for (int m = 0; m < M; ++m)
#pragma unroll
                for (int h = 0; h < XH; ++h) {
                    float xf[F::kVec];
                    F::unpack(xv[u][m][h], xf);
#pragma unroll
                    for (int e = 0; e < F::kVec; ++e) acc[m] = __builtin_fmaf(xf[e], wf[F::kVec * h + e], acc[m]);
                }
        }
    }
    const float sc = kInt8 ? a.scale[n] : 1.0f;
    const float bv = a.bias ? Fmt<T>::get(a.bias, n) : 0.0f;
#pragma unroll
    for (int m = 0; m < M; ++m) {
        float s = waveGroupReduce<kWave, SumOp>(acc[m]);
        if (lane == 0) {
            if constexpr (kInt8) s = sc * s;
            if (a.bias) s = s + bv;
            Fmt<T>::put(a.out, size_t(m) * a.N + n, s);
        }
    }
}

// One row (decode): linearGemv's sum -- per output channel one wave, lane chunks lane,
// lane + 64, ... in one FMA chain, then the same butterfly -- with every weight chunk of the
// wave's C channels requested before anything else (C x J per lane) and x staged once per
// block in LDS (kLds) or read through L1 / L2, so the loads are all in flight behind one x
// round trip.  Same bits as linearGemv (and
// as the fused rms_norm -> projection, which sums the same way).  Measured on MI355X (M = 1,
// >= 1 GiB of rotating weight sets): W8A16 [8960, 1536] 5.47 us against 6.79 us for
// linearSkinny and 7.55 us for linearGemv; bf16 [8960, 1536] 6.17 against 7.39 us; W8A16
// [1536, 8960] 6.41 against 7.00 us; bf16 [1536, 8960] 8.28 against 9.38 us.
template <typename T, bool kInt8, int J, int C, bool kLds, int NW>
__global__ void __launch_bounds__(NW * kWave)
    linearGemvRow(LinearArgs a) {
    using F = Fmt<T>;
    constexpr int E = kInt8 ? 16 : F::kVec; // weight elements per 16-byte chunk
    extern __shared__ __align__(16) char xs_raw[];
    const char *xs = kLds ? xs_raw : static_cast<const char *>(a.x);
    const int lane = int(threadIdx.x) % kWave;
    const int n0 = (int(blockIdx.x) * NW + int(threadIdx.x) / kWave) * C; // wave-uniform
    const int nc = a.K / E;
    // a channel past the last loads a valid row and stores nothing (its wave still joins the
    // block barrier); a chunk past the row end reads chunk 0 and is skipped
    v4u wv[C][J];
#pragma unroll
    for (int ci = 0; ci < C; ++ci) {
        const int n = n0 + ci;
        const char *wrow = static_cast<const char *>(a.w) + size_t(n < a.N ? n : a.N - 1) * a.K * (kInt8 ? 1 : F::kBytes);
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const int c = lane + kWave * j;
            wv[ci][j] = __builtin_nontemporal_load(reinterpret_cast<const v4u *>(wrow + size_t(c < nc ? c : 0) * 16));
        }
    }
    if constexpr (kLds) {
        for (int i = int(threadIdx.x); i < a.K / F::kVec; i += NW * kWave)
            reinterpret_cast<v4u *>(xs_raw)[i] = reinterpret_cast<const v4u *>(a.x)[i];
        __syncthreads();
    }
    // chunk-major: the lane's x chunk is unpacked once for the wave's C channels; each
    // channel still sums its chunks and elements in the same order (one FMA chain)
    float acc[C];
#pragma unroll
    for (int ci = 0; ci < C; ++ci) acc[ci] = 0.0f;
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int c = lane + kWave * j;
        if (c >= nc) continue; // (the lane's remaining chunks are past the end too)
        float xf[E];
#pragma unroll
        for (int h = 0; h < E / F::kVec; ++h) F::unpack(load16<T>(xs, c * E + F::kVec * h), xf + F::kVec * h);
#pragma unroll
        for (int ci = 0; ci < C; ++ci) {
            float wf[E];
            if constexpr (kInt8) {
                const uint32_t ww[4] = {wv[ci][j].x, wv[ci][j].y, wv[ci][j].z, wv[ci][j].w};
#pragma unroll
                for (int e = 0; e < E; ++e) wf[e] = float(int8_t(ww[e / 4] >> (8 * (e % 4))));
            } else {
                F::unpack(wv[ci][j], wf);
            }
#pragma unroll
            for (int e = 0; e < E; ++e) acc[ci] = __builtin_fmaf(xf[e], wf[e], acc[ci]);
        }
    }
#pragma unroll
    for (int ci = 0; ci < C; ++ci) {
        float t = waveGroupReduce<kWave, SumOp>(acc[ci]);
        const int n = n0 + ci;
        if (lane == 0 && n < a.N) {
            if constexpr (kInt8) t = a.scale[n] * t;
            if (a.bias) t = t + F::get(a.bias, n);
            F::put(a.out, n, t);
        }
    }
}

// Any shape and type: one thread per output, the sum in the reference's order.
template <typename T, bool kInt8>
__global__ void __launch_bounds__(256)
    linearScalar(LinearArgs a) {
    const size_t idx = size_t(blockIdx.x) * 256 + threadIdx.x;
    if (idx >= size_t(a.M) * a.N) return;
    const size_t m = idx / a.N, n = idx % a.N;
    float sum = 0.0f;
    for (int k = 0; k < a.K; ++k) {
        const float wv = kInt8 ? float(static_cast<const int8_t *>(a.w)[n * a.K + k]) : Fmt<T>::get(a.w, n * a.K + k);
        sum = sum + Fmt<T>::get(a.x, m * a.K + k) * wv;
    }
    if constexpr (kInt8) sum = a.scale[n] * sum;
    if (a.bias) sum = sum + Fmt<T>::get(a.bias, n);
    Fmt<T>::put(a.out, idx, sum);
}

// One row: linearGemvRow with J = ceil(chunks / 64) <= 24; false (linearGemv, the same sum)
// otherwise.  Variants (event timings of 5-16 rotating weight sets, all bit-identical):
//  - x staged in LDS by the block, except INT8 weights over at most 4096 channels, where the
//    block's staging is not hidden behind its 4 rows of codes and x is read from L1 / L2:
//    [3584, 3584] 5.54 -> 5.23 us, [1536, 8960] 6.26 -> 5.86 us, [3584, 18944] 18.7 -> 17.5 us
//    (larger N loses: [18944, 3584] 14.4 -> 15.3 us; bf16 [1536, 8960] 8.1 -> 8.7 us);
//  - 4 channels per wave for INT8 rows of at most 2 chunks per lane over 65536+ channels (the
//    lm_head), which spreads the block's x staging over 16 rows: [151936, 1536] 46.0 -> 40.0 us
//    (at [8960, 1536] it loses, 5.45 -> 6.57 us: too few blocks); 2 channels per wave in
//    4-wave blocks for such rows over 4097..65535 channels: [8960, 1536] 5.28-5.31 ->
//    4.99-5.03 us, [17920, 1536] 7.73-7.82 -> 7.66-7.68 us (same-box A/B, 3 runs each);
//  - waves per block: 8 where x is staged (the staging shared by more rows: bf16 [1536, 8960]
//    8.19 -> 7.70 us, [1536, 1536] 3.10 -> 2.95 us, [8960, 1536] 6.17 -> 6.09 us; 16 waves
//    10.5 us), 2 where it is read from L1 / L2 (INT8 [1536, 8960] 5.88 -> 5.68 us), 4 for
//    the 4-channel lm_head waves (8: 40.7 -> 42.6 us).
template <typename T, bool kInt8, int C, bool kLds, int NW, int J>
bool launchRowJ(const LinearArgs &a, int j, hipStream_t s) {
    if constexpr (J > 0) {
        if (j == J) {
            const unsigned blocks = unsigned((a.N + NW * C - 1) / (NW * C));
            linearGemvRow<T, kInt8, J, C, kLds, NW><<<blocks, NW * kWave, kLds ? size_t(a.K) * Fmt<T>::kBytes : 0, s>>>(a);
            return true;
        }
        return launchRowJ<T, kInt8, C, kLds, NW, J - 1>(a, j, s);
    }
    return false;
}

template <typename T, bool kInt8>
bool launchGemv1(const LinearArgs &a, hipStream_t s) {
    constexpr int E = kInt8 ? 16 : Fmt<T>::kVec;
    if (a.K % E != 0 || size_t(a.K) * Fmt<T>::kBytes > 64 * 1024) return false;
    const int j = (a.K / E + kWave - 1) / kWave;
    if (j < 1 || j > 24) return false;
    if constexpr (kInt8) {
        if (a.N <= 4096) return launchRowJ<T, true, 1, false, 2, 24>(a, j, s);
        if (a.N >= 65536 && j <= 2) return launchRowJ<T, true, 4, true, 4, 2>(a, j, s);
        if (j <= 2) return launchRowJ<T, true, 2, true, 4, 2>(a, j, s);
    }
    return launchRowJ<T, kInt8, 1, true, 8, 24>(a, j, s);
}

template <typename T, bool kInt8>
void launch(const LinearArgs &a, hipStream_t s) {
    if (a.M == 0 || a.N == 0) return;
    const auto al = [](const void *p, size_t n) { return (reinterpret_cast<uintptr_t>(p) % n) == 0; };
    constexpr bool kMfmaType = std::is_same_v<T, BF16> || std::is_same_v<T, F16>;
    // MFMA paths: 16-bit activations, 16-byte aligned rows (K % 8 == 0; INT8 codes K % 16 == 0)
    if (kMfmaType && a.K > 0 && a.K % (kInt8 ? 16 : 8) == 0 && al(a.x, 16) && al(a.w, 16)) {
        if constexpr (kMfmaType) {
            // one or two rows: the VALU GEMV (one wave per channel) while its f32 work stays
            // under the HBM time -- always for 16-bit weights; for INT8 weights (16 codes per
            // 16 bytes to convert) only when there are too few 16-channel tiles for the MFMA
            // kernel to occupy the chip
            // one row: the VALU sum of linearGemv (linearGemvRow when the row fits its
            // registers) -- also for INT8 weights, whatever N, so that the fused rms_norm ->
            // projection, which sums the same way, matches it bit for bit
            if (a.M == 1 && launchGemv1<T, kInt8>(a, s)) return;
            if (a.M == 1 || (a.M == 2 && (!kInt8 || (a.N + 15) / 16 < 256))) {
                const unsigned blocks = unsigned((a.N + 3) / 4);
                if (a.M == 1)
                    linearGemv<T, kInt8, 1><<<blocks, 256, 0, s>>>(a);
                else
                    linearGemv<T, kInt8, 2><<<blocks, 256, 0, s>>>(a);
                return;
            }
            if (a.M <= 16) {
                // waves per block: enough blocks x waves to fill the chip, at most one wave
                // per group of 128 k
                const int tiles = (a.N + 15) / 16, nw = skinnyWaves(a.N, a.K);
                const size_t lds = size_t(nw) * (16 * skinnyPitch(kInt8) + 256 * sizeof(float));
                if (a.swiglu)
                    linearSkinny<T, kInt8, true><<<unsigned(tiles), unsigned(nw * kWave), 2 * lds, s>>>(a);
                else
                    linearSkinny<T, kInt8, false><<<unsigned(tiles), unsigned(nw * kWave), lds, s>>>(a);
                return;
            }
        }
        return;
    }
    // f32, one row: the same GEMV (several rows: linear_gemm.hip)
    if constexpr (std::is_same_v<T, F32> && !kInt8) {
        if (a.M == 1 && a.K > 0 && a.K % 4 == 0 && al(a.x, 16) && al(a.w, 16)) {
            if (launchGemv1<F32, false>(a, s)) return;
            linearGemv<F32, false, 1><<<unsigned((a.N + 3) / 4), 256, 0, s>>>(a);
            return;
        }
    }
    const size_t n = size_t(a.M) * a.N;
    linearScalar<T, kInt8><<<unsigned((n + 255) / 256), 256, 0, s>>>(a);
}

template <bool kInt8>
void dispatch(const LinearArgs &a, llaisysDataType_t dt, hipStream_t s) {
    switch (dt) {
    case LLAISYS_DTYPE_F32: return launch<F32, kInt8>(a, s);
    case LLAISYS_DTYPE_BF16: return launch<BF16, kInt8>(a, s);
    case LLAISYS_DTYPE_F16: return launch<F16, kInt8>(a, s);
    default: return;
    }
}

} // namespace

// Rows 3 .. 16 of the 16-bit types: linearSkinny for one launch and for two alike (its waves' share
// of K depends on N and K only), while the block's transpose tiles and partials fit LDS.
bool linearSwigluFused(const LinearCall &c) {
    const auto al = [](const void *p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    if (gemmTakes(c)) return true;
    if (c.dt == LLAISYS_DTYPE_F32 || c.rows <= 2 || c.rows > 16 || c.K == 0 || c.K % (c.scale ? 16 : 8) || !al(c.x) || !al(c.w))
        return false;
    return 2 * skinnyWaves(int(c.N), int(c.K)) * (16 * skinnyPitch(c.scale != nullptr) + 1024) <= 150 * 1024;
}

size_t linearWorkspaceBytes(const LinearCall &c) { return gemmTakes(c) ? gemmWorkspaceBytes(c) : 0; }

void linear(const LinearCall &c, void *ws, size_t ws_bytes, hipStream_t s) {
    if (gemmTakes(c)) return gemm(c, ws, ws_bytes, s);
    const LinearArgs a{c.out, c.x, c.w, c.scale, c.bias, int(c.rows), int(c.N), int(c.K), c.swiglu};
    if (c.scale)
        dispatch<true>(a, c.dt, s);
    else
        dispatch<false>(a, c.dt, s);
}

} // namespace llaisys::kernels
