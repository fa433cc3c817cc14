// Kernels of the tiled linear layers, included by the translation units that instantiate them for
// one element type each (linear_gemm*.hip).
//
// Semantics: reference src/ops/linear/cpu/linear_cpu.cpp:11-41 (dense) and the W8A16 rule of
// linear.hip; the sums run in f32 in the order of the tiles' k, split sums added in split order.
//
// Design.  A block owns a tile of BW weight rows x BX activation rows and one of `splits` ranges
// of K.  Per stage of KS k, both operands move HBM -> LDS with global_load_lds_dwordx4 (1 KB per
// instruction, no register staging) through a ring of S stages, so S - 1 stages are in flight
// while the MFMAs run on one.  The load fills LDS contiguously, so rows cannot be padded: the lane
// that fills slot c of row r fetches chunk c ^ swz(r), and the operand reads apply the same XOR (no
// bank conflicts).  The MFMA computes out^T = w x^T, so a lane ends with 4 consecutive channels of
// one row.  INT8 codes stay codes in LDS and become exact bf16 / f16 values in registers.  f32
// runs on v_mfma_f32_32x32x2_f32 (f32 products and sums, 154 TFLOP/s on this card) with the same
// tiles: a 16-byte chunk is 4 k.
// When the tiles alone leave CUs idle, K is split over blocks; the partial sums go to the
// workspace in f32 and linearReduce adds them in split order, so results do not depend on
// which block ends first.  swiglu runs in the epilogue (of the tile, or of the reduction) on gate
// and up rounded to the element type, as the separate op would read them.
//
// What bounds a tile: neither unit, but its waves meeting at a barrier per stage.  192 x 256 on 2048 x
// 1536 -> 17920 (132 us, 854 TFLOP/s; 128 x 128 tiles of 64 x 64 per wave 146 us): the MFMA pipe is busy 47%
// of the cycles of a CU, LDS moves 74 of 128 B per cycle (operands and fill) without bank conflicts, and
// a wave spends 30% of its time in waits and barriers.  192 x 128 on 2048 x 8960 -> 1536, one block per
// CU: 42%, 96 B and 46%.
#pragma once

#include "common.hpp"
#include "launch.hpp"
#include "linear_common.hpp"
#include "linear_gemm.hpp"

#include <type_traits>

namespace llaisys::kernels {

using namespace lin;
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kXcds = 8; // accelerator complex dies, each with its own L2

// A chunk of K past the row end is read from here: zeros add nothing to a sum.
static __device__ const __align__(16) uint32_t kZeroChunk[4] = {0u, 0u, 0u, 0u};

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

// ldsBarrier with the wait and the barrier as builtins: the compiler then knows that the LDS reads
// issued before it have landed, and does not wait for the first one after it in their place.
__device__ __forceinline__ void stageBarrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F); // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
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

template <typename T, bool kInt8, bool kSw, int BW, int BX, int NWW, int NWX, int NWK, int KS, int S, bool kPipe = false>
__global__ void __launch_bounds__(NWW *NWX *NWK * 64)
    linearTile(GemmArgs a) {
    constexpr int kE = Fmt<T>::kBytes;
    constexpr int NWV = NWW * NWX * NWK;
    constexpr int WW = BW / NWW, WX = BX / NWX, TW = WW / 32, TX = WX / 32;
    constexpr int WB = KS * (kInt8 ? 1 : kE), XB = KS * kE; // bytes of a row per stage
    constexpr int WC = WB / 16, XC = XB / 16;               // chunks of a row per stage
    constexpr int kStageB = BW * WB + BX * XB;
    constexpr int WI = BW * WB / 1024, XI = BX * XB / 1024, kLoads = (WI + XI + NWV - 1) / NWV;
    static_assert(kLoads * (S - 2) < 64 && TW >= 1 && TX >= 1, "load split");
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
    const int ww0 = (wave % NWW) * WW, wx0 = (wave / NWW % NWX) * WX, wk = wave / (NWW * NWX);
    const int nk_all = (a.K + KS - 1) / KS;
    const int kt0 = sp * a.per, nk = min(nk_all - kt0, a.per);

    // weight row of tile row tr; with swiglu 8 gate rows and the 8 up rows of the same channels take
    // turns, so that one lane's sums hold both of a channel (q and q + 1 of the MFMA's D)
    const auto wrow = [&](int tr) {
        if constexpr (kSw) {
            return min(w0 / 2 + 8 * (tr / 16) + tr % 8, a.N - 1) + (tr & 8 ? a.N : 0);
        } else {
            return min(w0 + tr, a.N - 1);
        }
    };
    // load i of this wave fills KB slot(i) of a stage (a last one may be filled twice, with the same)
    const auto slot = [&](int i) { return min(wave * kLoads + i, WI + XI - 1); };
    const char *src[kLoads];
    int left[kLoads]; // chunks of the row from the lane's first one on
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const int q = slot(i);
        if (q < WI) {
            const int tr = q * (64 / WC) + lane / WC, c = (lane % WC) ^ swz<WC>(tr);
            src[i] = static_cast<const char *>(a.w) + size_t(wrow(tr)) * a.K * (kInt8 ? 1 : kE) + size_t(kt0) * WB + 16 * c;
            left[i] = int(size_t(a.K) * (kInt8 ? 1 : kE) / 16) - kt0 * WC - c;
        } else {
            const int tr = (q - WI) * (64 / XC) + lane / XC, c = (lane % XC) ^ swz<XC>(tr);
            src[i] = static_cast<const char *>(a.x) + size_t(min(x0 + tr, a.M - 1)) * a.K * kE + size_t(kt0) * XB + 16 * c;
            left[i] = int(size_t(a.K) * kE / 16) - kt0 * XC - c;
        }
    }
    const bool tail = a.K % KS != 0 && kt0 + nk == nk_all; // the last stage reaches past the rows
    // Called for kt = 0, 1, ..: the sources move on with it.  `steady`, here and in the stages below,
    // is a compile-time promise that kt is not the last stage: the loop over all but the last S
    // stages then has no branch around its loads and one constant wait, and the compiler places the
    // loads among the LDS reads and MFMAs (2048 rows of gate / up / swiglu 129.8 -> 127.1 us, one
    // [8960, 1536] 83.2 -> 79.4 in tiles of 192 x 256, 79.8 -> 79.0 in 192 x 128).
    const auto issue = [&](int kt, auto steady) {
        char *dst = lds + (kt % S) * kStageB;
        if (!steady && tail && kt == nk - 1) {
#pragma unroll
            for (int i = 0; i < kLoads; ++i) {
                const int q = slot(i);
                const char *p = kt * (q < WI ? WC : XC) < left[i] ? src[i] : reinterpret_cast<const char *>(kZeroChunk);
                __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1))) *)(p),
                                                 (void __attribute__((address_space(3))) *)(dst + q * 1024), 16, 0, 0);
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const int q = slot(i);
            __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1))) *)(src[i]),
                                             (void __attribute__((address_space(3))) *)(dst + q * 1024), 16, 0, 0);
            src[i] += q < WI ? WB : XB;
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
        if (st < nk) issue(st, std::false_type{});
    if constexpr (kPipe) {
        // One or two waves per SIMD: the operands of a pair of steps (one 16-code chunk per weight row) are
        // read from LDS while the MFMAs of the pair before run, also across stages, so a stage is
        // complete in LDS one stage before its MFMAs.
        static_assert(NWK == 1 && kE == 2 && S >= 3, "pipelined tiles");
        constexpr int kPairs = XC / 4, CW = kInt8 ? 1 : 2; // chunks of a weight row per pair
        constexpr int kReads = TW * CW + 2 * TX, kMfmas = 2 * TW * TX, kPaired = kReads < kMfmas ? kReads : kMfmas;
        struct Ops {
            v4u w[TW][CW], x[TX][2];
        };
        const auto fetch = [&](Ops &o, int kt, int p) {
            const char *tile = lds + (kt % S) * kStageB;
#pragma unroll
            for (int i = 0; i < TW; ++i)
#pragma unroll
                for (int c = 0; c < CW; ++c)
                    o.w[i][c] = *reinterpret_cast<const v4u *>(tile + wbase + 32 * i * WB + 16 * ((kInt8 ? 2 * p + h2 : 4 * p + 2 * h2 + c) ^ wsz));
#pragma unroll
            for (int j = 0; j < TX; ++j)
#pragma unroll
                for (int c = 0; c < 2; ++c)
                    o.x[j][c] = *reinterpret_cast<const v4u *>(tile + xbase + 32 * j * XB + 16 * ((4 * p + 2 * h2 + c) ^ xsz));
        };
        const auto multiply = [&](const Ops &o) {
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int i = 0; i < TW; ++i) {
                    const v4u fa = kInt8 ? codesToT<T>(c ? v2u{o.w[i][0].z, o.w[i][0].w} : v2u{o.w[i][0].x, o.w[i][0].y}) : o.w[i][CW == 1 ? 0 : c];
#pragma unroll
                    for (int j = 0; j < TX; ++j) acc[i][j] = mfmaChunk<T>(fa, o.x[j][c], acc[i][j]);
                }
        };
        const auto stage = [&](int kt, Ops &cur, Ops &nxt, auto steady) {
            if (steady || kt + S - 2 < nk) // stage kt + 1 has landed
                waitVmcnt<kLoads * (S - 3)>();
            else
                waitVmcnt<0>();
            stageBarrier(); // for every wave; stage kt - 1 is no longer read
            if (steady || kt + S - 1 < nk) issue(kt + S - 1, steady);
#pragma unroll
            for (int p = 0; p < kPairs; ++p) {
                Ops &c = p % 2 ? nxt : cur, &n = p % 2 ? cur : nxt;
                if (p + 1 < kPairs)
                    fetch(n, kt, p + 1);
                else
                    fetch(n, kt + 1, 0); // past the last stage: read, not used
                multiply(c);
                // one LDS read behind each of the first MFMAs (behind the last one what is left of them)
#pragma unroll
                for (int r = 0; r < kPaired; ++r) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0); // MFMA
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0); // LDS read
                }
                if constexpr (kReads > kPaired) __builtin_amdgcn_sched_group_barrier(0x100, kReads - kPaired, 0);
                if constexpr (kMfmas > kPaired) __builtin_amdgcn_sched_group_barrier(0x008, kMfmas - kPaired, 0);
            }
        };
        Ops o0, o1;
        if (S - 1 <= nk)
            waitVmcnt<kLoads * (S - 2)>();
        else
            waitVmcnt<0>();
        ldsBarrier();
        fetch(o0, 0, 0);
        if constexpr (kPairs % 2 == 0) {
            int kt = 0;
            for (; kt + S < nk; ++kt) stage(kt, o0, o1, std::true_type{});
            for (; kt < nk; ++kt) stage(kt, o0, o1, std::false_type{});
        } else {
            int kt = 0;
            for (; kt + 1 + S < nk; kt += 2) {
                stage(kt, o0, o1, std::true_type{});
                stage(kt + 1, o1, o0, std::true_type{});
            }
            for (; kt < nk; kt += 2) {
                stage(kt, o0, o1, std::false_type{});
                if (kt + 1 < nk) stage(kt + 1, o1, o0, std::false_type{});
            }
        }
    } else {
        const auto stage = [&](int kt, auto steady) {
            // this wave's loads of stage kt have landed (the stages after it may be in flight)
            if (steady || kt + S - 2 < nk)
                waitVmcnt<kLoads * (S - 2)>();
            else
                waitVmcnt<0>();
            ldsBarrier(); // every wave's have; stage kt - 1 is no longer read
            if (steady || kt + S - 1 < nk) issue(kt + S - 1, steady);
            const char *tile = lds + (kt % S) * kStageB;
            // k order of a stage: 16-bit types, step st and half h: chunk 4 (st / 2) + 2 h + st % 2, so
            // that the 16 codes of an INT8 chunk serve two steps; f32: chunk 2 st + h
            constexpr int kSteps = XC / 2;
            static_assert(kSteps % NWK == 0 && (kE == 4 || kSteps / 2 % NWK == 0), "the waves of a tile share its steps evenly");
            if constexpr (kInt8) {
#pragma unroll
                for (int pw = 0; pw < kSteps / 2 / NWK; ++pw) {
                    const int p = wk * (kSteps / 2 / NWK) + pw;
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
                for (int sw = 0; sw < kSteps / NWK; ++sw) {
                    const int st = wk * (kSteps / NWK) + sw;
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
        };
        int kt = 0;
        for (; kt + S < nk; ++kt) stage(kt, std::true_type{});
        for (; kt < nk; ++kt) stage(kt, std::false_type{});
    }
    if constexpr (NWK > 1) { // the waves' shares of a tile, added in wave order
        constexpr int kAcc = TW * TX * 16;
        static_assert((NWK - 1) * BW * BX * 4 <= S * kStageB, "the partial tiles fit the stages");
        float *xch = reinterpret_cast<float *>(lds) + size_t(wave % (NWW * NWX)) * kAcc * kWave;
        ldsBarrier(); // no wave reads a stage any more, and every load has landed
        if (wk > 0) {
#pragma unroll
            for (int i = 0; i < kAcc / 4; ++i) {
                const f32x16 &t = acc[i / 4 / TX][i / 4 % TX];
                *reinterpret_cast<f32x4 *>(xch + size_t(wk - 1) * BW * BX + (i * kWave + lane) * 4) =
                    f32x4{t[4 * (i % 4)], t[4 * (i % 4) + 1], t[4 * (i % 4) + 2], t[4 * (i % 4) + 3]};
            }
        }
        ldsBarrier();
        if (wk > 0) return;
#pragma unroll
        for (int k = 0; k < NWK - 1; ++k)
#pragma unroll
            for (int i = 0; i < kAcc / 4; ++i) {
                const f32x4 t = *reinterpret_cast<const f32x4 *>(xch + size_t(k) * BW * BX + (i * kWave + lane) * 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[i / 4 / TX][i / 4 % TX][4 * (i % 4) + e] += t[e];
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
                    n = (w0 + ww0 + 32 * i) / 2 + 8 * (q / 2) + 4 * h2 + (q % 2 ? a.N : 0);
                    top = q % 2 ? a.Nw : a.N;
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
#pragma unroll
    for (int i = 0; i < TW; ++i)
#pragma unroll
        for (int q = 0; q < 4; q += kSw ? 2 : 1) {
            const int n = kSw ? (w0 + ww0 + 32 * i) / 2 + 4 * q + 4 * h2 : w0 + ww0 + 32 * i + 8 * q + 4 * h2;
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
                        o[e] = SwigluOp::apply(Fmt<T>::round(o[e]), Fmt<T>::round(finish<T, kInt8>(a, acc[i][j][4 * (q + 1) + e], ne + a.N)));
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

template <typename T, bool kInt8, bool kSw, int BW, int BX, int NWW, int NWX, int NWK, int KS, int S, bool kPipe = false>
void launchTile(const GemmArgs &a, hipStream_t s) {
    const unsigned tiles = unsigned((a.Nw + BW - 1) / BW) * unsigned((a.M + BX - 1) / BX);
    linearTile<T, kInt8, kSw, BW, BX, NWW, NWX, NWK, KS, S, kPipe><<<tiles * unsigned(a.splits), NWW * NWX * NWK * kWave, 0, s>>>(a);
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

// The tile shapes of GemmTile for a 16-bit type
template <typename T, bool kInt8, bool kSw>
void launch16(GemmTile t, const GemmArgs &a, hipStream_t s) {
    if constexpr (kInt8) {
        switch (t) {
        case GemmTile::k64x64Deep: launchTile<T, true, kSw, 64, 64, 2, 1, 2, 128, 2>(a, s); break;
        case GemmTile::k64x64: launchTile<T, true, kSw, 64, 64, 2, 2, 1, 64, 3>(a, s); break;
        case GemmTile::k128x64: launchTile<T, true, kSw, 128, 64, 4, 1, 1, 64, 2>(a, s); break;
        case GemmTile::k128x128: launchTile<T, true, kSw, 128, 128, 4, 1, 1, 64, 2>(a, s); break;
        case GemmTile::k192x128: launchTile<T, true, kSw, 192, 128, 6, 1, 1, 64, 3, true>(a, s); break;
        case GemmTile::k256x128: launchTile<T, true, kSw, 256, 128, 4, 2, 1, 64, 2>(a, s); break;
        default: launchTile<T, true, kSw, 192, 256, 2, 4, 1, 64, 3, true>(a, s); break;
        }
    } else {
        switch (t) {
        case GemmTile::k64x64Deep: launchTile<T, false, kSw, 64, 64, 2, 1, 2, 128, 2>(a, s); break;
        case GemmTile::k64x64: launchTile<T, false, kSw, 64, 64, 2, 2, 1, 64, 3>(a, s); break;
        case GemmTile::k128x64: launchTile<T, false, kSw, 128, 64, 2, 2, 1, 64, 2>(a, s); break;
        case GemmTile::k128x128: launchTile<T, false, kSw, 128, 128, 2, 2, 1, 64, 2>(a, s); break;
        case GemmTile::k192x128: launchTile<T, false, kSw, 192, 128, 2, 4, 1, 64, 3, true>(a, s); break;
        default: launchTile<T, false, kSw, 192, 256, 2, 4, 1, 32, 5, true>(a, s); break;
        }
    }
    if (a.part) launchReduce<T, kInt8, kSw>(a, s);
}

template <typename T>
void gemm16(GemmTile t, const GemmArgs &a, bool swiglu, hipStream_t s) {
    if (a.scale)
        swiglu ? launch16<T, true, true>(t, a, s) : launch16<T, true, false>(t, a, s);
    else
        swiglu ? launch16<T, false, true>(t, a, s) : launch16<T, false, false>(t, a, s);
}

} // namespace llaisys::kernels
