// Causal GQA self-attention for gfx950, over a cache in the element type or in INT8.
//
// Semantics: reference src/ops/self_attention/cpu/self_attention_cpu.cpp:13-115.  q [seq,
// nh, d], k [total, nkvh, d], v [total, nkvh, dv], out [seq, nh, dv]; q head h reads kv
// head h / (nh / nkvh); query i sits at current_pos = total - seq + i in size_t arithmetic
// (so seq > total wraps and the early queries see every key) and sees keys t <=
// current_pos; scores are (q . k) * scale in f32, softmax in f32, out = sum_t p_t v_t
// rounded to the element type; total == 0 gives zeros.  The INT8 form reads k and v as
// codes [total, nkvh, d] I8 plus scales [total, nkvh] F32 and rounds code * scale to the
// element type first, i.e. it is attention over llaisysDequantizeInt8 of the caches.
//
// Arithmetic differs from the reference in order only: fused multiply-adds in a lane tree
// for q . k, an online softmax (running max, rescaled sum and output) over batches of keys,
// exp through the hardware exp2, and (sum p v) / (sum p) instead of sum (p / sum) v.  The
// tests bound the difference by the f32 accumulation error of the reference itself.
//
// Design (the launcher at the end picks the kernel):
//  - attnPrefill (bf16 / f16, head_dim 64 or 128, >= 16 queries): 32 queries of two q heads per
//    block on v_mfma_f32_32x32x16, the keys split over the block's waves and, where the blocks
//    leave CUs idle, over blocks (merged by attnCombineFew / attnCombine).
//  - attnPrefill16 (bf16, head_dim 128, >= 16 queries): 16 queries of 1, 2 or 4 q heads per block on
//    v_mfma_f32_16x16x32, for the calls that are over before attnPrefill's larger blocks pay (planPrefill).
//  - attnDecodeMfma (bf16 q, head_dim 128, fewer queries: decode, cache in bf16 or INT8):
//    HBM-bound; the key range is cut into chunks, one block per (query, kv head, chunk) with
//    the kv head's q heads as the MFMA columns; attnCombine merges the chunk partials.
//  - attnGroup (f32, fewer queries in f16 or with head_dim 64, and short prefills of these): one wavefront per q head, the
//    waves of a block being q heads of one kv head (they read the same K / V rows).  A key row of D elements
//    is spread over R = D / 8 lanes, 8 elements per lane, so one load instruction covers
//    64 / R keys; per batch of U instructions the wave forms its scores (8 FMAs, a butterfly
//    over R lanes), updates the running max once and folds p * v into per-lane
//    accumulators.  Long key ranges with few (query, head) pairs are split and merged by
//    attnCombine as well.
//  - attnScalar: any other head_dim / v_head_dim, one wave per (query, head).
#include "common.hpp"
#include "launch.hpp"
#include "rowplan.hpp"

#include <algorithm>
#include <cstdio>
#include <mutex>
#include <cmath>
#include <type_traits>

namespace llaisys::kernels {

namespace {


// Row reader: 8 consecutive elements of a K or V row as f32.
template <typename T, bool kInt8>
struct RowIO;

template <typename T>
struct RowIO<T, false> {
    static constexpr int kRegs = Fmt<T>::kBytes == 2 ? 1 : 2; // 16-byte loads per lane
    struct Raw {
        v4u r[kRegs];
    };
    __device__ static Raw load(const void *base, size_t row, int d, int col) {
        const char *p = static_cast<const char *>(base) + (row * size_t(d) + col) * Fmt<T>::kBytes;
        Raw x;
#pragma unroll
        for (int k = 0; k < kRegs; ++k) x.r[k] = *reinterpret_cast<const v4u *>(p + 16 * k);
        return x;
    }
    __device__ static void unpack(const Raw &x, float sc, float *f) {
        (void)sc;
        if constexpr (kRegs == 1) {
            Fmt<T>::unpack(x.r[0], f);
        } else {
            Fmt<T>::unpack(x.r[0], f);
            Fmt<T>::unpack(x.r[1], f + 4);
        }
    }
};

template <typename T>
struct RowIO<T, true> {
    typedef uint32_t v2u __attribute__((ext_vector_type(2)));
    struct Raw {
        v2u r;
    };
    __device__ static Raw load(const void *base, size_t row, int d, int col) {
        const int8_t *p = static_cast<const int8_t *>(base) + row * size_t(d) + col;
        return Raw{*reinterpret_cast<const v2u *>(p)};
    }
    // code * scale rounded to the element type, as llaisysDequantizeInt8 stores it
    __device__ static void unpack(const Raw &x, float sc, float *f) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            f[e] = Fmt<T>::round(float(int8_t(x.r.x >> (8 * e))) * sc);
            f[4 + e] = Fmt<T>::round(float(int8_t(x.r.y >> (8 * e))) * sc);
        }
    }
};

struct AttnArgs {
    void *out;
    const void *q;
    const void *k;  // elements, or codes
    const void *v;
    const float *ks; // scales (INT8 only)
    const float *vs;
    float *part;     // partials of a split launch: [(i * nh + h) * nchunks + c][D + 2]
    size_t seq, total;
    int nh, nkvh, group, slices, nchunks, chunk;
    float scale;
};

// Visible keys of query i: [0, vis).
__device__ __forceinline__ size_t visibleKeys(size_t total, size_t seq, size_t i) {
    const size_t cur = total - seq + i; // size_t arithmetic, as the reference
    return cur >= total ? total : cur + 1;
}

constexpr int kWaves = 8; // waves per block of the vector kernel

// One block per (query, kv head, slice of G q heads, key chunk); its kWaves waves take the
// chunk's key tiles (KPW * U keys) in turn, every wave holding the G heads' q, running max,
// sum and output columns in registers, so each K / V row is loaded once per block.  The
// waves' states merge through LDS; the block then writes the output (one chunk) or the
// chunk's partial (split launch).
template <typename T, bool kInt8, int D, int G, int U>
__global__ void __launch_bounds__(kWave * kWaves)
    attnGroup(AttnArgs a) {
    using IO = RowIO<T, kInt8>;
    constexpr int R = D / 8;       // lanes per key row
    constexpr int KPW = kWave / R; // keys per load instruction
    constexpr int TILE = KPW * U;  // keys per wave per step
    __shared__ float st[kWaves][G][D + 2];

    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / kWave);
    const int lane = int(threadIdx.x) % kWave;
    const int rs = lane / R, col = (lane % R) * 8;

    // block -> (query, kv head, head slice, chunk); the latest queries (most keys) first
    unsigned b = blockIdx.x;
    const int c = int(b % unsigned(a.nchunks));
    b /= unsigned(a.nchunks);
    const int sl = int(b % unsigned(a.slices));
    b /= unsigned(a.slices);
    const int g = int(b % unsigned(a.nkvh));
    const size_t i = a.seq - 1 - size_t(b / unsigned(a.nkvh));
    const int h0 = g * a.group + sl * G; // first q head of the slice

    const size_t vis = visibleKeys(a.total, a.seq, i);
    const size_t k0 = size_t(c) * size_t(a.chunk);
    const size_t k1 = min(vis, k0 + size_t(a.chunk));

    float qv[G][8];
#pragma unroll
    for (int j = 0; j < G; ++j) {
        const char *qp = static_cast<const char *>(a.q) + ((i * a.nh + h0 + j) * D + col) * Fmt<T>::kBytes;
        typename RowIO<T, false>::Raw r;
#pragma unroll
        for (int k = 0; k < RowIO<T, false>::kRegs; ++k) r.r[k] = *reinterpret_cast<const v4u *>(qp + 16 * k);
        RowIO<T, false>::unpack(r, 0.0f, qv[j]);
    }
    float m[G], l[G], o[G][8];
#pragma unroll
    for (int j = 0; j < G; ++j) {
        m[j] = -INFINITY;
        l[j] = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[j][e] = 0.0f;
    }

    for (size_t kb = k0 + size_t(wave) * TILE; kb < k1; kb += size_t(kWaves) * TILE) {
        typename IO::Raw kr[U], vr[U];
        float ksc[U], vsc[U];
        bool ok[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const size_t key = kb + size_t(u * KPW + rs);
            ok[u] = key < k1;
            const size_t row = (ok[u] ? key : k0) * size_t(a.nkvh) + size_t(g);
            kr[u] = IO::load(a.k, row, D, col);
            vr[u] = IO::load(a.v, row, D, col);
            if constexpr (kInt8) {
                ksc[u] = a.ks[row];
                vsc[u] = a.vs[row];
            } else {
                ksc[u] = vsc[u] = 0.0f;
            }
        }
        float s[G][U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            float kf[8];
            IO::unpack(kr[u], ksc[u], kf);
#pragma unroll
            for (int j = 0; j < G; ++j) {
                float dot = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; ++e) dot = __builtin_fmaf(qv[j][e], kf[e], dot);
                dot = waveGroupReduce<R, SumOp>(dot);
                s[j][u] = ok[u] ? dot * a.scale : -INFINITY;
            }
        }
#pragma unroll
        for (int j = 0; j < G; ++j) {
            float mx = m[j];
#pragma unroll
            for (int u = 0; u < U; ++u) mx = fmaxf(mx, s[j][u]);
            // a -inf score is weight 0 (reference :111-113); m == mx keeps the state as is
            const float corr = mx == m[j] ? 1.0f : __expf(m[j] - mx);
            l[j] *= corr;
#pragma unroll
            for (int e = 0; e < 8; ++e) o[j][e] *= corr;
            m[j] = mx;
#pragma unroll
            for (int u = 0; u < U; ++u) s[j][u] = s[j][u] == -INFINITY ? 0.0f : __expf(s[j][u] - mx);
        }
        if (kb + TILE > k1) { // the filler rows weigh 0, and 0 * Inf would not be 0
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (!ok[u]) vr[u] = typename IO::Raw{}, vsc[u] = 0.0f;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            float vf[8];
            IO::unpack(vr[u], vsc[u], vf);
#pragma unroll
            for (int j = 0; j < G; ++j) {
                l[j] += s[j][u];
#pragma unroll
                for (int e = 0; e < 8; ++e) o[j][e] = __builtin_fmaf(s[j][u], vf[e], o[j][e]);
            }
        }
    }

    // merge the KPW key slots of the wave (lanes R, 2R, ... apart hold the same columns)
#pragma unroll
    for (int off = R; off < kWave; off *= 2) {
#pragma unroll
        for (int j = 0; j < G; ++j) {
            const float mo = __shfl_xor(m[j], off, kWave), lo = __shfl_xor(l[j], off, kWave);
            const float M = fmaxf(m[j], mo);
            // a slot that saw no key has m = -inf, l = 0, o = 0; its factor is 1 only when M
            // is -inf too, and then every term is 0
            const float fa = m[j] == M ? 1.0f : __expf(m[j] - M);
            const float fb = mo == M ? 1.0f : __expf(mo - M);
            l[j] = l[j] * fa + lo * fb;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float oo = __shfl_xor(o[j][e], off, kWave);
                o[j][e] = o[j][e] * fa + oo * fb;
            }
            m[j] = M;
        }
    }
    if (lane < R) {
#pragma unroll
        for (int j = 0; j < G; ++j) {
#pragma unroll
            for (int e = 0; e < 8; ++e) st[wave][j][col + e] = o[j][e];
            if (lane == 0) {
                st[wave][j][D] = m[j];
                st[wave][j][D + 1] = l[j];
            }
        }
    }
    __syncthreads();
    // merge the waves: thread t -> (head j, column e) pairs
    for (int p = threadIdx.x; p < G * D; p += kWave * kWaves) {
        const int j = p / D, e = p % D;
        float M = -INFINITY;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) M = fmaxf(M, st[w][j][D]);
        float L = 0.0f, O = 0.0f;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const float mw = st[w][j][D];
            const float f = mw == M ? 1.0f : __expf(mw - M); // 1 for M = -inf, where l = o = 0
            L += st[w][j][D + 1] * f;
            O += st[w][j][e] * f;
        }
        const size_t ih = i * a.nh + size_t(h0 + j);
        if (a.nchunks == 1) {
            // put: the reference rounding, also for a NaN carrying the caller's scale payload
            Fmt<T>::put(a.out, ih * D + e, L == 0.0f ? 0.0f : O / L);
        } else {
            float *pp = a.part + (ih * size_t(a.nchunks) + c) * (D + 2);
            pp[e] = O;
            if (e == 0) {
                pp[D] = M;
                pp[D + 1] = L;
            }
        }
    }
}

// Merge of the chunk partials of a split launch: one 1024-thread block per (query, head,
// slab of 32 output columns); thread t takes column t % 32 of the slab for the chunks c =
// t / 32 (mod 32), so a thread reads at most nchunks / 32 partial values and the (query,
// head) pairs of a decode launch spread over D / 32 times as many blocks.  Every block of a
// pair forms the same maximum and sum from the chunks' (m, l).  Up to 256 chunks (kPer = 8
// per thread) the partial values are requested together with the (m, l) loads, so the
// merge waits for one round of loads rather than two; the sum runs in the same order
// either way.
constexpr int kCombineThreads = 1024;
constexpr int kCombineCols = 32; // output columns per block (head_dim is 64 or 128)

template <typename T, int kPer>
__global__ void __launch_bounds__(kCombineThreads)
    attnCombine(void *out, const float *part, int nchunks, int D) {
    __shared__ float w[1024];  // per-chunk factor exp(m_c - M), nchunks <= 1024
    __shared__ float red[kCombineThreads];
    __shared__ float wred[kCombineThreads / kWave];
    constexpr int kGroups = kCombineThreads / kCombineCols;
    const int slabs = D / kCombineCols;
    const size_t ih = blockIdx.x / unsigned(slabs); // i * nh + h
    const int col0 = int(blockIdx.x % unsigned(slabs)) * kCombineCols;
    const float *pp = part + ih * size_t(nchunks) * (D + 2);
    const int t = threadIdx.x;
    const int e = col0 + t % kCombineCols, grp = t / kCombineCols;
    const float mc = t < nchunks ? pp[size_t(t) * (D + 2) + D] : -INFINITY;
    const float lc = t < nchunks ? pp[size_t(t) * (D + 2) + D + 1] : 0.0f;
    float v[kPer > 0 ? kPer : 1];
#pragma unroll
    for (int j = 0; j < kPer; ++j) { // unconditional (clamped) loads, used only for k < nchunks
        const int k = grp + j * kGroups;
        v[j] = pp[size_t(k < nchunks ? k : 0) * (D + 2) + e];
    }
    const float M = groupReduce<kCombineThreads, MaxOp>(mc, wred); // every thread gets it
    const float f = mc == M ? 1.0f : __expf(mc - M);                // mc = -inf: l = o = 0
    if (t < nchunks) w[t] = f;
    const float L = groupReduce<kCombineThreads, SumOp>(t < nchunks ? lc * f : 0.0f, wred);
    __syncthreads();
    float acc = 0.0f;
    if constexpr (kPer > 0) {
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const int k = grp + j * kGroups;
            if (k < nchunks) acc += v[j] * w[k];
        }
    } else {
#pragma unroll 8
        for (int k = grp; k < nchunks; k += kGroups) acc += pp[size_t(k) * (D + 2) + e] * w[k];
    }
    red[t] = acc;
    __syncthreads();
    if (t < kCombineCols) {
        float O = 0.0f;
        for (int g = 0; g < kGroups; ++g) O += red[g * kCombineCols + t];
        Fmt<T>::put(out, ih * D + col0 + t, L == 0.0f ? 0.0f : O / L);
    }
}

template <typename T>
void launchCombine(void *out, const float *part, int nchunks, int D, size_t pairs, hipStream_t s) {
    const unsigned blocks = unsigned(pairs) * unsigned(D / kCombineCols);
    if (nchunks <= 8 * (kCombineThreads / kCombineCols))
        attnCombine<T, 8><<<blocks, kCombineThreads, 0, s>>>(out, part, nchunks, D);
    else
        attnCombine<T, 0><<<blocks, kCombineThreads, 0, s>>>(out, part, nchunks, D);
}

// Any head_dim / v_head_dim / group: one wave per (query, head), keys one at a time with an
// online softmax; the output accumulates in LDS (dv floats per wave, lane j owns the
// columns j, j + 64, ...).  For the shapes the vector kernel does not take.
template <typename T, bool kInt8>
__global__ void __launch_bounds__(kWave)
    attnScalar(AttnArgs a, int d, int dv) {
    extern __shared__ float acc[]; // dv
    const size_t ih = blockIdx.x;
    const size_t i = ih / size_t(a.nh);
    const int h = int(ih % size_t(a.nh));
    const int g = h / a.group;
    const int lane = threadIdx.x;
    const size_t vis = visibleKeys(a.total, a.seq, i);
    const auto kval = [&](size_t t, int e) {
        const size_t row = t * size_t(a.nkvh) + size_t(g);
        if constexpr (kInt8)
            return Fmt<T>::round(float(static_cast<const int8_t *>(a.k)[row * d + e]) * a.ks[row]);
        else
            return Fmt<T>::get(a.k, row * d + e);
    };
    const auto vval = [&](size_t t, int e) {
        const size_t row = t * size_t(a.nkvh) + size_t(g);
        if constexpr (kInt8)
            return Fmt<T>::round(float(static_cast<const int8_t *>(a.v)[row * dv + e]) * a.vs[row]);
        else
            return Fmt<T>::get(a.v, row * dv + e);
    };
    for (int e = lane; e < dv; e += kWave) acc[e] = 0.0f;
    float m = -INFINITY, l = 0.0f;
    for (size_t t = 0; t < vis; ++t) {
        float dot = 0.0f;
        for (int e = lane; e < d; e += kWave) dot = __builtin_fmaf(Fmt<T>::get(a.q, (i * a.nh + h) * d + e), kval(t, e), dot);
        dot = waveGroupReduce<kWave, SumOp>(dot);
        const float s = dot * a.scale;
        if (s == -INFINITY) continue; // weight 0
        const float mx = fmaxf(m, s);
        const float corr = mx == m ? 1.0f : __expf(m - mx);
        const float p = __expf(s - mx);
        l = l * corr + p;
        for (int e = lane; e < dv; e += kWave) acc[e] = acc[e] * corr + p * vval(t, e);
        m = mx;
    }
    const float inv = l == 0.0f ? 0.0f : 1.0f / l; // (NaN for a NaN score)
    for (int e = lane; e < dv; e += kWave) Fmt<T>::put(a.out, ih * dv + e, acc[e] * inv);
}

// 8 consecutive elements of a cache row (128 per row) as raw bits: bf16 (16 bytes) or INT8
// codes (8 bytes, in .x / .y).
template <bool kInt8>
__device__ __forceinline__ v4u loadRow8(const void *base, size_t row, int col) {
    if constexpr (kInt8) {
        typedef uint32_t v2u __attribute__((ext_vector_type(2)));
        const v2u c = *reinterpret_cast<const v2u *>(static_cast<const int8_t *>(base) + row * 128 + col);
        return v4u{c.x, c.y, 0u, 0u};
    } else {
        return *reinterpret_cast<const v4u *>(static_cast<const uint16_t *>(base) + row * 128 + col);
    }
}

// 8 INT8 codes -> bf16(code * sc) as 4 packed words.  code = u - 128 for the unsigned byte
// u of code ^ 0x80, and fma(u, sc, -128 sc) rounds u * sc - 128 sc = code * sc once (-128 sc
// is exact), i.e. exactly float(code) * sc; the pair conversion then rounds to bf16 as the
// reference does for every non-NaN value.
__device__ __forceinline__ v4u codesToBf16(const v4u &raw, float sc) {
    const uint32_t ux = raw.x ^ 0x80808080u, uy = raw.y ^ 0x80808080u;
    const float off = -128.0f * sc;
    const auto cv = [&](uint32_t u, int k) {
        const float b = float((u >> (8 * k)) & 0xFFu); // v_cvt_f32_ubyte{k}
        return __builtin_fmaf(b, sc, off);
    };
    return v4u{Bf16Cvt::narrow2Q(cv(ux, 0), cv(ux, 1)), Bf16Cvt::narrow2Q(cv(ux, 2), cv(ux, 3)),
               Bf16Cvt::narrow2Q(cv(uy, 0), cv(uy, 1)), Bf16Cvt::narrow2Q(cv(uy, 2), cv(uy, 3))};
}

// ---- prefill on MFMA (bf16 / f16, head_dim 64 or 128, cache in the type or INT8) --------------
// A block takes 32 queries of 2 q heads of one kv head (odd groups: 64 queries of one q head), a
// "unit" each, and its 2 x kSplits waves walk the keys in steps of kSplits x 32: wave (unit u,
// split s) takes keys 32 s .. + 31 of every step, so the splits of a unit stay balanced up to the
// causal diagonal and merge through LDS at the end.  Per step a wave forms S^T = K Q^T (32 keys x
// 32 queries) and O^T += V^T P^T with v_mfma_f32_32x32x16: A[m = l % 32][k = 8 (l / 32) + j],
// B[k = 8 (l / 32) + j][n = l % 32], D[m = 8 (i / 4) + 4 (l / 32) + i % 4][n = l % 32].  Row m =
// 16 g + 8 a + 4 h + b of K is key 16 g + 8 h + 4 a + b, so lane half h ends with the scores of keys
// 16 g + 8 h + 0 .. 7 of its query -- the 8 consecutive k of the P V product's B operand -- and the
// softmax needs one exchange between the two lanes of a query.  P enters as two 16-bit parts (hi +
// lo: 2^-17 relative in bf16, 2^-22 in f16), which is less than the f32 weights of the vector kernel:
// over 12 to 32 heads and 16 to 1500 keys the error against 64 bits is the vector kernel's to five
// digits in bf16 (4 to 15 in 10000 outputs are not the exact value's rounding, 1 to 4 there) and within
// 0.5% in f16.  In f16 the weights carry a factor 2^8, which keeps the low parts of weights down to 2^-11
// normal numbers and cancels in O / l.
//
// K and V tiles move HBM -> LDS with global_load_lds_dwordx4 (1 KB per instruction, two stages, the
// next step's loads in flight during this one's math).  V stays row-major; its transposed operand
// is two ds_read_b64_tr_b16: within 16 lanes, lane j's element e is element j % 4 of the 8 bytes
// that lane 4 e + j / 4 addresses.  Rows cannot be padded (the load fills LDS contiguously), so the
// 16-byte chunks of a row are XOR-swizzled: K so that 16 rows' reads of one chunk touch all banks,
// V so that the 64-byte pieces of 4 rows do.  The codes of an INT8 cache are converted on their way into
// LDS, or the cache is dequantized into the workspace first (planPrefill; the same operands, the same bits).
// Keys past the cache read row 0 and weigh 0, as masked keys do; what a non-finite V element of
// such a row leaves in the sums is replaced at the end (visibleSum).
//
// What bounds it: a step is 24 MFMAs (about 950 cycles) and 800 cycles of VALU work (16 exponentials
// per lane and their two parts) per wave, two waves on a SIMD walking the same phases between barriers:
// 1.9 us a step, near the sum of the phases.  Waves with tiles of their own and no barrier (two units
// per wave), or four waves on a SIMD, came to the same 3.8 us per 256 keys, and running one unit half a
// step behind the other spilled registers.
// 2048 queries, 12 / 2 heads, bf16: 44.9 us with 16-query tiles and one wave per q head on 16 x 16
// x 32 MFMAs (1 KB of LDS read per 16 MFMA cycles, CUs with early queries idle) -> 36.4 us; f16, 300
// queries over 1500 INT8 keys: 479 us on the vector kernel -> 25.5 us.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));

constexpr int kMfmaQ = 16;   // fewest queries that take the prefill kernel
constexpr int kSplits = 4;   // waves per unit, each with 32 keys of a step
constexpr int kStepKeys = 32 * kSplits;

__device__ __forceinline__ bf16x8 asBf16x8(const v4u &r) { return __builtin_bit_cast(bf16x8, r); }

typedef short v4s __attribute__((ext_vector_type(4)));
__device__ __forceinline__ int swzV(int r) { return ((r & 3) | (((r >> 3) & 1) << 2)) << 1; }
__device__ __forceinline__ uint64_t ldsReadTr16(const char *p) {
    const v4s r = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s *)(p));
    return __builtin_bit_cast(uint64_t, r);
}

// Two f32 as two elements of T (hi), and what is left of them as two more (lo)
template <typename T>
__device__ __forceinline__ void splitPair(float x0, float x1, uint32_t &hi, uint32_t &lo) {
    if constexpr (std::is_same_v<T, BF16>) {
        hi = Bf16Cvt::narrow2Q(x0, x1);
        lo = Bf16Cvt::narrow2Q(x0 - __uint_as_float(hi << 16), x1 - __uint_as_float(hi & 0xFFFF0000u));
    } else {
        const v2h h = __builtin_convertvector(v2f{x0, x1}, v2h);
        hi = __builtin_bit_cast(uint32_t, h);
        lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f{x0 - float(h[0]), x1 - float(h[1])}, v2h));
    }
}

template <typename T>
__device__ __forceinline__ f32x16 mfma32(const v4u &a, const v4u &b, const f32x16 &c) {
    if constexpr (std::is_same_v<T, BF16>)
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(asBf16x8(a), asBf16x8(b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// 16 INT8 codes -> T(code * sc) as 8 packed words (bf16: codesToBf16's exact product)
template <typename T>
__device__ __forceinline__ void codesToRow(const v4u &raw, float sc, v4u (&out)[2]) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const v4u half = h ? v4u{raw.z, raw.w, 0u, 0u} : v4u{raw.x, raw.y, 0u, 0u};
        if constexpr (std::is_same_v<T, BF16>) {
            out[h] = codesToBf16(half, sc);
        } else {
            float f[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) f[e] = float(int8_t(half[e / 4] >> (8 * (e % 4)))) * sc;
            out[h] = Fmt<F16>::pack(f);
        }
    }
}

// Keys that the queries [q0, q1] see: the most and the fewest.  Where seq > total the first seq -
// total queries wrap and see every key (visibleKeys).
__device__ __forceinline__ void visibleRange(size_t total, size_t seq, size_t q0, size_t q1, size_t &most, size_t &least) {
    const size_t wrapped = seq > total ? seq - total : 0;
    most = q0 < wrapped ? total : visibleKeys(total, seq, q1);
    least = q1 < wrapped ? total : visibleKeys(total, seq, q0 < wrapped ? wrapped : q0);
}

// The value of the lane 32 away
__device__ __forceinline__ float otherHalf(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(threadIdx.x & 32 ? r[0] : r[1]);
}

// Column col of sum p V over the keys [k0, end) of kv head g for one q row, p = 2^(dot c2 - mc):
// a wave's work, 64 keys' weights at a time, only those keys' rows read.
template <typename T, bool kInt8, int D>
__device__ __forceinline__ float visibleSum(const AttnArgs &a, const uint16_t *qrow, int g, int col, size_t k0,
                                            size_t end, float c2, float mc) {
    using IO = RowIO<T, kInt8>;
    using QO = RowIO<T, false>;
    const int lane = int(threadIdx.x) % kWave;
    float acc = 0.0f;
    for (size_t kb = k0; kb < end; kb += kWave) {
        const size_t krow = min(kb + size_t(lane), end - 1) * size_t(a.nkvh) + size_t(g);
        float dot = 0.0f;
#pragma unroll 1
        for (int c = 0; c < D; c += 8) {
            float qf[8], kf[8];
            QO::unpack(QO::load(qrow, 0, D, c), 0.0f, qf);
            IO::unpack(IO::load(a.k, krow, D, c), kInt8 ? a.ks[krow] : 0.0f, kf);
#pragma unroll
            for (int e = 0; e < 8; ++e) dot = __builtin_fmaf(qf[e], kf[e], dot);
        }
        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(dot, c2, -mc));
        const int keys = int(min(end - kb, size_t(kWave)));
#pragma unroll 1
        for (int j = 0; j < keys; ++j) {
            const size_t vrow = (kb + size_t(j)) * size_t(a.nkvh) + size_t(g);
            float v;
            if constexpr (kInt8)
                v = Fmt<T>::round(float(static_cast<const int8_t *>(a.v)[vrow * D + col]) * a.vs[vrow]);
            else
                v = Fmt<T>::get(a.v, vrow * D + col);
            acc = __builtin_fmaf(__shfl(p, j, kWave), v, acc);
        }
    }
    return acc;
}

template <typename T, bool kInt8, int D, bool kHeads>
__global__ void __launch_bounds__(kWave * 2 * kSplits, 2)
    attnPrefill(AttnArgs a) {
    constexpr int RB = 2 * D, C = RB / 16;       // bytes and chunks of a key row
    constexpr int QS = D / 16, DT = D / 32;      // MFMA steps of q . k, column tiles of O
    constexpr int kTileB = 32 * RB;              // one K or V tile of a wave's step
    constexpr int kStageB = kSplits * 2 * kTileB; // [split][K tile | V tile]
    constexpr int kLoads = kTileB / 1024;        // loads per wave: unit 0 the K tile, unit 1 the V tile
    constexpr float kBias = std::is_same_v<T, F16> ? 8.0f : 0.0f; // base-2 exponent added to the weights
    __shared__ __align__(16) char lds[2 * kStageB];
    __shared__ float ml[2][kSplits][2][32];
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / kWave);
    const int unit = wave / kSplits, split = wave % kSplits;
    const int lane = int(threadIdx.x) % kWave;
    const int n = lane % 32, h2 = lane / 32;

    constexpr int kBlockQ = kHeads ? 32 : 64;
    const size_t nqb = (a.seq + kBlockQ - 1) / kBlockQ;
    unsigned b = blockIdx.x;
    const int c = int(b % unsigned(a.nchunks));
    b /= unsigned(a.nchunks);
    const int sl = int(b % unsigned(a.slices));
    b /= unsigned(a.slices);
    const int g = int(b % unsigned(a.nkvh));
    const size_t qb = nqb - 1 - size_t(b / unsigned(a.nkvh)); // latest queries (most keys) first
    const int h = g * a.group + (kHeads ? 2 * sl + unit : sl);
    const size_t q0 = qb * kBlockQ + (kHeads ? 0 : 32 * unit);
    const size_t qi = min(q0 + size_t(n), a.seq - 1); // this lane's query (clamped for loads)
    const size_t vis_q = visibleKeys(a.total, a.seq, qi);
    size_t most, least;
    visibleRange(a.total, a.seq, qb * kBlockQ, min(qb * kBlockQ + kBlockQ - 1, a.seq - 1), most, least);
    const size_t k0 = size_t(c) * size_t(a.chunk); // a multiple of kStepKeys
    const size_t k1 = a.nchunks == 1 ? most : min(most, k0 + size_t(a.chunk));
    const int steps = k1 > k0 ? int((k1 - k0 + kStepKeys - 1) / kStepKeys) : 0;
    const float c2 = a.scale * 1.4426950408889634f; // scores to base-2 exponents

    v4u qreg[QS];
#pragma unroll
    for (int st = 0; st < QS; ++st)
        qreg[st] = *reinterpret_cast<const v4u *>(static_cast<const uint16_t *>(a.q) + (qi * a.nh + h) * D + 16 * st + 8 * h2);
    float m = -INFINITY, lsum = 0.0f; // m: running max of the raw dots (scaled by c2 in use)
    f32x16 o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[dt][i] = 0.0f;

    const auto swzRow = [](bool v, int r) { // chunk XOR of row r of a tile
        if (D == 128) return v ? 4 * (r & 3) : r & 15;
        return v ? 4 * ((r >> 1) & 1) : (r >> 1) & 7;
    };
    // This wave's share of a step's loads: its split's K tile (unit 0) or V tile (unit 1).  Elements:
    // load j fills 1 KB, rows j kRows + lane / C: the row swizzles are those of lane / C, with bits 2 and 3 of
    // the chunk flipped by j % 4 for K, so the lane offsets are formed once and the rest of an address is
    // wave-uniform.  Codes: lane l takes 16-code pieces l, l + 64, ...
    constexpr int kRows = 1024 / RB;
    const uint32_t rowB = uint32_t(a.nkvh) * RB;
    uint32_t off[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) off[j] = uint32_t(lane / C) * rowB + 16 * ((lane % C) ^ swzRow(unit, j * kRows + lane / C));
    const char *cache = static_cast<const char *>(unit ? a.v : a.k);
    const float *cscale = unit ? a.vs : a.ks;
    char *const mine = lds + split * 2 * kTileB + unit * kTileB;
    constexpr int kCodeLoads = 32 * D / 16 / kWave;
    v4u craw[kInt8 ? kCodeLoads : 1];
    float csc[kInt8 ? kCodeLoads : 1];
    const auto issue = [&](int step, int stage) {
        const size_t t0 = k0 + size_t(step) * kStepKeys + size_t(32 * split);
        if constexpr (kInt8) {
#pragma unroll
            for (int j = 0; j < kCodeLoads; ++j) {
                const int piece = lane + kWave * j, row = piece / (D / 16), col = 16 * (piece % (D / 16));
                const size_t key = (t0 + row < a.total ? t0 + row : 0) * size_t(a.nkvh) + size_t(g);
                const v2u lo = *reinterpret_cast<const v2u *>(cache + key * D + col); // 8-byte aligned codes
                const v2u hi = *reinterpret_cast<const v2u *>(cache + key * D + col + 8);
                craw[j] = v4u{lo.x, lo.y, hi.x, hi.y};
                csc[j] = cscale[key];
            }
        } else {
            const char *base = cache + (t0 * size_t(a.nkvh) + size_t(g)) * RB; // wave-uniform
            // in scalar registers, formed anew each time: no per-load pointers are kept across the loop
            const uint64_t bits = reinterpret_cast<uint64_t>(base);
            base = reinterpret_cast<const char *>(uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(int(bits)))) |
                                                  uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(int(bits >> 32)))) << 32);
            char *dst = mine + stage * kStageB;
            if (t0 + 32 <= a.total) {
#pragma unroll
                for (int j = 0; j < kLoads; ++j)
                    __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1))) *)(base + size_t(j * kRows) * rowB + off[j % 4]),
                                                     (void __attribute__((address_space(3))) *)(dst + j * 1024), 16, 0, 0);
            } else { // rows past the cache read row 0
#pragma unroll
                for (int j = 0; j < kLoads; ++j) {
                    const bool in = t0 + size_t(j * kRows + lane / C) < a.total;
                    const char *src = in ? base + size_t(j * kRows) * rowB + off[j % 4]
                                         : cache + size_t(g) * RB + (off[j % 4] - uint32_t(lane / C) * rowB);
                    __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1))) *)(src),
                                                     (void __attribute__((address_space(3))) *)(dst + j * 1024), 16, 0, 0);
                }
            }
        }
    };
    const auto land = [&](int stage) { // the loads issued last are in LDS (this wave's)
        if constexpr (kInt8) {
#pragma unroll
            for (int j = 0; j < kCodeLoads; ++j) {
                const int piece = lane + kWave * j, row = piece / (D / 16), col = 2 * (piece % (D / 16));
                v4u el[2];
                codesToRow<T>(craw[j], csc[j], el);
#pragma unroll
                for (int e = 0; e < 2; ++e)
                    *reinterpret_cast<v4u *>(mine + stage * kStageB + row * RB + 16 * ((col + e) ^ swzRow(unit, row))) = el[e];
            }
        } else {
            waitVmcnt<0>();
        }
    };

    // This lane's operand addresses within a tile: K row krow (A row n), the chunk of step st by XOR with
    // 32 st; V pieces (4 columns of a row) of rows 8 h2 + (lane % 16) / 4, + 4 and + 16, the column tile dt
    // by XOR with 64 dt.
    const int krow = 16 * (n / 16) + 8 * ((n >> 2) & 1) + 4 * ((n >> 3) & 1) + n % 4;
    const int kaddr = krow * RB + 16 * (h2 ^ swzRow(false, krow));
    const int vrow = 8 * h2 + (lane % 16) / 4;
    const int vaddr = vrow * RB + 16 * ((2 * (lane / 16 % 2) + (lane % 4) / 2) ^ swzRow(true, vrow)) + 8 * (lane % 2);
    if (steps > 0) issue(0, 0);
    for (int it = 0; it < steps; ++it) {
        const int buf = it & 1;
        land(buf);
        ldsBarrier(); // every wave's tiles of this step are in LDS, and the other stage is no longer read
        if (it + 1 < steps) issue(it + 1, buf ^ 1);
        const size_t kt0 = k0 + size_t(it) * kStepKeys + size_t(32 * split);
        if (kt0 >= k1) continue; // the last step may not reach this split
        const char *kt = lds + buf * kStageB + split * 2 * kTileB, *vt = kt + kTileB;
        f32x16 s;
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = 0.0f;
#pragma unroll
        for (int st = 0; st < QS; ++st)
            s = mfma32<T>(*reinterpret_cast<const v4u *>(kt + (kaddr ^ (32 * st))), qreg[st], s);
        if (kt0 + 32 > least) { // the causal diagonal or the cache's end (block-uniform): mask
            const int nvis = int(min(vis_q - min(vis_q, kt0), size_t(32))) - 8 * h2;
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = 16 * (i / 8) + i % 8 < nvis ? s[i] : -INFINITY;
        }
        float mx = m;
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[i]);
        mx = fmaxf(mx, otherHalf(mx));
        // exp(scale (s - max)) as 2^(s c2 - max c2); a masked key (-inf) gets weight 0: mc = 0 while
        // every score is -inf keeps it 0 rather than NaN, with no per-score select
        const float mc = (mx == -INFINITY ? 0.0f : mx * c2) - kBias;
        float ps = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            s[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], c2, -mc));
            ps += s[i];
        }
        if (__builtin_expect(__any(mx != m), 0)) { // rescale only when a max moved
            const float corr = mx == m ? 1.0f : __builtin_amdgcn_exp2f(__builtin_fmaf(m, c2, -mc - kBias));
            lsum *= corr;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) o[dt] *= corr;
        }
        m = mx;
        lsum += ps;
#pragma unroll
        for (int kg = 0; kg < 2; ++kg) {
            uint32_t hw[4], lw[4];
#pragma unroll
            for (int w = 0; w < 4; ++w) splitPair<T>(s[8 * kg + 2 * w], s[8 * kg + 2 * w + 1], hw[w], lw[w]);
            const v4u phi = {hw[0], hw[1], hw[2], hw[3]}, plo = {lw[0], lw[1], lw[2], lw[3]};
            v4u vv[DT];
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                const char *vp = vt + (vaddr ^ (64 * dt)) + 16 * kg * RB;
                const uint64_t e0 = ldsReadTr16(vp), e1 = ldsReadTr16(vp + 4 * RB);
                vv[dt] = v4u{uint32_t(e0), uint32_t(e0 >> 32), uint32_t(e1), uint32_t(e1 >> 32)};
            }
            // (all column tiles before the second part: no MFMA waits for the one before it)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) o[dt] = mfma32<T>(vv[dt], phi, o[dt]);
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) o[dt] = mfma32<T>(vv[dt], plo, o[dt]);
        }
    }
    lsum += otherHalf(lsum);

    // merge the splits: every wave leaves (max, sum, output) in LDS, then wave (u, s) finishes the
    // column tiles s, s + kSplits, .. of unit u
    ldsBarrier(); // the tiles are no longer read
    float *const xo = reinterpret_cast<float *>(lds); // [unit][split][dt][i / 4][lane][4]
    static_assert(2 * kSplits * DT * 16 * kWave * 4 <= 2 * kStageB, "the outputs fit the tiles' storage");
    if (h2 == 0) {
        ml[unit][split][0][n] = m;
        ml[unit][split][1][n] = lsum;
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            *reinterpret_cast<f32x4 *>(xo + ((((unit * kSplits + split) * DT + dt) * 4 + q) * kWave + lane) * 4) =
                f32x4{o[dt][4 * q], o[dt][4 * q + 1], o[dt][4 * q + 2], o[dt][4 * q + 3]};
    ldsBarrier();
    const bool live = q0 + size_t(n) < a.seq;
    float M = -INFINITY, L = 0.0f, f[kSplits];
#pragma unroll
    for (int k = 0; k < kSplits; ++k) M = fmaxf(M, ml[unit][k][0][n]);
#pragma unroll
    for (int k = 0; k < kSplits; ++k) {
        const float mk = ml[unit][k][0][n];
        f[k] = mk == M ? 1.0f : __builtin_amdgcn_exp2f((mk - M) * c2); // 1 for M = -inf, where l = o = 0
        L += ml[unit][k][1][n] * f[k];
    }
    const size_t ih = qi * a.nh + size_t(h);
    float *const part = a.nchunks > 1 ? a.part + (ih * size_t(a.nchunks) + c) * (D + 2) : nullptr;
    static_assert(DT <= kSplits, "a wave finishes one column tile at most");
    if (split < DT) {
        const int dt = split;
        f32x4 O[4];
        float z = 0.0f; // NaN where an output is not finite
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            O[q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int k = 0; k < kSplits; ++k)
                O[q] += f[k] * *reinterpret_cast<const f32x4 *>(xo + ((((unit * kSplits + k) * DT + dt) * 4 + q) * kWave + lane) * 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) z = __builtin_fmaf(O[q][e], 0.0f, z);
        }
        // The MFMA also multiplies V rows that a query does not see (past the diagonal, and the filler past
        // the cache) by 0, and a visible infinity by a low part that may be 0 or negative: where an output is
        // not finite though the weights are (L), the query's 32 columns are summed again over its own keys.
        uint64_t redo = __ballot(live && z != z && L == L);
        if (__builtin_expect(redo != 0, 0)) {
            const float mc = (M == -INFINITY ? 0.0f : M * c2) - kBias;
            uint32_t rows = uint32_t(redo) | uint32_t(redo >> 32);
            while (rows) {
                const int r = __builtin_ctz(rows);
                rows &= rows - 1;
                const size_t i = q0 + size_t(r);
                const float y = visibleSum<T, kInt8, D>(a, static_cast<const uint16_t *>(a.q) + (i * a.nh + h) * D, g, 32 * dt + n, k0,
                                                        min(k1, visibleKeys(a.total, a.seq, i)), c2, __shfl(mc, r, kWave));
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float ye = __shfl(y, 8 * q + 4 * h2 + e, kWave);
                        O[q][e] = n == r ? ye : O[q][e];
                    }
            }
        }
        const float inv = L == 0.0f ? 0.0f : 1.0f / L;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (!live) break;
            const int col = 32 * dt + 8 * q + 4 * h2;
            if (part) {
#pragma unroll
                for (int e = 0; e < 4; ++e) part[col + e] = O[q][e];
            } else {
                using Cv = std::conditional_t<std::is_same_v<T, BF16>, Bf16Cvt, F16Cvt>; // the reference rounding
                *reinterpret_cast<v2u *>(static_cast<uint16_t *>(a.out) + ih * D + col) =
                    v2u{Cv::narrow(O[q][0] * inv) | (Cv::narrow(O[q][1] * inv) << 16), Cv::narrow(O[q][2] * inv) | (Cv::narrow(O[q][3] * inv) << 16)};
            }
        }
    }
    if (part && live && split == 0 && h2 == 0) {
        part[D] = M * a.scale; // the scaled units attnCombine works in
        part[D + 1] = L;
    }
}

// ---- prefill of few heads per kv head: 16 queries per block (bf16, head_dim 128) -------------
// A block takes 16 queries of W q heads of one kv head, a wave each (kSplit: two, each walking half
// of the 64-key tiles), on v_mfma_f32_16x16x32: S^T = K Q^T in 4 score tiles per step, lane (n, g4) with
// the scores of query n, then O^T += V^T P^T with P in two bf16 parts as attnPrefill's.  A[m = l % 16]
// [k = 8 (l / 16) + j], B[k = 8 (l / 16) + j][n = l % 16], D[m = 4 (l / 16) + i][n = l % 16]; row m of
// score tile t is key 32 (t / 2) + 8 (m / 4) + 4 (t % 2) + m % 4, so lane group g4 holds the 8
// consecutive keys its part of the P V product takes.  Tiles come by global_load_lds_dwordx4 in two
// stages, chunks swizzled by swzK / swzV.
constexpr int kTileKeys = 64;
__device__ __forceinline__ int swzK(int r) { return (r & 3) | (((r >> 3) & 3) << 2); }

template <int W>
__global__ void __launch_bounds__(kWave * W * 2)
    attnPrefill16(AttnArgs a) {
    constexpr int D = 128, KB = D / 32, DT = D / 16;
    constexpr int kRowB = 2 * D;               // bytes of a key row
    constexpr int kTileB = kTileKeys * kRowB;  // one K or V tile
    constexpr int kLoads = 2 * kTileB / 1024;  // 1 KB load instructions per stage
    constexpr int kPer = (kLoads + W - 1) / W;
    __shared__ __align__(16) char lds_all[2][2][2 * kTileB]; // [half][stage][K tile | V tile]
    const int wave_all = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / kWave);
    const int half = wave_all / W, wave = wave_all % W;
    const int lane = int(threadIdx.x) % kWave;
    const int n = lane % 16, g4 = lane / 16;

    const size_t nqb = (a.seq + 15) / 16;
    unsigned b = blockIdx.x;
    const int sl = int(b % unsigned(a.slices));
    b /= unsigned(a.slices);
    const int g = int(b % unsigned(a.nkvh));
    const size_t qb = nqb - 1 - size_t(b / unsigned(a.nkvh)); // latest queries first
    const int h = g * a.group + sl * W + wave;
    const size_t q0 = qb * 16;
    const size_t qi = min(q0 + size_t(n), a.seq - 1);
    const size_t vis_q = visibleKeys(a.total, a.seq, qi);
    size_t most, least;
    visibleRange(a.total, a.seq, q0, min(q0 + 15, a.seq - 1), most, least);
    const size_t ntiles = (most + kTileKeys - 1) / kTileKeys;
    const float c2 = a.scale * 1.4426950408889634f;

    bf16x8 qreg[KB];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
        const uint16_t *qp = static_cast<const uint16_t *>(a.q) + (qi * a.nh + h) * D + 32 * kb + 8 * g4;
        qreg[kb] = asBf16x8(*reinterpret_cast<const v4u *>(qp));
    }
    float m = -INFINITY, lsum = 0.0f;
    f32x4 o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[dt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // load instruction j of this wave is stage load q = wave + W j (K rows for q < 16, then
    // V rows): rows 4 (q % 16) + lane / 16 of the tile, LDS slot lane % 16 receiving chunk
    // slot ^ swizzle(row) of the kv head's row
    const size_t rowB = size_t(a.nkvh) * kRowB; // bytes between consecutive keys
    const char *cache[2] = {static_cast<const char *>(a.k), static_cast<const char *>(a.v)};
    // (byte offsets within a tile fit 32 bits: the launcher checks 64 rows * rowB < 2^31)
    int lrow[kPer];
    uint32_t loff[kPer], lcol[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int q = wave + W * j;
        const int row = 4 * (q % 16) + lane / 16, slot = lane % 16;
        const int chunk = slot ^ (q < 16 ? swzK(row) : swzV(row));
        lrow[j] = row;
        lcol[j] = uint32_t(g * kRowB + chunk * 16);
        loff[j] = uint32_t(row) * uint32_t(rowB) + lcol[j];
    }
    const auto issue = [&](size_t t0, int stage) {
        char *dst = &lds_all[half][stage][0];
        const size_t left = a.total - t0; // keys of the cache from t0 on (> 0)
        const bool full = left >= size_t(kTileKeys);
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const int q = wave + W * j;
            if (q >= kLoads) break;
            // the tile's rows from the tile base; in the cache's last tile, rows past it read row 0
            const char *src = full || size_t(lrow[j]) < left ? cache[q / 16] + t0 * rowB + loff[j]
                                                            : cache[q / 16] + lcol[j];
            __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1))) *)(src),
                                             (void __attribute__((address_space(3))) *)(dst + q * 1024), 16, 0, 0);
        }
    };

    const size_t nsteps = (ntiles + 1) / 2;
    const size_t tbeg = half ? nsteps : 0;
    const size_t tcount = half ? ntiles - nsteps : nsteps;
    if (tcount > 0) issue(tbeg * kTileKeys, 0);
    for (size_t it = 0; it < nsteps; ++it) {
        const int buf = int(it & 1);
        const size_t kt0 = (tbeg + it) * kTileKeys;
        waitVmcnt<0>(); // this wave's loads of tile it have landed
        ldsBarrier();   // every wave's have; every wave is past the step that read the other stage
        if (it + 1 < tcount) issue(kt0 + kTileKeys, buf ^ 1);
        if (it >= tcount) continue;
        const char *kt = &lds_all[half][buf][0], *vt = kt + kTileB;
        const bool whole = kt0 + kTileKeys <= least;
        const int nvis = int(min(vis_q - min(vis_q, kt0), size_t(kTileKeys)));
        float p[4][4];
        float mx = m;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int krow = 32 * (t / 2) + 8 * (n / 4) + 4 * (t % 2) + n % 4; // A row n
            const char *kr = kt + krow * kRowB;
            const int sw = swzK(krow);
            f32x4 acc = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int kb = 0; kb < KB; ++kb) {
                const v4u kv = *reinterpret_cast<const v4u *>(kr + 16 * ((4 * kb + g4) ^ sw));
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(asBf16x8(kv), qreg[kb], acc, 0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) p[t][i] = acc[i];
        }
        if (!whole) {
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int off = 32 * (t / 2) + 8 * g4 + 4 * (t % 2) + i;
                    p[t][i] = off < nvis ? p[t][i] : -INFINITY;
                }
        }
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) mx = fmaxf(mx, p[t][i]);
        mx = fmaxf(mx, __shfl_xor(mx, 16, kWave));
        mx = fmaxf(mx, __shfl_xor(mx, 32, kWave));
        const float mc = mx == -INFINITY ? 0.0f : mx * c2;
        float ps = 0.0f;
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                p[t][i] = __builtin_amdgcn_exp2f(__builtin_fmaf(p[t][i], c2, -mc));
                ps += p[t][i];
            }
        if (__builtin_expect(__any(mx != m), 0)) {
            const float corr = mx == m ? 1.0f : __builtin_amdgcn_exp2f(__builtin_fmaf(m, c2, -mc));
            lsum *= corr;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) o[dt] *= corr;
        }
        m = mx;
        lsum += ps;
        // the transposing reads' rows and column offset: keys 32 p2 + 8 g + n / 4 (and + 4),
        // columns 16 dt + 4 (n % 4) .. + 3, i.e. half n % 2 of chunk 2 dt + (n % 4) / 2
#pragma unroll
        for (int p2 = 0; p2 < 2; ++p2) {
            uint32_t hw[4], lw[4];
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const float x0 = p[2 * p2 + w / 2][2 * (w % 2)], x1 = p[2 * p2 + w / 2][2 * (w % 2) + 1];
                splitPair<BF16>(x0, x1, hw[w], lw[w]);
            }
            const bf16x8 bhi = asBf16x8(v4u{hw[0], hw[1], hw[2], hw[3]});
            const bf16x8 blo = asBf16x8(v4u{lw[0], lw[1], lw[2], lw[3]});
            const int r0 = 32 * p2 + 8 * g4 + n / 4;
            const char *v0 = vt + r0 * kRowB + 8 * (n % 2), *v1 = v0 + 4 * kRowB;
            const int sw = swzV(r0); // rows r0 and r0 + 4 share it
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                const int cofs = 16 * ((2 * dt + (n % 4) / 2) ^ sw);
                const uint64_t e0 = ldsReadTr16(v0 + cofs), e1 = ldsReadTr16(v1 + cofs);
                const v4u vv = v4u{uint32_t(e0), uint32_t(e0 >> 32), uint32_t(e1), uint32_t(e1 >> 32)};
                o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(asBf16x8(vv), bhi, o[dt], 0, 0, 0);
                o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(asBf16x8(vv), blo, o[dt], 0, 0, 0);
            }
        }
    }
    float lt = lsum + __shfl_xor(lsum, 16, kWave);
    lt += __shfl_xor(lt, 32, kWave);
    float *xch = reinterpret_cast<float *>(&lds_all[0][0][0]) + size_t(wave) * kWave * (2 + 4 * DT);
    __syncthreads();
    if (half == 1) {
        xch[lane] = m;
        xch[kWave + lane] = lt;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int i = 0; i < 4; ++i) xch[(2 + 4 * dt + i) * kWave + lane] = o[dt][i];
    }
    __syncthreads();
    if (half == 1) return;
    const float m1 = xch[lane], l1 = xch[kWave + lane];
    const float M = fmaxf(m, m1);
    const float f0 = m == M ? 1.0f : __builtin_amdgcn_exp2f(__builtin_fmaf(m, c2, -M * c2));
    const float f1 = m1 == M ? 1.0f : __builtin_amdgcn_exp2f(__builtin_fmaf(m1, c2, -M * c2));
    lt = lt * f0 + l1 * f1;
    m = M;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) o[dt][i] = o[dt][i] * f0 + xch[(2 + 4 * dt + i) * kWave + lane] * f1;
    // as attnPrefill: a query whose outputs are not finite though its weights are is summed again over
    // its own keys, 64 columns at a time
    const bool live = q0 + size_t(n) < a.seq;
    float z = 0.0f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) z = __builtin_fmaf(o[dt][i], 0.0f, z);
    const uint64_t redo = __ballot(live && z != z && lt == lt);
    if (__builtin_expect(redo != 0, 0)) {
        const float mc = m == -INFINITY ? 0.0f : m * c2;
        uint32_t rows = uint32_t(redo | redo >> 16 | redo >> 32 | redo >> 48) & 0xFFFFu;
        while (rows) {
            const int r = __builtin_ctz(rows);
            rows &= rows - 1;
            const size_t i = q0 + size_t(r);
            const uint16_t *qrow = static_cast<const uint16_t *>(a.q) + (i * a.nh + h) * D;
#pragma unroll
            for (int ch = 0; ch < 2; ++ch) {
                const float y = visibleSum<BF16, false, D>(a, qrow, g, kWave * ch + lane, 0, visibleKeys(a.total, a.seq, i), c2,
                                                           __shfl(mc, r, kWave));
#pragma unroll
                for (int dt = 0; dt < DT / 2; ++dt)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float ye = __shfl(y, 16 * dt + 4 * g4 + e, kWave);
                        f32x4 &od = o[DT / 2 * ch + dt];
                        od[e] = n == r ? ye : od[e];
                    }
            }
        }
    }
    if (!live) return;
    const float inv = lt == 0.0f ? 0.0f : 1.0f / lt;
    uint16_t *op = static_cast<uint16_t *>(a.out) + (qi * a.nh + h) * D + 4 * g4;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
        const uint32_t w0 = f32ToBf16(o[dt][0] * inv) | (f32ToBf16(o[dt][1] * inv) << 16);
        const uint32_t w1 = f32ToBf16(o[dt][2] * inv) | (f32ToBf16(o[dt][3] * inv) << 16);
        *reinterpret_cast<v2u *>(op + 16 * dt) = v2u{w0, w1};
    }
}

// Merge of few chunk partials for many (query, head) pairs: a thread per 4 columns of a pair.
// (attnCombine spends 1024 threads on 32 columns of a pair, for up to 1024 chunks.)
template <typename T>
__global__ void __launch_bounds__(256)
    attnCombineFew(void *out, const float *part, int nchunks, int D, size_t pairs) {
    const size_t idx = size_t(blockIdx.x) * 256 + threadIdx.x;
    const int per = D / 4;
    const size_t ih = idx / per;
    if (ih >= pairs) return;
    const int col = 4 * int(idx % per);
    const float *pp = part + ih * size_t(nchunks) * (D + 2);
    float M = -INFINITY, L = 0.0f, O[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int c = 0; c < nchunks; ++c) M = fmaxf(M, pp[size_t(c) * (D + 2) + D]);
    for (int c = 0; c < nchunks; ++c) {
        const float *pc = pp + size_t(c) * (D + 2);
        const float f = pc[D] == M ? 1.0f : __expf(pc[D] - M); // 1 for M = -inf, where l = o = 0
        L += pc[D + 1] * f;
#pragma unroll
        for (int e = 0; e < 4; ++e) O[e] += pc[col + e] * f;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) Fmt<T>::put(out, ih * D + col + e, L == 0.0f ? 0.0f : O[e] / L);
}

// ---- decode on MFMA (bf16 q / out, head_dim 128, cache in bf16 or INT8) ---------------
// Few queries, long cache.  Block = (query, kv head, key chunk), NW waves; each wave takes
// 32-key steps of the chunk on its own.  The MFMA columns are the G (<= 16) q heads of the
// kv head (columns past G hold zero queries and are never written): S^T = K Q^T over 2
// tiles of 16 keys (row m of tile t is key 8(m / 4) + 4t + m % 4, so lane group g holds keys
// 8g .. 8g + 7 and P^T is the B operand of one 32-key P V product as the lanes hold it),
// then O^T += V^T P^T with the V rows staged through the wave's own LDS slice and read
// back transposed (no block barrier inside the loop).  K enters the A operand straight
// from memory: bf16 rows, or INT8 codes turned into bf16(code * scale) (codesToBf16) with
// the step's scales shared by shuffles.  The waves merge in LDS; a split launch writes
// chunk partials in the layout attnCombine merges (max in scaled units).
constexpr int kDecWaves = 2;
constexpr int kDecKT = 32;   // keys per wave step

template <bool kInt8, int NW>
__global__ void __launch_bounds__(kWave * NW)
    attnDecodeMfma(AttnArgs a) {
    constexpr int D = 128, KB = D / 32, DT = D / 16;
    __shared__ __align__(16) char vrow[NW][kDecKT * 2 * D]; // the wave's V rows, chunks swizzled (swzV)
    __shared__ float st[NW][16][D + 2];
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / kWave);
    const int lane = int(threadIdx.x) % kWave;
    const int n = lane % 16, g4 = lane / 16;

    unsigned b = blockIdx.x;
    const int c = int(b % unsigned(a.nchunks));
    b /= unsigned(a.nchunks);
    const int g = int(b % unsigned(a.nkvh));
    const size_t i = a.seq - 1 - size_t(b / unsigned(a.nkvh));
    const size_t vis = visibleKeys(a.total, a.seq, i);
    const size_t k0 = size_t(c) * size_t(a.chunk);
    const size_t k1 = min(vis, k0 + size_t(a.chunk));
    const bool col_ok = n < a.group;
    const int hq = g * a.group + (col_ok ? n : 0); // this column's q head (clamped)
    const float c2 = a.scale * 1.4426950408889634f;
    const size_t rstride = size_t(a.nkvh);          // rows between keys

    bf16x8 qreg[KB];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
        v4u r = v4u{0u, 0u, 0u, 0u};
        if (col_ok)
            r = *reinterpret_cast<const v4u *>(static_cast<const uint16_t *>(a.q) + (i * a.nh + hq) * D + 32 * kb + 8 * g4);
        qreg[kb] = asBf16x8(r);
    }
    float m = -INFINITY, lsum = 0.0f; // m: max of the raw dots
    f32x4 o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[dt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    for (size_t kt0 = k0 + size_t(wave) * kDecKT; kt0 < k1; kt0 += size_t(NW) * kDecKT) {
        const int nk = int(min(k1 - kt0, size_t(kDecKT)));
        const bool part = nk < kDecKT; // the chunk's last, partial step (wave-uniform)
        // Loads are unconditional: a key past the step reads the step's first key and is
        // zeroed after the load (partial steps only).  Loads under per-lane branches were
        // issued one round trip at a time.
        // V pieces: piece r of a lane is key 4r + lane / 16, columns 8 (lane % 16) .. + 7, so
        // 16 lanes read one row contiguously
        v4u vr[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            const int kr = 4 * r + lane / 16;
            const int key = kr < nk ? kr : 0;
            vr[r] = loadRow8<kInt8>(a.v, (kt0 + key) * rstride + g, 8 * (lane % 16));
        }
        // K operands: tile t, row n -> key 8(n / 4) + 4t + n % 4
        v4u ka[2][KB];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int off = 8 * (n / 4) + 4 * t + n % 4;
            const int key = off < nk ? off : 0;
#pragma unroll
            for (int kb = 0; kb < KB; ++kb)
                ka[t][kb] = loadRow8<kInt8>(a.k, (kt0 + key) * rstride + g, 32 * kb + 8 * g4);
        }
        if (part) {
#pragma unroll
            for (int r = 0; r < 8; ++r)
                if (4 * r + lane / 16 >= nk) vr[r] = v4u{0u, 0u, 0u, 0u};
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int kb = 0; kb < KB; ++kb)
                    if (8 * (n / 4) + 4 * t + n % 4 >= nk) ka[t][kb] = v4u{0u, 0u, 0u, 0u};
        }
        if constexpr (kInt8) {
            // the step's scales, one load per lane (K for lanes 0-31, V for 32-63), handed
            // to the lanes that convert a row by lane shuffles
            const int sk = lane % kDecKT;
            float sreg = (lane < kDecKT ? a.ks : a.vs)[(kt0 + (sk < nk ? sk : 0)) * rstride + g];
            if (sk >= nk) sreg = 0.0f;
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const float sc = __shfl(sreg, 8 * (n / 4) + 4 * t + n % 4, kWave);
#pragma unroll
                for (int kb = 0; kb < KB; ++kb) ka[t][kb] = codesToBf16(ka[t][kb], sc);
            }
#pragma unroll
            for (int r = 0; r < 8; ++r) vr[r] = codesToBf16(vr[r], __shfl(sreg, kDecKT + 4 * r + lane / 16, kWave));
        }
        float p[2][4];
        float mx = m;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            f32x4 acc = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int kb = 0; kb < KB; ++kb)
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(asBf16x8(ka[t][kb]), qreg[kb], acc, 0, 0, 0);
#pragma unroll
            for (int ii = 0; ii < 4; ++ii) p[t][ii] = acc[ii];
        }
        if (nk < kDecKT) { // the chunk's last, partial step: keys past its end are masked
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int ii = 0; ii < 4; ++ii) // key of D row 4g + ii
                    p[t][ii] = 8 * g4 + 4 * t + ii < nk ? p[t][ii] : -INFINITY;
        }
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int ii = 0; ii < 4; ++ii) mx = fmaxf(mx, p[t][ii]);
        mx = fmaxf(mx, __shfl_xor(mx, 16, kWave));
        mx = fmaxf(mx, __shfl_xor(mx, 32, kWave));
        // a masked key (-inf) gets weight 0; mc = 0 while every score is -inf keeps it 0
        // rather than NaN, with no per-score select
        const float mc = mx == -INFINITY ? 0.0f : mx * c2;
        float ps = 0.0f;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int ii = 0; ii < 4; ++ii) {
                p[t][ii] = __builtin_amdgcn_exp2f(__builtin_fmaf(p[t][ii], c2, -mc));
                ps += p[t][ii];
            }
        if (__builtin_expect(__any(mx != m), 0)) {
            const float corr = mx == m ? 1.0f : __builtin_amdgcn_exp2f(__builtin_fmaf(m, c2, -mc));
            lsum *= corr;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) o[dt] *= corr;
        }
        m = mx;
        lsum += ps;
        // V rows into this wave's slice as loaded (the previous step's reads of it are done:
        // one wave, in order; the fences keep the compiler from moving accesses across); 16
        // lanes write one row's 16 chunks, whatever the swizzle: no bank conflicts
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            const int kr = 4 * r + lane / 16;
            *reinterpret_cast<v4u *>(&vrow[wave][kr * 2 * D + 16 * ((lane % 16) ^ swzV(kr))]) = vr[r];
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        // P as bf16 hi + lo, two keys per conversion (key 8g + j is p[j / 4][j % 4])
        uint32_t hw[4], lw[4];
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const float x0 = p[w / 2][2 * (w % 2)], x1 = p[w / 2][2 * (w % 2) + 1];
            hw[w] = Bf16Cvt::narrow2Q(x0, x1);
            lw[w] = Bf16Cvt::narrow2Q(x0 - __uint_as_float(hw[w] << 16), x1 - __uint_as_float(hw[w] & 0xFFFF0000u));
        }
        const bf16x8 bhi = asBf16x8(v4u{hw[0], hw[1], hw[2], hw[3]});
        const bf16x8 blo = asBf16x8(v4u{lw[0], lw[1], lw[2], lw[3]});
        // V^T operands by transposing reads: lane n of group g gets keys 8g .. 8g + 7 of column
        // 16 dt + n from lanes reading key rows 8g + n / 4 (and + 4), columns 16 dt + 4 (n % 4) ..
        const int r0 = 8 * g4 + n / 4;
        const char *v0 = &vrow[wave][r0 * 2 * D + 8 * (n % 2)], *v1 = v0 + 4 * 2 * D;
        const int vsw = swzV(r0); // rows r0 and r0 + 4 share it
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            const int cofs = 16 * ((2 * dt + (n % 4) / 2) ^ vsw);
            const uint64_t e0 = ldsReadTr16(v0 + cofs), e1 = ldsReadTr16(v1 + cofs);
            const v4u vv = v4u{uint32_t(e0), uint32_t(e0 >> 32), uint32_t(e1), uint32_t(e1 >> 32)};
            o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(asBf16x8(vv), bhi, o[dt], 0, 0, 0);
            o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(asBf16x8(vv), blo, o[dt], 0, 0, 0);
        }
    }
    float lt = lsum + __shfl_xor(lsum, 16, kWave);
    lt += __shfl_xor(lt, 32, kWave);
    if (col_ok) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int ii = 0; ii < 4; ++ii) st[wave][n][16 * dt + 4 * g4 + ii] = o[dt][ii];
        if (g4 == 0) {
            st[wave][n][D] = m;
            st[wave][n][D + 1] = lt;
        }
    }
    __syncthreads();
    for (int pi = threadIdx.x; pi < a.group * D; pi += kWave * NW) {
        const int j = pi / D, e = pi % D;
        float M = -INFINITY;
#pragma unroll
        for (int w = 0; w < NW; ++w) M = fmaxf(M, st[w][j][D]);
        float L = 0.0f, O = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const float mw = st[w][j][D];
            const float f = mw == M ? 1.0f : __builtin_amdgcn_exp2f((mw - M) * c2); // 1 for M = -inf, where l = o = 0
            L += st[w][j][D + 1] * f;
            O += st[w][j][e] * f;
        }
        const size_t ih = i * a.nh + size_t(g * a.group + j);
        if (a.nchunks == 1) {
            Fmt<BF16>::put(a.out, ih * D + e, L == 0.0f ? 0.0f : O / L);
        } else {
            float *pp = a.part + (ih * size_t(a.nchunks) + c) * (D + 2);
            pp[e] = O;
            if (e == 0) {
                pp[D] = M * a.scale; // the scaled units attnCombine works in
                pp[D + 1] = L;
            }
        }
    }
}

// Heads per wave for a kv group: the largest supported count that divides it.
int sliceOf(int group) {
    for (int g : {8, 6, 4, 2})
        if (group % g == 0) return g;
    return 1;
}

// Load instructions per step of the vector kernel: 16 bytes of K and V codes per lane, or 32 of elements
constexpr int groupLoads(bool int8) { return int8 ? 8 : 4; }

template <typename T, bool kInt8, int D, int G>
void launchGroup(const AttnArgs &a, size_t blocks, hipStream_t s) {
    attnGroup<T, kInt8, D, G, groupLoads(kInt8)><<<unsigned(blocks), kWave * kWaves, 0, s>>>(a);
}

template <typename T, bool kInt8, int D>
void launchD(const AttnArgs &a, int G, size_t blocks, hipStream_t s) {
    switch (G) {
    case 8: return launchGroup<T, kInt8, D, 8>(a, blocks, s);
    case 6: return launchGroup<T, kInt8, D, 6>(a, blocks, s);
    case 4: return launchGroup<T, kInt8, D, 4>(a, blocks, s);
    case 2: return launchGroup<T, kInt8, D, 2>(a, blocks, s);
    default: return launchGroup<T, kInt8, D, 1>(a, blocks, s);
    }
}

// The vector kernels' shape and alignment condition.
bool vecShape(const AttnArgs &a, int d, int dv, bool int8) {
    const auto aligned = [](const void *p, size_t n) { return (reinterpret_cast<uintptr_t>(p) % n) == 0; };
    return d == dv && (d == 64 || d == 128) && aligned(a.q, 16) && aligned(a.out, 16) &&
           (int8 ? aligned(a.k, 8) && aligned(a.v, 8) : aligned(a.k, 16) && aligned(a.v, 16));
}

// Chunks of the vector kernel's keys.  A block's waves each take one step of keys (U loads) per chunk when
// the launch is split: about 2048 waves for decode, partials within the workspace and at most 1024 per
// (query, head).
size_t vectorChunks(const AttnArgs &a, int d, int U, size_t ws_bytes) {
    const size_t tile = size_t(kWave / (d / 8)) * size_t(U) * kWaves; // keys per block step
    const size_t groups = a.seq * size_t(a.nkvh) * size_t(a.group / sliceOf(a.group));
    if (groups >= 512 || a.total <= tile) return 1;
    const size_t n = std::min<size_t>((a.total + tile - 1) / tile, 1024);
    const size_t per = size_t(d + 2) * sizeof(float) * a.seq * size_t(a.nh);
    return std::max<size_t>(1, std::min(n, ws_bytes / per));
}

// Expected time in us of a launch of one block per CU at a time: the launch, and for each block `block` and,
// per 128 keys, `step` + `busy` times the share of CUs that have one.  The blocks with the most keys
// start first; of more than kCUs blocks, the longest that starts second starts after the shortest of
// the first kCUs.
constexpr double kLaunchUs = 2.4;
constexpr int kCUs = 256;
struct BlockTime {
    double block, step, busy;
    double stepUs(size_t blocks) const { return step + busy * std::min(1.0, double(blocks) / kCUs); }
};
double roundsUs(const BlockTime &t, size_t blocks, size_t longest, size_t shortest) {
    const double full = double(blocks) / kCUs, lo = double(shortest), hi = double(longest), step = t.stepUs(blocks);
    double us = t.block + step * hi;
    // (1.07: rounds do not follow on each other without a gap)
    if (full > 1.0)
        us = std::max({us, 1.07 * full * (t.block + step * (lo + hi) / 2), 1.07 * 2 * (t.block + step * (hi - (hi - lo) / full))});
    return kLaunchUs + us;
}

// How a call of 16 or more queries runs (bf16 or f16, head_dim 64 or 128, a non-empty cache and a
// positive finite scale: the MFMA kernels track the max of the raw dot products).
enum class PrefillKernel { k32, k16, kGroup, kGroup8 }; // attnPrefill, attnPrefill16, attnGroup with 4 and 8 loads per step
struct Prefill {
    PrefillKernel kernel;
    int heads;     // q heads per block; attnPrefill: 2, or 1 of 64 queries
    int chunk, nchunks;
    size_t blocks, part_bytes;
    bool elements; // an INT8 cache is dequantized into the workspace first
    size_t need;   // bytes of workspace it cannot do without
};
constexpr size_t kPrefillPartBytes = size_t(8) << 20;

// attnPrefill's times by type, head_dim and cache (Codes: INT8 converted in the kernel), with those of
// a launch whose keys are split: a chunk's merge and its 10000 partials.  From sweeps over 16 to 512
// (bf16, 128: 2048) queries, 0 to 1600 (4096) earlier keys and ten head counts; rms error 3 to 5%.
struct PrefillTime {
    BlockTime t;
    double merge, partials;
};
constexpr PrefillTime kBf16D128{{4.32, 1.62, 0.32}, 0.88, 3.4}, kBf16D128Codes{{3.96, 2.29, 0.18}, 0.84, 3.2};
constexpr PrefillTime kBf16D64{{2.78, 1.20, 0.24}, 1.10, 1.5}, kBf16D64Codes{{2.63, 1.51, 0.19}, 1.10, 1.5};
constexpr PrefillTime kF16D128{{5.17, 1.60, 0.51}, 0.77, 2.9}, kF16D64{{4.15, 1.19, 0.24}, 0.72, 1.4};
// attnPrefill16 with 1, 2 and 4 heads per block; rms error 2 to 3%
constexpr BlockTime kTiles16[3] = {{2.03, 1.95, 0.0}, {2.07, 1.62, 0.04}, {2.82, 1.68, 0.13}};
// attnGroup over elements with 1 and 2 heads per block (more heads, and f16 with head_dim 64, are slower
// than attnPrefill at every size measured): a launch, a round of kCUs blocks, 100000 block keys, a key tile, and split as above
struct GroupTime {
    double base, round, keys, tile, merge, partials;
};
constexpr GroupTime kGroupBf16D64[2] = {{1.09, 0.70, 1.12, 0.24, 3.6, 15.2}, {1.25, 1.46, 0.98, 0.95, 2.9, 23.7}};
constexpr GroupTime kGroupF16D128[2] = {{3.39, 1.60, 6.41, 1.06, 3.1, 42.7}, {3.60, 2.75, 0.0, 2.45, 2.5, 60.0}};

// Dequantizing an INT8 cache of `el` elements (K and V): a launch, which small caches are not much more than
double dequantizeUs(size_t el) {
    const double m = double(el) * 1e-6;
    return 2.0 + std::min(5.0 * m, 3.0 + 1.3 * m);
}

// How the prefill is cut; false where it does not apply.  Kernel and cut depend on the shape only, not
// on the entry point or on how the cache is kept, so that all of them give the same bits.
//  - attnPrefill: keys are split over blocks where the query blocks alone would leave CUs idle, into
//    chunks of at least 4 steps (512 keys): 16 queries over 32768 keys would otherwise be 256 steps in
//    each of 6 blocks.
//  - Its block costs about 4 us beside its steps, so calls of few steps and of less than two rounds of
//    small blocks run faster on attnPrefill16 (bf16, 128; 100 queries, 32 / 8 heads 8.3 -> 6.2 us) or
//    attnGroup (16 queries, 16 / 16 heads of 64, bf16 6.2 -> 4.7 us).
//  - attnPrefill converts a bf16 INT8 cache in the kernel until the query blocks that convert a tile again
//    cost more than one launch that dequantizes it (16 / 16 heads of 128, 64 queries over 1264 keys 28.8 ->
//    21.6 us; from about 3000 queries the other way round).  f16 codes cost five times as much.
bool planPrefill(Prefill &p, const AttnArgs &a, int d, int dv, bool int8, llaisysDataType_t dt) {
    const bool bf16 = dt == LLAISYS_DTYPE_BF16;
    if ((!bf16 && dt != LLAISYS_DTYPE_F16) || !vecShape(a, d, dv, int8)) return false;
    if (a.total == 0 || a.seq < size_t(kMfmaQ) || !(a.scale > 0.0f) || !std::isfinite(a.scale)) return false;
    // the kernel's lane offsets within one 1 KB load (512 / d key rows) have 32 bits
    if (size_t(a.nkvh) * 1024 >= size_t(1) << 32) return false;
    const size_t nh = size_t(a.nh), bq = a.group % 2 == 0 ? 32 : 64;
    p.kernel = PrefillKernel::k32;
    p.heads = a.group % 2 == 0 ? 2 : 1;
    p.blocks = (a.seq + bq - 1) / bq * (nh / p.heads);
    const size_t steps = (a.total + kStepKeys - 1) / kStepKeys;
    const size_t partial = a.seq * nh * size_t(d + 2) * sizeof(float);
    size_t n = std::max<size_t>(1, std::min({256 / p.blocks, steps / 4, kPrefillPartBytes / partial, size_t(1024)}));
    const size_t per = (steps + n - 1) / n;
    n = (steps + per - 1) / per;
    if (per * kStepKeys > size_t(INT32_MAX)) return false;
    p.chunk = int(per * kStepKeys);

    const size_t past = a.total > a.seq ? a.total - a.seq : 0;
    const double partials = double(a.seq * nh) * 1e-4;
    // steps of the block of the first q queries, the fewest
    const auto first = [&](size_t q) { return (std::min(a.total, past + q) + kStepKeys - 1) / kStepKeys; };
    const auto prefillUs = [&](const PrefillTime &t) {
        // (odd groups, up to 32 queries: the second unit's queries are repeats)
        if (n == 1) return (p.heads == 1 && a.seq <= 32 ? 0.9 : 1.0) * roundsUs(t.t, p.blocks, steps, first(bq));
        return kLaunchUs + t.t.block + t.t.stepUs(p.blocks * n) * double(per) + (t.merge + t.partials * partials) * double(n);
    };
    double us = prefillUs(bf16 ? (d == 128 ? kBf16D128 : kBf16D64) : (d == 128 ? kF16D128 : kF16D64));
    const size_t el = 2 * a.total * size_t(a.nkvh) * size_t(d), el_bytes = el * sizeof(uint16_t);
    const double deq = dequantizeUs(el);
    p.elements = int8 && !(bf16 && prefillUs(d == 128 ? kBf16D128Codes : kBf16D64Codes) < us + deq);
    // attnPrefill16 reads elements only: caches that an INT8 call can dequantize, whichever entry point it has
    const size_t ws = std::min(kNoAllocScratchBytes, selfAttentionWorkspaceBytes(a.seq, nh, size_t(d)));
    if (bf16 && d == 128 && el_bytes <= ws && size_t(a.nkvh) * 256 * kTileKeys < size_t(1) << 31) {
        for (int w : {4, 2, 1}) {
            if (a.group % w != 0 || (w == 1 && a.group % 2 == 0)) continue;
            const size_t blocks = (a.seq + 15) / 16 * (nh / size_t(w));
            const double t = roundsUs(kTiles16[w / 2], blocks, steps, first(16));
            if (blocks > 2 * kCUs || t >= us) continue;
            us = t;
            p.kernel = PrefillKernel::k16;
            p.heads = w;
            p.blocks = blocks;
            p.elements = int8;
        }
    }
    const int G = sliceOf(a.group);
    if (bf16 == (d == 64) && G <= 2) {
        const GroupTime &t = bf16 ? kGroupBf16D64[G - 1] : kGroupF16D128[G - 1];
        const size_t groups = a.seq * (nh / size_t(G)), tile = size_t(kWave / (d / 8)) * groupLoads(false) * kWaves;
        // one round of blocks over one to two tiles of keys: twice the loads per step and no split (64 queries
        // over 464 keys, 4 / 4 heads, bf16 10.1 -> 5.8 us, INT8 11.3 -> 7.7 us)
        const bool twice = bf16 && groups <= kCUs && a.total > tile && a.total <= 2 * tile;
        const size_t c = twice ? 1 : vectorChunks(a, d, groupLoads(false), selfAttentionWorkspaceBytes(a.seq, nh, size_t(d)));
        const double keys = double(a.total) - double(std::min(a.seq, a.total)) / 2;
        const double tiles = double(a.total) / double(tile);
        double g = kLaunchUs + t.base + t.round * std::ceil(double(groups * c) / kCUs) + t.keys * double(groups) * keys * 1e-5;
        g += c > 1 ? t.tile + t.merge + t.partials * partials * double(c) : t.tile * (tiles < 1 ? tiles : std::ceil(tiles));
        if ((twice || g < us) && groups * c < size_t(1) << 31) {
            p.kernel = twice ? PrefillKernel::kGroup8 : PrefillKernel::kGroup;
            p.heads = G;
            p.blocks = groups;
            p.chunk = int(c == 1 ? std::min<size_t>(a.total, size_t(INT32_MAX)) : (a.total + c - 1) / c);
            n = c;
            // 0.5 us and 1.5e-5 us per block and key is what the kernel takes longer over codes
            p.elements = int8 && !twice && (!bf16 || 0.5 + 1.5e-5 * double(groups * a.total) > deq);
        }
    }
    if (p.kernel == PrefillKernel::k16) n = 1;
    p.nchunks = int(n);
    p.blocks *= n;
    p.part_bytes = n > 1 ? partial * n : 0;
    p.need = int8 && p.kernel == PrefillKernel::k16 ? el_bytes : p.part_bytes;
    return p.blocks < (size_t(1) << 31);
}

template <typename T, bool kInt8, int D>
void launchPrefillKernel(const AttnArgs &a, const Prefill &p, hipStream_t s) {
    const unsigned blocks = unsigned(p.blocks);
    if (p.kernel == PrefillKernel::kGroup8) {
        if constexpr (std::is_same_v<T, BF16> && D == 64)
            p.heads == 2 ? attnGroup<T, kInt8, D, 2, 8><<<blocks, kWave * kWaves, 0, s>>>(a)
                         : attnGroup<T, kInt8, D, 1, 8><<<blocks, kWave * kWaves, 0, s>>>(a);
    } else if (p.kernel == PrefillKernel::kGroup) {
        // (the loads per step of elements also for codes, so that both sum in the same order)
        if constexpr (std::is_same_v<T, F16> == (D == 128))
            p.heads == 2 ? attnGroup<T, kInt8, D, 2, groupLoads(false)><<<blocks, kWave * kWaves, 0, s>>>(a)
                         : attnGroup<T, kInt8, D, 1, groupLoads(false)><<<blocks, kWave * kWaves, 0, s>>>(a);
    } else if (p.kernel == PrefillKernel::k16) {
        if constexpr (std::is_same_v<T, BF16> && !kInt8 && D == 128) {
            switch (p.heads) {
            case 4: attnPrefill16<4><<<blocks, kWave * 8, 0, s>>>(a); return;
            case 2: attnPrefill16<2><<<blocks, kWave * 4, 0, s>>>(a); return;
            default: attnPrefill16<1><<<blocks, kWave * 2, 0, s>>>(a); return;
            }
        }
    } else {
        constexpr unsigned threads = kWave * 2 * kSplits;
        p.heads == 2 ? attnPrefill<T, kInt8, D, true><<<blocks, threads, 0, s>>>(a)
                     : attnPrefill<T, kInt8, D, false><<<blocks, threads, 0, s>>>(a);
    }
}

template <typename T, bool kInt8>
void launchPrefill(const AttnArgs &a, const Prefill &p, int d, hipStream_t s) {
    if (d == 128)
        launchPrefillKernel<T, kInt8, 128>(a, p, s);
    else
        launchPrefillKernel<T, kInt8, 64>(a, p, s);
    if (p.nchunks == 1) return;
    const size_t pairs = a.seq * size_t(a.nh);
    if (p.nchunks <= 16 && p.kernel != PrefillKernel::kGroup)
        attnCombineFew<T><<<unsigned((pairs * size_t(d / 4) + 255) / 256), 256, 0, s>>>(a.out, a.part, p.nchunks, d, pairs);
    else
        launchCombine<T>(a.out, a.part, p.nchunks, d, pairs, s);
}

template <typename T, bool kInt8>
void launch(AttnArgs a, int d, int dv, void *ws, size_t ws_bytes, hipStream_t s) {
    if (a.seq == 0 || a.nh == 0) return;
    const bool vec = vecShape(a, d, dv, kInt8);
    if (!vec) {
        a.nchunks = 1;
        attnScalar<T, kInt8><<<unsigned(a.seq * size_t(a.nh)), kWave, size_t(dv) * sizeof(float), s>>>(a, d, dv);
        return;
    }
    const int G = sliceOf(a.group);
    a.slices = a.group / G;
    if constexpr (!std::is_same_v<T, F32>) {
        constexpr auto dt = std::is_same_v<T, BF16> ? LLAISYS_DTYPE_BF16 : LLAISYS_DTYPE_F16;
        Prefill p;
        if (planPrefill(p, a, d, dv, kInt8, dt) && p.need <= ws_bytes) {
            a.slices = a.group / p.heads;
            a.chunk = p.chunk;
            a.nchunks = p.nchunks;
            a.part = static_cast<float *>(ws);
            if constexpr (kInt8) {
                // Both caches in one launch, T(code * scale) as the tiles would be staged: the same
                // operands, the same bits.  A cache whose 16-bit form does not fit the workspace behind
                // the partials is converted in the kernel.
                const size_t cache_el = a.total * size_t(a.nkvh) * size_t(d), off = (p.part_bytes + 255) / 256 * 256;
                if (p.elements && off + 2 * cache_el * sizeof(uint16_t) <= ws_bytes) {
                    uint16_t *kd = reinterpret_cast<uint16_t *>(static_cast<char *>(ws) + off), *vd = kd + cache_el;
                    dequantizeInt8Pair(kd, static_cast<const int8_t *>(a.k), a.ks, a.total * size_t(a.nkvh), vd,
                                       static_cast<const int8_t *>(a.v), a.vs, a.total * size_t(a.nkvh),
                                       size_t(d), dt, s);
                    a.k = kd;
                    a.v = vd;
                    return launchPrefill<T, false>(a, p, d, s);
                }
            }
            return launchPrefill<T, kInt8>(a, p, d, s);
        }
    }
    // bf16 decode (fewer than 16 queries): the MFMA decode kernel, one 32-key step per wave
    // when the chunks allow (up to 1024 per (query, head), partials within the workspace)
    if constexpr (std::is_same_v<T, BF16>) {
        if (d == 128 && a.total > 0 && a.seq < size_t(kMfmaQ) && a.group <= 16 && a.scale > 0.0f &&
            std::isfinite(a.scale)) {
            // waves per block: 8 for caches of 16K+ keys (half the partials to merge: 32K
            // decode 14.6 -> 13.3 us INT8 KV, 14.4 -> 13.8 us bf16 KV), 2 below (more blocks
            // for the shorter chains: the 4096-key decode step took 1.157 ms with 4, 1.122 ms
            // with 2, 1.144 ms with 1; it lost with 8)
            const int nw = a.total >= 16384 ? 8 : kDecWaves;
            const size_t bk = size_t(nw) * kDecKT; // keys per block step
            const size_t pairs = a.seq * size_t(a.nh);
            size_t nchunks = std::min<size_t>((a.total + bk - 1) / bk, 1024);
            nchunks = std::max<size_t>(1, std::min(nchunks, ws_bytes / (size_t(d + 2) * sizeof(float) * pairs)));
            a.nchunks = int(nchunks);
            a.chunk = int(std::min<size_t>((a.total + nchunks - 1) / nchunks, size_t(INT32_MAX)));
            a.part = static_cast<float *>(ws);
            const unsigned blocks = unsigned(a.seq * size_t(a.nkvh) * nchunks);
            if (nw == 8)
                attnDecodeMfma<kInt8, 8><<<blocks, kWave * 8, 0, s>>>(a);
            else
                attnDecodeMfma<kInt8, kDecWaves><<<blocks, kWave * kDecWaves, 0, s>>>(a);
            if (nchunks > 1)
                launchCombine<T>(a.out, a.part, a.nchunks, d, pairs, s);
            return;
        }
    }
    const size_t nchunks = vectorChunks(a, d, groupLoads(kInt8), ws_bytes);
    a.nchunks = int(nchunks);
    a.chunk = int(std::min<size_t>(nchunks == 1 ? std::max<size_t>(a.total, 1)
                                                : (a.total + nchunks - 1) / nchunks,
                                   size_t(INT32_MAX)));
    a.part = static_cast<float *>(ws);
    const size_t blocks = a.seq * size_t(a.nkvh) * size_t(a.slices) * nchunks;
    if (d == 64)
        launchD<T, kInt8, 64>(a, G, blocks, s);
    else
        launchD<T, kInt8, 128>(a, G, blocks, s);
    if (nchunks > 1)
        launchCombine<T>(a.out, a.part, a.nchunks, d, a.seq * size_t(a.nh), s);
}

template <bool kInt8>
void dispatch(AttnArgs a, int d, int dv, llaisysDataType_t dt, void *ws, size_t ws_bytes, hipStream_t s) {
    switch (dt) {
    case LLAISYS_DTYPE_F32: return launch<F32, kInt8>(a, d, dv, ws, ws_bytes, s);
    case LLAISYS_DTYPE_BF16: return launch<BF16, kInt8>(a, d, dv, ws, ws_bytes, s);
    case LLAISYS_DTYPE_F16: return launch<F16, kInt8>(a, d, dv, ws, ws_bytes, s);
    default: return;
    }
}

} // namespace

extern "C" void llaisysTestAttentionRoute(size_t seq, size_t total, size_t nh, size_t nkvh, size_t d, int int8, int dt, int route[6]) {
    AttnArgs a{};
    a.seq = seq;
    a.total = total;
    a.nh = int(nh);
    a.nkvh = int(nkvh);
    a.group = int(nh / nkvh);
    a.scale = 1.0f;
    Prefill p{};
    const bool takes = planPrefill(p, a, int(d), int(d), int8 != 0, llaisysDataType_t(dt));
    route[0] = takes ? 1 + int(p.kernel) : 0;
    route[1] = takes ? p.nchunks : 0;
    route[2] = takes ? p.chunk : 0;
    route[3] = takes ? int(p.blocks) : 0;
    route[4] = takes ? p.heads : 0;
    route[5] = takes && p.elements;
}

// ---- scratch of the allocation-free entry point -----------------------------------------
// File-scope device array holding the split attention's partials for
// llaisysSelfAttentionInt8KVNoAlloc.  Each GPU the library runs on holds its own copy (at its
// own address) until the process ends.  In host code the name `scratch` is only a stand-in:
// its device address comes from hipGetSymbolAddress, resolved once per device with that
// device current, and only that address is ever handed to kernels.  Nothing in it needs to
// start at zero: every partial a launch reads was written earlier in the same launch pair.
static __device__ __align__(256) char scratch[kNoAllocScratchBytes];

namespace {
constexpr int kScratchDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[kScratchDevices] = {};
} // namespace

void *noAllocScratch(int device, char *err, size_t err_len) {
    if (device < 0 || device >= kScratchDevices) {
        snprintf(err, err_len, "device id %d out of range", device);
        return nullptr;
    }
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
        void *ptr = nullptr;
        const hipError_t st = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (st != hipSuccess || ptr == nullptr) {
            snprintf(err, err_len, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(st));
            return nullptr;
        }
        g_scratch_ptr[device] = ptr;
    }
    return g_scratch_ptr[device];
}

size_t selfAttentionInt8KVScratchBytes(const void *out, const void *q, const void *k, const void *v,
                                       size_t seq, size_t total, size_t nh, size_t nkvh, size_t d,
                                       size_t dv, float scale, llaisysDataType_t dt, size_t cap) {
    AttnArgs a{};
    a.out = const_cast<void *>(out);
    a.q = q;
    a.k = k;
    a.v = v;
    a.seq = seq;
    a.total = total;
    a.nh = int(nh);
    a.nkvh = int(nkvh);
    a.group = int(nh / nkvh);
    a.scale = scale;
    const size_t most = selfAttentionWorkspaceBytes(seq, nh, d);
    // a bf16 prefill with head_dim 128 is always accepted
    if (nh > 0 && dt == LLAISYS_DTYPE_BF16 && d == 128 && seq >= size_t(kMfmaQ) && total > 0 && scale > 0.0f &&
        std::isfinite(scale) && vecShape(a, int(d), int(dv), true)) {
        Prefill p;
        if (planPrefill(p, a, int(d), int(dv), true, dt)) {
            const size_t part = (p.part_bytes + 255) / 256 * 256, cache = 2 * total * nkvh * d * sizeof(uint16_t);
            return p.elements && part + cache <= cap ? part + cache : part;
        }
        const size_t n = vectorChunks(a, int(d), groupLoads(true), most);
        return n > 1 ? std::min(cap, n * seq * nh * (d + 2) * sizeof(float)) : 0;
    }
    return most;
}

size_t selfAttentionWorkspaceBytes(size_t seq, size_t nh, size_t head_dim) {
    // up to 1024 partials of head_dim + 2 floats per (query, head), capped at 64 MiB: a
    // smaller workspace only lowers the chunk count (decode: 12 heads x 1024 x 520 B)
    return std::min<size_t>(std::min<size_t>(seq * nh, 4096) * 1024 * (head_dim + 2) * sizeof(float),
                            size_t(64) << 20);
}

void selfAttention(void *out, const void *q, const void *k, const void *v, const float *k_scale,
                   const float *v_scale, size_t seq, size_t total, size_t nh, size_t nkvh,
                   size_t d, size_t dv, float scale, llaisysDataType_t dt, void *ws,
                   size_t ws_bytes, hipStream_t s) {
    AttnArgs a{};
    a.out = out;
    a.q = q;
    a.k = k;
    a.v = v;
    a.ks = k_scale;
    a.vs = v_scale;
    a.seq = seq;
    a.total = total;
    a.nh = int(nh);
    a.nkvh = int(nkvh);
    a.group = int(nh / nkvh);
    a.scale = scale;
    if (k_scale)
        dispatch<true>(a, int(d), int(dv), dt, ws, ws_bytes, s);
    else
        dispatch<false>(a, int(d), int(dv), dt, ws, ws_bytes, s);
}

} // namespace llaisys::kernels
