// The tiled linear kernels: several rows, any of the element types (linear_gemm.hip picks the tile,
// linear_gemm_kernels.hpp holds the kernels).
#pragma once

#include "launch.hpp"

namespace llaisys::kernels {

// The rows, types and alignments the tiled kernels take.
bool gemmTakes(const LinearCall &c);
// Workspace that lets the launch split K as it would like to; with less it does not split.
size_t gemmWorkspaceBytes(const LinearCall &c);
void gemm(const LinearCall &c, void *ws, size_t ws_bytes, hipStream_t s);

// For the tests.  The plan of a call: tile, splits, stages per split, k per stage (no GPU needed).
extern "C" int llaisysTestLinearPlan(size_t rows, size_t K, size_t N, int int8, int swiglu, int dt, int plan[4]);
// A 16-bit call on the tile and split given, on the default stream and waited for, with `ws` for its
// partial sums: the splits it ran with, 0 for a tile or call that there is none for.
extern "C" int llaisysTestLinearTile(void *out, const void *x, const void *w, const float *scale, const void *bias, size_t rows,
                                     size_t K, size_t N, int swiglu, int dt, int tile, size_t splits, void *ws, size_t ws_bytes);

// ---- between linear_gemm.hip and the kernels ---------------------------------------------------

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

// Tile shapes of the 16-bit types, weight rows x activation rows (64x64Deep: stages of 128 k shared
// by two waves per tile quarter).
enum class GemmTile { k64x64Deep, k64x64, k128x64, k128x128, k192x128, k256x128, k192x256 };

void gemmBf16(GemmTile t, const GemmArgs &a, bool swiglu, hipStream_t s);
void gemmF16(GemmTile t, const GemmArgs &a, bool swiglu, hipStream_t s);

} // namespace llaisys::kernels
