// Production tile shapes of the GEMM variants (kernels in gemm_kernels.hpp)
// and their launchers.
#include "gemm_kernels.hpp"

namespace dhx {
namespace {

using gemm::Tile;
using gemm::tiles_for;

// Tiles of the launches of several rounds of workgroups (the rings' follow
// below). The patch embedding stages both operands in LDS (its A operand is
// gathered from pixels); the others take activations in fragment order
// straight into registers, waves stacked along M. The residual GEMMs (N = 384:
// too few 128x128 tiles to fill 256 CUs) use 128x64 tiles, twice as many
// workgroups of a quarter of the registers.
using PatchTile = Tile<64, 128, 2, 2>;
// QKV on 32-deep stages (24 KB of weight buffers; its RoPE angles wait in
// LDS, not registers): four workgroups per CU, so a batch of 64 (909 tiles)
// runs as one round of workgroups.
using QkvTile = Tile<128, 128, 4, 1, 32>;
// QKV for launches of fewer rows (the image groups of batch 32 and of 512x512
// batch 8): 128x64 tiles (one head per wave), twice the workgroups. Same stage
// depth, and the LayerNorm fold is applied in the epilogue, so a row's result
// is bitwise the same on either shape.
using QkvTileS = Tile<128, 64, 4, 1, 32>;
constexpr int kQkvSmallRows = 5120;
using ResidTile = Tile<128, 64, 4, 1>;
using ResidTileK = Tile<128, 64, 4, 1, 128>;  // down projection (k = 1536)
using SwigluTile = Tile<256, 128, 4, 1, 64>;
// SwiGLU for launches of fewer rows (batch 32's and 512x512 batch 8's image
// groups of 3216 and 4116 rows; below 2048 the rings): 128-row tiles, three
// workgroups per CU instead of two. Measured in the two-group forward: the
// 128-row tiles win at 3216 and 4116 rows (at 4116 the 256-row tiling's
// last tile holds 20 rows), the 256-row ones at 6432 (batch 64's groups).
using SwigluTileS = Tile<128, 128, 4, 1, 64>;
constexpr int kSwigluSmallRows = 5120;
// Launches of up to this many rows take four XCD N slices, larger ones two.
constexpr int kSwigluSplit4Rows = 8192;
// The folded LayerNorm's -mean * wsum term joins column block i's
// accumulators at K step i + 1, so where it enters the fp32 sum depends on
// the stage depth. Both tile shapes must share it for a row's result to be
// bitwise the same whichever shape its launch takes (the image groupings of
// the forward and the allocation-free entry point rely on that).
static_assert(SwigluTile::BK == SwigluTileS::BK, "one stage depth for every SwiGLU tile shape");
using SplitTile = Tile<128, 128, 4, 1>;

// Tiles of the ring kernels, two to eight waves of 32x32 or 32x64.
using ResidRing32 = Tile<32, 64, 1, 2, 128>;
using ResidRing32K = Tile<32, 64, 1, 2, 64>;
using ResidRing64 = Tile<64, 64, 2, 2, 64>;
using ResidRing128 = Tile<128, 64, 4, 2, 64>;
using ResidRing128W = Tile<128, 128, 4, 2, 64>;
using SwigluRing64 = Tile<64, 128, 2, 2, 32>;
using SwigluRing128 = Tile<128, 128, 4, 2, 32>;
using SwigluRing128W = Tile<128, 192, 4, 3, 32>;
using QkvRing64 = Tile<64, 64, 2, 1, 64>;
using QkvRing64W = Tile<64, 128, 2, 2, 64>;
using QkvRing128 = Tile<128, 128, 4, 2, 64>;
constexpr int kRound = 256;  // workgroups of one per CU
constexpr int kResidRing128Rows = 5120;
constexpr int kQkvSharedRing = 22 * 128;  // QkvRing128's most rows beside other kernels

template <class T, class Kernel, class Args>
hipError_t launch(Kernel kernel, int tiles, const Args& a, hipStream_t s) {
    return start(kernel, dim3(gemm::tile_grid(tiles)), dim3(T::THREADS), 0, s, a);
}

}  // namespace

hipError_t launch_patch_embed(const PatchEmbedArgs& a, hipStream_t s) {
    const int ring = (a.images * a.grid * a.grid + gemm::kPatchRingRows - 1) / gemm::kPatchRingRows *
                     (kHidden / gemm::kPatchRingCols);
    if (ring <= kRound) {
        const dim3 grid(gemm::tile_grid(ring)), block(128);
        return a.stats ? start(gemm::patch_ring_kernel<true>, grid, block, 0, s, a)
                       : start(gemm::patch_ring_kernel<false>, grid, block, 0, s, a);
    }
    const int tiles = tiles_for<PatchTile>(a.images * a.grid * a.grid, kHidden);
    return a.stats ? launch<PatchTile>(gemm::patch_embed_kernel<PatchTile, true>, tiles, a, s)
                   : launch<PatchTile>(gemm::patch_embed_kernel<PatchTile, false>, tiles, a, s);
}

template <class T>
static hipError_t launch_qkv_tiles(const QkvArgs& a, hipStream_t s) {
    const int tiles = tiles_for<T>(a.images * (a.grid * a.grid + kPrefix), 3 * kHidden);
    const dim3 grid(gemm::tile_grid(tiles));
    const size_t lds = gemm::rope_lds_bytes(a.grid);
    return a.stats ? start(gemm::qkv_rope_kernel<T, true>, grid, dim3(T::THREADS), lds, s, a)
                   : start(gemm::qkv_rope_kernel<T, false>, grid, dim3(T::THREADS), lds, s, a);
}

template <class T, int NST>
static hipError_t launch_qkv_ring(const QkvArgs& a, hipStream_t s) {
    const dim3 grid(gemm::tile_grid(tiles_for<T>(a.images * (a.grid * a.grid + kPrefix), 3 * kHidden)));
    const size_t lds = gemm::rope_lds_bytes(a.grid);
    return a.stats ? start(gemm::qkv_ring_kernel<T, NST, true>, grid, dim3(T::THREADS), lds, s, a)
                   : start(gemm::qkv_ring_kernel<T, NST, false>, grid, dim3(T::THREADS), lds, s, a);
}

// As for the residual GEMMs: the smallest ring tile that one round of
// workgroups covers. Whole forward (one chain, graph replay), the tiles
// below / 64x64 / 64x128 / 128x128: 201 rows 418 / 390 / 395 / 405 us, 603
// rows 426 / 401 / 406 / 420, 1005 rows 411 / 434 / 400 / 415, 1608 rows 446
// / 461 / 427 / 440, 2412 rows 466 / 509 / 481 / 453, 3216 rows 503 / 586 /
// 519 / 487, 4020 rows 513 / 645 / 583 / 559. Beside another image group's
// kernels the 128x128 ring, which takes most of a CU's LDS, only to 2816 rows
// (two groups, the tiles below / 128x128: 2 x 2412 rows 590 / 578 us, 2 x 2610
// 685 / 644, 2 x 2814 667 / 632; 2 x 2835 711 / 728, 2 x 3216 684 / 681, 2 x
// 3240 739 / 768, 3393 and 3654 732 / 756).
hipError_t launch_qkv_rope(const QkvArgs& a, hipStream_t s) {
    const int rows = a.images * (a.grid * a.grid + kPrefix);
    if (rows <= kRound / 18 * 64) return launch_qkv_ring<QkvRing64, 4>(a, s);
    if (rows <= kRound / 9 * 64) return launch_qkv_ring<QkvRing64W, 4>(a, s);
    if (rows <= (a.shared ? kQkvSharedRing : kRound / 9 * 128)) return launch_qkv_ring<QkvRing128, 3>(a, s);
    return rows < kQkvSmallRows ? launch_qkv_tiles<QkvTileS>(a, s) : launch_qkv_tiles<QkvTile>(a, s);
}

template <class T, int NST, int K>
static hipError_t launch_resid_ring(const ResidArgs& a, hipStream_t s) {
    const int tiles = tiles_for<T>(a.rows, kHidden);
    return a.stats ? launch<T>(gemm::resid_ring_kernel<T, NST, true, K / T::BK>, tiles, a, s)
                   : launch<T>(gemm::resid_ring_kernel<T, NST, false, K / T::BK>, tiles, a, s);
}

hipError_t launch_resid(const ResidArgs& a, hipStream_t s) {
    // Launches that one round of workgroups covers, one per CU, take the
    // smallest ring tile that does (N = 384 is six 64-column tiles): a smaller
    // one needs a second round, a larger one leaves CUs idle. Whole forward
    // (one chain, graph replay), against resid_kernel: o-projection 32x64 at
    // 201 rows 412 -> 403 us (64x64 406); down projection 64x64 at 201 / 1005
    // / 2412 rows 412 -> 376, 404 -> 368, 488 -> 455, at 3216 rows 528 -> 551;
    // 128x64 there 528 -> 517, at 4020 rows 539 -> 527, at 5025 rows 563 ->
    // 549, but not to the end of its round: 512x512 batch 5 (5145 rows) 803 ->
    // 839 us, 384x384 batch 9 (5229 rows) 732 -> 753. To 1344 rows the
    // down projection's 32x64 tile with five 64-deep stages in flight takes
    // 8.5 us off each of these (201 rows 295.3 -> 286.8, 1005 rows 315.6 ->
    // 308.5; three or four 128-deep stages 294, 293, 1608 rows 355 -> 377).
    // Beside another image group's kernels (a.shared) the 128x64 ring, which
    // takes a CU's LDS whole, loses to the tiles below (620 -> 629 us at 2 x
    // 2814 rows, 667 -> 728 at 2 x 3216).
    // One more size for the down projection, 128x128 tiles to 10880 rows: 6432
    // rows 736 -> 699 us, 8643 rows 886 -> 858, 8232 rows 1029 -> 1008 (one
    // chain); beside another group 1003 -> 992 at 2 x 5427 rows, 1100 -> 1105 at
    // 2 x 6432. The o-projection, with three stages to a tile, gains nothing
    // from it.
    const int round = a.rows <= kRound / 6 * 32   ? 32
                      : a.rows <= kRound / 6 * 64 ? 64
                      : a.shared                  ? 0
                      : a.rows < kResidRing128Rows ? 128
                      : a.rows <= kRound / 6 * 128 ? 0
                      : a.rows <= kRound / 3 * 128 ? 256 : 0;
    if (a.k == kHidden && round == 32) return launch_resid_ring<ResidRing32, 4, kHidden>(a, s);
    if (a.k == kHidden && round == 64) return launch_resid_ring<ResidRing64, 5, kHidden>(a, s);
    if (a.k == kHidden && round == 128) return launch_resid_ring<ResidRing128, 4, kHidden>(a, s);
    if (a.k == kFF && round == 32) return launch_resid_ring<ResidRing32K, 6, kFF>(a, s);
    if (a.k == kFF && round == 64) return launch_resid_ring<ResidRing64, 5, kFF>(a, s);
    if (a.k == kFF && round == 128) return launch_resid_ring<ResidRing128, 4, kFF>(a, s);
    if (a.k == kFF && round == 256) return launch_resid_ring<ResidRing128W, 4, kFF>(a, s);
    // The K loop walks its stages six at a time (gemm_main_dma).
    if (a.k % (6 * ResidTile::BK) != 0) return hipErrorInvalidValue;
    if (a.k == kHidden) {  // the o-projection: three 128-deep stages, unrolled
        const int tiles = tiles_for<ResidTileK>(a.rows, kHidden);
        return a.stats ? launch<ResidTileK>(gemm::resid_kernel<ResidTileK, true, kHidden / 128>, tiles, a, s)
                       : launch<ResidTileK>(gemm::resid_kernel<ResidTileK, false, kHidden / 128>, tiles, a, s);
    }
    if (a.k == kFF) {  // the down projection: twelve 128-deep stages, unrolled
        const int tiles = tiles_for<ResidTileK>(a.rows, kHidden);
        return a.stats ? launch<ResidTileK>(gemm::resid_kernel<ResidTileK, true, kFF / 128>, tiles, a, s)
                       : launch<ResidTileK>(gemm::resid_kernel<ResidTileK, false, kFF / 128>, tiles, a, s);
    }
    if (a.k % (6 * ResidTileK::BK) == 0) {
        const int tiles = tiles_for<ResidTileK>(a.rows, kHidden);
        return a.stats ? launch<ResidTileK>(gemm::resid_kernel<ResidTileK, true>, tiles, a, s)
                       : launch<ResidTileK>(gemm::resid_kernel<ResidTileK, false>, tiles, a, s);
    }
    const int tiles = tiles_for<ResidTile>(a.rows, kHidden);
    return a.stats ? launch<ResidTile>(gemm::resid_kernel<ResidTile, true>, tiles, a, s)
                   : launch<ResidTile>(gemm::resid_kernel<ResidTile, false>, tiles, a, s);
}

template <class T, int NS>
static hipError_t launch_swiglu_tiles(const SwigluArgs& a, hipStream_t s) {
    static_assert(kHidden % (6 * T::BK) == 0, "the K loop walks its stages six at a time");
    const int grid = gemm::tile_grid_split<NS>((a.rows + T::BM - 1) / T::BM, 2 * kFF / T::BN);
    return a.stats ? start(gemm::swiglu_kernel<T, true, NS>, dim3(grid), dim3(T::THREADS), 0, s, a)
                   : start(gemm::swiglu_kernel<T, false, NS>, dim3(grid), dim3(T::THREADS), 0, s, a);
}

template <class T, int NST>
static hipError_t launch_swiglu_ring(const SwigluArgs& a, hipStream_t s) {
    const dim3 grid(gemm::tile_grid(tiles_for<T>(a.rows, 2 * kFF)));
    return a.stats ? start(gemm::swiglu_ring_kernel<T, NST, true>, grid, dim3(T::THREADS), 0, s, a)
                   : start(gemm::swiglu_ring_kernel<T, NST, false>, grid, dim3(T::THREADS), 0, s, a);
}

// As for the residual GEMMs: the smallest ring tile that one round of
// workgroups covers, to 2048 rows. Whole forward (one chain, graph replay),
// the 128x128 tiles below / 64x128 / 128x128 / 128x192 rings: 201 rows 336 /
// 329 / 336 / - us, 603 rows 345 / 337 / 343 / -, 1005 rows 349 / 355 / 346 /
// -, 1206 rows 375 / 359 / 353 / -, 1608 rows 379 / - / 381 / 371, 2010 rows
// 391 / - / 394 / 385, 2412 rows 404 / - / 407 / 457. Above, several rounds
// overlap one tile's epilogue with another's K loop, which the rings, taking
// most of a CU's LDS, do not.
//
// For the larger launches, the XCD split (each XCD's L2 keeps 1/NS of the
// weights): two N slices for the whole batch-64 launch, four for the image groups of 5120 - 8191 rows
// that the forward runs concurrently (measured: forward +0.9 % at batch 64,
// the whole-batch launch 2 % slower with four).
hipError_t launch_swiglu(const SwigluArgs& a, hipStream_t s) {
    if (a.rows <= kRound / 24 * 64) return launch_swiglu_ring<SwigluRing64, 4>(a, s);
    if (a.rows <= kRound / 24 * 128) return launch_swiglu_ring<SwigluRing128, 4>(a, s);
    if (a.rows <= kRound / 16 * 128) return launch_swiglu_ring<SwigluRing128W, 4>(a, s);
    if (a.rows < kSwigluSmallRows) return launch_swiglu_tiles<SwigluTileS, 2>(a, s);
    return a.rows < kSwigluSplit4Rows ? launch_swiglu_tiles<SwigluTile, 4>(a, s) : launch_swiglu_tiles<SwigluTile, 2>(a, s);
}

hipError_t launch_splitk(const SplitKArgs& a, hipStream_t s) {
    // Each split's K loop walks its stages six at a time (gemm_main_dma).
    if (a.splits < 1 || a.k % a.splits != 0 || (a.k / a.splits) % (6 * SplitTile::BK) != 0) return hipErrorInvalidValue;
    const int tiles = tiles_for<SplitTile>(a.rows, kHidden) * a.splits;
    if (a.k / a.splits == kHidden)  // the model's b = 1 down projection: 4 splits of 384, six stages unrolled
        return launch<SplitTile>(gemm::splitk_kernel<SplitTile, kHidden / SplitTile::BK>, tiles, a, s);
    return launch<SplitTile>(gemm::splitk_kernel<SplitTile>, tiles, a, s);
}

}  // namespace dhx
