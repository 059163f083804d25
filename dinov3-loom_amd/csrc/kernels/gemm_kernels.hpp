// The GEMM variants of the forward pass, as kernels templated on the tile
// shape (gemm.hip instantiates the shapes used in production). Replaces the
// reference's Loom GEMMs: kernels/matmul_bias_f16_wmma.loom (patch embed,
// with the embed scatter of kernels/embed_scatter_f32.loom fused in),
// matmul_qkv_rope_f16_wmma.loom, matmul_resid_f16_wmma.loom,
// matmul_swiglu_f16_wmma.loom and matmul_splitk_f16_wmma.loom.
//
// Activations (x, h, attn, act) are kept in fragment order (common.hpp). The
// GEMMs of several rounds of workgroups load them straight into registers
// (ActFrags) and stage only the weights in LDS, with the workgroup's waves
// stacked along M; the rings of the small launches (*_ring_kernel) move both
// operands through LDS, and the patch embedding gathers its own from pixels.
#pragma once
#include "gemm_core.hpp"
#include "launch.hpp"

namespace dhx {
namespace gemm {

// A operand of the patch embedding, gathered from NCHW f32 pixels (the im2col
// of lib.rs:265-280): row m = image*P + gy*G + gx, column k = c*256 + dy*16 +
// dx. A 64-wide stage covers one channel and four pixel rows of the patch;
// consecutive lanes read consecutive 16-byte pieces of a pixel row, and the
// patches of one grid row are adjacent in memory. Pixels are narrowed to f16
// on the way to LDS.
template <class T>
struct PatchRows {
    static constexpr bool kInRegs = false;
    static_assert(T::BK == 64, "a stage is one channel x four pixel rows");
    static constexpr int CHUNKS = T::BM * T::BK / 4 / T::THREADS;
    static_assert(T::BM * T::BK / 4 % T::THREADS == 0, "patch tile splits evenly");
    const float* px;
    int M, G, P, S;
    float4_t r[CHUNKS];
    __device__ __forceinline__ void load(int m0, int /*n0*/, int kt, int tid) {
#pragma unroll
        for (int i = 0; i < CHUNKS; ++i) {
            const int c = tid + i * T::THREADS;
            const int dxq = c & 3, row = (c >> 2) % T::BM, dyl = c / (4 * T::BM);
            const int m = min(m0 + row, M - 1);  // rows past M feed unstored outputs
            const int img = m / P, p = m - img * P, gy = p / G, gx = p - gy * G;
            const int ch = kt >> 2, dy = (kt & 3) * 4 + dyl;
            r[i] = *(const float4_t*)(px + (((size_t)img * 3 + ch) * S + gy * 16 + dy) * S + gx * 16 + dxq * 4);
        }
    }
    __device__ __forceinline__ void store(half_t* s, int tid) const {
#pragma unroll
        for (int i = 0; i < CHUNKS; ++i) {
            const int c = tid + i * T::THREADS;
            const int dxq = c & 3, row = (c >> 2) % T::BM, dyl = c / (4 * T::BM);
            *(half4_t*)(s + row * T::LDK + dyl * 16 + dxq * 4) = to_half4(r[i]);
        }
    }
};

// (mean, M2) partial of one row over a 64-column statistics slot whose
// values are split between this lane (32 of them, already rounded to the f16
// values stored in x) and its partner lane l ^ 32. Both partners call this;
// the lane with hi == 0 writes.
__device__ __forceinline__ void pair_stats(float* stats, size_t m, int slot, const float (&v)[32], int hi, bool store) {
    float s = 0.f;
#pragma unroll
    for (int e = 0; e < 32; ++e) s += v[e];
    s = half_pair_sum(s);
    const float mean = s * (1.0f / 64.0f);
    float d[32];
#pragma unroll
    for (int e = 0; e < 32; ++e) d[e] = v[e] - mean;
    const float q = half_pair_sum(sum_of_squares(d));
    if (store && hi == 0) *(float2_t*)(stats + m * kStatFloats + slot * 2) = float2_t{mean, q};
}

// A wave's 32 x 64 block of patch rows m_base .., rounded to f16 in LDS (st,
// of pitch sp halfs), written to x as fragment pieces; with STATS also its
// statistics slot.
template <bool STATS>
__device__ __forceinline__ void patch_rows(const PatchEmbedArgs& p, const half_t* st, int sp, int m_base, int n_base, int M,
                                           int P) {
    const int lane = threadIdx.x & 63, l32 = lane & 31, hi = lane >> 5;
    const int m = m_base + l32;
    const bool valid = m < M;
    const size_t row = valid ? (size_t)m + (size_t)(m / P + 1) * kPrefix : 0;  // image*Tok + kPrefix + patch
    // The wave's 32 patch rows land in x rows row(m_base) .. at most
    // 32 + 5 * (32 / P + 1) rows further: within 8 row blocks.
    const size_t rb0 = ((size_t)m_base + (size_t)(m_base / P + 1) * kPrefix) / 32;
    const WtOut xo(p.x + rb0 * (kHidden / 16) * 512, 8 * (kHidden / 16) * 1024);
    float v[32];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
        const half8_t h = *(const half8_t*)(st + l32 * sp + ks * 16 + hi * 8);
        if (valid)
            xo.store((uint32_t)(frag_piece((int)row, n_base + ks * 16 + hi * 8, kHidden) - rb0 * (kHidden / 16) * 512) * 2, h);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[ks * 8 + e] = (float)h[e];
    }
    if constexpr (STATS) pair_stats(p.stats, row, n_base / 64, v, hi, valid);
}

// CLS + registers, columns n0 .. n0 + BN - 1, of every image whose first patch
// row lies in m0 .. m_end - 1, by threads tid of THREADS.
template <int BN, int THREADS, bool STATS>
__device__ __forceinline__ void patch_prefix(const PatchEmbedArgs& p, int tid, int m0, int m_end, int n0, int P, int Tok) {
    for (int img = (m0 + P - 1) / P; img * P < m_end; ++img) {
        for (int idx = tid; idx < kPrefix * BN; idx += THREADS) {
            const int r = idx / BN, col = n0 + idx % BN;
            p.x[frag_piece(img * Tok + r, col & ~7, kHidden) + (col & 7)] = (half_t)p.prefix[r * kHidden + col];
        }
        if constexpr (STATS) {
            constexpr int slots = BN / 64;
            for (int idx = tid; idx < kPrefix * slots * 2; idx += THREADS) {
                const int r = idx / (slots * 2), e = idx % (slots * 2);
                const int off = (n0 / 64) * 2 + e;
                p.stats[((size_t)img * Tok + r) * kStatFloats + off] = p.prefix_stats[r * kStatFloats + off];
            }
        }
    }
}

// Patch embedding + CLS/register scatter into the f16 residual stream x
// (fragment order; with STATS, also the LayerNorm row statistics of x). Each
// wave rounds its 32 x 64 block to f16 into LDS, then writes it as fragment
// pieces, lane (l, hi) taking row l and the half hi of each 16-column block.
template <class T, bool STATS>
__global__ __launch_bounds__(T::THREADS) void patch_embed_kernel(DHX_PATCH_PARAMS) {
    const PatchEmbedArgs p{pixels_, w_, bias_, prefix_, x_, images_, grid_, prefix_stats_, stats_};
    static_assert(T::TN == 64 && T::TM == 32, "one 32-row block and one statistics slot per wave");
    constexpr int SP = T::TN + 8;  // staging pitch in halfs
    static_assert(T::WAVES * T::TM * SP <= T::LDS_HALFS, "staging fits the stage buffers");
    __shared__ __attribute__((aligned(16))) half_t lds[T::LDS_HALFS];
    const int P = p.grid * p.grid, Tok = P + kPrefix, M = p.images * P;
    constexpr int NT = kHidden / T::BN;
    const int S = 16 * p.grid;
    PatchRows<T> al[2] = {{p.pixels, M, p.grid, P, S}, {p.pixels, M, p.grid, P, S}};
    WeightRows<T> wl[2] = {{{}, p.w, 768, 0}, {{}, p.w, 768, 0}};
    gemm_tile<T>(al, wl, NT, NT * ((M + T::BM - 1) / T::BM), 768 / T::BK, lds, [&](const Acc<T>& acc, int m0, int n0) {
        const Frag<T> f(m0, n0);
        half_t* const st = lds + (threadIdx.x >> 6) * (T::TM * SP);
#pragma unroll
        for (int i = 0; i < T::FN; ++i)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int n = f.col(i, g);
                const float4_t b = ld4(p.bias + n);
                *(half4_t*)(st + f.l32 * SP + (n - f.n_base)) = to_half4(group4(acc.v[i][0], g) + b);
            }
        wave_lds_sync();
        patch_rows<STATS>(p, st, SP, f.m_base, f.n_base, M, P);
        patch_prefix<T::BN, T::THREADS, STATS>(p, threadIdx.x, m0, min(m0 + T::BM, M), n0, P, Tok);
    });
}

// Patch embedding for launches that one round of workgroups covers (see the
// launcher): 32x64 tiles of two waves (one column block each) and a ring of
// eight 64-deep stages, pixels as they are (float32) and weights, both by DMA.
// patch_embed_kernel's twelve steps wait for loads issued one step ahead, on
// 12 workgroups at 196 patches; here seven stages are in flight on 42:
// alone at 196 patches 8.4 -> 5.6 us, at 1176 8.6 -> 6.0, and 3 us less of
// the forward at one image. Left are the launch, one cold load, twelve barriers
// and the stores. A stage holds four pixel rows of one channel of 32 patches as [row][patch]
// [16 pixels], 16-byte chunk c of patch r at slot c ^ (r / 4) % 4, and 64
// weight rows of 64 columns, chunk c of row r at slot c ^ (r / 2) % 8, so that
// 16 consecutive rows' reads of one chunk cover all banks. The same MFMAs in
// the same order as patch_embed_kernel: a row's result is bitwise the same.
// Offsets into the pixels are 32 bits: the launcher bounds the launch.
constexpr int kPatchRing = 8, kPatchRingRows = 32, kPatchRingCols = 64;
constexpr int kPatchRingW = 32 * 64 * 2;  // halfs of a stage's pixels, after which its weights follow
constexpr int kPatchRingHalfs = kPatchRingW + 64 * 64;

// The K loop of one tile; see gemm_main_ring for the waits.
__device__ __forceinline__ void patch_ring(const PatchEmbedArgs& p, half_t* const (&bufs)[kPatchRing], int m0, int n0, int M,
                                           int P, float16_t& acc) {
    constexpr int KT = 768 / 64;
    const int S = 16 * p.grid;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, hi = lane >> 5;
    const __amdgpu_buffer_rsrc_t rp = dma_src(p.pixels, p.images * 3 * S * S * 4);
    const __amdgpu_buffer_rsrc_t rw = dma_src(p.w + (size_t)n0 * 768, kPatchRingCols * 768 * 2);
    // Each wave moves two of a stage's four pixel rows (16 patches a load) and
    // 32 of its 64 weight rows (8 a load).
    int ap[2], aw[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int m = min(m0 + 16 * h + (lane >> 2), M - 1);  // rows past M feed unstored outputs
        const int img = m / P, q = m - img * P, gy = q / p.grid, gx = q - gy * p.grid;
        ap[h] = ((img * 3 * S + gy * 16) * S + gx * 16) * 4 + ((lane & 3) ^ (lane >> 4)) * 16;
        aw[h] = (lane >> 3) * 1536 + ((lane & 7) ^ (4 * h + (lane >> 4))) * 16;
    }
    auto lds = [](half_t* a) { return (__attribute__((address_space(3))) void*)a; };
    auto load = [&](half_t* stage, int kt) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int dy = wave * 2 + (j >> 1);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rp, lds(stage + (dy * 2 + (j & 1)) * 512), 16, ap[j & 1],
                                                     ((kt >> 2) * S + (kt & 3) * 4 + dy) * S * 4, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, lds(stage + kPatchRingW + (wave * 4 + j) * 512), 16, aw[j & 1],
                                                     (wave * 4 + j) * 8 * 1536 + kt * 128, 0, 0);
    };
    acc = float16_t{};
    static_for<kPatchRing - 1>([&](auto I) { load(bufs[decltype(I)::value], decltype(I)::value); });
    static_for<KT>([&](auto I) {
        constexpr int s = decltype(I)::value;
        constexpr int ahead = KT - 1 - s < kPatchRing - 2 ? KT - 1 - s : kPatchRing - 2;  // later stages in flight
        vm_barrier<ahead * 8>();
        if constexpr (s + kPatchRing - 1 < KT) load(bufs[(s + kPatchRing - 1) % kPatchRing], s + kPatchRing - 1);
        const half_t* const stage = bufs[s % kPatchRing];
        const float* const a = (const float*)stage + l32 * 16;
        const half_t* const w = stage + kPatchRingW + (wave * 32 + l32) * 64;
        half8_t af[4], wf[4];
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            const half4_t lo = to_half4(*(const float4_t*)(a + kk * 512 + ((2 * hi) ^ ((l32 >> 2) & 3)) * 4));
            const half4_t up = to_half4(*(const float4_t*)(a + kk * 512 + ((2 * hi + 1) ^ ((l32 >> 2) & 3)) * 4));
            af[kk] = __builtin_shufflevector(lo, up, 0, 1, 2, 3, 4, 5, 6, 7);
            wf[kk] = *(const half8_t*)(w + ((2 * kk + hi) ^ ((l32 >> 1) & 7)) * 8);
        }
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) acc = mfma32x32x16(wf[kk], af[kk], acc);
    });
}

template <bool STATS>
__global__ __launch_bounds__(128, 1) void patch_ring_kernel(DHX_PATCH_PARAMS) {
    const PatchEmbedArgs p{pixels_, w_, bias_, prefix_, x_, images_, grid_, prefix_stats_, stats_};
    constexpr int NT = kHidden / kPatchRingCols, SP = kPatchRingCols + 8;
    __shared__ __attribute__((aligned(16))) half_t ring0[kPatchRingHalfs], ring1[kPatchRingHalfs], ring2[kPatchRingHalfs],
        ring3[kPatchRingHalfs], ring4[kPatchRingHalfs], ring5[kPatchRingHalfs], ring6[kPatchRingHalfs],
        ring7[kPatchRingHalfs];
    __shared__ __attribute__((aligned(16))) half_t st[32 * SP];
    __shared__ __attribute__((aligned(16))) float bias[dma_copy_bytes(kPatchRingCols * 4) / 4];
    half_t* const bufs[kPatchRing] = {ring0, ring1, ring2, ring3, ring4, ring5, ring6, ring7};
    const int P = p.grid * p.grid, M = p.images * P;
    const int t = xcd_tile(NT * ((M + kPatchRingRows - 1) / kPatchRingRows));
    if (t < 0) return;  // uniform per workgroup
    const int n0 = (t % NT) * kPatchRingCols, m0 = (t / NT) * kPatchRingRows;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    dma_copy<kPatchRingCols * 4, 2>(dma_src(p.bias + n0, kPatchRingCols * 4), bias, tid);
    float16_t acc;
    patch_ring(p, bufs, m0, n0, M, P, acc);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const int n = wave * 32 + g * 8 + (lane >> 5) * 4;
        *(half4_t*)(st + (lane & 31) * SP + n) = to_half4(group4(acc, g) + *(const float4_t*)&bias[n]);
    }
    lds_barrier();
    if (wave == 0)
        patch_rows<STATS>(p, st, SP, m0, n0, M, P);
    else
        patch_prefix<kPatchRingCols, 64, STATS>(p, lane, m0, min(m0 + kPatchRingRows, M), n0, P, P + kPrefix);
}

template <class T>
__device__ __forceinline__ void init_frags(ActFrags<T> (&al)[2], const half_t* a, int rows, int k, int ks_off = 0) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        al[i].a = a;
        al[i].ksteps = k / 16;
        al[i].mblocks = (rows + 31) / 32;
        al[i].ks_off = ks_off;
    }
}

// RoPE angles in LDS. DINOv3's tables are separable (weights.rs:127-144):
// the angle of channel c < 16 of patch (gy, gx) depends on gy only, that of
// channel 16 <= c < 32 on gx only, and channels 32..63 repeat 0..31. Four
// [R][16] float tables (R = the grid side rounded up to 16) hold every angle
// the QKV epilogue needs: cos and sin of the row part (table row gy, from
// patch (gy, 0) of the full [P][64] tables) and of the column part (table
// row gx, from patch (0, gx)), the same float values the full tables hold.
__host__ __device__ constexpr int rope_table_rows(int grid) { return (grid + 15) / 16 * 16; }
__host__ __device__ constexpr int rope_lds_bytes(int grid) { return 4 * rope_table_rows(grid) * 16 * 4; }

// Table w (cos row part, sin row part, cos column part, sin column part) is
// filled by wave w % WAVES with DMA loads of 16 table rows each: lane i moves
// 16 bytes, channels 4(i % 4) .. +3 of table row 16q + i / 4, to LDS byte
// 16i of the load's 1 KB. Rows past the grid read beyond the source table's
// bounds, which the buffer descriptor turns into zeros, or other patches'
// angles (grids under 16), and are never read back.
template <int WAVES>
__device__ __forceinline__ void rope_table_dma(const float* cos, const float* sin, int grid, float* lds, int tid) {
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int rows = rope_table_rows(grid);
#pragma unroll
    for (int i = 0; i < (4 + WAVES - 1) / WAVES; ++i) {
        const int w = wave + i * WAVES;  // uniform
        if (w >= 4) break;
        const __amdgpu_buffer_rsrc_t r = dma_src(w & 1 ? sin : cos, grid * grid * kHeadDim * 4);
        float* const table = lds + w * rows * 16;
        for (int q = 0; q < rows / 16; ++q) {  // uniform, 1..4
            const int row = q * 16 + (lane >> 2);
            const int src = (w < 2 ? row * grid * kHeadDim : row * kHeadDim + 16) + (lane & 3) * 4;  // floats
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)(table + q * 256), 16,
                                                     src * 4, 0, 0, 0);
        }
    }
}

// Epilogue of the QKV GEMM (see qkv_rope_kernel): bias and wsum hold the
// tile's columns, rope_lds the tables of rope_table_dma, norm(j) is the
// LayerNorm (mean, rstd) of this lane's row of row block j.
template <class T, bool LN, class Norm>
__device__ __forceinline__ void qkv_epilogue(const QkvArgs& p, const Acc<T>& acc, const Frag<T>& f, int m0, int n0,
                                             const float* bias, const float* wsum, const float* rope_lds, Norm&& norm) {
    const int P = p.grid * p.grid, Tok = P + kPrefix, M = p.images * Tok;
    const int part = f.n_base / kHidden, head0 = (f.n_base % kHidden) / kHeadDim;
    // By value: between the members themselves the choice is one of addresses,
    // which keeps the whole struct in scratch memory.
    half_t* const q = p.q;
    half_t* const k = p.k;
    half_t* const v = p.v;
    half_t* out = q;
    if (part == 1) out = k;
    if (part == 2) out = v;
    const size_t head_elems = (size_t)p.tpad * kHeadDim;
    const int rows16 = rope_table_rows(p.grid);
    // The tile's rows lie in images img0 .. img0 + BM / Tok + 1 (img0
    // from the tile origin, so it is uniform); the descriptor covers
    // those.
    const int img0 = min(m0, M - 1) / Tok;
    const int span = min(p.images - img0, T::BM / Tok + 2);
    const WtOut wo(out + (size_t)img0 * kHeads * head_elems, (uint32_t)(span * kHeads * head_elems * 2));
#pragma unroll
    for (int j = 0; j < T::FM; ++j) {
        const int mr = f.row(j);
        const int m = min(mr, M - 1);  // rows past M are computed but never written out
        const int img = m / Tok, tok = m - img * Tok;
        // This row's angles (cos, sin of channels 8g + 4hi .. +3, g =
        // 0..3); v tiles and prefix rows rotate by cos 1, sin 0.
        const bool rot = part < 2 && tok >= kPrefix;
        const int pt = max(tok - kPrefix, 0), gy = pt / p.grid, gx = pt - gy * p.grid;
        float4_t co[4], si[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            co[g] = float4_t{1.f, 1.f, 1.f, 1.f};
            si[g] = float4_t{};
        }
        if (rot) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int at = (g < 2 ? gy * 16 : 2 * rows16 * 16 + gx * 16) + (g & 1) * 8 + f.hi * 4;
                co[g] = *(const float4_t*)&rope_lds[at];
                si[g] = *(const float4_t*)&rope_lds[at + rows16 * 16];
            }
        }
        const RowNorm rn = norm(j);
#pragma unroll
        for (int h2 = 0; h2 < T::TN / kHeadDim; ++h2) {
            half4_t lo_h[4], up_h[4];
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int c = g * 8 + f.hi * 4;  // channel in the head (0..31); partner c + 32
                const int nl = f.n_base - n0 + h2 * kHeadDim + c;  // column in the tile
                float4_t lo = group4(acc.v[2 * h2][j], g), up = group4(acc.v[2 * h2 + 1][j], g);
                const float4_t b_lo = *(const float4_t*)&bias[nl], b_up = *(const float4_t*)&bias[nl + 32];
                float4_t w_lo{}, w_up{};
                if constexpr (LN) {
                    w_lo = *(const float4_t*)&wsum[nl];
                    w_up = *(const float4_t*)&wsum[nl + 32];
                }
                // Explicit FMAs: a row's result is the same on every tile
                // shape, however the compiler would contract each. lo's
                // products are the fused ones in both outputs.
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if constexpr (LN) {
                        lo[e] = fmaf(fmaf(-rn.mean, w_lo[e], lo[e]), rn.rstd, b_lo[e]);
                        up[e] = fmaf(fmaf(-rn.mean, w_up[e], up[e]), rn.rstd, b_up[e]);
                    } else {
                        lo[e] += b_lo[e];
                        up[e] += b_up[e];
                    }
                    const float l = lo[e];
                    lo[e] = fmaf(l, co[g][e], -(up[e] * si[g][e]));  // x[c] cos - x[c+32] sin
                    up[e] = fmaf(l, si[g][e], up[e] * co[g][e]);     // x[c+32] cos + x[c] sin
                }
                lo_h[g] = to_half4(lo);
                up_h[g] = to_half4(up);
            }
            // Channels 16kk + 8hi .. +7 of the head for kk = 0..3.
            const half8_t c0 = frag_swap(lo_h[0], lo_h[1]), c1 = frag_swap(lo_h[2], lo_h[3]);
            const half8_t c2 = frag_swap(up_h[0], up_h[1]), c3 = frag_swap(up_h[2], up_h[3]);
            const uint32_t hm = (uint32_t)(((img - img0) * kHeads + head0 + h2) * head_elems) * 2;
            if (mr < M) {
                wo.store(hm + (uint32_t)frag_piece(tok, f.hi * 8, kHeadDim) * 2, c0);
                wo.store(hm + (uint32_t)frag_piece(tok, 16 + f.hi * 8, kHeadDim) * 2, c1);
                wo.store(hm + (uint32_t)frag_piece(tok, 32 + f.hi * 8, kHeadDim) * 2, c2);
                wo.store(hm + (uint32_t)frag_piece(tok, 48 + f.hi * 8, kHeadDim) * 2, c3);
            }
        }
    }
}

// QKV + bias + 2D RoPE. A wave's 64 or 128 columns are one or two heads of
// q, k or v (a tile never straddles two of them); channel c and its rotation
// partner c+32 of a head are acc.v[2h] / acc.v[2h+1] of the same lane, and
// both use angle column c of the RoPE tables (DINOv3's tables repeat columns
// 0..31 in 32..63; only the first half is read, from the LDS tables of
// rope_table_dma). Results are rounded to f16 and regrouped in registers
// (frag_swap) so each lane holds 8 consecutive channels of its row. q, k
// and v are [image][head] matrices of tpad rows x 64 channels, each in
// fragment order: a lane's 8 channels are one 16-byte piece of a fragment,
// so the 64 lanes of a store cover one or two runs of whole rows' pieces per
// half-fragment (a row-major head row would take 32 separate 32-byte writes
// per store instead). Launched with rope_lds_bytes(grid) of dynamic LDS.
template <class T, bool LN>
__global__ __launch_bounds__(T::THREADS, T::FM == 1 ? (T::BK == 32 ? 4 : 3) : 2) void qkv_rope_kernel(DHX_QKV_PARAMS) {
    const QkvArgs p{h_, w_, bias_, cos_, sin_, q_, k_, v_, images_, grid_, tpad_, stats_, wsum_};
    static_assert(T::TN % kHeadDim == 0 && kHidden % T::BN == 0 && T::WGN == 1,
                  "whole heads per wave and tile, whole rows per wave");
    __shared__ __attribute__((aligned(16))) half_t wb0[T::WF_HALFS], wb1[T::WF_HALFS], wb2[T::WF_HALFS];
    __shared__ __attribute__((aligned(16))) float cst[2][T::BN];  // bias, wsum of the tile's columns
    __shared__ float2_t rows_norm[T::BM];                          // (mean, rstd) of the tile's rows
    extern __shared__ __attribute__((aligned(16))) float rope_lds[];  // rope_table_dma's four tables
    static_assert(T::BN <= T::THREADS, "one thread per column constant");
    const int P = p.grid * p.grid, Tok = P + kPrefix, M = p.images * Tok;
    constexpr int NT = 3 * kHidden / T::BN;
    const int tid = threadIdx.x;
    ActFrags<T> al[2];
    init_frags(al, p.h, M, kHidden);
    WeightDma<T> wd(p.w, 3 * kHidden, kHidden);
    // The epilogue's own operands are loaded ahead of the K loop: the RoPE
    // tables (DMA, first: they are the oldest loads every later wait covers),
    // the tile's column constants and its rows' LayerNorm (mean, rstd), all
    // of which wait in LDS.
    float4_t raw[T::FM][3];
    float cb = 0.f, cw = 0.f;
    gemm_tile_dma<T, 1, kHidden / T::BK>(
        al, wd, wb0, wb1, wb2, NT, NT * ((M + T::BM - 1) / T::BM), kHidden / T::BK,
        [&](int m0, int n0) {
            rope_table_dma<T::WAVES>(p.cos, p.sin, p.grid, rope_lds, tid);
            const Frag<T> f(m0, n0);
            if constexpr (LN) {
#pragma unroll
                for (int j = 0; j < T::FM; ++j) {
                    const float4_t* sp = (const float4_t*)(p.stats + (size_t)min(f.row(j), M - 1) * kStatFloats);
                    raw[j][0] = sp[0];
                    raw[j][1] = sp[1];
                    raw[j][2] = sp[2];
                }
            }
            if (tid < T::BN) {
                cb = p.bias[n0 + tid];
                if constexpr (LN) cw = p.wsum[n0 + tid];
            }
        },
        [&] {
            if (tid < T::BN) {
                cst[0][tid] = cb;
                cst[1][tid] = cw;
            }
            if constexpr (LN) {
                const int lane = tid & 63, r0 = (tid >> 6) % T::WGM * T::TM;
#pragma unroll
                for (int j = 0; j < T::FM; ++j) {
                    const RowNorm rn = row_norm<true>(raw[j][0], raw[j][1], raw[j][2]);
                    if (lane < 32) rows_norm[r0 + j * 32 + lane] = float2_t{rn.mean, rn.rstd};
                }
            }
        },
        [&](const Acc<T>& acc, int m0, int n0) {
        const Frag<T> f(m0, n0);
        qkv_epilogue<T, LN>(p, acc, f, m0, n0, cst[0], cst[1], rope_lds, [&](int j) {
            if constexpr (!LN) return RowNorm{0.f, 1.f};
            const float2_t v = rows_norm[f.m_base - m0 + j * 32 + f.l32];
            return RowNorm{v[0], v[1]};
        });
    });
}

// The QKV GEMM on a ring, for launches that fit one round of workgroups (see
// the launcher and resid_ring_kernel): everything the epilogue needs comes
// through LDS by DMA ahead of the stages. In a forward the launch starts with
// cold L2s, and qkv_rope_kernel's twelve 32-deep steps then each wait for a
// load; here three 64-deep stages are in flight (two on 128-row tiles). At 201
// rows 5.1 -> 4.7 us alone with warm caches, 2.3 us per launch less in the forward.
template <class T, int NST, bool LN>
__global__ __launch_bounds__(T::THREADS, (Ring<T, NST>::MIN_WAVES)) void qkv_ring_kernel(DHX_QKV_PARAMS) {
    const QkvArgs p{h_, w_, bias_, cos_, sin_, q_, k_, v_, images_, grid_, tpad_, stats_, wsum_};
    static_assert(T::TN % kHeadDim == 0 && kHidden % T::BN == 0, "whole heads per wave and tile");
    DHX_RING_BUFS(T, NST);
    __shared__ __attribute__((aligned(16))) float bias[dma_copy_bytes(T::BN * 4) / 4], wsum[dma_copy_bytes(T::BN * 4) / 4];
    __shared__ __attribute__((aligned(16))) float stats[dma_copy_bytes(T::BM * kStatFloats * 4) / 4];
    extern __shared__ __attribute__((aligned(16))) float rope_lds[];  // rope_table_dma's four tables
    const int M = p.images * (p.grid * p.grid + kPrefix);
    constexpr int NT = 3 * kHidden / T::BN;
    const int tid = threadIdx.x;
    const int t = xcd_tile(NT * ((M + T::BM - 1) / T::BM));
    if (t < 0) return;  // uniform per workgroup
    const int n0 = (t % NT) * T::BN, m0 = (t / NT) * T::BM;
    const Frag<T> f(m0, n0);
    rope_table_dma<T::WAVES>(p.cos, p.sin, p.grid, rope_lds, tid);
    dma_copy<T::BN * 4, T::WAVES>(dma_src(p.bias + n0, T::BN * 4), bias, tid);
    if constexpr (LN) {
        dma_copy<T::BN * 4, T::WAVES>(dma_src(p.wsum + n0, T::BN * 4), wsum, tid);
        dma_copy<T::BM * kStatFloats * 4, T::WAVES>(
            dma_src(p.stats + (size_t)m0 * kStatFloats, min(T::BM, M - m0) * kStatFloats * 4), stats, tid);
    }
    const Ring<T, NST> ring(p.h, p.w, M, kHidden, m0, n0);
    RowNorm rn[T::FM];
    Acc<T> acc;
    gemm_main_ring<T, NST, kHidden / T::BK>(ring, bufs, acc, [&](Acc<T>&, auto S) {
        if constexpr (LN && decltype(S)::value == 0) {
#pragma unroll
            for (int j = 0; j < T::FM; ++j) rn[j] = row_norm<true>(stats, f.row(j) - m0);
        }
    });
    qkv_epilogue<T, LN>(p, acc, f, m0, n0, bias, wsum, rope_lds,
                        [&](int j) { return LN ? rn[j] : RowNorm{0.f, 1.f}; });
}

// This lane's piece of the first fragment of row block j of the wave's part
// of x (a row block past the rows repeats the last one); the next fragments
// follow 64 pieces apart.
template <class T>
__device__ __forceinline__ half8_t* resid_frag(const ResidArgs& p, const Frag<T>& f, int mblocks, int j) {
    const int mb = min(f.m_base / 32 + j, mblocks - 1);
    return (half8_t*)(p.x + ((size_t)mb * (kHidden / 16) + f.n_base / 16) * 512) + (threadIdx.x & 63);
}

// Epilogue of the residual GEMMs: x += ls * acc + ls * b (cst[0] = ls * b,
// cst[1] = ls of the tile's columns), with STATS also the row statistics of
// the updated x. Each 16-column half of an MFMA result becomes a fragment in
// registers (frag_swap), and x is read (xold, loaded before the K loop: each
// element belongs to one tile, so nothing else writes it meanwhile) and
// written fragment by fragment, 1 KB contiguous per wave access. A statistics
// slot is 64 columns: waves of 32 columns come in pairs, and the second
// hands its rounded values to the first through LDS (hand: 2 KB per row
// block; every load must have landed), which then sums all 64 in the same
// order as a 64-column wave.
template <class T, bool STATS>
__device__ __forceinline__ void resid_epilogue(const ResidArgs& p, const Acc<T>& acc,
                                               const half8_t (&xold)[T::FM][T::TN / 16], const float (&cst)[2][T::BN],
                                               const Frag<T>& f, int n0, int mblocks, half8_t* hand) {
    static_assert(T::TN == 64 || (T::TN == 32 && T::WGN == 2 && T::FM == 1), "one statistics slot per wave or pair");
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < T::FM; ++j) {
        const int m = f.m_base + j * 32 + f.l32;
        const bool valid = m < p.rows;
        float v[32];
        half8_t h[T::TN / 16];
        half8_t* const x = resid_frag(p, f, mblocks, j);
#pragma unroll
        for (int i = 0; i < T::FN; ++i) {
            float4_t u[4];
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int nt = f.col(i, g) - n0;  // column in the tile
                const float4_t bl = *(const float4_t*)&cst[0][nt], l = *(const float4_t*)&cst[1][nt];
#pragma unroll
                for (int e = 0; e < 4; ++e) u[g][e] = fmaf(acc.v[i][j][4 * g + e], l[e], bl[e]);
            }
            frag_swap(u[0], u[1]);
            frag_swap(u[2], u[3]);
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) {
                const half8_t old = xold[j][2 * i + kk];
                half8_t& n = h[2 * i + kk];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    n[e] = (half_t)((float)old[e] + u[2 * kk][e]);
                    n[e + 4] = (half_t)((float)old[e + 4] + u[2 * kk + 1][e]);
                }
                if (valid) x[(2 * i + kk) * 64] = n;
#pragma unroll
                for (int e = 0; e < 8; ++e) v[(2 * i + kk) * 8 + e] = (float)n[e];
            }
        }
        if constexpr (STATS && T::TN == 32) {
            half8_t* const pair = hand + (f.m_base % T::BM) / 32 * 128;
            const bool first = f.n_base % 64 == 0;  // uniform per wave
            lds_barrier();                          // every wave is done reading the LDS behind hand
            if (!first) {
                pair[lane] = h[0];
                pair[64 + lane] = h[1];
            }
            lds_barrier();
            if (first) {
#pragma unroll
                for (int kk = 0; kk < 2; ++kk) {
                    const half8_t other = pair[kk * 64 + lane];
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[16 + kk * 8 + e] = (float)other[e];
                }
            }
            if (first) pair_stats(p.stats, m, f.n_base / 64, v, f.hi, valid);
        } else if constexpr (STATS) {
            pair_stats(p.stats, m, f.n_base / 64, v, f.hi, valid);
        }
    }
}

// Residual GEMM: x += ls * (A W^T + b), in place on the f16 residual stream
// in fragment order (with STATS, also the LayerNorm row statistics of the
// updated x); LDS holds only the weight stages and the column constants.
template <class T, bool STATS, int KT = 0>
__global__ __launch_bounds__(T::THREADS, T::BK == 128 ? 3 : 4) void resid_kernel(DHX_RESID_PARAMS) {
    const ResidArgs p{a_, w_, bias_, ls_, x_, rows_, k_, stats_};
    static_assert(T::TN % 64 == 0 && T::TM == 32, "whole statistics slots, one 32-row block per wave");
    static_assert(T::BN <= T::THREADS, "one thread per column constant");
    constexpr int XF = T::TN / 16;  // x fragments per wave
    __shared__ __attribute__((aligned(16))) half_t wb0[T::WF_HALFS], wb1[T::WF_HALFS], wb2[T::WF_HALFS];
    __shared__ __attribute__((aligned(16))) float cst[2][T::BN];  // bias * ls, ls of the tile's columns
    constexpr int NT = kHidden / T::BN;
    const int tid = threadIdx.x, mblocks = (p.rows + 31) / 32;
    ActFrags<T> al[2];
    init_frags(al, p.a, p.rows, p.k);
    WeightDma<T> wd(p.w, kHidden, p.k);
    // The epilogue's own operands are loaded ahead of the K loop: the old x
    // fragments of the wave's 32 x TN block and the column constants (into
    // LDS).
    half8_t xold[1][XF];
    float cb = 0.f, cl = 0.f;
    gemm_tile_dma<T, 1, KT>(
        al, wd, wb0, wb1, wb2, NT, NT * ((p.rows + T::BM - 1) / T::BM), p.k / T::BK,
        [&](int m0, int n0) {
            const Frag<T> f(m0, n0);
#pragma unroll
            for (int i = 0; i < XF; ++i) xold[0][i] = resid_frag(p, f, mblocks, 0)[i * 64];
            if (tid < T::BN) {
                cb = p.bias[n0 + tid];
                cl = p.ls[n0 + tid];
            }
        },
        [&] {
            if (tid < T::BN) {
                cst[0][tid] = cb * cl;  // ls * (acc + b) = acc * ls + b * ls: one FMA per output
                cst[1][tid] = cl;
            }
        },
        [&](const Acc<T>& acc, int m0, int n0) {
            const Frag<T> f(m0, n0);
            if (f.m_base / 32 >= mblocks) return;  // uniform per wave
            resid_epilogue<T, STATS>(p, acc, xold, cst, f, n0, mblocks, nullptr);
        });
}

// The residual GEMMs on a ring, for launches that fit one round of workgroups
// (see the launcher). There the time is the latency of a chain of stage
// loads, and of a workgroup's loads through its CU's 64 bytes per clock:
// small tiles spread the bytes over the chip and NST - 1 stages in flight
// hide the latency that resid_kernel, with its activations one step ahead,
// waits for in every step. Down projection at 201 rows 8.5 -> 5.8 us, at 1608
// rows 8.7 -> 6.0 us; o-projection 4.3 -> 3.6 and 4.45 -> 3.9 us (HIP events,
// alone). The column constants come through LDS by DMA as well, so that the
// old x fragments, used only after every load has landed, are the only
// register loads.
template <class T, int NST, bool STATS, int KT>
__global__ __launch_bounds__(T::THREADS, (Ring<T, NST>::MIN_WAVES)) void resid_ring_kernel(DHX_RESID_PARAMS) {
    const ResidArgs p{a_, w_, bias_, ls_, x_, rows_, k_, stats_};
    static_assert(T::BN <= T::THREADS, "one thread per column constant");
    DHX_RING_BUFS(T, NST);
    __shared__ __attribute__((aligned(16))) float raw_b[dma_copy_bytes(T::BN * 4) / 4], raw_l[dma_copy_bytes(T::BN * 4) / 4];
    __shared__ __attribute__((aligned(16))) float cst[2][T::BN];  // bias * ls, ls of the tile's columns
    constexpr int NT = kHidden / T::BN;
    const int tid = threadIdx.x, mblocks = (p.rows + 31) / 32;
    const int t = xcd_tile(NT * ((p.rows + T::BM - 1) / T::BM));
    if (t < 0) return;  // uniform per workgroup
    const int n0 = (t % NT) * T::BN, m0 = (t / NT) * T::BM;
    const Frag<T> f(m0, n0);
    half8_t xold[T::FM][T::TN / 16];
#pragma unroll
    for (int j = 0; j < T::FM; ++j)
#pragma unroll
        for (int i = 0; i < T::TN / 16; ++i) xold[j][i] = resid_frag(p, f, mblocks, j)[i * 64];
    compiler_fence();
    dma_copy<T::BN * 4, T::WAVES>(dma_src(p.bias + n0, T::BN * 4), raw_b, tid);
    dma_copy<T::BN * 4, T::WAVES>(dma_src(p.ls + n0, T::BN * 4), raw_l, tid);
    const Ring<T, NST> ring(p.a, p.w, p.rows, p.k, m0, n0);
    Acc<T> acc;
    gemm_main_ring<T, NST, KT>(ring, bufs, acc, [&](Acc<T>&, auto S) {
        if (decltype(S)::value == 0 && tid < T::BN) {
            cst[0][tid] = raw_b[tid] * raw_l[tid];
            cst[1][tid] = raw_l[tid];
        }
    });
    resid_epilogue<T, STATS>(p, acc, xold, cst, f, n0, mblocks, (half8_t*)ring0);
}

// Epilogue of the SwiGLU GEMM (see swiglu_kernel): bias holds the tile's
// column constants, gate columns scaled by -log2(e) and up columns by -ln(2).
template <class T>
__device__ __forceinline__ void swiglu_epilogue(const SwigluArgs& p, const Acc<T>& acc, const Frag<T>& f, int n0,
                                                const float* bias, const RowNorm (&rn)[T::FM]) {
    const int lane = threadIdx.x & 63, mblocks = (p.rows + 31) / 32;
    // Pair q of the wave: gate = acc.v[2q], up = acc.v[2q + 1], outputs
    // 32q .. 32q+31 of the wave's OW, i.e. act fragments 2q and 2q + 1.
    // With gate g and up u (after LayerNorm folding and bias), the output
    // silu(g) u = g u / (1 + e^-g) is computed from gs = -g log2(e) and
    // us = -u ln(2) as gs us / (1 + 2^gs) (gs us = g u): the scales ride
    // on the FMAs that apply rstd and the bias, which saves the multiply
    // that would otherwise form the exponent.
#pragma unroll
    for (int j = 0; j < T::FM; ++j) {
        const int mb = f.m_base / 32 + j;
        if (mb >= mblocks) break;  // uniform per wave
        const float sg = rn[j].rstd * -kLog2e, su = rn[j].rstd * -kLn2;
        const WtOut act(p.act + (size_t)mb * (kFF / 16) * 512, 32 * kFF * 2);
#pragma unroll
        for (int q = 0; q < T::FN / 2; ++q) {
            half4_t y[4];
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int c = g * 8 + f.hi * 4, nl = f.n_base - n0 + 64 * q + c;
                float4_t gate = group4(acc.v[2 * q][j], g), up = group4(acc.v[2 * q + 1][j], g);
                const float4_t bg = *(const float4_t*)&bias[nl], bu = *(const float4_t*)&bias[nl + 32];
                float4_t r;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float gs = fmaf(gate[e], sg, bg[e]), us = fmaf(up[e], su, bu[e]);
                    r[e] = gs * us * fast_rcp(1.0f + fast_exp2(gs));
                }
                y[g] = to_half4(r);
            }
#pragma unroll
            for (int kk = 0; kk < 2; ++kk)
                act.store(((f.n_base / 32 + 2 * q + kk) * 512 + lane * 8) * 2, frag_swap(y[2 * kk], y[2 * kk + 1]));
        }
    }
}

// The scale a column's bias is kept with (the first 32 of each 64 are gates).
__device__ __forceinline__ float swiglu_scale(int column) { return column % 64 < 32 ? -kLog2e : -kLn2; }

// Adds the folded LayerNorm's -mean * wsum to column block i of the
// accumulators; wsum: the 32 columns of the block.
template <class T>
__device__ __forceinline__ void swiglu_mean(Acc<T>& acc, int i, const float* wsum, const RowNorm (&rn)[T::FM]) {
    const int hi = (threadIdx.x & 63) >> 5;
    float4_t w[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) w[g] = *(const float4_t*)&wsum[8 * g + 4 * hi];
#pragma unroll
    for (int j = 0; j < T::FM; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc.v[i][j][4 * g + e] = fmaf(-rn[j].mean, w[g][e], acc.v[i][j][4 * g + e]);
}

// SwiGLU dual GEMM. W rows are packed as blocks of 32 gate rows followed by
// the 32 matching up rows, so a wave's 128 columns are two gate/up pairs of
// 32 outputs each. The tile's column constants (bias, and wsum with the
// folded LayerNorm) and its rows' statistics are loaded before the K loop;
// the constants wait in LDS. The epilogue turns each 16-column half of a
// 32-column act block into a fragment in registers (frag_swap) and writes
// it whole (act is in fragment order).
// NS: N slices of the XCD tile split (xcd_tile_split); the launcher picks
// it by the launch's size.
template <class T, bool LN, int NS>
__global__ __launch_bounds__(T::THREADS, T::FM == 1 ? 3 : 2) void swiglu_kernel(DHX_SWIGLU_PARAMS) {
    const SwigluArgs p{h_, w_, bias_, act_, rows_, stats_, wsum_};
    static_assert(T::TN % 64 == 0 && T::WGN == 1, "whole gate/up pairs, whole rows per wave");
    static_assert(T::BN <= T::THREADS, "one thread per column constant");
    static_assert(kHidden / T::BK > T::FN, "a K-loop step for every column block's LayerNorm mean term");
    __shared__ __attribute__((aligned(16))) half_t wb0[T::WF_HALFS], wb1[T::WF_HALFS], wb2[T::WF_HALFS];
    __shared__ __attribute__((aligned(16))) float cst[2][T::BN];  // bias, wsum
    constexpr int NT = 2 * kFF / T::BN;
    const int tid = threadIdx.x;
    ActFrags<T> al[2];
    init_frags(al, p.h, p.rows, kHidden);
    WeightDma<T> wd(p.w, 2 * kFF, kHidden);
    float4_t raw[T::FM][3];
    RowNorm rn[T::FM];
    float cb = 0.f, cw = 0.f;
    gemm_tile_dma<T, NS, kHidden / T::BK>(
        al, wd, wb0, wb1, wb2, NT, NT * ((p.rows + T::BM - 1) / T::BM), kHidden / T::BK,
        [&](int m0, int n0) {
            const Frag<T> f(m0, n0);
            if constexpr (LN) {
#pragma unroll
                for (int j = 0; j < T::FM; ++j) {
                    const float4_t* sp = (const float4_t*)(p.stats + (size_t)min(f.row(j), p.rows - 1) * kStatFloats);
                    raw[j][0] = sp[0];
                    raw[j][1] = sp[1];
                    raw[j][2] = sp[2];
                }
            }
            if (tid < T::BN) {
                cb = p.bias[n0 + tid];
                if constexpr (LN) cw = p.wsum[n0 + tid];
            }
        },
        [&] {
            if (tid < T::BN) {
                cst[0][tid] = cb * swiglu_scale(tid);
                cst[1][tid] = cw;
            }
#pragma unroll
            for (int j = 0; j < T::FM; ++j) rn[j] = LN ? row_norm<false>(raw[j][0], raw[j][1], raw[j][2]) : RowNorm{0.f, 1.f};
        },
        [&](const Acc<T>& acc, int m0, int n0) {
        const Frag<T> f(m0, n0);
        swiglu_epilogue<T>(p, acc, f, n0, cst[0], rn);
    },
    // The folded LayerNorm's -mean * wsum, added to column block i of the
    // accumulators at step i + 1 of the K loop (an additive term may join
    // the sum at any point), where its FMAs issue beside the MFMAs instead
    // of lengthening the epilogue.
    [&](Acc<T>& acc, int s) {
        if constexpr (LN) {
            static_for<T::FN>([&](auto I) {
                constexpr int i = decltype(I)::value;
                if (s == i + 1) swiglu_mean<T>(acc, i, &cst[1][32 * i], rn);
            });
        }
    });
}

// The SwiGLU GEMM on a ring, for launches that fit one round of workgroups
// (see the launcher and resid_ring_kernel), its column constants and row
// statistics through LDS by DMA; alone at 201 rows 5.3 -> 4.9 us, at 1206
// rows 7.4 -> 5.7, at 1608 rows 7.4 -> 6.8. The folded LayerNorm's mean term joins column
// block b (of each 128 columns) before K step 64(b + 1), as in swiglu_kernel,
// so a row's result is bitwise the same on either.
template <class T, int NST, bool LN>
__global__ __launch_bounds__(T::THREADS, (Ring<T, NST>::MIN_WAVES)) void swiglu_ring_kernel(DHX_SWIGLU_PARAMS) {
    const SwigluArgs p{h_, w_, bias_, act_, rows_, stats_, wsum_};
    static_assert(T::TN % 64 == 0, "whole gate/up pairs");
    static_assert(T::BN <= T::THREADS && T::BK <= 64, "one thread per column constant");
    DHX_RING_BUFS(T, NST);
    __shared__ __attribute__((aligned(16))) float raw[dma_copy_bytes(T::BN * 4) / 4], wsum[dma_copy_bytes(T::BN * 4) / 4];
    __shared__ __attribute__((aligned(16))) float stats[dma_copy_bytes(T::BM * kStatFloats * 4) / 4], bias[T::BN];
    constexpr int NT = 2 * kFF / T::BN;
    const int tid = threadIdx.x;
    const int t = xcd_tile(NT * ((p.rows + T::BM - 1) / T::BM));
    if (t < 0) return;  // uniform per workgroup
    const int n0 = (t % NT) * T::BN, m0 = (t / NT) * T::BM;
    const Frag<T> f(m0, n0);
    dma_copy<T::BN * 4, T::WAVES>(dma_src(p.bias + n0, T::BN * 4), raw, tid);
    if constexpr (LN) {
        dma_copy<T::BN * 4, T::WAVES>(dma_src(p.wsum + n0, T::BN * 4), wsum, tid);
        dma_copy<T::BM * kStatFloats * 4, T::WAVES>(
            dma_src(p.stats + (size_t)m0 * kStatFloats, min(T::BM, p.rows - m0) * kStatFloats * 4), stats, tid);
    }
    const Ring<T, NST> ring(p.h, p.w, p.rows, kHidden, m0, n0);
    const int nb = __builtin_amdgcn_readfirstlane(f.n_base / 32);  // first column block of the wave
    RowNorm rn[T::FM];
    Acc<T> acc;
    gemm_main_ring<T, NST, kHidden / T::BK>(ring, bufs, acc, [&](Acc<T>& a, auto S) {
        constexpr int s = decltype(S)::value;
        if constexpr (s == 0) {
            if (tid < T::BN) bias[tid] = raw[tid] * swiglu_scale(tid);
#pragma unroll
            for (int j = 0; j < T::FM; ++j) rn[j] = LN ? row_norm<false>(stats, f.row(j) - m0) : RowNorm{0.f, 1.f};
        }
        if constexpr (LN && s > 0 && s * T::BK % 64 == 0 && s * T::BK <= 256) {
            static_for<T::FN>([&](auto I) {
                constexpr int i = decltype(I)::value;
                if ((nb + i) % 4 == s * T::BK / 64 - 1) swiglu_mean<T>(a, i, &wsum[f.n_base - n0 + 32 * i], rn);
            });
        }
    });
    swiglu_epilogue<T>(p, acc, f, n0, bias, rn);
}

// Split-K GEMM into f32 slabs [split][rows][384]; no atomics, so results do
// not depend on scheduling. The tile space is (split, m tile) x n tile: a
// tile's m origin runs over splits * padded rows, and both loaders decode the
// split (their K offset) from it.
template <class T>
struct SplitDecode {
    int mt, kc;
    __device__ __forceinline__ int split(int m0) const { return m0 / T::BM / mt; }
    __device__ __forceinline__ int row0(int m0) const { return m0 - split(m0) * mt * T::BM; }
};

template <class T>
struct SplitActFrags : ActFrags<T> {
    SplitDecode<T> d;
    __device__ __forceinline__ void load(int m0, int n0, int kt, int tid) {
        this->ks_off = d.split(m0) * (d.kc / 16);
        ActFrags<T>::load(d.row0(m0), n0, kt, tid);
    }
};

template <class T, int KT = 0>
__global__ __launch_bounds__(T::THREADS, 3) void splitk_kernel(DHX_SPLITK_PARAMS) {
    const SplitKArgs p{a_, w_, partials_, rows_, k_, splits_};
    __shared__ __attribute__((aligned(16))) half_t wb0[T::WF_HALFS], wb1[T::WF_HALFS], wb2[T::WF_HALFS];
    constexpr int NT = kHidden / T::BN;
    const int MT = (p.rows + T::BM - 1) / T::BM;
    const SplitDecode<T> d{MT, p.k / p.splits};
    ActFrags<T> base[2];
    init_frags(base, p.a, p.rows, p.k);
    SplitActFrags<T> al[2] = {{base[0], d}, {base[1], d}};
    WeightDma<T> wd(p.w, kHidden, p.k);
    gemm_tile_dma<T, 1, KT>(
        al, wd, wb0, wb1, wb2, NT, NT * MT * p.splits, d.kc / T::BK,
        [&](int m0, int) { wd.ks_off = d.split(m0) * (d.kc / 16); }, [] {},
        [&](const Acc<T>& acc, int m0, int n0) {
            const Frag<T> f(d.row0(m0), n0);
            float* slab = p.partials + (size_t)d.split(m0) * p.rows * kHidden;
            const int m = f.row(0);
            if (m >= p.rows) return;
#pragma unroll
            for (int i = 0; i < T::FN; ++i)
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    *(float4_t*)(slab + (size_t)m * kHidden + f.col(i, g)) = group4(acc.v[i][0], g);
        });
}

}  // namespace gemm
}  // namespace dhx
