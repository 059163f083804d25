// Host-side launchers for the forward-pass kernels. Each launcher assumes the
// engine has already checked every binding's size against the shapes below
// (engine.cpp: required_bytes); they only derive grids and launch.
//
// The f16 activations x, h, attn and act are stored in fragment order
// (common.hpp: frag_piece), rows padded to a multiple of 32; "[rows][K] frag"
// below means that layout.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstring>

#include "common.hpp"

namespace dhx {

// Row LayerNorm over 384 channels, eps 1e-5, fp32 statistics.
// x [rows][384] frag -> out [rows][384] frag f16 (or row-major f32 when
// f32_out).
struct LayerNormArgs {
    const half_t* x;
    const float* gamma;
    const float* beta;
    void* out;
    int rows;
    int f32_out;
};

// Fused patch embedding: im2col of NCHW f32 pixels (patch order (gy, gx),
// k order (c, dy, dx)), GEMM with patch_w [384][768] f16, + bias, narrowed to
// f16 and scattered into x [images*T][384] frag after the CLS + 4 register
// rows, which are copied from prefix [5][384] f32.
struct PatchEmbedArgs {
    const float* pixels;
    const half_t* w;
    const float* bias;
    const float* prefix;
    half_t* x;
    int images;
    int grid;  // patches per side G; image side 16*G, T = G*G + 5
    // Optional (both or neither): row statistics of x for a fused LayerNorm
    // consumer; prefix_stats holds those of the 5 prefix rows [5][6][2].
    const float* prefix_stats = nullptr;
    float* stats = nullptr;
};

// Row statistics of the residual stream x for LayerNorm fused into the next
// GEMM: stats[row][slot][2] = (mean, M2) of the f16 values of x in columns
// 64*slot .. 64*slot+63, slot 0..5 (M2 = sum of squared deviations from that
// slot's mean). A consumer combines the six slots (Chan et al.'s pairwise
// update) into the row mean and variance.
constexpr int kStatSlots = kHidden / 64;
constexpr int kStatFloats = 2 * kStatSlots;

// h [rows][384] frag . Wqkv[1152][384]^T + b, 2D RoPE on q and k of patch
// tokens, written per (image, head): q, k, v [images][6] matrices of
// [tpad][64] in fragment order (rows past the image's tokens are never
// written). cos / sin are [patches][64] with columns
// 32..63 repeating 0..31 (the rotation of channels c and c+32 uses angle c);
// only columns 0..31 are read.
// With stats == nullptr: h = LN1(x) is given and out = h.W^T + bias. With
// stats: h is the raw residual x, w holds W' = gamma (.) W (per input
// channel), wsum[n] = sum_k W'[n][k] and bias holds t = b + beta.W^T, so
// out = rstd * (x.W'^T - mean * wsum) + t = LN(x).W^T + b.
struct QkvArgs {
    const half_t* h;
    const half_t* w;
    const float* bias;
    const float* cos;
    const float* sin;
    half_t* q;
    half_t* k;
    half_t* v;
    int images;
    int grid;
    int tpad;
    const float* stats = nullptr;
    const float* wsum = nullptr;
    // Other kernels run beside this launch (concurrent image groups); chooses
    // the tile shape only, not the result.
    bool shared = false;
};

// softmax(q k^T / 8) v per (image, head) over that image's T tokens, with
// q, k, v as written by the QKV kernel; rows T .. tpad-1 of v must be finite
// (the engine zeroes buffers at allocation and nothing writes those rows).
// out [images*T][384] frag (head h in columns 64h .. 64h+63).
struct AttentionArgs {
    const half_t* q;
    const half_t* k;
    const half_t* v;
    half_t* out;
    int images;
    int tokens;
    int tpad;
    bool shared = false;  // as in QkvArgs
};

// x[rows][384] += ls * (a[rows][k] . W[384][k]^T + b), f16 residual in place
// (a and x frag).
struct ResidArgs {
    const half_t* a;
    const half_t* w;
    const float* bias;
    const float* ls;
    half_t* x;
    int rows;
    int k;
    float* stats = nullptr;  // optional: row statistics of the updated x
    bool shared = false;     // as in QkvArgs
};

// act[rows][1536] frag = silu(h.Wg^T + bg) * (h.Wu^T + bu), h frag; W and b are packed
// with gate and up rows interleaved in blocks of 32.
// stats / wsum: LayerNorm fused as in QkvArgs.
struct SwigluArgs {
    const half_t* h;
    const half_t* w;
    const float* bias;
    half_t* act;
    int rows;
    const float* stats = nullptr;
    const float* wsum = nullptr;
};

// partials[s][rows][384] = a[:, s*k/splits ...] . W[:, s*k/splits ...]^T
// (f32 row-major; a frag).
struct SplitKArgs {
    const half_t* a;
    const half_t* w;
    float* partials;
    int rows;
    int k;
    int splits;
};

// x[rows][384] frag += ls * (sum_s partials[s] + b).
struct ReduceArgs {
    const float* partials;
    const float* bias;
    const float* ls;
    half_t* x;
    int rows;
    int splits;
    float* stats = nullptr;  // optional: row statistics of the updated x
};

// Rows tokens .. tpad-1 of q, k and v ([images][6] fragment-order [tpad][64]
// matrices) set to zero:
// attention reads them as masked keys, so they must be finite. For buffers
// that did not come zeroed from the engine (the allocation-free forward's
// scratch, which keeps earlier calls' data). A fill kernel, not a memset, so
// that the launch can be captured into a graph.
struct PadRowsArgs {
    half_t* q;
    half_t* k;
    half_t* v;
    int images;
    int tokens;
    int tpad;
};

// Kernels take their arguments one by one, in the order of first use: the
// first fourteen words are then in scalar registers when a wave starts
// (-amdgpu-kernarg-preload-count, build.py), where a struct is read with
// scalar loads whose first one misses every cache. A chain of dependent
// launches in a graph took 1.96 us per launch with the loads, 1.83 without.
// DHX_<kernel>_PARAMS declares the parameters, from which each kernel gathers
// its struct, and start() launches a kernel on one.

// A device pointer as a kernel parameter that the runtime takes for a number
// (a parameter of pointer type costs host time in every launch, see enqueue).
// To the kernel it is a pointer to global memory either way.
struct Addr {
    uint64_t a;
    Addr() = default;
    Addr(const void* p) : a(reinterpret_cast<uint64_t>(p)) {}
    template <class T>
    __device__ __forceinline__ operator T*() const {
        return (T*)(__attribute__((address_space(1))) T*)a;
    }
};

#define DHX_LAYERNORM_PARAMS Addr x_, Addr gamma_, Addr beta_, Addr out_, int rows_, int f32_out_
#define DHX_PATCH_PARAMS Addr pixels_, Addr w_, Addr bias_, Addr prefix_, Addr x_, Addr stats_, int images_, int grid_, Addr prefix_stats_
#define DHX_QKV_PARAMS Addr cos_, Addr sin_, Addr h_, Addr w_, Addr bias_, Addr stats_, int images_, int grid_, Addr wsum_, Addr q_, Addr k_, Addr v_, int tpad_
#define DHX_ATTENTION_PARAMS Addr q_, Addr k_, Addr v_, Addr out_, int images_, int tokens_, int tpad_
#define DHX_RESID_PARAMS Addr x_, Addr a_, Addr w_, Addr bias_, Addr ls_, Addr stats_, int rows_, int k_
#define DHX_SWIGLU_PARAMS Addr h_, Addr w_, Addr bias_, Addr stats_, Addr wsum_, Addr act_, int rows_
#define DHX_SPLITK_PARAMS Addr a_, Addr w_, Addr partials_, int rows_, int k_, int splits_
#define DHX_REDUCE_PARAMS Addr partials_, Addr bias_, Addr ls_, Addr x_, Addr stats_, int rows_, int splits_
#define DHX_PAD_ROWS_PARAMS Addr q_, Addr k_, Addr v_, int images_, int tokens_, int tpad_

// Launches a kernel on its arguments packed into one buffer, each at its
// natural alignment, as they lie in the kernel's argument segment. Host time
// of the allocation-free call at one image (63 launches), with pointers passed
// one by one / packed / packed as Addr: captured 111 / 82 / 81 us, the
// capture's end and instantiation 123 / 104 / 87, queued directly 246 / 237 /
// 202; one struct per kernel, without the preload, took 85, 87 and 208.
template <class... P, class... A>
hipError_t enqueue(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t s, A... args) {
    static_assert(sizeof...(P) == sizeof...(A), "one argument per parameter");
    static_assert(((sizeof(P) <= 8) && ...), "the buffer holds every argument");
    alignas(8) unsigned char packed[8 * sizeof...(P)];
    size_t size = 0;
    auto put = [&](auto value) {
        size = (size + sizeof(value) - 1) / sizeof(value) * sizeof(value);
        std::memcpy(packed + size, &value, sizeof(value));
        size += sizeof(value);
    };
    (put(static_cast<P>(args)), ...);
    void* extra[] = {HIP_LAUNCH_PARAM_BUFFER_POINTER, packed, HIP_LAUNCH_PARAM_BUFFER_SIZE, &size, HIP_LAUNCH_PARAM_END};
    hipFunction_t f = nullptr;
    hipError_t err = hipGetFuncBySymbol(&f, reinterpret_cast<const void*>(kernel));
    if (err == hipSuccess)
        err = hipModuleLaunchKernel(f, grid.x, grid.y, grid.z, block.x, block.y, block.z, (unsigned)lds, s, nullptr, extra);
    if (err != hipSuccess) (void)hipGetLastError();  // reported by the caller, once
    return err;
}

template <class... P>
hipError_t start(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t s, const LayerNormArgs& a) {
    return enqueue(kernel, grid, block, lds, s, a.x, a.gamma, a.beta, a.out, a.rows, a.f32_out);
}
template <class... P>
hipError_t start(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t s, const PatchEmbedArgs& a) {
    return enqueue(kernel, grid, block, lds, s, a.pixels, a.w, a.bias, a.prefix, a.x, a.stats, a.images, a.grid, a.prefix_stats);
}
template <class... P>
hipError_t start(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t s, const QkvArgs& a) {
    return enqueue(kernel, grid, block, lds, s, a.cos, a.sin, a.h, a.w, a.bias, a.stats, a.images, a.grid, a.wsum, a.q, a.k, a.v, a.tpad);
}
template <class... P>
hipError_t start(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t s, const AttentionArgs& a) {
    return enqueue(kernel, grid, block, lds, s, a.q, a.k, a.v, a.out, a.images, a.tokens, a.tpad);
}
template <class... P>
hipError_t start(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t s, const ResidArgs& a) {
    return enqueue(kernel, grid, block, lds, s, a.x, a.a, a.w, a.bias, a.ls, a.stats, a.rows, a.k);
}
template <class... P>
hipError_t start(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t s, const SwigluArgs& a) {
    return enqueue(kernel, grid, block, lds, s, a.h, a.w, a.bias, a.stats, a.wsum, a.act, a.rows);
}
template <class... P>
hipError_t start(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t s, const SplitKArgs& a) {
    return enqueue(kernel, grid, block, lds, s, a.a, a.w, a.partials, a.rows, a.k, a.splits);
}
template <class... P>
hipError_t start(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t s, const ReduceArgs& a) {
    return enqueue(kernel, grid, block, lds, s, a.partials, a.bias, a.ls, a.x, a.stats, a.rows, a.splits);
}
template <class... P>
hipError_t start(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t s, const PadRowsArgs& a) {
    return enqueue(kernel, grid, block, lds, s, a.q, a.k, a.v, a.images, a.tokens, a.tpad);
}

hipError_t launch_layernorm(const LayerNormArgs& a, hipStream_t s);
hipError_t launch_zero_pad_rows(const PadRowsArgs& a, hipStream_t s);
hipError_t launch_patch_embed(const PatchEmbedArgs& a, hipStream_t s);
hipError_t launch_qkv_rope(const QkvArgs& a, hipStream_t s);
hipError_t launch_attention(const AttentionArgs& a, hipStream_t s);
hipError_t launch_resid(const ResidArgs& a, hipStream_t s);
hipError_t launch_swiglu(const SwigluArgs& a, hipStream_t s);
hipError_t launch_splitk(const SplitKArgs& a, hipStream_t s);
hipError_t launch_splitk_reduce(const ReduceArgs& a, hipStream_t s);

}  // namespace dhx
