// Online-softmax attention for gfx950 (replaces the reference's
// kernels/attention_online_f16_wmma_cf16.loom).
//
// Three kernels share one step (attend32), each wave owning 32 queries of one
// (image, head) and taking 32 keys a step: attention_kernel (four waves walk
// all keys), attention_parallel_kernel (a wave per key block, for short
// sequences in small launches) and attention_split_kernel (two key halves, for
// long sequences); the launcher says which runs when. Keys stream through LDS in blocks of 32 or 64 (K and
// V both as [key][ch]). q, k and v come per (image, head) as [tpad][64]
// matrices in fragment order (a wave's Q fragments are then 1 KB contiguous
// loads). The blocks move from global memory straight into LDS with DMA loads
// (buffer_load ... lds), two blocks ahead or more; each 128-byte key row is
// stored with its 16-byte chunks XOR-swizzled by the
// row (swz below), so the row reads of K and the transpose reads of V hit
// distinct banks.
//
// Everything is computed transposed so that a lane owns one query:
//   S^T = K . Q^T      (MFMA a = K rows from LDS, b = Q^T held in registers)
//   O^T += V^T . P^T   (MFMA a = V^T rows, read out of the [key][ch] V block
//                       with LDS transpose reads; b = P^T straight from the
//                       S^T accumulators)
// Lane l holds query (l % 32) and 16 of every 32 keys; the other 16 are in
// lane l ^ 32, so each row max / row sum is 15 in-register ops plus one
// cross-half exchange, and the running rescale of O^T is a per-lane scalar.
// Q is scaled by 1/8 in registers and log2(e) is folded into one FMA per
// score, so the softmax runs on v_exp_f32; the running max is updated lazily
// (only when a block's weights against it sum past e^8), which skips
// most rescales of O and, on the common path, the block max itself.
// P is rounded to f16 for the PV product; the denominator keeps the fp32
// weights (as in the reference, attention_online_f16_wmma_cf16.loom:195-216).
#include <type_traits>

#include "launch.hpp"

namespace dhx {
namespace {

constexpr int kThreads = 256;
constexpr int QB = 128;                  // queries per workgroup
// The lazy rescaling's slack: the running max moves only when a block's
// weights against it sum past e^8 (some score more than 8 above it).
constexpr float kLazySum = 2980.957987f;  // e^8

// LDS on gfx950 has 64 banks of 4 bytes: two 128-byte key rows per bank
// cycle. Chunk c of key row r sits at slot c ^ swz_slot(r), with
// swz_slot(r) = f((r / 2) % 8), f(t) = 4 (t % 2) + t / 2 (a bijection). The
// K row reads of 16 lanes (16 consecutive rows, one chunk) then cover all
// 64 banks, and so do the V transpose reads (4 consecutive rows x 4 aligned
// chunks per 32 lanes: rows 2 apart differ in bit 2 of the slot).
__device__ __forceinline__ int swz_slot(int r) {
    const int t = (r >> 1) & 7;
    return ((t & 1) << 2) | (t >> 1);
}

// Element offset of channel ch (a multiple of 4) of key row r inside a
// swizzled block.
__device__ __forceinline__ int swz(int r, int ch) {
    return r * kHeadDim + ((((ch >> 3) ^ swz_slot(r)) & 7) << 3) + (ch & 7);
}

// Waits until at most N of this wave's vector-memory operations are
// outstanding and its LDS traffic is done, then joins the workgroup barrier.
template <int N>
__device__ __forceinline__ void vm_barrier() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// The running softmax state of one lane's query (lane l holds query l % 32
// and half of each 32-key sub-block's scores; see the top of this file).
struct QueryState {
    half8_t qf[4];                      // Q^T fragments, pre-scaled by 1/8
    float16_t o[2];                     // O^T accumulators: channels 32ct + 8(r/4) + 4hi + r%4
    float m_run = -1e30f, l_run = 0.f;  // running max (lazy) and denominator
};

// Transpose-read position of this lane inside a 4-key x 32-channel patch of
// a V block: lane j of each 16-lane group receives channel 16*(group%2) + j
// of four consecutive keys.
__device__ __forceinline__ int tr_row_of(int lane) { return (lane & 15) >> 2; }
__device__ __forceinline__ int tr_col_of(int lane) { return 16 * ((lane >> 4) & 1) + 4 * (lane & 3); }

// This lane's element offsets inside a 32-key sub-block: of its four K
// fragments, k(kk), and of its V transpose reads of 32-channel half ct, key
// rows 4hi + tr_row and 8 further, v(ct, r) (the key rows 16 further have the
// same swizzle). Computed once per kernel: the walks' steps are conditional,
// and the compiler does not share address arithmetic between them.
struct LaneOffsets {
    int k_[4], v_[2][2];
    __device__ __forceinline__ explicit LaneOffsets(int lane) {
        const int l32 = lane & 31, hi = lane >> 5;
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) k_[kk] = swz(l32, kk * 16 + hi * 8);
#pragma unroll
        for (int ct = 0; ct < 2; ++ct)
#pragma unroll
            for (int r = 0; r < 2; ++r) v_[ct][r] = swz(4 * hi + tr_row_of(lane) + 8 * r, ct * 32 + tr_col_of(lane));
    }
    __device__ __forceinline__ void step() {}
    __device__ __forceinline__ int k(int kk) const { return k_[kk]; }
    __device__ __forceinline__ int v(int ct, int r) const { return v_[ct][r]; }
};

// The same offsets from two registers instead of eight, for the kernel that
// would not fit its 128 otherwise: the others differ from the first by one
// exclusive or (chunk 2kk or 4ct, and a slot that changes in bit 1 with 8
// rows), taken anew in every step.
struct LaneOffsetsXor {
    int k_, v_;
    __device__ __forceinline__ explicit LaneOffsetsXor(int lane) {
        const int l32 = lane & 31, hi = lane >> 5;
        k_ = swz(l32, hi * 8);
        v_ = swz(4 * hi + tr_row_of(lane), tr_col_of(lane));
    }
    // Keeps the compiler from computing the other offsets ahead of the steps.
    __device__ __forceinline__ void step() { asm volatile("" : "+v"(k_), "+v"(v_)); }
    __device__ __forceinline__ int k(int kk) const { return k_ ^ (kk << 4); }
    __device__ __forceinline__ int v(int ct, int r) const { return (v_ ^ (ct << 5) ^ (r << 4)) + r * 8 * kHeadDim; }
};

// The pieces of one step over a 32-key block (keys key0 .. key0+31 of the
// sequence of T). Scores: s[r] is that of key key0 + 8(r/4) + 4*hi + r%4 for
// query l32 (S^T = K Q^T), -inf past T.
template <class Offsets>
__device__ __forceinline__ float16_t scores32(const half_t* sK, const half8_t (&qf)[4], const Offsets& at) {
    float16_t s = {};
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) s = mfma32x32x16(*(const half8_t*)(sK + at.k(kk)), qf[kk], s);
    return s;
}

__device__ __forceinline__ void mask32(float16_t& s, int key0, int T, int hi) {
    if (key0 + 32 > T) {  // the last, partial block of keys (uniform)
#pragma unroll
        for (int r = 0; r < 16; ++r)
            if (key0 + 8 * (r >> 2) + 4 * hi + (r & 3) >= T) s[r] = -__builtin_inff();
    }
}

// V^T operand of channels ct*32 + l32 and keys key0 + 16ks + (j < 4 ? 4hi + j
// : 8 + 4hi + j - 4).
template <class Offsets>
__device__ __forceinline__ half8_t v_frag(const half_t* sV, int ct, int ks, const Offsets& at) {
    const half4_t a0 = lds_read_tr16(sV + ks * 16 * kHeadDim + at.v(ct, 0));
    const half4_t a1 = lds_read_tr16(sV + ks * 16 * kHeadDim + at.v(ct, 1));
    return __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7);
}

// p = 2^(s log2e - m log2e); returns the sum over the lane pair.
__device__ __forceinline__ float weights32(const float16_t& s, float m, float (&p)[16]) {
    const float mb = m * kLog2e;
    float sum = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        p[r] = fast_exp2(fmaf(s[r], kLog2e, -mb));
        sum += p[r];
    }
    return half_pair_sum(sum);
}

__device__ __forceinline__ float block_max32(const float16_t& s) {
    float mx = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
    return half_pair_max(mx);  // every block holds a valid key of each pair
}

// P^T as the b operand: k-slice element j of this lane is the key of v_frag's
// element j.
__device__ __forceinline__ half8_t p_frag(const float (&p)[16], int ks) {
    half8_t b;
#pragma unroll
    for (int e = 0; e < 8; ++e) b[e] = (half_t)p[8 * ks + e];
    return b;
}

// One step over a 32-key block (rows row0 .. row0+31 of the swizzled K and V
// blocks in LDS): scores, lazy running max, weights P = 2^(s log2e - m log2e),
// O^T += V^T P^T with P in f16 and the denominator in f32. FIRST: the first
// block of a walk (O and l still zero), whose weights against the initial max
// of -1e30 would all overflow: its block max becomes the running max directly,
// with one pass of exponentials instead of two (the same values and rounding
// as the rescale path).
template <bool FIRST = false, class Offsets>
__device__ __forceinline__ void attend32(QueryState& st, const half_t* sK, const half_t* sV, int row0, int key0,
                                         int T, int lane, Offsets& at) {
    at.step();
    sK += row0 * kHeadDim;
    sV += row0 * kHeadDim;
    float16_t s = scores32(sK, st.qf, at);
    // The V^T operands do not depend on the softmax: read them now so their
    // LDS latency hides under the exponentials.
    half8_t va[2][2];
#pragma unroll
    for (int ct = 0; ct < 2; ++ct)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) va[ct][ks] = v_frag(sV, ct, ks, at);
    mask32(s, key0, T, lane >> 5);
    // Weights against the running max; after the first block (which takes its
    // own max), the block max is needed only when some lane's weights sum past
    // e^8 (a weight may then exceed it): blocks whose scores grew by more than
    // 8. Those lanes move their max to the block's, rescale O and l, and
    // recompute; every weight is then at most its sum, at most e^8, well
    // inside f16.
    float p[16], sum;
    if constexpr (FIRST) {
        st.m_run = fmaxf(block_max32(s), st.m_run);  // as below, also for a block whose scores are all -inf
        sum = weights32(s, st.m_run, p);
    } else {
        sum = weights32(s, st.m_run, p);
        const bool grow = !(sum <= kLazySum);
        if (__any(grow)) {  // uniform across the wave
            const float m_new = grow ? fmaxf(block_max32(s), st.m_run) : st.m_run;
            const float alpha = fast_exp2((st.m_run - m_new) * kLog2e);
            st.l_run *= alpha;
            st.o[0] *= alpha;
            st.o[1] *= alpha;
            st.m_run = m_new;
            sum = weights32(s, m_new, p);
        }
    }
    st.l_run += sum;
    const half8_t pb[2] = {p_frag(p, 0), p_frag(p, 1)};
#pragma unroll
    for (int ct = 0; ct < 2; ++ct)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) st.o[ct] = mfma32x32x16(va[ct][ks], pb[ks], st.o[ct]);
}

// Output of one lane's query, channel half ct: O / l in f16 into out (fragment
// order): each 16-channel half of the block becomes one 8-channel piece per
// lane after frag_swap. row0: the first query row of the wave (wave-uniform);
// the wave's 32 rows lie in its 32-row block and the next, which the
// write-through descriptor covers.
__device__ __forceinline__ void store_half(const float16_t& a, float inv, half_t* out, int row0, int row, int head,
                                           int ct, int hi) {
    const size_t base = (size_t)(row0 / 32) * (kHidden / 16) * 512;
    const WtOut o(out + base, 2 * (kHidden / 16) * 1024);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
        const half4_t g0 = {(half_t)(a[8 * kk] * inv), (half_t)(a[8 * kk + 1] * inv),
                            (half_t)(a[8 * kk + 2] * inv), (half_t)(a[8 * kk + 3] * inv)};
        const half4_t g1 = {(half_t)(a[8 * kk + 4] * inv), (half_t)(a[8 * kk + 5] * inv),
                            (half_t)(a[8 * kk + 6] * inv), (half_t)(a[8 * kk + 7] * inv)};
        const half8_t piece = frag_swap(g0, g1);
        const int c = head * kHeadDim + ct * 32 + kk * 16 + hi * 8;
        o.store((uint32_t)(frag_piece(row, c, kHidden) - base) * 2, piece);
    }
}

__device__ __forceinline__ void store_query(const QueryState& st, half_t* out, int row0, int row, int head, int hi) {
    const float inv = 1.0f / st.l_run;
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) store_half(st.o[ct], inv, out, row0, row, head, ct, hi);
}

// NKB > 0: the number of key blocks of KB = 32 keys, known at compile time
// (the block loop is then unrolled, which keeps the compiler's wait counts
// exact; used for 201 tokens, whose 24 KB of LDS also leave room for other
// image groups' kernels). NKB = 0: any count of KB = 64-key blocks.
template <int NKB>
struct KeyBlock {
    static constexpr int KB = NKB > 0 ? 32 : 64;   // keys per LDS block
    static constexpr int BLK = KB * kHeadDim;      // halfs per K (or V) block
    static constexpr int LOADS = KB / 32;          // DMA loads of 8 rows per matrix and wave
};

// DMA offsets for moving 8 key rows (one 1 KB load) out of a
// fragment-order [tpad][64] matrix: lane i lands at LDS slot (row i/8, chunk
// slot i%8) of rows r0 .. r0+7 and fetches the chunk c the swizzle puts
// there (r0 % 8 == 0, so row % 16 = r0 % 16 + i/8). Chunk c (channels 8c ..
// 8c+7) of row r sits at byte ((r/32)*4 + c/2)*1024 + ((c%2)*32 + r%32)*16:
// the lane part holds c and i/8, the scalar part (dma_row_offset) r0's
// 32-row block and r0 % 32 (no carry: r0 % 32 + 7 < 32). A load reads 8
// runs of 128 bytes (8 rows of one chunk each).
__device__ __forceinline__ int dma_lane_offset(int lane, int r0) {
    const int c = (lane & 7) ^ swz_slot(r0 % 16 + (lane >> 3));
    return ((c >> 1) << 10) + ((c & 1) << 9) + (lane >> 3) * 16;
}
__device__ __forceinline__ int dma_row_offset(int r0) { return (r0 >> 5) * 4096 + (r0 & 31) * 16; }

// Buffer descriptors of one (image, head)'s q, k and v matrices.
struct HeadSrc {
    __amdgpu_buffer_rsrc_t q, k, v;
    __device__ __forceinline__ HeadSrc(const AttentionArgs& p, int img, int head) {
        const size_t mat = ((size_t)img * kHeads + head) * p.tpad * kHeadDim;
        const int bytes = p.tpad * kHeadDim * 2;
        q = __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t*>(p.q + mat), 0, bytes, kBufferRsrcWord3);
        k = __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t*>(p.k + mat), 0, bytes, kBufferRsrcWord3);
        v = __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t*>(p.v + mat), 0, bytes, kBufferRsrcWord3);
    }
};

template <int NKB>
__global__ __launch_bounds__(kThreads, 3) void attention_kernel(DHX_ATTENTION_PARAMS) {
    const AttentionArgs p{q_, k_, v_, out_, images_, tokens_, tpad_};
    using KBT = KeyBlock<NKB>;
    __shared__ __attribute__((aligned(16))) half_t sK0[KBT::BLK], sK1[KBT::BLK], sK2[KBT::BLK];
    __shared__ __attribute__((aligned(16))) half_t sV0[KBT::BLK], sV1[KBT::BLK], sV2[KBT::BLK];
    // 1-D grid, XCD-aware: the tile space (query block fastest, then head,
    // then image) is cut into 8 contiguous chunks, one per XCD, so the query
    // blocks of one (image, head) share K and V in that XCD's L2.
    const int nqb = (p.tokens + QB - 1) / QB, total = nqb * kHeads * p.images;
    const int per = (total + 7) >> 3, g = blockIdx.x, t = (g & 7) * per + (g >> 3);
    if ((g >> 3) >= per || t >= total) return;  // uniform per workgroup
    const int qb = t % nqb, head = (t / nqb) % kHeads, img = t / (nqb * kHeads);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, hi = lane >> 5;
    const int T = p.tokens;
    const size_t bh = (size_t)img * kHeads + head;
    const half_t* qg = p.q + bh * p.tpad * kHeadDim;
    const int nkb = NKB > 0 ? NKB : (T + KBT::KB - 1) / KBT::KB;  // nkb * KB <= tpad, so every block row exists

    // Block kb of K and V: each wave moves KB/4 key rows of each, as 1 KB
    // DMA loads of 8 rows.
    const uint32_t bytes = (uint32_t)p.tpad * kHeadDim * 2;
    const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<half_t*>(p.k + bh * p.tpad * kHeadDim), 0, bytes, kBufferRsrcWord3);
    const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<half_t*>(p.v + bh * p.tpad * kHeadDim), 0, bytes, kBufferRsrcWord3);
    // Wave w moves key rows (KB/4) w .. +KB/4-1 as KB/32 loads of 8 rows per
    // matrix; load j covers rows (KB/4) w + 8j.
    // Sized 2, not KBT::LOADS: with a local array whose size depends on the
    // template parameter this compiler silently drops the host launch stub.
    int voff[2];
#pragma unroll
    for (int j = 0; j < KBT::LOADS; ++j) voff[j] = dma_lane_offset(lane, (tid >> 6) * (KBT::KB / 4) + 8 * j);
    auto dma = [&](half_t* k_buf, half_t* v_buf, int kb) {
#pragma unroll
        for (int j = 0; j < KBT::LOADS; ++j) {
            const int row = wave * (KBT::KB / 4) + j * 8, soff = dma_row_offset(kb * KBT::KB + row);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (__attribute__((address_space(3))) void*)(k_buf + row * kHeadDim),
                                                     16, voff[j], soff, 0, 0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (__attribute__((address_space(3))) void*)(v_buf + row * kHeadDim),
                                                     16, voff[j], soff, 0, 0);
        }
    };
    constexpr int kDmaPerBlock = 2 * KBT::LOADS;  // per wave

    // Block 0 first, then the Q fragments (registers), then block 1: the
    // wait for block 0 counts only the DMA loads of block 1 (DMA loads land
    // in issue order among themselves, but not in order with register loads).
    dma(sK0, sV0, 0);
    // Queries past T load row T-1 (unconditional loads keep the wait counts
    // exact); their results are never stored.
    const int qrow = qb * QB + wave * 32 + l32;
    QueryState st;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
        st.qf[kk] = *(const half8_t*)(qg + frag_piece(min(qrow, T - 1), kk * 16 + hi * 8, kHeadDim));
    asm volatile("" ::: "memory");
    if (NKB == 0 || nkb > 1) {  // with a runtime count, block 1 repeats block 0 when there is one block
        dma(sK1, sV1, min(1, nkb - 1));
        vm_barrier<kDmaPerBlock>();
    } else {
        vm_barrier<0>();
    }

    LaneOffsets at(lane);
    // Scores are s = (q / 8) . k: Q is scaled by 1/8 once (a power of two,
    // exact for normal f16 values), and the softmax weight of a score is
    // 2^(s*log2e - m*log2e), one FMA and one v_exp_f32.
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) st.qf[kk] *= (half_t)0.125f;
    st.o[0] = st.o[1] = float16_t{};
    // Waves whose 32 queries all lie past T only help move K and V.
    const bool active = qb * QB + wave * 32 < T;

    auto block = [&](const half_t* sK, const half_t* sV, int kb) {
#pragma unroll
        for (int sub = 0; sub < KBT::KB / 32 && active; ++sub) {
            const int key0 = kb * KBT::KB + sub * 32;
            if (key0 >= T) break;  // uniform across the workgroup
            if (NKB > 0 && kb == 0 && sub == 0)  // the unrolled walk: its first block is known at compile time
                attend32<true>(st, sK, sV, 0, key0, T, lane, at);
            else
                attend32(st, sK, sV, sub * 32, key0, T, lane, at);
        }
    };
    // Block kb is computed from buffer kb % 3 while the DMA of block kb+2
    // fills the buffer of block kb-1 (released by the previous barrier). The
    // barrier after block kb waits until only block kb+2's DMA may be in
    // flight, so block kb+1 has landed for every wave.
    auto step = [&](const half_t* k_cur, const half_t* v_cur, half_t* k_fill, half_t* v_fill, int kb) {
        const bool more = kb + 2 < nkb;  // uniform
        if (more) dma(k_fill, v_fill, kb + 2);
        block(k_cur, v_cur, kb);
        if (more)
            vm_barrier<kDmaPerBlock>();
        else if (kb + 1 < nkb)
            vm_barrier<0>();
    };
    if constexpr (NKB > 0) {
        half_t* const kbuf[3] = {sK0, sK1, sK2};
        half_t* const vbuf[3] = {sV0, sV1, sV2};
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) step(kbuf[kb % 3], vbuf[kb % 3], kbuf[(kb + 2) % 3], vbuf[(kb + 2) % 3], kb);
    } else {
        // Runtime block count: every step issues its DMA (past the last block
        // it repeats the last one into the buffer just released) and waits
        // the same way, so no branch makes the compiler's counts conservative;
        // the repeats are drained before the workgroup ends.
        auto step_rt = [&](const half_t* k_cur, const half_t* v_cur, half_t* k_fill, half_t* v_fill, int kb) {
            dma(k_fill, v_fill, min(kb + 2, nkb - 1));
            block(k_cur, v_cur, kb);
            vm_barrier<kDmaPerBlock>();
        };
        for (int kb = 0; kb < nkb; kb += 3) {
            step_rt(sK0, sV0, sK2, sV2, kb);
            if (kb + 1 >= nkb) break;
            step_rt(sK1, sV1, sK0, sV0, kb + 1);
            if (kb + 2 >= nkb) break;
            step_rt(sK2, sV2, sK1, sV1, kb + 2);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }

    if (qrow < T) store_query(st, p.out, img * T + qb * QB + wave * 32, img * T + qrow, head, hi);
}

// Short sequences in small launches: a workgroup holds 32 queries, and wave j
// of its N = ceil(T / 32) takes key block j. In attention_kernel a wave walks
// the blocks one after another, and a small launch waits for that chain of N
// softmax steps (about 0.4 us each) on a few SIMDs. Here the blocks' scores,
// weights and weight sums are taken side by side, against the first block's
// max: where no later block's weights against it sum past e^8, that is the
// running max attention_kernel keeps too. Then two waves, one per 32
// channels, run the PV products over the blocks in order, and the sums are
// added in order, so a query's result is bitwise that of attention_kernel.
// Where some block's weights do sum past e^8, the first wave walks the blocks
// as attention_kernel would. All loads are DMA, with exact waits. Alone: 201
// tokens 5.1 -> 4.2 us to 6 images, 69 tokens 4.25 -> 3.0, 261 tokens 6.5 ->
// 5.2, 405 tokens 8.0 -> 6.4; what is left is the launch, the loads, one
// softmax step and the 2 N MFMAs of a PV chain.
constexpr int kMaxParallel = 14;  // 446 tokens; the next square grid's 489 take 16 blocks

template <int N>
struct ParallelLds {
    static constexpr int KV = N * 32 * kHeadDim;  // halfs of K (or V)
    static constexpr int P = N * 2 * 512;         // halfs of P^T fragments
    static constexpr int SUMS = N * 32;
};

template <int N>
__device__ __forceinline__ void parallel_blocks(const AttentionArgs& p, half_t* sk, half_t* sv, half_t* sq, half_t* sp,
                                                float* smax, float* sums, int* grew, int qb, int head, int img) {
    constexpr int BLK = 32 * kHeadDim;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, hi = lane >> 5, T = p.tokens, q0 = qb * 32;
    const HeadSrc src(p, img, head);
    auto lds = [](half_t* a) { return (__attribute__((address_space(3))) void*)a; };
    // Q fragment kk by wave kk % N (rows past T are tpad's padding: finite, and
    // never stored), then the wave's own K block and V block.
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
        if (kk % N == wave)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(src.q, lds(sq + kk * 512), 16, lane * 16, (qb * 4 + kk) * 1024, 0, 0);
    half_t* const k_own = sk + wave * BLK;
    half_t* const v_own = sv + wave * BLK;
    const int even = dma_lane_offset(lane, 0), odd = dma_lane_offset(lane, 8);
#pragma unroll
    for (int i = 0; i < 4; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(src.k, lds(k_own + 8 * i * kHeadDim), 16, i & 1 ? odd : even,
                                                 dma_row_offset(wave * 32 + 8 * i), 0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(src.v, lds(v_own + 8 * i * kHeadDim), 16, i & 1 ? odd : even,
                                                 dma_row_offset(wave * 32 + 8 * i), 0, 0);
    if (tid == 0) *grew = 0;
    LaneOffsets at(lane);
    QueryState st;
    vm_barrier<4>();  // Q and K have landed; V may be outstanding
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) st.qf[kk] = *(const half8_t*)(sq + kk * 512 + lane * 8) * (half_t)0.125f;
    float16_t s = scores32(k_own, st.qf, at);
    mask32(s, wave * 32, T, hi);
    if (wave == 0) smax[l32] = fmaxf(block_max32(s), st.m_run);  // both lanes of a pair hold the pair's
    vm_barrier<0>();
    float w[16];
    const float sum = weights32(s, smax[l32], w);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) *(half8_t*)(sp + (wave * 2 + ks) * 512 + lane * 8) = p_frag(w, ks);
    sums[wave * 32 + l32] = sum;
    if (wave > 0 && __any(!(sum <= kLazySum))) *grew = 1;
    vm_barrier<0>();
    const int row0 = img * T + q0, row = row0 + l32;
    if (*grew) {  // uniform across the workgroup
        if (wave > 0) return;
        st.o[0] = st.o[1] = float16_t{};
        attend32<true>(st, sk, sv, 0, 0, T, lane, at);
        for (int kb = 1; kb < N; ++kb) attend32(st, sk + kb * BLK, sv + kb * BLK, 0, kb * 32, T, lane, at);
        if (q0 + l32 < T) store_query(st, p.out, row0, row, head, hi);
        return;
    }
    float l = sums[l32];
#pragma unroll
    for (int kb = 1; kb < N; ++kb) l += sums[kb * 32 + l32];
    const float inv = 1.0f / l;
    if (wave > 1) return;
#pragma unroll
    for (int c = 0; c < (N == 1 ? 2 : 1); ++c) {
        const int ct = N == 1 ? c : wave;
        // Channel half 1 sits 4 chunks from half 0 (LaneOffsets, one exclusive or).
        const half_t* const v0 = sv + (at.v(0, 0) ^ (ct << 5));
        const half_t* const v1 = sv + (at.v(0, 1) ^ (ct << 5));
        float16_t o = {};
#pragma unroll
        for (int b = 0; b < 2 * N; ++b) {  // 16-key slices: block b / 2
            const half4_t a0 = lds_read_tr16(v0 + b * 16 * kHeadDim), a1 = lds_read_tr16(v1 + b * 16 * kHeadDim);
            o = mfma32x32x16(__builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7),
                             *(const half8_t*)(sp + b * 512 + lane * 8), o);
        }
        if (q0 + l32 < T) store_half(o, inv, p.out, row0, row, head, ct, hi);
    }
}

// As many waves per SIMD as two workgroups per CU have (one from eight blocks
// on, by its LDS).
template <int N>
__global__ __launch_bounds__(N * kWave, N > 7 ? (N + 3) / 4 : N > 3 ? (N + 1) / 2 : 2) void attention_parallel_kernel(
    DHX_ATTENTION_PARAMS) {
    const AttentionArgs p{q_, k_, v_, out_, images_, tokens_, tpad_};
    using L = ParallelLds<N>;
    __shared__ __attribute__((aligned(16))) half_t sk[L::KV], sv[L::KV], sq[4 * 512], sp[L::P];
    __shared__ float smax[32], sums[L::SUMS];
    __shared__ int grew;
    const int nqb = (p.tokens + 31) / 32, total = nqb * kHeads * p.images;
    const int per = (total + 7) >> 3, g = blockIdx.x, t = (g & 7) * per + (g >> 3);
    if ((g >> 3) >= per || t >= total) return;  // uniform per workgroup
    parallel_blocks<N>(p, sk, sv, sq, sp, smax, sums, &grew, t % nqb, (t / nqb) % kHeads, t / (nqb * kHeads));
}

// Long sequences: workgroups of 2 QW waves hold 32 QW queries as QW query
// waves x 2 key halves. Half h walks key blocks h*nh .. h*nh+nh-1 (32 keys
// each, nh = ceil(blocks / 2)) through its own three K and three V buffers;
// both halves meet at the same barriers. At the end the second half's
// (running max, denominator, O^T) go through LDS to the first half, which
// merges them (rescaling both to the larger max) and writes the output. What
// bounds it is the wave's own chain of score MFMAs, about 85 vector
// instructions (16 of them exponentials) and PV MFMAs, some 700 - 850 cycles
// per 32 keys, MFMA and vector issue hardly overlapping: two waves per SIMD
// take the time of one twice, so a launch is as fast as its keys per SIMD are
// few. Halves and 64-query workgroups spread them (512x512 batch 1: 54
// workgroups of 8 waves -> 102 of 4, 13.1 -> 10.6 us); deeper rings did not
// help (four to eight buffers per half: 13.1 -> 13.3 - 14.3 us).
constexpr int kSplitBlk = 32 * kHeadDim;  // halfs per 32-key K (or V) block

// One key half's walk from block `first` on (past the sequence's last block
// the DMA repeats that block and the compute is skipped). The buffers are
// separate LDS variables chosen at compile time (the caller branches on the
// half), so the compiler can tell the buffer being read from the ones being
// filled and adds no waits of its own for the DMA in flight. The Q fragments
// come through LDS too (sq, 4 KB, one of the third buffers): with DMA loads
// only, every wait is an exact count. NH > 0: nh = NH, unrolled.
template <int NH, int QW>
__device__ __forceinline__ void split_walk(QueryState& st, half_t* const (&kbuf)[3], half_t* const (&vbuf)[3],
                                           const HeadSrc& src, half_t* sq, int first, int nh_rt, int nkb, int q0, int T,
                                           int hwave, int lane) {
    constexpr int LOADS = 4 / QW;  // 8-row DMA loads per matrix, wave and block
    const int nh = NH > 0 ? NH : nh_rt, last = min(first + nh, nkb) - 1;
    int voff[4];  // sized 4, not LOADS (see attention_kernel)
#pragma unroll
    for (int i = 0; i < LOADS; ++i) voff[i] = dma_lane_offset(lane, 8 * (hwave * LOADS + i));
    auto lds = [](half_t* a) { return (__attribute__((address_space(3))) void*)a; };
    auto dma = [&](int buf, int s) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int row = 8 * (hwave * LOADS + i), soff = dma_row_offset(min(first + s, last) * 32 + row);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(src.k, lds(kbuf[buf] + row * kHeadDim), 16, voff[i], soff, 0, 0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(src.v, lds(vbuf[buf] + row * kHeadDim), 16, voff[i], soff, 0, 0);
        }
    };
    constexpr int kPerBlock = 2 * LOADS;
    // Query rows past T are tpad's padding: finite, and never stored. Each
    // wave takes its fragments before the barrier after which sq is filled
    // with a block.
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(src.q, lds(sq + kk * 512), 16, lane * 16, (q0 / 32 * 4 + kk) * 1024, 0, 0);
    dma(0, 0);
    dma(1, 1);
    st.o[0] = st.o[1] = float16_t{};
    std::conditional_t<NH == 0 && QW == 4, LaneOffsetsXor, LaneOffsets> at(lane);
    const bool active = q0 < T;  // waves whose queries all lie past T only move K and V
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * kPerBlock) : "memory");
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) st.qf[kk] = *(const half8_t*)(sq + kk * 512 + lane * 8) * (half_t)0.125f;
    vm_barrier<kPerBlock>();
    // Step s: block first+s from buffer s % 3 while block s+2's DMA fills
    // the buffer that the previous barrier released; the barrier leaves only
    // that DMA in flight, so block s+1 has landed for every wave.
    auto attend = [&](int b, int s, bool first_block) {
        const int kb = first + s;
        if (!active || kb >= nkb) return;
        if (first_block)
            attend32<true>(st, kbuf[b], vbuf[b], 0, kb * 32, T, lane, at);
        else
            attend32(st, kbuf[b], vbuf[b], 0, kb * 32, T, lane, at);
    };
    if constexpr (NH > 0) {
#pragma unroll
        for (int s = 0; s < NH; ++s) {
            if (s + 2 < NH) dma((s + 2) % 3, s + 2);
            attend(s % 3, s, s == 0);
            if (s + 2 < NH)
                vm_barrier<kPerBlock>();
            else
                vm_barrier<0>();
        }
    } else {
        // As in attention_kernel: every step issues its DMA (past the last
        // block it repeats it) and waits the same way; the repeats are drained
        // at the end.
        auto step = [&](int b, int s) {
            dma((b + 2) % 3, s + 2);
            attend(b, s, false);
            vm_barrier<kPerBlock>();
        };
        for (int s = 0; s < nh; s += 3) {
            step(0, s);
            if (s + 1 >= nh) break;
            step(1, s + 1);
            if (s + 2 >= nh) break;
            step(2, s + 2);
        }
        vm_barrier<0>();
    }
}

// QW = 4: two workgroups per CU, four waves per SIMD, which caps the kernel
// at 128 VGPRs; one register more halves the resident workgroups.
template <int NH, int QW>
__global__ __launch_bounds__(2 * QW * kWave, QW == 4 ? 4 : 2) void attention_split_kernel(DHX_ATTENTION_PARAMS) {
    const AttentionArgs p{q_, k_, v_, out_, images_, tokens_, tpad_};
    // Per half three K and three V blocks of 4 KB (48 KB), as separate
    // variables (the compiler tells distinct variables apart, not the rows of
    // one array); reused at the end for the merge.
    __shared__ __attribute__((aligned(16))) half_t k00[kSplitBlk], k01[kSplitBlk], k02[kSplitBlk];
    __shared__ __attribute__((aligned(16))) half_t v00[kSplitBlk], v01[kSplitBlk], v02[kSplitBlk];
    __shared__ __attribute__((aligned(16))) half_t k10[kSplitBlk], k11[kSplitBlk], k12[kSplitBlk];
    __shared__ __attribute__((aligned(16))) half_t v10[kSplitBlk], v11[kSplitBlk], v12[kSplitBlk];
    constexpr int Q = 32 * QW;  // queries per workgroup
    const int nqb = (p.tokens + Q - 1) / Q, total = nqb * kHeads * p.images;
    const int per = (total + 7) >> 3, g = blockIdx.x, t = (g & 7) * per + (g >> 3);
    if ((g >> 3) >= per || t >= total) return;  // uniform per workgroup
    const int qb = t % nqb, head = (t / nqb) % kHeads, img = t / (nqb * kHeads);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int qw = wave % QW, half = wave / QW;  // query wave; key half (uniform per wave)
    const int l32 = lane & 31, hi = lane >> 5;
    const int T = p.tokens, nkb = (T + 31) / 32;  // nkb <= 2 * nh and nkb * 32 <= tpad
    const int nh = NH > 0 ? NH : (nkb + 1) / 2;
    const HeadSrc src(p, img, head);
    const int q0 = qb * Q + qw * 32, qrow = q0 + l32;
    // Query wave qw's Q fragments (both halves' waves load the same).
    half_t* const sq = qw == 0 ? k02 : qw == 1 ? v02 : qw == 2 ? k12 : v12;
    QueryState st;
    if (half == 0) {
        half_t* const kb[3] = {k00, k01, k02};
        half_t* const vb[3] = {v00, v01, v02};
        split_walk<NH, QW>(st, kb, vb, src, sq, 0, nh, nkb, q0, T, qw, lane);
    } else {
        half_t* const kb[3] = {k10, k11, k12};
        half_t* const vb[3] = {v10, v11, v12};
        split_walk<NH, QW>(st, kb, vb, src, sq, nh, nh, nkb, q0, T, qw, lane);
    }
    // Merge: the second half hands its 34 values per lane (max, denominator,
    // O^T) to the first through LDS; both are rescaled to the larger max.
    // Every wave passed the walk's last barrier, which waited for all of its
    // DMA loads, so the buffers are free. Value f of query wave qw sits in
    // buffer f / 4 at [(f % 4) * QW + qw][lane] (f is a constant, so each
    // access names its buffer).
    half_t* const bufs[12] = {k00, k01, k02, v00, v01, v02, k10, k11, k12, v10, v11, v12};
    auto slot = [&](int f) -> float* {
        return reinterpret_cast<float*>(bufs[f / 4]) + ((f % 4) * QW + qw) * 64 + lane;
    };
    if (half == 1) {
        *slot(0) = st.m_run;
        *slot(1) = st.l_run;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            *slot(2 + r) = st.o[0][r];
            *slot(18 + r) = st.o[1][r];
        }
    }
    __syncthreads();
    if (half == 1 || qrow >= T) return;
    const float m1 = *slot(0), m = fmaxf(st.m_run, m1);
    const float a0 = fast_exp2((st.m_run - m) * kLog2e), a1 = fast_exp2((m1 - m) * kLog2e);
    st.l_run = fmaf(st.l_run, a0, *slot(1) * a1);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        st.o[0][r] = fmaf(st.o[0][r], a0, *slot(2 + r) * a1);
        st.o[1][r] = fmaf(st.o[1][r], a0, *slot(18 + r) * a1);
    }
    store_query(st, p.out, img * T + q0, img * T + qrow, head, hi);
}

// The longest sequences attention_kernel takes: from here on the keys are
// walked in two halves (attention_split_kernel). The walk is part of a result's
// arithmetic, so it depends on the sequence only, not on the launch.
constexpr int kSplitBlocks = 16;  // blocks of 32 keys, from 481 tokens on
constexpr int kRound = 256;       // workgroups of one per CU

template <int N>
hipError_t launch_parallel(const AttentionArgs& a, int nkb, int groups, hipStream_t s) {
    if constexpr (N > 1)
        if (nkb < N) return launch_parallel<N - 1>(a, nkb, groups, s);
    return start(attention_parallel_kernel<N>, dim3((groups + 7) & ~7), dim3(N * kWave), 0, s, a);
}

template <int NH, int QW>
hipError_t launch_split(const AttentionArgs& a, int groups, hipStream_t s) {
    return start(attention_split_kernel<NH, QW>, dim3((groups + 7) & ~7), dim3(2 * QW * kWave), 0, s, a);
}

}  // namespace

// To 446 tokens, where one round of 32-query workgroups covers the launch, one
// wave per key block (whole forward, against the walks below: 224x224 batch 1
// 304 -> 294 us, batch 6 332 -> 322, 128x128 batch 4 302 -> 286, 256x256 batch
// 4 351 -> 334, 320x320 batch 3 368 -> 349; in two rounds 224x224 batch 8 351
// -> 361). From 481 tokens on two key halves, on workgroups of 64 queries
// where one round of them covers the launch, which then runs on twice the CUs
// with one wave per SIMD (128 -> 64 queries: 384x384 batch 3 439 -> 421 us,
// 512x512 batch 1 455 -> 424, 720x720 batch 1 620 -> 569; attention_kernel with
// its run-time count before: 443, -, 666), else of 128 (1024x1024 batch 2 1852
// -> 1800; equal to attention_kernel from 581 tokens on, 5 % slower at 405).
// 512x512 (17 blocks per half) in more than one round takes the unrolled walk
// (batch 8 975 -> 964 us); in one round its 80 KB of code cost more to fetch
// than they save (batch 1 449 against 424, batch 4 636 against 629). Beside
// another image group's kernels (a.shared) there are CUs to share and code to
// fetch once for both: batch 8 in two groups 1005 -> 985 us unrolled, and 64
// queries are the better workgroup to 192 of them only (two groups, 64 | 128:
// 2 x 192 workgroups, 352x352 batch 8, 580 | 611 us; 216 and 270, 368x368
// batch 9, 675 | 664; 2 x 240, 352x352 batch 10, 684 | 659, 400x400 batch 8,
// 720 | 684). 201 tokens: seven blocks of 32 keys, unrolled. Otherwise blocks
// of 64 keys with a run-time count.
hipError_t launch_attention(const AttentionArgs& a, hipStream_t s) {
    const int nqb = (a.tokens + QB - 1) / QB, total = nqb * kHeads * a.images;
    const int total64 = (a.tokens + 63) / 64 * kHeads * a.images;
    const dim3 grid((total + 7) & ~7), block(kThreads);
    const int nkb = (a.tokens + 31) / 32;
    const int total32 = nkb * kHeads * a.images;
    if (nkb <= kMaxParallel && total32 <= kRound) return launch_parallel<kMaxParallel>(a, nkb, total32, s);
    if (nkb >= kSplitBlocks) {
        if ((nkb + 1) / 2 == 17 && (a.shared || total > kRound)) return launch_split<17, 4>(a, total, s);
        if (total64 <= (a.shared ? kRound * 3 / 4 : kRound)) return launch_split<0, 2>(a, total64, s);
        return launch_split<0, 4>(a, total, s);
    }
    return nkb == 7 ? start(attention_kernel<7>, grid, block, 0, s, a) : start(attention_kernel<0>, grid, block, 0, s, a);
}

}  // namespace dhx
