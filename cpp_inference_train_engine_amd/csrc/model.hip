// Batched MLA decode step on gfx950: everything of CpuDecoder::decode around the
// attention (src/infer/inference.cpp:76-173) for B sessions at once, one new token
// each.
//
// Per layer, in launch order (y = x.W for every projection, as in ops.cpp:8-18):
//   g1_kernel   RMSNorm(x, attn_norm) . [w_dq | w_dkv]  (inference.cpp:85-95)
//   g2_kernel   per head, q_norm(cq) . w_uq, RoPE of the rope columns (q_rope) and the absorption
//               q_latent = W_uk_h^T q_nope (inference.cpp:85-90,121-124), both stored in the
//               cache dtype as the MPS graph does (mps_backend.mm:561); one more workgroup
//               kv_norms the latent, RoPEs the key, rounds both and appends them to the paged
//               cache (inference.cpp:91-103)
//   (decode attention partials + merge: decode.hip)
//   g4_kernel   latent_ctx [H*kv_rank] . out_proj + x  (inference.cpp:154-156; out_proj
//               is the combined W_uv.W_o of prepare_projections, inference.cpp:28-46)
//   g5_kernel   RMSNorm(ffn_norm) -> [w_gate | w_up] -> SwiGLU  (inference.cpp:157-161)
//   g6_kernel   . w_down + residual  (inference.cpp:162-165)
// Per step: embed_kernel (token rows, RoPE rows), g7_kernel or g7_rows_kernel (final RMSNorm,
// tied logits h.E^T, inference.cpp:166-168, with a greedy partial per 64 columns) and argmax_kernel
// (sample_token's greedy rule, inference.cpp:345-380).
//
// Every projection is a skinny GEMM on v_mfma_f32_16x16x32_f16 (fp16 operands, fp32
// accumulation).  A workgroup owns 16 rows (64 for the logits) and one to four 16-column
// output tiles; its 8 waves split K and the partial sums meet in LDS (g2_kernel, a head a workgroup,
// and g7_rows_kernel, 64 columns a wave, do not split K).  Each wave fetches its weight tiles (fp16,
// TILED: each wave load reads 1 KB contiguously) and its slice of the activation rows into
// registers at kernel start, so a GEMM pays about one memory round trip.  Small row blocks keep
// the bytes each CU must pull low: the load phase, not the arithmetic, is what these kernels wait
// on.
//
// RMSNorm (ops.cpp:33-45) is RMSNorm(x)_k = x_k * inv * w_k with inv = 1/rms(x) per row,
// so RMSNorm(x).W = inv * ((x o w).W): the kernel that writes an activation x also
// writes (x o w) in fp16 for the consumer's A operand (w = the norm weight of the next
// consumer) and, per row and 16-column tile, the sum of squares of x; the consumer adds
// those partials (in a fixed order) into inv and scales its output rows by it.
#include "mla_common.hpp"
#include "mla_internal.hpp"
#include "mla_model.hpp"

#include <cmath>

namespace mla {
namespace {

using V8 = half8;
constexpr int kWaves = 8;  // waves per GEMM workgroup

__device__ __forceinline__ floatx4 mma(V8 a, V8 b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// ---- L2 prefetch for the next kernel on the stream -------------------------------------
// Workgroups b of a launch (x-fastest linear id) with one residue b % 8 run on one XCD:
// the dispatcher deals workgroups to the 8 XCDs in turn, starting on an XCD that depends
// on the hardware queue (constant for the queue, so the same residue lands on the same
// XCD in consecutive kernels of one stream).  Each XCD has its own L2, which keeps its lines across
// kernel boundaries, while the attention's page stream evicts every layer's weights from
// it.  So the kernel that runs before a weight-latency-bound one touches, from each XCD,
// the 1 KB weight blocks that the next kernel's workgroups on that XCD will read; the next
// kernel's grid is padded to a multiple of 8 columns, so that each of its column tiles runs
// on one fixed XCD.  The loads go straight to a scratch block of LDS (global_load_lds: no
// VGPR is written behind the compiler's back), issued by the split-K waves that have handed
// their partial sums over and have nothing left to do: issued any earlier, the compiler's
// waits for the kernel's own operands would wait for them too (vmcnt retires in order),
// which measured slower than no prefetch.  A different placement only costs the prefetch
// its effect, never a result.
constexpr int kXcds = 8;

__device__ __forceinline__ int block_xcd() {
    return (int)((blockIdx.y * gridDim.x + blockIdx.x) % kXcds);
}

// Blocks [0, n) of this XCD's list (block k at addr(k)), spread over waves
// [first, blockDim/64) of all of this launch's workgroups on the XCD.
template <typename F>
__device__ __forceinline__ void l2_prefetch(int n, F&& addr, uint16_t* scratch, int first) {
    const int lin = blockIdx.y * gridDim.x + blockIdx.x, total = gridDim.x * gridDim.y;
    const int x = lin % kXcds, wgs = (total - x + kXcds - 1) / kXcds;
    const int nw = (blockDim.x >> 6) - first, lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) - first;
    for (int k = (lin / kXcds) * nw + wave; k < n; k += wgs * nw)
        copy_block_to_lds(addr(k), lane * 16, scratch);
}

// Sums over aligned groups of G = 4, 8 or 16 lanes of a 16-lane row, left in every lane
// of the group, on DPP lane moves (VALU) instead of LDS permutes: the two quad swaps give
// every lane its quad's sum, then the half-row mirror pairs the quads of each half and the
// row mirror the halves (each pairs lanes that hold equal partial sums, so every lane ends
// with the same bits).  Every lane of the row must be active.
template <int CTRL>
__device__ __forceinline__ float dpp_mov(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, false));
}
template <int G>
__device__ __forceinline__ float group_sum(float v) {
    static_assert(G == 4 || G == 8 || G == 16, "group of 4, 8 or 16 lanes");
    v += dpp_mov<0xB1>(v);  // quad_perm [1,0,3,2]
    v += dpp_mov<0x4E>(v);  // quad_perm [2,3,0,1]
    if constexpr (G >= 8)
        v += dpp_mov<0x141>(v);  // row_half_mirror
    if constexpr (G >= 16)
        v += dpp_mov<0x140>(v);  // row_mirror
    return v;
}
// Sum over the 16 lanes of an MFMA output row group (lanes with equal g hold the same
// rows, one column each).
__device__ __forceinline__ float sum16(float v) { return group_sum<16>(v); }

template <int MT, int NT>
__device__ __forceinline__ void zero(floatx4 (&acc)[MT][NT]) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int j = 0; j < NT; ++j)
            acc[mt][j] = floatx4{0, 0, 0, 0};
}

// ---- operand prefetch ----------------------------------------------------------
// A wave's k-steps are kt0, kt0 + ks, kt0 + 2ks, ... (KW of them; kt0 = the wave's
// K group and ks = the number of K groups, so uneven K spreads evenly).
//
// Every load of a step kernel's operands and side inputs is unconditional: k-steps past
// KT read the zero block as their weights (and add nothing), other out-of-range indices are
// clamped, and what a clamped load read is dropped where it would be used.  A load behind a
// condition becomes a branch, at whose join the compiler waits for loads in flight (the
// conditional form of qkv_kernel waited for nearly all of its weights, and only then issued the
// last two loads): every such wait is one more memory round trip of the kernel.  The wave
// index is made scalar (wave_index), so the weight addresses and the choices are scalar too.
__device__ __forceinline__ int wave_index() {
    return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
}

// operands_issued() keeps the compiler from moving loads below it, behind the MFMAs (it does,
// to save registers, and the loads it moved then start a round trip of their own).
__device__ __forceinline__ void operands_issued() { __builtin_amdgcn_sched_barrier(0); }

// Weight (B operand) registers of one wave: its k-steps of tiles [nt0, nt0+NT), of which
// ntv >= 1 exist (the others repeat the last one).  Tile (nt, kt) of a tiled W
// (mla_model.hpp) is 512 contiguous fp16 words; lane l reads 16 bytes at 8l.
__device__ __forceinline__ V8 load_w(const uint16_t* w, const uint16_t* zeros, int nt, int kt,
                                     int KT, int lane) {
    const uint16_t* p = kt < KT ? w + ((long long)nt * KT + kt) * 512 : zeros;
    return *reinterpret_cast<const V8*>(p + lane * 8);
}
template <int NT, int KW>
struct BPre {
    V8 b[KW][NT];
    __device__ __forceinline__ void load(const uint16_t* w, const uint16_t* zeros, int nt0,
                                         int ntv, int KT, int kt0, int ks, int lane) {
#pragma unroll
        for (int kk = 0; kk < KW; ++kk)
#pragma unroll
            for (int j = 0; j < NT; ++j)
                b[kk][j] = load_w(w, zeros, nt0 + min(j, ntv - 1), kt0 + kk * ks, KT, lane);
    }
};

// Activation (A operand) registers: lane (g, n) needs rows 16mt + n (mt < MT) and
// columns 32kt + 8g .. +7 of each of its k-steps of the activation rows from X on (a whole
// 16-row tile's first word; KT 32-column blocks a row).  Rows past `rows` (>= 1) repeat the last
// one: their products are dropped, and the lanes that share its address add no traffic.
template <int KW, int MT>
struct APre16 {
    V8 x[KW][MT];
    __device__ __forceinline__ void load(const uint16_t* X, int rows, int KT, int kt0, int ks,
                                         int lane) {
        const int g = lane >> 4, n = lane & 15;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int r = min(16 * mt + n, rows - 1);
            const uint16_t* p = X + act_word(r, 8 * g, KT);
#pragma unroll
            for (int kk = 0; kk < KW; ++kk)
                x[kk][mt] = *reinterpret_cast<const V8*>(p + min(kt0 + kk * ks, KT - 1) * 512);
        }
    }
};

template <int MT, int NT, int KW, typename AOp>
__device__ __forceinline__ void mma_steps(floatx4 (&acc)[MT][NT], const BPre<NT, KW>& b,
                                          AOp aop) {
#pragma unroll
    for (int kk = 0; kk < KW; ++kk)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const V8 a = aop(kk, mt);
#pragma unroll
            for (int j = 0; j < NT; ++j)
                acc[mt][j] = mma(a, b.b[kk][j], acc[mt][j]);
        }
}

// 1/rms of `rows` rows (ops.cpp:33-45: inv = 1/sqrt(mean(x^2) + eps)) from the
// producer's per-tile partial sums of squares (n_tiles <= 64): TPR threads a row each
// load every TPR-th tile, then combine in a fixed order.  Threads [0, TPR*rows) take
// part (whole waves).  issue() goes before the kernel's operand loads and finish()
// after its MFMAs, so the sums travel with the operands instead of delaying them by a
// round trip; inv_s is visible after the next barrier.
template <int TPR>
struct RmsPrefetch {
    static_assert(TPR >= 4 && TPR <= 16 && (TPR & (TPR - 1)) == 0, "threads per row");
    static constexpr int kPer = 64 / TPR;
    float v[kPer];
    __device__ __forceinline__ void issue(const float* ss, int n_tiles, int row0, int rows) {
        const int t = threadIdx.x;
        const float* p = ss + (long long)(row0 + min(t / TPR, rows - 1)) * n_tiles;
#pragma unroll
        for (int i = 0; i < kPer; ++i)
            v[i] = p[min(t % TPR + TPR * i, n_tiles - 1)];
    }
    __device__ __forceinline__ void finish(int n_tiles, int K, float eps, float* inv_s, int rows) {
        const int t = threadIdx.x;
        float sum = 0.0f;
#pragma unroll
        for (int i = 0; i < kPer; ++i)
            sum += t % TPR + TPR * i < n_tiles ? v[i] : 0.0f;
        sum = group_sum<TPR>(sum);
        if (t < TPR * rows && t % TPR == 0)
            inv_s[t / TPR] = 1.0f / sqrtf(sum / (float)K + eps);
    }
};

// Split-K reduction through LDS `part` (kWaves*MT*NTW*64 floatx4).  Wave w computed K
// group w % KG of tiles [(w / KG) * NTW, +NTW); after the barrier wave mt < MT sums all
// K groups of M-tile mt into v[t] for the workgroup's NT = NTW * kWaves / KG tiles
// (lane (g, n): C[16mt + 4g + i][16t + n]); other waves get false.
template <int MT, int NTW, int KG>
__device__ __forceinline__ bool splitk_reduce(floatx4 (&acc)[MT][NTW], floatx4* part, int& mt,
                                              floatx4 (&v)[NTW * (kWaves / KG)]) {
    const int wave = wave_index(), lane = threadIdx.x & 63;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int j = 0; j < NTW; ++j)
            part[((wave * MT + m) * NTW + j) * 64 + lane] = acc[m][j];
    __syncthreads();
    if (wave >= MT)
        return false;
    mt = wave;
#pragma unroll
    for (int ng = 0; ng < kWaves / KG; ++ng)
#pragma unroll
        for (int j = 0; j < NTW; ++j) {
            floatx4 sum = {0, 0, 0, 0};
#pragma unroll
            for (int kg = 0; kg < KG; ++kg)
                sum += part[(((ng * KG + kg) * MT + mt) * NTW + j) * 64 + lane];
            v[ng * NTW + j] = sum;
        }
    return true;
}

// Per-row sum of squares of this lane group's 16 columns (y holds rows 4g+i of one
// column; columns that do not count add 0), written by lane n == 0 to
// ss[row * n_tiles + tile] for rows < B.
__device__ __forceinline__ void write_ss(floatx4 y, bool col_counts, float* ss, int n_tiles,
                                         int tile, int row0, int B) {
    const int lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float q = sum16(col_counts ? y[i] * y[i] : 0.0f);
        const int row = row0 + 4 * g + i;
        if (n == 0 && row < B)
            ss[(long long)row * n_tiles + tile] = q;
    }
}

__device__ __forceinline__ float2 rope_table(const StepArgs& s, int pos, int j2) {
    const ModelDims& m = s.dims;
    pos = min(max(pos, 0), m.max_seq - 1);  // the caller rejects others (inference.cpp:71-75)
    return s.rope_tab[(long long)pos * (m.rope / 2) + j2];
}

// ------------------------------------------------------------------ embed ----
// x[b] = E[token[b]] (fp32), xw[b] = x o attn_norm of layer 0 (fp16), the per-tile sums
// of squares of x, and the (cos, sin) row of b's position for every layer's RoPE; rows
// [B, m_pad) are zeroed.  E is read from its tiled logits layout (K = d_model, N = vocab).
__global__ __launch_bounds__(256) void embed_kernel(StepArgs s, const float* norm0) {
    const int b = blockIdx.x;
    const ModelDims& m = s.dims;
    const int d_tiles = m.d_pad / 16, KT = m.d_pad / 32, half = m.rope / 2;
    int tok = b < s.B ? s.tokens[b] : 0;
    tok = tok < 0 || tok >= m.vocab ? 0 : tok;  // the caller validates tokens
    if ((int)threadIdx.x < half)
        s.rope_rows[(long long)b * half + threadIdx.x] =
            b < s.B ? rope_table(s, s.positions[b], threadIdx.x) : float2{1.0f, 0.0f};
    for (int c0 = 0; c0 < m.d_pad; c0 += 256) {
        const int c = c0 + threadIdx.x;
        float v = 0.0f, w = 0.0f;
        if (b < s.B && c < m.d_model) {
            const long long e = ((long long)(tok >> 4) * KT + (c >> 5)) * 512 +
                                (((c & 31) >> 3) * 16 + (tok & 15)) * 8 + (c & 7);
            v = (float)__builtin_bit_cast(_Float16, s.embed[e]);
            w = norm0[c];
        }
        if (c < m.d_pad) {
            s.x[(long long)b * m.d_pad + c] = v;
            s.xw[act_word(b, c, KT)] = F16::from_float(v * w);
        }
        const float q = sum16(v * v);
        if ((threadIdx.x & 15) == 0 && c < m.d_pad)
            s.ss_x[(long long)b * d_tiles + c / 16] = q;
    }
}

// --------------------------------------------------------------- g1 and g2 ----
// Between the residual stream x and the attention (inference.cpp:85-103).  g1: per 16 rows and
// 16-column tile, y = RMSNorm(x, attn_norm) . [w_dq | w_dkv], 8 waves splitting K.  The norms
// that follow are RMSNorm(v)_c = v_c * inv * w_c with one inv per row, so g1 leaves v o w (cq:
// fp16, g2's A operand; latent: fp32) with the rows' sums of squares per tile, and g2 applies inv
// to its products.  g2: workgroup h computes head h's queries for 16 rows (q_head), W_uq and W_uk
// as two products: their product as one fp16 weight falls into fp16's subnormals for small
// weights (std 0.001: error of q_latent 3.2e-4 -> 2.5e-3) and past its range for large ones.
// Smaller batches run both in one launch (qkv_kernel, below), with the same results bit for bit
// (the same K groups, summed in the same order).
// Block k < head_blocks of head h's w_uq and w_uk tiles (each contiguous per head).
__device__ __forceinline__ int uq_blocks(const ModelDims& m) {
    return (m.qk_pad / 16) * (m.q_pad / 32);
}
__device__ __forceinline__ int uk_blocks(const ModelDims& m) {
    return (m.kv_pad / 16) * (m.nope_pad / 32);
}
__device__ __forceinline__ int head_blocks(const ModelDims& m) { return uq_blocks(m) + uk_blocks(m); }
__device__ __forceinline__ const uint16_t* head_block(const ModelDims& m, const uint16_t* w_uq,
                                                      const uint16_t* w_uk, int h, int k) {
    const int nq = uq_blocks(m), nk = uk_blocks(m);
    return k < nq ? w_uq + ((long long)h * nq + k) * 512
                  : w_uk + ((long long)h * nk + k - nq) * 512;
}

template <int KW>
__global__ __launch_bounds__(64 * kWaves) void g1_kernel(StepArgs s, LayerWeights L) {
    __shared__ __attribute__((aligned(16))) floatx4 part[kWaves * 64];
    __shared__ __attribute__((aligned(16))) uint16_t scratch[512];
    __shared__ float inv_s[16];
    const ModelDims& m = s.dims;
    const int wave = wave_index(), lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15;
    const int q_tiles = m.q_pad / 16, tiles = q_tiles + m.kvw_pad / 16, nt = blockIdx.x;
    const int row0 = blockIdx.y * 16, KT = m.d_pad / 32;
    if (nt >= tiles)
        return;  // columns are padded to a multiple of 8 (see l2_prefetch)
    RmsPrefetch<16> rms;
    rms.issue(s.ss_x, m.d_pad / 16, row0, 16);
    BPre<1, KW> bw;
    bw.load(L.w_dq_dkv, s.zeros, nt, 1, KT, wave, kWaves, lane);
    APre16<KW, 1> a;
    a.load(s.xw + (long long)row0 * m.d_pad, s.B - row0, KT, wave, kWaves, lane);
    // column c of cq (c < q_rank counts in its norm) or of [latent | key] (c < kv_rank)
    const bool kv = nt >= q_tiles;
    const int c = 16 * (kv ? nt - q_tiles : nt) + n, norm_cols = kv ? m.kv_rank : m.q_rank;
    const float wn = (kv ? L.kv_norm : L.q_norm)[min(c, norm_cols - 1)];
    operands_issued();
    floatx4 acc[1][1];
    zero(acc);
    mma_steps(acc, bw, [&](int kk, int mt) { return a.x[kk][mt]; });
    rms.finish(m.d_pad / 16, m.d_model, m.eps, inv_s, 16);
    int mt;
    floatx4 v[1];
    if (!splitk_reduce<1, 1, kWaves>(acc, part, mt, v)) {
        // g2 (next on the stream) runs head h with residue h % 8
        const int x = block_xcd(), per = head_blocks(m);
        l2_prefetch(x < m.H ? (m.H - x + kXcds - 1) / kXcds * per : 0, [&](int k) {
            return head_block(m, L.w_uq, L.w_uk, x + kXcds * (k / per), k % per);
        }, scratch, 1);
        return;
    }
    floatx4 y;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = row0 + 4 * g + i;
        y[i] = v[0][i] * inv_s[4 * g + i];
        if (row < s.B) {
            if (kv)
                s.ckv[(long long)row * m.kvw_pad + c] = y[i] * (c < m.kv_rank ? wn : 1.0f);
            else
                s.cqw[act_word(row, c, m.q_pad / 32)] =
                    F16::from_float(as_stored(c < m.q_rank ? y[i] * wn : 0.0f));
        }
    }
    if (kv)
        write_ss(y, c < m.kv_rank, s.ss_kv, m.kvw_pad / 16, nt - q_tiles, row0, s.B);
    else
        write_ss(y, c < m.q_rank, s.ss_cq, q_tiles, nt, row0, s.B);
}

// RoPE of the adjacent columns (a0, a1) (ops.cpp:88-108).  One form for every kernel: the
// kernels that a row can go through, depending on the batch, give the same bits.
__device__ __forceinline__ float rope_even(float a0, float a1, float2 cs) {
    return fmaf(a0, cs.x, -(a1 * cs.y));
}
__device__ __forceinline__ float rope_odd(float a0, float a1, float2 cs) {
    return fmaf(a0, cs.y, a1 * cs.x);
}

// The appended rows row0 .. row0 + 15: kv_norm of the latent, RoPE of the key, rounding, and the
// paged store.  Everything comes from LDS: y (rows of ld: v o kv_norm, then the key), the rows'
// kv_norm factors, slots (-1: none) and rotations [16][rope / 2].
__device__ __forceinline__ void append_rows(const StepArgs& s, uint16_t* pool, const float* y,
                                            int ld, const float* inv_s, const int32_t* slot_s,
                                            const float2* cs_s) {
    const ModelDims& m = s.dims;
    const bool tiled = page_tiled(m.page_size, m.kv_rank, m.rope);
    const int width = m.kv_rank + m.rope, per = blockDim.x / 16;  // threads of a row
    const int r = threadIdx.x / per;
    const int slot = slot_s[r];
    const int page = slot / m.page_size, off = slot % m.page_size;
    if (slot < 0 || page >= s.num_pool_pages)
        return;
    const float* yr = y + r * ld;
    const float inv = inv_s[r];
    uint16_t* base = pool + (long long)page * m.page_size * width;
    for (int c = threadIdx.x % per; c < width; c += per) {
        if (c < m.kv_rank) {
            base[latent_word(tiled, off, c, m.page_size, m.kv_rank)] =
                F16::from_float(as_stored(yr[c] * inv));
        } else {
            const int j = c - m.kv_rank;
            const float2 cs = cs_s[r * (m.rope / 2) + j / 2];
            const float a = yr[m.kv_rank + (j & ~1)], b = yr[m.kv_rank + (j | 1)];
            base[rope_word(tiled, off, j, m.page_size, m.kv_rank, m.rope)] =
                F16::from_float(as_stored(j & 1 ? rope_odd(a, b, cs) : rope_even(a, b, cs)));
        }
    }
}
constexpr int kMaxHalfRope = 32;  // rope <= 64 (mla_model_create checks)

// The sum of a row's n <= 16 partial sums of squares v[0 .. 15], in tile order (one order for every
// kernel that forms q_norm or kv_norm).
__device__ __forceinline__ float sum_tiles(const float (&v)[16], int n) {
    float ss = 0.0f;
#pragma unroll
    for (int j = 0; j < 16; ++j)
        ss += j < n ? v[j] : 0.0f;
    return ss;
}

// Head h's queries for rows row0 .. row0 + 15 from the rows' activation cq o q_norm (xq(k): lane
// (g, n)'s operand of k-step k: row n, columns 32k + 8g ..), by WAVES waves.  Wave w computes column
// tiles w, w + WAVES, .. of q = cq . w_uq transposed (lane (g, n): columns 4g + i of row n) into LDS
// (qf, 16 rows of qk_pad + 4 floats, free before the call); after the barrier RoPE of the rope
// columns goes to q_rope and the nope columns, rounded to fp16, are the operand of q_latent =
// W_uk_h^T q_nope, of which wave w computes column tiles w, w + WAVES, ...  inv_s, cs_s: the rows'
// q_norm factors and rotations in LDS, visible after the barrier.  bq / bu: this wave's weight
// tiles, loaded with the caller's operands.
constexpr int kQkTiles = 4, kKvTiles = 8, kNopeSteps = 2;  // limits (mla_model_create checks)

template <int WAVES, int KQ>
struct HeadWeights {
    static constexpr int QT = (kQkTiles + WAVES - 1) / WAVES, UT = (kKvTiles + WAVES - 1) / WAVES;
    V8 bq[QT][KQ], bu[UT][kNopeSteps];
    __device__ __forceinline__ void load(const ModelDims& m, const LayerWeights& L,
                                         const uint16_t* zeros, int h, int wave, int lane) {
        const int qk_tiles = m.qk_pad / 16, kv_tiles = m.kv_pad / 16;
        const int KTQ = m.q_pad / 32, KTU = m.nope_pad / 32;
#pragma unroll
        for (int t = 0; t < QT; ++t)
            if (wave + WAVES * t < qk_tiles)  // scalar, and nothing else writes the registers
#pragma unroll
                for (int k = 0; k < KQ; ++k)
                    bq[t][k] = load_w(L.w_uq, zeros, h * qk_tiles + wave + WAVES * t, k, KTQ, lane);
#pragma unroll
        for (int t = 0; t < UT; ++t)
            if (wave + WAVES * t < kv_tiles)
#pragma unroll
                for (int k = 0; k < kNopeSteps; ++k)
                    bu[t][k] = load_w(L.w_uk, zeros, h * kv_tiles + wave + WAVES * t, k, KTU, lane);
    }
};

template <int WAVES, int KQ, typename XQ>
__device__ __forceinline__ void q_head(const StepArgs& s, const HeadWeights<WAVES, KQ>& w, int h,
                                       int row0, XQ&& xq, const float* inv_s, const float2* cs_s,
                                       float* qf) {
    constexpr int QT = HeadWeights<WAVES, KQ>::QT, UT = HeadWeights<WAVES, KQ>::UT;
    const ModelDims& m = s.dims;
    const int wave = wave_index(), lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15;
    const int KTQ = m.q_pad / 32, ld = m.qk_pad + 4;
#pragma unroll
    for (int t = 0; t < QT; ++t) {
        const int tile = wave + WAVES * t;
        if (tile >= m.qk_pad / 16)
            break;
        floatx4 q = {0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < KQ; ++k)
            if (k < KTQ)
                q = mma(w.bq[t][k], xq(k), q);
        *reinterpret_cast<floatx4*>(qf + n * ld + 16 * tile + 4 * g) = q;
    }
    __syncthreads();
    // q_latent first: nothing waits for RoPE's stores
    const float inv = inv_s[n];
    V8 qn[kNopeSteps];
#pragma unroll
    for (int k = 0; k < kNopeSteps; ++k) {
        const int c0 = min(32 * k + 8 * g, m.qk_pad - 8);  // past nope: dropped below
        const floatx4 a = *reinterpret_cast<const floatx4*>(qf + n * ld + c0);
        const floatx4 b = *reinterpret_cast<const floatx4*>(qf + n * ld + c0 + 4);
#pragma unroll
        for (int e = 0; e < 8; ++e)
            qn[k][e] = (_Float16)(32 * k + 8 * g + e < m.nope ? (e < 4 ? a[e] : b[e - 4]) * inv : 0.0f);
    }
#pragma unroll
    for (int t = 0; t < UT; ++t) {
        const int tile = wave + WAVES * t, c = 16 * tile + 4 * g, row = row0 + n;
        if (tile >= m.kv_pad / 16)
            break;
        floatx4 ql = {0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < kNopeSteps; ++k)
            if (k < m.nope_pad / 32)
                ql = mma(w.bu[t][k], qn[k], ql);
        if (row >= s.B)
            continue;
        uint16_t* out = s.q_latent + ((long long)row * m.H + h) * m.kv_rank + c;
        if (m.kv_rank % 4 == 0) {  // a lane's four columns, 8 bytes
            if (c < m.kv_rank)
                *reinterpret_cast<u32x2*>(out) = __builtin_bit_cast(
                    u32x2, half4{(_Float16)ql[0], (_Float16)ql[1], (_Float16)ql[2], (_Float16)ql[3]});
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (c + i < m.kv_rank)
                    out[i] = F16::from_float(ql[i]);
        }
    }
    const int rhalf = m.rope / 2;
    for (int e = threadIdx.x; e < 16 * rhalf; e += 64 * WAVES) {
        const int r = e / rhalf, jp = 2 * (e % rhalf), row = row0 + r;
        if (row >= s.B)
            continue;
        const float a0 = qf[r * ld + m.nope + jp] * inv_s[r];
        const float a1 = qf[r * ld + m.nope + jp + 1] * inv_s[r];
        uint16_t* qr = s.q_rope + ((long long)row * m.H + h) * m.rope + jp;
        qr[0] = F16::from_float(rope_even(a0, a1, cs_s[e]));
        qr[1] = F16::from_float(rope_odd(a0, a1, cs_s[e]));
    }
}

constexpr int kG2Waves = 4;

template <int KW>
__global__ __launch_bounds__(64 * kG2Waves) void g2_kernel(StepArgs s, LayerWeights L,
                                                           uint16_t* pool) {
    __shared__ __attribute__((aligned(16))) float qf[16 * (192 + 4)];  // or the appended rows
    __shared__ float inv_s[16];
    __shared__ int32_t slot_s[16];
    __shared__ float2 cs_s[16 * kMaxHalfRope];
    const ModelDims& m = s.dims;
    const int tid = threadIdx.x, wave = wave_index(), lane = tid & 63, g = lane >> 4, n = lane & 15;
    const int row0 = blockIdx.y * 16, h = blockIdx.x, rh = m.rope / 2;
    if (h > m.H)
        return;  // columns are padded to a multiple of 8 (see l2_prefetch)
    // every load in flight at once, the rows' rotations (two a thread) and, in the last wave, the
    // sums of squares of row n among them
    const bool kv = h == m.H;
    const int ss_tiles = (kv ? m.kvw_pad : m.q_pad) / 16;
    float sv[16];
    if (wave == kG2Waves - 1) {  // scalar, and nothing else writes the registers
        const float* ss = (kv ? s.ss_kv : s.ss_cq) + (long long)(row0 + n) * ss_tiles;
#pragma unroll
        for (int j = 0; j < 16; ++j)
            sv[j] = ss[min(j, ss_tiles - 1)];
    }
    float2 r2[2];
#pragma unroll
    for (int k = 0; k < 2; ++k)
        r2[k] = s.rope_rows[(long long)row0 * rh + min(tid + 256 * k, 16 * rh - 1)];
    auto row_inputs = [&]() {  // q_norm / kv_norm factors and rotations of the rows, to LDS
        if (wave == kG2Waves - 1 && g == 0) {
            const int cols = kv ? m.kv_rank : m.q_rank;
            inv_s[n] = 1.0f / sqrtf(sum_tiles(sv, ss_tiles) / (float)cols + m.eps);
        }
#pragma unroll
        for (int k = 0; k < 2; ++k)
            if (tid + 256 * k < 16 * rh)
                cs_s[tid + 256 * k] = r2[k];
    };
    if (kv) {  // the append workgroup: a thread loads 12 columns of row tid / 16 and its slot
        const int row = row0 + tid / 16, ld = m.kvw_pad + 4;
        float v[12];
#pragma unroll
        for (int k = 0; k < 12; ++k)
            v[k] = s.ckv[(long long)row * m.kvw_pad + min(16 * k + tid % 16, m.kvw_pad - 1)];
        const int32_t slot = s.slot_mapping[min(row, s.B - 1)];
        operands_issued();
        row_inputs();
#pragma unroll
        for (int k = 0; k < 12; ++k)
            if (16 * k < m.kvw_pad)
                qf[tid / 16 * ld + 16 * k + tid % 16] = v[k];
        if (tid % 16 == 0)
            slot_s[tid / 16] = row < s.B ? slot : -1;
        __syncthreads();
        append_rows(s, pool, qf, ld, inv_s, slot_s, cs_s);
        return;
    }
    HeadWeights<kG2Waves, KW> w;
    w.load(m, L, s.zeros, h, wave, lane);
    APre16<KW, 1> a;
    a.load(s.cqw + (long long)row0 * m.q_pad, s.B - row0, m.q_pad / 32, 0, 1, lane);
    operands_issued();
    row_inputs();
    q_head(s, w, h, row0, [&](int k) { return a.x[k][0]; }, inv_s, cs_s, qf);
}

// qkv_kernel -- g1 and g2 in one launch for smaller batches: workgroup h < H computes head h's
// queries, workgroup H the cache append.  Both start with g1's split-K GEMM over their column
// range, so no other workgroup's output is waited for: each head workgroup recomputes the whole
// cq row it needs for q_norm.  Each of the 9 workgroups (at 8 heads) of 16 rows then pulls 230 KB
// of weights through one CU's load path, and one workgroup fills a CU; that costs less than a
// second launch and its round trip until some XCD has more workgroups than CUs (an XCD runs the
// columns of one residue, see l2_prefetch).  A step of sessions of 100 to 200 tokens, one launch /
// two, us: 8 heads (the line lies at 256 rows) 17 rows 263 / 276, 64 273 / 287, 128 295 / 308, 256
// 358 / 374, 320 471 / 439, 640 657 / 589; 16 heads (160 rows) 160 rows 357 / 370, 176 405 / 378; 4
// heads (512 rows) 512 rows 474 / 492, 528 556 / 533.
constexpr int kQkvRows = 16;
constexpr int kXcdCus = 32;
__host__ __device__ inline bool qkv_one_launch(const ModelDims& m, int rows) {
    return (rows + kQkvRows - 1) / kQkvRows * ((m.H + kXcds) / kXcds) <= kXcdCus;
}
constexpr int kQkvMaxTiles = 16;  // q_pad <= 256, kvw_pad <= 192: at most 16 column tiles
constexpr int kQkvPad = 8;        // fp16 pad of the LDS A-operand rows
// fp32 pad of the LDS y rows: with a pitch of 36 mod 64 words, the split-K reduction's
// writes (rows 4g + i of lane group g) fall 16 banks apart per group, conflict-free.
constexpr int kQkvYPad = 36;

// LDS layout of qkv_kernel (bytes), from the model dims.
struct QkvLds {
    int part, y, ya, qf, total;
};
__host__ __device__ inline QkvLds qkv_lds(const ModelDims& m) {
    const int nt = max(m.q_pad, m.kvw_pad) / 16;
    const int ncol = max(m.q_pad, m.kvw_pad);
    // A head workgroup writes ya where the append workgroup keeps y (neither needs the other).
    QkvLds l;
    l.part = 0;                      // [8 waves][nt][64] floatx4
    l.qf = 0;                        // [16][qk_pad + 4] fp32, once the partials are summed
    l.y = kWaves * nt * 64 * 16;     // [16][ncol + kQkvYPad] fp32
    l.ya = l.y;                      // [16][q_pad + pad] fp16
    l.total = l.y + kQkvRows * (ncol + kQkvYPad) * 4;
    return l;
}

// KC: chunks of two k-steps per wave (KT <= 16 * KC); NT >= the workgroup's column tiles
// (q_pad <= 16 NT).
template <int KC, int NT>
__global__ __launch_bounds__(64 * kWaves) void qkv_kernel(StepArgs s, LayerWeights L,
                                                          uint16_t* pool) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    constexpr int KQ = NT / 2;  // k-steps of w_uq
    const ModelDims& m = s.dims;
    const QkvLds lay = qkv_lds(m);
    floatx4* part = reinterpret_cast<floatx4*>(smem + lay.part);
    float* y = reinterpret_cast<float*>(smem + lay.y);
    _Float16* ya = reinterpret_cast<_Float16*>(smem + lay.ya);
    float* qf = reinterpret_cast<float*>(smem + lay.qf);
    __shared__ float inv_x[kQkvRows];
    __shared__ float inv_n[kQkvRows];  // q_norm / kv_norm factor per row
    // row sums of squares per column tile (a pitch of 20: the rows' reads start in different banks)
    __shared__ __attribute__((aligned(16))) float ss_part[kQkvRows][kQkvMaxTiles + 4];
    __shared__ int32_t slot_s[kQkvRows];
    __shared__ float2 cs_s[kQkvRows * kMaxHalfRope];

    const int h = blockIdx.x, row0 = blockIdx.y * kQkvRows;
    const int tid = threadIdx.x, wave = wave_index(), lane = tid & 63, g = lane >> 4, n = lane & 15;
    if (h > m.H)
        return;  // the heads' columns are padded to a multiple of 8 (head h: residue h % 8)
    const bool kv = h == m.H;
    const int KT = m.d_pad / 32, q_tiles = m.q_pad / 16;
    const int nt0 = kv ? q_tiles : 0, ntv = kv ? m.kvw_pad / 16 : q_tiles;
    const int ldy = max(m.q_pad, m.kvw_pad) + kQkvYPad;
    RmsPrefetch<16> rms;
    rms.issue(s.ss_x, m.d_pad / 16, row0, kQkvRows);
    // The norm weights of the two columns this thread reduces (16 * (wave + 8k) + n), the rows'
    // slots and rotations travel with the GEMM operands.
    const int ncols = kv ? m.kv_rank : m.q_rank;
    const float* nwp = kv ? L.kv_norm : L.q_norm;
    float nw[2];
#pragma unroll
    for (int k = 0; k < 2; ++k)
        nw[k] = nwp[min(16 * (wave + kWaves * k) + n, ncols - 1)];
    const int rhalf = m.rope / 2;
    const int32_t slot_pf = s.slot_mapping[min(row0 + tid, s.B - 1)];
    const float2 rcs = s.rope_rows[(long long)row0 * rhalf + min(tid, kQkvRows * rhalf - 1)];

    // ---- GEMM 1: every operand of this wave in flight at once, chunk by chunk ----
    floatx4 acc[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j)
        acc[j] = floatx4{0, 0, 0, 0};
    const uint16_t* xw = s.xw + act_word(min(row0 + n, s.B - 1), 8 * g, KT);
    HeadWeights<kWaves, KQ> hw;  // head workgroups: used after the reduction
#pragma unroll
    for (int c = 0; c < KC; ++c) {
        V8 a[2], b[2][NT];
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const int kt = wave + kWaves * (2 * c + kk);
            a[kk] = *reinterpret_cast<const V8*>(xw + min(kt, KT - 1) * 512);
#pragma unroll
            for (int j = 0; j < NT; ++j)
                b[kk][j] = load_w(L.w_dq_dkv, s.zeros, nt0 + min(j, ntv - 1), kt, KT, lane);
        }
        if (c == 0 && !kv)
            hw.load(m, L, s.zeros, h, wave, lane);
        operands_issued();
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
            for (int j = 0; j < NT; ++j)
                acc[j] = mma(a[kk], b[kk][j], acc[j]);
    }
    rms.finish(m.d_pad / 16, m.d_model, m.eps, inv_x, kQkvRows);
#pragma unroll
    for (int j = 0; j < NT; ++j)
        if (j < ntv)
            part[(wave * ntv + j) * 64 + lane] = acc[j];
    if (tid < kQkvRows)
        slot_s[tid] = row0 + tid < s.B ? slot_pf : -1;
    if (tid < kQkvRows * rhalf)
        cs_s[tid] = rcs;
    if (tid < kQkvRows * kQkvMaxTiles && tid % kQkvMaxTiles >= ntv)
        ss_part[tid / kQkvMaxTiles][tid % kQkvMaxTiles] = 0.0f;
    __syncthreads();
    // v[r][c] = inv_x[r] * sum over the waves (rows 4g+i, column 16j+n of lane group e);
    // head: ya = v o q_norm weight (fp16 A operand); kv: y = v o kv_norm weight (1 for the
    // key's RoPE columns).  ss_part[r][j] = sum of v^2 over tile j's norm columns.
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int j = wave + kWaves * k, col = 16 * j + n;
        if (j >= ntv)
            break;
        floatx4 v = {0, 0, 0, 0};
#pragma unroll
        for (int w = 0; w < kWaves; ++w)
            v += part[(w * ntv + j) * 64 + lane];
        const float wc = col < ncols ? nw[k] : kv ? 1.0f : 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = 4 * g + i;
            const float yv = v[i] * inv_x[r];
            if (kv)
                y[r * ldy + col] = yv * wc;
            else
                ya[r * (m.q_pad + kQkvPad) + col] = (_Float16)as_stored(yv * wc);
            const float sq = sum16(col < ncols ? yv * yv : 0.0f);
            if (n == 0)
                ss_part[r][j] = sq;
        }
    }
    __syncthreads();
    // the norm factors of the rows (ops.cpp:37-44: 1/sqrt(mean(v^2) + eps))
    if (wave == kWaves - 1 && g == 0) {
        float ssv[kQkvMaxTiles];
#pragma unroll
        for (int j = 0; j < kQkvMaxTiles; ++j)
            ssv[j] = ss_part[n][j];
        inv_n[n] = 1.0f / sqrtf(sum_tiles(ssv, kQkvMaxTiles) / (float)ncols + m.eps);
    }

    if (kv) {  // ---- kv_norm, RoPE of the key, rounding and the paged append ----
        __syncthreads();
        append_rows(s, pool, y, ldy, inv_n, slot_s, cs_s);
        return;
    }
    q_head(s, hw, h, row0, [&](int k) {
        return *reinterpret_cast<const V8*>(ya + n * (m.q_pad + kQkvPad) + 32 * k + 8 * g);
    }, inv_n, cs_s, qf);
}

// ----------------------------------------------------------- g4 and g6 ----
// y = A . W + residual for 16 rows and one 16-column tile (8 waves split K): y to `out`
// (fp32), y o wnorm to `outw` (fp16, the next consumer's normalised A operand), and
// y's per-tile sums of squares.  The residual and norm columns are fetched with the
// operands.
template <int KW, typename ALoad, typename Pf>
__device__ __forceinline__ void splitk_residual(ALoad&& aload, const uint16_t* w,
                                                const uint16_t* zeros, int KT, int N,
                                                const float* residual, const float* wnorm,
                                                float* out, uint16_t* outw, float* ss,
                                                int n_tiles, int ld, int row0, int B,
                                                Pf&& prefetch) {
    __shared__ __attribute__((aligned(16))) floatx4 part[kWaves * 64];
    const int wave = wave_index(), lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15;
    const int nt = blockIdx.x, col = nt * 16 + n;
    BPre<1, KW> bw;
    bw.load(w, zeros, nt, 1, KT, wave, kWaves, lane);
    floatx4 res;
    float wn;
    if (wave == 0) {  // the wave that uses them
#pragma unroll
        for (int i = 0; i < 4; ++i)
            res[i] = residual[(long long)(row0 + 4 * g + i) * ld + min(col, N - 1)];
        wn = wnorm[min(col, N - 1)];
    }
    floatx4 acc[1][1];
    zero(acc);
    aload(acc, bw, wave, lane);
    int mt;
    floatx4 v[1];
    if (!splitk_reduce<1, 1, kWaves>(acc, part, mt, v)) {
        prefetch();  // waves 1.. have nothing left to do but this
        return;
    }
    floatx4 y;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const long long row = row0 + 4 * g + i;
        y[i] = col < N ? v[0][i] + res[i] : 0.0f;
        if (row < B && col < N) {
            out[row * ld + col] = y[i];
            outw[act_word(row, col, ld >> 5)] = F16::from_float(y[i] * wn);
        }
    }
    write_ss(y, col < N, ss, n_tiles, nt, row0, B);
}

template <int KW>
__global__ __launch_bounds__(64 * kWaves) void g4_kernel(StepArgs s, LayerWeights L) {
    __shared__ __attribute__((aligned(16))) uint16_t pf_scratch[512];
    const ModelDims& m = s.dims;
    const int row0 = blockIdx.y * 16;
    const int KT = m.ctx_pad / 32;
    splitk_residual<KW>(
        [&](floatx4(&acc)[1][1], const BPre<1, KW>& bw, int kt0, int lane) {
            APre16<KW, 1> a;
            a.load(s.ctx + (long long)row0 * m.ctx_pad, s.B - row0, KT, kt0, kWaves, lane);
            operands_issued();
            mma_steps(acc, bw, [&](int kk, int mt) { return a.x[kk][mt]; });
        },
        L.w_out, s.zeros, KT, m.d_model, s.x, L.ffn_norm, s.res, s.resw, s.ss_res, m.d_pad / 16, m.d_pad,
        row0, s.B, [&]() {
            // g5 (next on the stream) runs column pair p with residue p % 8: its two tiles of
            // every k-step are 2 * KT5 contiguous blocks
            const int x = block_xcd(), np = m.ff_pad / 16, KT5 = m.d_pad / 32, per = 2 * KT5;
            const int pairs = x < np ? (np - x + kXcds - 1) / kXcds : 0;
            l2_prefetch(pairs * per, [&](int k) {
                const int p = x + kXcds * (k / per);
                return L.w_gate_up + ((long long)2 * p * KT5 + k % per) * 512;
            }, pf_scratch, 1);
        });
}

// next_norm: the norm weight of x's next consumer (attn_norm of the next layer, or
// final_norm after the last layer).  next: the next layer's weights (qkv_kernel or g1_kernel runs
// next on the stream), or null after the last layer.
template <int KW>
__global__ __launch_bounds__(64 * kWaves) void g6_kernel(StepArgs s, LayerWeights L,
                                                         const float* next_norm,
                                                         const uint16_t* next_dq_dkv,
                                                         const uint16_t* next_uq,
                                                         const uint16_t* next_uk) {
    __shared__ __attribute__((aligned(16))) uint16_t pf_scratch[512];
    const ModelDims& m = s.dims;
    const int row0 = blockIdx.y * 16, KT = m.ff_pad / 32;
    splitk_residual<KW>(
        [&](floatx4(&acc)[1][1], const BPre<1, KW>& bw, int kt0, int lane) {
            APre16<KW, 1> a;
            a.load(s.u + (long long)row0 * m.ff_pad, s.B - row0, KT, kt0, kWaves, lane);
            operands_issued();
            mma_steps(acc, bw, [&](int kk, int mt) { return a.x[kk][mt]; });
        },
        L.w_down, s.zeros, KT, m.d_model, s.res, next_norm, s.x, s.xw, s.ss_x, m.d_pad / 16, m.d_pad,
        row0, s.B, [&]() {
            if (!next_dq_dkv)
                return;
            if (qkv_one_launch(m, s.B)) {
                // qkv_kernel runs head h with residue h % 8 and the append workgroup (h = H) with
                // H % 8: head workgroups read the w_dq tiles, the append one the w_dkv tiles, and
                // head h its w_uq and w_uk blocks
                const int x = block_xcd(), KTq = m.d_pad / 32, q_tiles = m.q_pad / 16;
                const int n_dq = x < m.H ? q_tiles * KTq : 0;
                const int n_dkv = m.H % kXcds == x ? (m.kvw_pad / 16) * KTq : 0;
                const int per = head_blocks(m);
                const int heads = x < m.H ? (m.H - x + kXcds - 1) / kXcds : 0;
                l2_prefetch(n_dq + n_dkv + heads * per, [&](int k) {
                    if (k < n_dq)
                        return next_dq_dkv + (long long)k * 512;
                    k -= n_dq;
                    if (k < n_dkv)
                        return next_dq_dkv + ((long long)q_tiles * KTq + k) * 512;
                    k -= n_dkv;
                    return head_block(m, next_uq, next_uk, x + kXcds * (k / per), k % per);
                }, pf_scratch, 1);
                return;
            }
            // g1_kernel runs column tile t with residue t % 8 (its KT blocks are contiguous)
            const int x = block_xcd(), KT1 = m.d_pad / 32, tiles = (m.q_pad + m.kvw_pad) / 16;
            l2_prefetch(x < tiles ? (tiles - x + kXcds - 1) / kXcds * KT1 : 0, [&](int k) {
                return next_dq_dkv + ((long long)(x + kXcds * (k / KT1)) * KT1 + k % KT1) * 512;
            }, pf_scratch, 1);
        });
}

// --------------------------------------------------------------------- g5 ----
// RMSNorm(res, ffn_norm) . [w_gate | w_up] for 16 rows: w_gate_up interleaves 16-column
// tiles of gate and up (tile 2j = gate columns 16j.., tile 2j+1 = up columns 16j..); one
// pair per workgroup, 8 waves split K, then SwiGLU (ops.cpp:65-77: gate*sigmoid(gate)*up).
__device__ __forceinline__ float silu_stable(float x) {
    if (x >= 0.0f)
        return x * (1.0f / (1.0f + expf(-x)));
    const float e = expf(x);
    return x * (e / (1.0f + e));
}

template <int KW>
__global__ __launch_bounds__(64 * kWaves) void g5_kernel(StepArgs s, LayerWeights L) {
    __shared__ __attribute__((aligned(16))) floatx4 part[kWaves * 2 * 64];
    __shared__ float inv_s[16];
    const ModelDims& m = s.dims;
    const int row0 = blockIdx.y * 16, p = blockIdx.x;
    if (p >= m.ff_pad / 16)
        return;  // the grid's columns are padded to a multiple of 8 (one XCD per pair)
    const int wave = wave_index(), lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15;
    const int KT = m.d_pad / 32;
    RmsPrefetch<16> rms;
    rms.issue(s.ss_res, m.d_pad / 16, row0, 16);
    BPre<2, KW> bw;
    bw.load(L.w_gate_up, s.zeros, 2 * p, 2, KT, wave, kWaves, lane);
    APre16<KW, 1> a;
    a.load(s.resw + (long long)row0 * m.d_pad, s.B - row0, KT, wave, kWaves, lane);
    operands_issued();
    floatx4 acc[1][2];
    zero(acc);
    mma_steps(acc, bw, [&](int kk, int mt) { return a.x[kk][mt]; });
    rms.finish(m.d_pad / 16, m.d_model, m.eps, inv_s, 16);
    int mt;
    floatx4 v[2];
    if (!splitk_reduce<1, 2, kWaves>(acc, part, mt, v))
        return;
    const int col = p * 16 + n;
    if (col < m.d_ff)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = row0 + 4 * g + i;
            const float inv = inv_s[4 * g + i];
            if (row < s.B)
                s.u[act_word(row, col, m.ff_pad / 32)] =
                    F16::from_float(silu_stable(v[0][i] * inv) * (v[1][i] * inv));
        }
}

// --------------------------------------------------------------------- g7 ----
// Final RMSNorm + tied logits h . E^T for 64 rows and four 16-column tiles per
// workgroup (the waves split K eight ways: measured 11.7 us at config 3 against 13.1 us
// for four ways times two tile groups, whose waves each loaded twice the activation
// rows); each workgroup also leaves, per row, the greedy winner of its 64 columns
// (strict >, so the lowest index wins ties; banned ids never win) and whether all of
// them were finite (banned or not: sample_token checks every logit,
// inference.cpp:352-353).
constexpr int kG7Tiles = 4, kG7KG = 8;

// Greedy key of a logit: larger value first, then lower column.  The value's bits are
// mapped to an order-preserving unsigned (after -0 -> +0, which compares equal to it),
// the column to its complement; 0 marks "no candidate" (every real key is larger).
__device__ __forceinline__ uint64_t greedy_key(float y, int col) {
    const uint32_t b = __float_as_uint(y + 0.0f);
    const uint32_t ord = b ^ ((uint32_t)((int32_t)b >> 31) | 0x80000000u);
    return ((uint64_t)ord << 32) | (uint32_t)~(uint32_t)col;
}
template <int CTRL>
__device__ __forceinline__ uint64_t dpp_shr64(uint64_t v) {  // lanes without a source get 0
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), CTRL, 0xf, 0xf, true);
    return ((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo;
}
// Running maximum along each row of 16 lanes: lane 15 of the row ends with the row's max.
__device__ __forceinline__ uint64_t row_max16(uint64_t v) {
    uint64_t t = dpp_shr64<0x111>(v);
    v = t > v ? t : v;
    t = dpp_shr64<0x112>(v);
    v = t > v ? t : v;
    t = dpp_shr64<0x114>(v);
    v = t > v ? t : v;
    t = dpp_shr64<0x118>(v);
    return t > v ? t : v;
}

// A wave's 16 rows x 64 columns of logits: the values, and per row the greedy winner of the
// group's columns.  v[j]: lane (g, n) holds rows row0 + 4g + i of column 16j + n.
__device__ __forceinline__ void logits_out(const StepArgs& s, const floatx4 (&v)[kG7Tiles], int row0,
                                           const float* inv, int part, int parts) {
    const ModelDims& m = s.dims;
    const int lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15;
    uint64_t best[4] = {0, 0, 0, 0};
    uint64_t nonfinite[4] = {0, 0, 0, 0};  // 1 when some logit of the row is not finite
#pragma unroll
    for (int j = 0; j < kG7Tiles; ++j) {
        const int col = (part * kG7Tiles + j) * 16 + n;
        const bool valid = col < m.vocab;
        const bool open = valid && !(s.ban && ((s.ban[col >> 5] >> (col & 31)) & 1u));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = row0 + 4 * g + i;
            const float y = v[j][i] * inv[4 * g + i];
            if (valid && row < s.B)
                s.logits[(long long)row * m.vocab + col] = y;
            if (valid && !isfinite(y))
                nonfinite[i] = 1;
            const uint64_t k = open ? greedy_key(y, col) : 0;
            best[i] = k > best[i] ? k : best[i];
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        // the 16 lanes of a row hold 16 columns each; lane 15 gathers the row's winner
        const uint64_t k = row_max16(best[i]);
        const uint64_t bad = row_max16(nonfinite[i]);
        const int row = row0 + 4 * g + i;
        if (n == 15 && row < s.B) {
            const long long idx = (long long)row * parts + part;
            const uint32_t ord = (uint32_t)(k >> 32);
            const uint32_t b = ord & 0x80000000u ? ord ^ 0x80000000u : ~ord;
            s.arg_v[idx] = k ? __uint_as_float(b) : -INFINITY;
            s.arg_c[idx] = bad ? -1 : k ? (int)~(uint32_t)k : 0x7fffffff;
        }
    }
}

template <int KW>
__global__ __launch_bounds__(64 * kWaves) void g7_kernel(StepArgs s) {
    constexpr int NTW = kG7Tiles / (kWaves / kG7KG);
    __shared__ __attribute__((aligned(16))) floatx4 part[kWaves * 4 * NTW * 64];
    __shared__ float inv_s[64];
    const ModelDims& m = s.dims;
    const int row0 = blockIdx.y * 64;
    const int wave = wave_index(), lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15;
    const int KT = m.d_pad / 32, kg = wave % kG7KG, ng = wave / kG7KG;
    const int n_tiles = m.vocab_pad / 16, nt0 = blockIdx.x * kG7Tiles;
    RmsPrefetch<8> rms;
    rms.issue(s.ss_x, m.d_pad / 16, row0, 64);
    BPre<NTW, KW> bw;
    bw.load(s.embed, s.zeros, nt0 + ng * NTW, min(NTW, n_tiles - nt0 - ng * NTW), KT, kg, kG7KG, lane);
    APre16<KW, 4> a;
    a.load(s.xw + (long long)row0 * m.d_pad, s.B - row0, KT, kg, kG7KG, lane);
    operands_issued();
    floatx4 acc[4][NTW];
    zero(acc);
    mma_steps(acc, bw, [&](int kk, int mt) { return a.x[kk][mt]; });
    rms.finish(m.d_pad / 16, m.d_model, m.eps, inv_s, 64);
    int mt;
    floatx4 v[kG7Tiles];
    if (!splitk_reduce<4, NTW, kG7KG>(acc, part, mt, v))
        return;
    logits_out(s, v, row0 + 16 * mt, inv_s + 16 * mt, blockIdx.x, gridDim.x);
}

// The same product for many 64 x 64 blocks: each of a workgroup's four waves computes one by
// itself, K group after K group in g7_kernel's order (the same bits).  g7_kernel's exchange of
// partial sums takes 131 KB of LDS, so a CU runs one workgroup at a time, about 7 us a round,
// with nothing to hide its loads and stores behind; here nothing is exchanged, two workgroups
// share a CU (256 VGPRs), the waves read the same activations, and a column group's workgroups
// all run on one XCD (grid padded to its count), whose L2 keeps its share of the embedding.
// d_model 512, vocabulary 16384: 200 rows 28.0 -> 16.7 us, 1000 rows 100 -> 43 us, about 24 us of
// it products, 11 the 64 MB of logits, 8 the greedy keys.
constexpr int kG7RowsWaves = 4;

template <int KW>
__global__ __launch_bounds__(64 * kG7RowsWaves, 2) void g7_rows_kernel(StepArgs s, int parts) {
    __shared__ float inv_s[64];
    const ModelDims& m = s.dims;
    const int row0 = blockIdx.y * 64, part0 = blockIdx.x * kG7RowsWaves;
    if (part0 >= parts)
        return;  // the grid is padded to a multiple of the XCDs
    const int wave = wave_index(), lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15;
    const int KT = m.d_pad / 32, n_tiles = m.vocab_pad / 16;
    const int part = min(part0 + wave, parts - 1), nt0 = part * kG7Tiles;
    RmsPrefetch<8> rms[2];  // 32 rows each
    rms[0].issue(s.ss_x, m.d_pad / 16, row0, 32);
    rms[1].issue(s.ss_x, m.d_pad / 16, row0 + 32, 32);
    const uint16_t *x[4], *w[kG7Tiles];
#pragma unroll
    for (int j = 0; j < kG7Tiles; ++j)
        w[j] = s.embed + (long long)min(nt0 + j, n_tiles - 1) * KT * 512 + lane * 8;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
        x[mt] = s.xw + act_word(min(row0 + 16 * mt + n, s.B - 1), 8 * g, KT);
    // Step kk of a K group uses buffer kk % kBufs and refills it for the step kBufs later.  The
    // loop over the groups stays rolled: unrolled, the compiler gathers the loads of all
    // groups at its top and spills.
    constexpr int kBufs = KW < 2 ? KW : 2;  // divides KW
    static_assert(KW % kBufs == 0, "buffers");
    V8 a[kBufs][4], b[kBufs][kG7Tiles];
    auto load = [&](int kg, int kk) {
        const int kt = min(kg + kk * kG7KG, KT - 1) * 512;
#pragma unroll
        for (int j = 0; j < kG7Tiles; ++j)
            b[kk % kBufs][j] = *reinterpret_cast<const V8*>(w[j] + kt);
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
            a[kk % kBufs][mt] = *reinterpret_cast<const V8*>(x[mt] + kt);
    };
#pragma unroll
    for (int kk = 0; kk < kBufs; ++kk)
        load(0, kk);
    floatx4 sum[4][kG7Tiles];
    zero(sum);
    auto group = [&](int kg, bool more) {
        floatx4 acc[4][kG7Tiles];
        zero(acc);
#pragma unroll
        for (int kk = 0; kk < KW; ++kk) {
            operands_issued();
            // The activations of a step past KT count as zeros (no branch: it would hold the
            // accumulators in two places).
            const uint32_t in = kg + kk * kG7KG < KT ? 0xffffffffu : 0u;
#pragma unroll
            for (int mt = 0; mt < 4; ++mt) {
                const V8 x0 = __builtin_bit_cast(
                    V8, __builtin_bit_cast(u32x4, a[kk % kBufs][mt]) & in);
#pragma unroll
                for (int j = 0; j < kG7Tiles; ++j)
                    acc[mt][j] = mma(x0, b[kk % kBufs][j], acc[mt][j]);
            }
            if (kk + kBufs < KW)
                load(kg, kk + kBufs);
            else if (more)
                load(kg + 1, kk + kBufs - KW);
        }
        operands_issued();
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
#pragma unroll
            for (int j = 0; j < kG7Tiles; ++j)
                sum[mt][j] += acc[mt][j];
    };
#pragma unroll 1
    for (int kg = 0; kg < kG7KG - 1; ++kg)
        group(kg, true);
    group(kG7KG - 1, false);
    rms[0].finish(m.d_pad / 16, m.d_model, m.eps, inv_s, 32);
    rms[1].finish(m.d_pad / 16, m.d_model, m.eps, inv_s + 32, 32);
    __syncthreads();
    if (part0 + wave >= parts)
        return;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
        logits_out(s, sum[mt], row0 + 16 * mt, inv_s + 16 * mt, part, parts);
}

// Last row of each session (cu_q[b+1] - 1) to row b of the logits operands: the
// normalised activation xw (fp16) and its per-tile sums of squares.  The reference
// returns the logits of a prefill's last position only (inference.cpp:64-66).  Rows
// [B, m_pad) are zeroed.
__global__ __launch_bounds__(256) void gather_last_kernel(StepArgs s, int B, const int32_t* cu_q,
                                                          uint16_t* xw_out, float* ss_out) {
    const ModelDims& m = s.dims;
    const int b = blockIdx.x, d_tiles = m.d_pad / 16;
    const int src = b < B ? cu_q[b + 1] - 1 : -1;
    for (int c = threadIdx.x; c < m.d_pad; c += 256)
        xw_out[act_word(b, c, m.d_pad / 32)] =
            src >= 0 ? s.xw[act_word(src, c, m.d_pad / 32)] : 0;
    for (int c = threadIdx.x; c < d_tiles; c += 256)
        ss_out[(long long)b * d_tiles + c] = src >= 0 ? s.ss_x[(long long)src * d_tiles + c] : 0.0f;
}

// Greedy token per row (inference.cpp:354-380 with no repetition penalty): the lowest
// column among the maxima of the ids not banned; -1 when a logit is not finite
// (numerical_error, checked first as the reference does), -2 when every id is banned
// ("All tokens are banned").  256
// threads load up to four partials each at once (parts <= 1024).
constexpr int kArgItems = 4;

__global__ __launch_bounds__(256) void argmax_kernel(StepArgs s, int parts) {
    __shared__ float sv[4];
    __shared__ int sc[4], sbad[4];
    const int row = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float pv[kArgItems];
    int pc[kArgItems];
#pragma unroll
    for (int i = 0; i < kArgItems; ++i) {
        const int p = threadIdx.x + 256 * i;
        pv[i] = -INFINITY;
        pc[i] = 0x7fffffff;
        if (p < parts) {
            pv[i] = s.arg_v[(long long)row * parts + p];
            pc[i] = s.arg_c[(long long)row * parts + p];
        }
    }
    float bv = -INFINITY;
    int bc = 0x7fffffff, bad = 0;
#pragma unroll
    for (int i = 0; i < kArgItems; ++i) {  // increasing columns
        if (pc[i] < 0)
            bad = 1;
        else if (pc[i] != 0x7fffffff && (bc == 0x7fffffff || pv[i] > bv)) {
            bv = pv[i];
            bc = pc[i];
        }
    }
    auto better = [](float ov, int oc, float v, int c) {
        return oc != 0x7fffffff && (c == 0x7fffffff || ov > v || (ov == v && oc < c));
    };
    for (int off = 32; off > 0; off >>= 1) {
        const float ov = __shfl_xor(bv, off, 64);
        const int oc = __shfl_xor(bc, off, 64);
        bad |= __shfl_xor(bad, off, 64);
        if (better(ov, oc, bv, bc)) {
            bv = ov;
            bc = oc;
        }
    }
    if (lane == 0) {
        sv[wave] = bv;
        sc[wave] = bc;
        sbad[wave] = bad;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 4; ++w) {
            bad |= sbad[w];
            if (better(sv[w], sc[w], bv, bc)) {
                bv = sv[w];
                bc = sc[w];
            }
        }
        s.next_tokens[row] = bad ? -1 : bc == 0x7fffffff ? -2 : bc;
    }
}

// k-steps per wave, rounded up to a compiled variant
int kw_variant(int ksteps) {
    return ksteps <= 1 ? 1 : ksteps <= 2 ? 2 : ksteps <= 3 ? 3 : ksteps <= 4 ? 4 : ksteps <= 6 ? 6 : 8;
}
int ceil_div(int a, int b) { return (a + b - 1) / b; }
int round_up_to(int a, int b) { return ceil_div(a, b) * b; }

}  // namespace

// ------------------------------------------------------------------ launches ----
int g7_parts(const ModelDims& m) { return ceil_div(m.vocab_pad / 16, kG7Tiles); }

#define MLA_KW_DISPATCH(kw, KERNEL, ...)                                                        \
    switch (kw) {                                                                                \
    case 1: hipLaunchKernelGGL(KERNEL<1>, __VA_ARGS__); break;                                   \
    case 2: hipLaunchKernelGGL(KERNEL<2>, __VA_ARGS__); break;                                   \
    case 3: hipLaunchKernelGGL(KERNEL<3>, __VA_ARGS__); break;                                   \
    case 4: hipLaunchKernelGGL(KERNEL<4>, __VA_ARGS__); break;                                   \
    case 6: hipLaunchKernelGGL(KERNEL<6>, __VA_ARGS__); break;                                   \
    default: hipLaunchKernelGGL(KERNEL<8>, __VA_ARGS__); break;                                  \
    }
// K = d_model <= 1024 over 8 K groups: at most 4 k-steps a wave
#define MLA_KW4_DISPATCH(kw, KERNEL, ...)                                                       \
    switch (kw) {                                                                                \
    case 1: hipLaunchKernelGGL(KERNEL<1>, __VA_ARGS__); break;                                   \
    case 2: hipLaunchKernelGGL(KERNEL<2>, __VA_ARGS__); break;                                   \
    case 3: hipLaunchKernelGGL(KERNEL<3>, __VA_ARGS__); break;                                   \
    default: hipLaunchKernelGGL(KERNEL<4>, __VA_ARGS__); break;                                  \
    }

int layer_pre_launches(const ModelDims& m, int rows) { return qkv_one_launch(m, rows) ? 1 : 2; }

size_t qkv_lds_bytes(const ModelDims& m) { return (size_t)qkv_lds(m).total; }

// Kernels whose dynamic LDS can exceed 64 KB: allow what this model's shape needs.
hipError_t model_kernel_attributes(const ModelDims& m) {
    const int bytes = (int)qkv_lds_bytes(m);
    const void* ks[] = {
        reinterpret_cast<const void*>(&qkv_kernel<1, 4>), reinterpret_cast<const void*>(&qkv_kernel<1, 8>),
        reinterpret_cast<const void*>(&qkv_kernel<1, 12>), reinterpret_cast<const void*>(&qkv_kernel<1, 16>),
        reinterpret_cast<const void*>(&qkv_kernel<2, 4>), reinterpret_cast<const void*>(&qkv_kernel<2, 8>),
        reinterpret_cast<const void*>(&qkv_kernel<2, 12>), reinterpret_cast<const void*>(&qkv_kernel<2, 16>)};
    for (const void* k : ks) {
        const hipError_t e =
            hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
        if (e != hipSuccess)
            return e;
    }
    return hipSuccess;
}

hipError_t launch_embed(const StepArgs& s, const float* first_norm, hipStream_t st) {
    hipLaunchKernelGGL(embed_kernel, dim3(s.m_pad), dim3(256), 0, st, s, first_norm);
    return hipGetLastError();
}

hipError_t launch_layer_pre(const StepArgs& s, const LayerWeights& w, uint16_t* pool,
                            hipStream_t st) {
    const ModelDims& m = s.dims;
    if (qkv_one_launch(m, s.B)) {
        const size_t lds = qkv_lds_bytes(m);
        const dim3 grid(round_up_to(m.H + 1, kXcds), ceil_div(s.B, kQkvRows));  // padded: see l2_prefetch
        const int nt = max(m.q_pad, m.kvw_pad) / 16;  // <= 16 (mla_model_create checks)
        const int tiles = nt <= 4 ? 4 : nt <= 8 ? 8 : nt <= 12 ? 12 : 16;
        // d_pad <= 512: one chunk of two k-steps per wave; <= 1024: two
        const int kc = m.d_pad / 32 <= 2 * kWaves ? 1 : 2;
#define MLA_QKV(KC, NT)                                                                         \
    hipLaunchKernelGGL((qkv_kernel<KC, NT>), grid, dim3(64 * kWaves), lds, st, s, w, pool)
        if (kc == 1) {
            if (tiles == 4) MLA_QKV(1, 4); else if (tiles == 8) MLA_QKV(1, 8);
            else if (tiles == 12) MLA_QKV(1, 12); else MLA_QKV(1, 16);
        } else {
            if (tiles == 4) MLA_QKV(2, 4); else if (tiles == 8) MLA_QKV(2, 8);
            else if (tiles == 12) MLA_QKV(2, 12); else MLA_QKV(2, 16);
        }
#undef MLA_QKV
        return hipGetLastError();
    }
    const int chunks = ceil_div(s.B, 16);
    const int tiles = (m.q_pad + m.kvw_pad) / 16;
    MLA_KW4_DISPATCH(kw_variant(ceil_div(m.d_pad / 32, kWaves)), g1_kernel,
                     dim3(round_up_to(tiles, kXcds), chunks), dim3(64 * kWaves), 0, st, s, w);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return e;
    MLA_KW_DISPATCH(kw_variant(m.q_pad / 32), g2_kernel, dim3(round_up_to(m.H + 1, kXcds), chunks),
                    dim3(64 * kG2Waves), 0, st, s, w, pool);
    return hipGetLastError();
}

hipError_t launch_layer_post(const StepArgs& s, const LayerWeights& w, const float* next_norm,
                             const LayerWeights* next, hipStream_t st) {
    const ModelDims& m = s.dims;
    const int chunks = ceil_div(s.B, 16), d_tiles = m.d_pad / 16;
    MLA_KW_DISPATCH(kw_variant(ceil_div(m.ctx_pad / 32, kWaves)), g4_kernel,
                    dim3(d_tiles, chunks), dim3(64 * kWaves), 0, st, s, w);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return e;
    MLA_KW4_DISPATCH(kw_variant(ceil_div(m.d_pad / 32, kWaves)), g5_kernel,
                     dim3(round_up_to(m.ff_pad / 16, kXcds), chunks), dim3(64 * kWaves), 0, st, s,
                     w);  // columns padded: see l2_prefetch
    e = hipGetLastError();
    if (e != hipSuccess)
        return e;
    MLA_KW_DISPATCH(kw_variant(ceil_div(m.ff_pad / 32, kWaves)), g6_kernel,
                    dim3(d_tiles, chunks), dim3(64 * kWaves), 0, st, s, w, next_norm,
                    next ? next->w_dq_dkv : nullptr, next ? next->w_uq : nullptr,
                    next ? next->w_uk : nullptr);
    return hipGetLastError();
}

hipError_t launch_gather_last(const StepArgs& s, int B, const int32_t* cu_q, uint16_t* xw_out,
                              float* ss_out, hipStream_t st) {
    hipLaunchKernelGGL(gather_last_kernel, dim3((B + 63) / 64 * 64), dim3(256), 0, st, s, B, cu_q,
                       xw_out, ss_out);
    return hipGetLastError();
}

hipError_t launch_logits(const StepArgs& s, hipStream_t st) {
    const ModelDims& m = s.dims;
    const int parts = g7_parts(m);
    const int kw = kw_variant(ceil_div(m.d_pad / 32, kG7KG)), chunks = ceil_div(s.B, 64);
    // g7_kernel up to two rounds of one workgroup a CU.  A step, one layer, us (g7_kernel /
    // g7_rows_kernel): 500 workgroups (128 rows of 16000 tokens, d_model 512) 53.0 / 53.3, 750
    // (129 rows) 60.5 / 54.9, 782 (1 row of 50000) 58.0 / 55.4; below, 32 (256 rows of 500)
    // 49.7 / 56.9.
    const dim3 rows_grid(round_up_to(ceil_div(parts, kG7RowsWaves), kXcds), chunks);
    if (parts * chunks <= 512)
        MLA_KW4_DISPATCH(kw, g7_kernel, dim3(parts, chunks), dim3(64 * kWaves), 0, st, s)
    else if (kw == 1)
        hipLaunchKernelGGL(g7_rows_kernel<1>, rows_grid, dim3(64 * kG7RowsWaves), 0, st, s, parts);
    else if (kw == 2)
        hipLaunchKernelGGL(g7_rows_kernel<2>, rows_grid, dim3(64 * kG7RowsWaves), 0, st, s, parts);
    else  // three buffers spill: a third step counts as a third and an empty fourth
        hipLaunchKernelGGL(g7_rows_kernel<4>, rows_grid, dim3(64 * kG7RowsWaves), 0, st, s, parts);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return e;
    if (s.B > 0)
        hipLaunchKernelGGL(argmax_kernel, dim3(s.B), dim3(256), 0, st, s, parts);
    return hipGetLastError();
}

}  // namespace mla
