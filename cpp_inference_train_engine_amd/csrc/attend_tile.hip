// (c) Absorbed MLA attention over tiled page records of any shape, gfx950: decode and
// chunked prefill for the architectures outside the page kernels (decode.hip, prefill.hip)
// and the wide kernel (decode_wide.hip): any head count, kv_rank % 32 == 0 up to 512,
// rope_dim % 8 == 0 up to 64, page_size % 16 == 0.
//
// Same math as decode_page_kernel and prefill_page_kernel (src/infer/inference.cpp:116-153;
// src/model/ops.cpp:109-142), with the probabilities in 22 bits (fp16) or 24 (bf16): the other
// route of these shapes, the portable kernels, keeps them in fp32.
//
// attend_tile_kernel -- a workgroup of 4 waves owns QT 16-row tiles of q-rows: 16 QT heads of
//   one query (decode; one work item of the split-K list), or 16 QT consecutive (query, head)
//   rows of one session's chunk (prefill).  Every wave holds all of the rows' Q^T operands in
//   registers and streams every 4th 32-token unit of the key range through its own LDS slot:
//   two 16-token tiles, each one contiguous latent run and one rope run of a page record,
//   copied as stored (global_load_lds_dwordx4; the tiles may lie on different pages, so any
//   page size that is a multiple of 16 works).  Per unit and row tile
//     S^T = K . Q^T     v_mfma_f32_16x16x32, K read from LDS as stored
//     online softmax    log2 domain, the reference max raised lazily
//     O^T += C^T . P^T  C^T through the transpose read ds_read_b64_tr_b16; P^T enters as the
//                       sum of 16-bit parts that together hold its 22 (fp16: 2 parts) or 24
//                       (bf16: 3 parts) bits
//   The waves' states meet in LDS once at the end.
// A key beyond a row's position, or of weight zero, adds nothing to the row, whatever its latent
// holds, as in the portable kernels.  The product adds 0 times the latent, so an infinite or NaN
// latent is zeroed in the slot first.  Such a latent makes the key's score non-finite in every row:
// a row that sees the key is NaN through its probability, or weighs it 0 (a score of -inf).
// One slot per wave and no second buffer: five, three and two workgroups fit a CU's LDS at kv_rank
// up to 64, 128 and 256, so that other waves' copies are in flight while one computes, and a second
// buffer would halve that count; above 256 one workgroup fits, whose four waves have only each other.
// What bounds it: the latency of the copies, and for wide kv_rank the LDS reads (each row tile
// reads the unit twice).  The portable kernels it replaces for these shapes are bound by 2-byte
// loads and serial VALU sums.  Measured, us against the portable kernels', and the error against 64
// bits (portable in brackets): decode with merge, 32 sessions of ~1.8k tokens: 32 heads, kv_rank
// 256, rope 32, 32-token pages, bf16 31.7 (1.03 TB/s) against 1543, 2.4e-7 (2.9e-7); 16 heads,
// kv_rank 512, rope 64, bf16 61.7 against 1655, 3.6e-7 (4.8e-7), fp16 58.5 against 1526, 4.0e-7
// (8.7e-7).  4 chunks of 129 tokens on contexts up to 1000, 16 heads: kv_rank 64, rope 16, fp16 15.5
// (62 TFLOP/s) against 839, 1.7e-7 (3.5e-7); kv_rank 512, rope 64, bf16 101 against 4843, 3.8e-7
// (5.2e-7).  Over kv_rank 32 to 512 and 2 to 1000 keys the error lies between 0.25 and 1.0 times
// the portable kernels', but for 2 to 4 keys at kv_rank 32 (7.6e-8, 6.6e-8); a third fp16 part
// changes none of these.
#include "mla_common.hpp"
#include "mla_internal.hpp"

#include <cmath>
#include <type_traits>

namespace mla {
namespace {

constexpr int kTileWaves = 4;
// Rows of odd 256-byte sub-chunks of a latent block sit at slot row ^ kTileRot in LDS, so that
// the transpose reads of a sub-chunk pair fall in disjoint banks (see decode_wide_kernel).
constexpr int kTileRot = 12;
// The reference max sits kTileHead below the row's max when it is set, and is raised again
// when a score passes it by more than kTileRise: probabilities are at most 2^kTileRise (within
// fp16), and at least 2^kTileHead at the max, so that the fp16 parts of the small ones do not
// fall among its subnormals.
constexpr float kTileHead = 6.0f, kTileRise = 14.0f;

__device__ __forceinline__ float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }

__device__ __forceinline__ u32x2 lds_read_tr16(const uint16_t* p) {
    typedef short s4 __attribute__((ext_vector_type(4)));
    const auto v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (s4 __attribute__((address_space(3)))*)((__attribute__((address_space(3))) char*)p));
    return __builtin_bit_cast(u32x2, v);
}

// KSM: latent k-steps (kv_rank / 32 <= KSM); QT: 16-row tiles; Args: DecodeArgs (grid: work
// items, row-tile groups of the heads) or PrefillArgs (grid: row blocks of the longest chunk,
// sessions).
template <typename T, int KSM, int QT, typename Args>
__global__ __launch_bounds__(64 * kTileWaves) __attribute__((amdgpu_waves_per_eu(
    KSM >= 16 ? 1 : 2, 8))) void attend_tile_kernel(Args a) {
    constexpr bool PREFILL = std::is_same_v<Args, PrefillArgs>;
    constexpr int RSM = 2;                          // rope k-steps (rope_dim <= 64)
    constexpr int NP = T::split_p ? 3 : 2;          // 16-bit parts of a probability
    constexpr int RTM = 2 * KSM;                    // 16-row latent tiles of O^T
    constexpr int SLOT = 32 * (32 * KSM + 32 * RSM);  // words of a wave's slot
    constexpr int THREADS = 64 * kTileWaves;
    using V8 = typename T::vec8;
    __shared__ __attribute__((aligned(16))) uint16_t slots[kTileWaves][SLOT];

    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, n = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int H = a.H, KV = a.kv_rank, RP = a.rope_dim, PS = a.page_size;
    const int ks = KV >> 5, rs = (RP + 31) >> 5, tpp = PS >> 4;

    // ---- the workgroup's rows and key range ----
    int s, n_rows, k_len, tile_begin, key_end, ctx = 0, ns = 1, rb = 0, h0 = 0, slot = 0;
    long long f0;  // flat (row, head) index of its first row
    if constexpr (PREFILL) {
        s = blockIdx.y;
        if (a.info[0] <= 0)
            return;  // failed metadata build (or an empty batch)
        const int q0 = a.cu_q[s], q_len = a.cu_q[s + 1] - q0;
        k_len = a.cu_k[s + 1] - a.cu_k[s];
        rb = (gridDim.x - 1 - blockIdx.x) * (16 * QT);  // later queries see more keys: first
        const int rows = min(q_len, a.max_q_len) * H;
        if (q_len < 2 || rb >= rows)
            return;
        n_rows = min(16 * QT, rows - rb);
        ctx = k_len - q_len;
        tile_begin = 0;
        key_end = ctx + (rb + n_rows - 1) / H + 1;
        f0 = (long long)q0 * H + rb;
    } else {
        // block -> (item, row-tile group): the groups of an item are 8 blocks apart, so they
        // run on one XCD and close in time, and all but one read the pages from its L2
        const int groups = (H + 16 * QT - 1) / (16 * QT);
        const int w = blockIdx.x / (8 * groups) * 8 + blockIdx.x % 8;
        if (w >= a.max_work)
            return;
        const int32_t* d = a.work_desc + (long long)w * kWorkDescInts;
        s = d[0];
        if (s < 0 || d[7] != 1)
            return;  // an empty slot, or not a decode row
        h0 = blockIdx.x / 8 % groups * (16 * QT);
        n_rows = min(16 * QT, H - h0);
        k_len = d[2];
        tile_begin = d[3] * tpp;
        key_end = min(k_len, d[4] * PS);
        ns = d[5];
        slot = d[6];
        f0 = (long long)d[1] * H + h0;
    }
    const int32_t* ptab = a.page_table + (long long)s * a.max_pages;
    const long long rec = (long long)PS * (KV + RP);
    const int n_units = (key_end - 16 * tile_begin + 31) >> 5;

    // ---- Q^T operands: row 16q + n, latent columns 32j + 8g .., then the rope key's ----
    V8 qv[QT][KSM + RSM];
    int lim[QT];  // lane's row n sees keys [0, lim]
#pragma unroll
    for (int q = 0; q < QT; ++q) {
        const int r = 16 * q + n;
        const bool ok = r < n_rows;
        const long long fr = f0 + r;
        lim[q] = PREFILL ? ctx + (rb + r) / H : k_len - 1;
#pragma unroll
        for (int j = 0; j < KSM; ++j)
            qv[q][j] = ok && j < ks
                           ? *reinterpret_cast<const V8*>(a.q_latent + fr * KV + 32 * j + 8 * g)
                           : V8{};
#pragma unroll
        for (int j = 0; j < RSM; ++j)
            qv[q][KSM + j] = ok && 32 * j + 8 * g < RP
                                 ? *reinterpret_cast<const V8*>(a.q_rope + fr * RP + 32 * j + 8 * g)
                                 : V8{};
    }

    // ---- a unit's copies into this wave's slot: tile t's latent, then the rope of both ----
    uint16_t* const sp = slots[wave];
    const uint32_t sp_lds = lds_u32(sp);
    const uint32_t lat_off =
        2 * ((lane >> 4) * 128 + ((lane & 15) ^ (((lane >> 4) & 1) * kTileRot)) * 8);
    // The page id of tile t (-1 past the keys); ids outside the pool are skipped like it.
    auto tile_page = [&](int t) {
        return 16 * t < key_end ? __builtin_amdgcn_readfirstlane(ptab[t / tpp]) : -1;
    };
    auto copy_tile = [&](int tt, int t, int page) {
        const uint16_t* base = a.pages + page * rec;
        const uint16_t* lat = base + (long long)(t % tpp) * 16 * KV;
        const uint32_t dst = sp_lds + tt * 32 * KV;
        int k = 0;
        for (; k + 4 <= ks; k += 4)
            copy_4blocks_to_lds_at(lat + k * 512, lat_off, dst + k * 1024);
        for (; k < ks; ++k)
            copy_block_to_lds_at(lat + k * 512, lat_off, dst + k * 1024);
        const uint16_t* key = base + (long long)PS * KV + (long long)(t % tpp) * 16 * RP;
        for (int b = 0; b < 32 * RP; b += 1024)
            if (b + 16 * lane < 32 * RP)
                copy_block_to_lds_at(key + b / 2, 16 * lane, sp_lds + 64 * KV + tt * 32 * RP + b);
    };
    // Tokens [valid, 16) of tile tt read as zero (their stored bits may be anything).
    auto clear_tile = [&](int tt, int valid) {
        const u32x4 zero = {0, 0, 0, 0};
        for (int k = 0; k < ks; ++k)
            if ((n ^ ((g & 1) * kTileRot)) >= valid)
                *reinterpret_cast<u32x4*>(sp + tt * 16 * KV + k * 512 + lane * 8) = zero;
        for (int c = lane; c < 2 * RP; c += 64)
            if ((c & 15) >= valid)
                *reinterpret_cast<u32x4*>(sp + 32 * KV + tt * 16 * RP + c * 8) = zero;
    };

    // Infinite and NaN latents of the unit become 0 (its scores have been computed).
    auto drop_nonfinite = [&]() {
        constexpr uint32_t kExp = T::exp_mask;
#pragma unroll 1
        for (int k = 0; k < 2 * ks; ++k) {  // both tiles' 512-word blocks are contiguous
            u32x4* p = reinterpret_cast<u32x4*>(sp + k * 512 + lane * 8);
            u32x4 v = *p;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if ((v[e] & kExp) == kExp)
                    v[e] &= 0xffff0000u;
                if (((v[e] >> 16) & kExp) == kExp)
                    v[e] &= 0x0000ffffu;
            }
            *p = v;
        }
        wave_lds_fence();
    };

    const int s_lane = g * 128 + (n ^ ((g & 1) * kTileRot)) * 8;
    const int tr_par = (n & 3) >> 1;
    const int tr_lane = tr_par * 128 + ((4 * g + (n >> 2)) ^ (tr_par * kTileRot)) * 8 + 4 * (n & 1);
    int rope_off[RSM];  // lanes past the rope columns read a valid chunk (their Q^T is zero)
#pragma unroll
    for (int j = 0; j < RSM; ++j)
        rope_off[j] = (32 * j + 8 * g < RP ? 4 * j + g : 0) * 128 + n * 8;

    float m_run[QT], l_run[QT];
    floatx4 acc[QT][RTM];
#pragma unroll
    for (int q = 0; q < QT; ++q) {
        m_run[q] = -INFINITY;
        l_run[q] = 0.0f;
#pragma unroll
        for (int rt = 0; rt < RTM; ++rt)
            acc[q][rt] = floatx4{0, 0, 0, 0};
    }

    int pg0 = 0, pg1 = 0;  // pages of the next unit's tiles, fetched a unit ahead
    if (wave < n_units) {
        pg0 = tile_page(tile_begin + 2 * wave);
        pg1 = tile_page(tile_begin + 2 * wave + 1);
    }
    for (int u = wave; u < n_units; u += kTileWaves) {
        const int t0 = tile_begin + 2 * u;
        const bool ok0 = (unsigned)pg0 < (unsigned)a.num_pool_pages;
        const bool ok1 = (unsigned)pg1 < (unsigned)a.num_pool_pages;
        if (ok0)
            copy_tile(0, t0, pg0);
        if (ok1)
            copy_tile(1, t0 + 1, pg1);
        if (u + kTileWaves < n_units) {
            pg0 = tile_page(t0 + 2 * kTileWaves);
            pg1 = tile_page(t0 + 2 * kTileWaves + 1);
        }
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the unit (and Q^T) landed
        wave_lds_fence();
        const int valid0 = ok0 ? min(16, k_len - 16 * t0) : 0;
        const int valid1 = ok1 ? max(0, min(16, k_len - 16 * t0 - 16)) : 0;
        if (valid0 < 16 || valid1 < 16) {
            clear_tile(0, valid0);
            clear_tile(1, valid1);
            wave_lds_fence();
        }

        floatx4 sc[2][QT];
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
            for (int q = 0; q < QT; ++q)
                sc[tt][q] = floatx4{0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < KSM; ++j)
            if (j < ks)
#pragma unroll
                for (int tt = 0; tt < 2; ++tt) {
                    const V8 ka =
                        *reinterpret_cast<const V8*>(sp + tt * 16 * KV + j * 512 + s_lane);
#pragma unroll
                    for (int q = 0; q < QT; ++q)
                        sc[tt][q] = T::mma32(ka, qv[q][j], sc[tt][q]);
                }
#pragma unroll
        for (int j = 0; j < RSM; ++j)
            if (j < rs)
#pragma unroll
                for (int tt = 0; tt < 2; ++tt) {
                    const V8 ka = *reinterpret_cast<const V8*>(sp + 32 * KV + tt * 16 * RP +
                                                               rope_off[j]);
#pragma unroll
                    for (int q = 0; q < QT; ++q)
                        sc[tt][q] = T::mma32(ka, qv[q][KSM + j], sc[tt][q]);
                }

        // Not 0 when a score of the first row tile is not finite; tested once the probabilities,
        // which do not wait for it, are done.
        floatx4 odd = sc[0][0] * 0.0f + sc[1][0] * 0.0f;
        odd[0] += odd[1] + (odd[2] + odd[3]);

        V8 pb[NP][QT];
#pragma unroll
        for (int q = 0; q < QT; ++q) {
            bool rise = false;
            float mp = -INFINITY;
#pragma unroll
            for (int tt = 0; tt < 2; ++tt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int tok = 4 * g + i;
                    float x = sc[tt][q][i] * a.scale_log2;
                    if (tok >= (tt ? valid1 : valid0) || 16 * (t0 + tt) + tok > lim[q])
                        x = -INFINITY;
                    sc[tt][q][i] = x;
                    rise |= x > m_run[q] + kTileRise;
                    mp = fmaxf(mp, x);
                }
            if (__builtin_amdgcn_ballot_w64(rise)) {
                const float m_new = fmaxf(m_run[q], rows_max(mp) - kTileHead);
                const bool had = m_run[q] != -INFINITY;  // the row has accumulated state
                if (__builtin_amdgcn_ballot_w64(had && m_new > m_run[q])) {
                    const float alpha = had ? exp2_fast(m_run[q] - m_new) : 1.0f;
                    l_run[q] *= alpha;
#pragma unroll
                    for (int rt = 0; rt < RTM; ++rt)
                        acc[q][rt] *= alpha;
                }
                m_run[q] = m_new;
            }
            const float m_ref = m_run[q] == -INFINITY ? 0.0f : m_run[q];
            float psum = 0.0f;
#pragma unroll
            for (int tt = 0; tt < 2; ++tt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float e = exp2_fast(sc[tt][q][i] - m_ref);
                    psum += e;
#pragma unroll
                    for (int k = 0; k < NP; ++k) {
                        const auto part = static_cast<typename T::scalar>(e);
                        pb[k][q][4 * tt + i] = part;
                        e -= static_cast<float>(part);
                    }
                }
            l_run[q] += psum;
        }
        if (__builtin_amdgcn_ballot_w64(odd[0] != 0.0f))
            drop_nonfinite();
#pragma unroll
        for (int rt = 0; rt < RTM; ++rt)
            if (rt < 2 * ks) {
                const int blk = ((rt >> 1) * 4 + 2 * (rt & 1)) * 128;  // latent rows 16rt..
                const u32x2 lo = lds_read_tr16(sp + blk + tr_lane);
                const u32x2 hi = lds_read_tr16(sp + 16 * KV + blk + tr_lane);
                const V8 ca = __builtin_bit_cast(V8, u32x4{lo[0], lo[1], hi[0], hi[1]});
#pragma unroll
                for (int k = 0; k < NP; ++k)
#pragma unroll
                    for (int q = 0; q < QT; ++q)
                        acc[q][rt] = T::mma32(ca, pb[k][q], acc[q][rt]);
            }
        wave_lds_fence();  // the slot's reads are done before the next copy into it
    }

    // ---- the waves' states meet in LDS, one row tile at a time; normalise and store ----
    // A wave parks its tile in its own slot: 16 rows of KV + 4 floats, then m and l of the
    // rows (64 KV + 256 + 128 bytes of the slot's 64 (32 KSM + 64)).
    const int pitch = KV + 4;
#pragma unroll
    for (int q = 0; q < QT; ++q) {
        const float l = rows_sum(l_run[q]);
        float* mine = reinterpret_cast<float*>(slots[wave]);
        if (q > 0)
            __syncthreads();  // the previous tile's rows have been read
#pragma unroll
        for (int rt = 0; rt < RTM; ++rt)
            if (rt < 2 * ks)
                *reinterpret_cast<floatx4*>(mine + n * pitch + 16 * rt + 4 * g) = acc[q][rt];
        if (g == 0) {
            mine[16 * pitch + n] = m_run[q];
            mine[16 * pitch + 16 + n] = l;
        }
        __syncthreads();
        const int per_row = KV / 4;
        for (int e = tid; e < 16 * per_row; e += THREADS) {
            const int r = e / per_row, c = (e % per_row) * 4, row = 16 * q + r;
            if (row >= n_rows)
                break;
            float M = -INFINITY;
#pragma unroll
            for (int v = 0; v < kTileWaves; ++v)
                M = fmaxf(M, reinterpret_cast<const float*>(slots[v])[16 * pitch + r]);
            float L = 0.0f;
            floatx4 o = {0, 0, 0, 0};
#pragma unroll
            for (int v = 0; v < kTileWaves; ++v) {
                const float* x = reinterpret_cast<const float*>(slots[v]);
                const float mv = x[16 * pitch + r];
                const float f = mv == -INFINITY ? 0.0f : exp2_fast(mv - M);
                L += x[16 * pitch + 16 + r] * f;
                o += *reinterpret_cast<const floatx4*>(x + r * pitch + c) * f;
            }
            if (ns == 1) {
                const float inv = L > 0.0f ? 1.0f / L : 0.0f;
                store_row<false, kRowAny>(a, (f0 + row) / H, (int)((f0 + row) % H), c, o * inv);
                if (a.lse && c == 0)
                    a.lse[f0 + row] = (M + __log2f(L)) * kLn2;
            } else if constexpr (!PREFILL) {
                const long long sl = slot;
                *reinterpret_cast<floatx4*>(a.part_o + (sl * H + h0 + row) * KV + c) = o;
                if (c == 0) {
                    float* ml = a.part_ml + sl * part_ml_stride(H) + 2 * (h0 + row);
                    ml[0] = M;
                    ml[1] = L;
                }
            }
        }
    }
}

template <typename T, int KSM, int QT, typename Args>
hipError_t launch_one(const Args& a, dim3 grid, hipStream_t stream) {
    hipLaunchKernelGGL((attend_tile_kernel<T, KSM, QT, Args>), grid, dim3(64 * kTileWaves), 0,
                       stream, a);
    return hipGetLastError();
}

// Rows of a workgroup: two row tiles share each copied unit up to kv_rank 128 when there are
// rows for both.  Two tiles against one in us: large calls 131.6 / 135.6 (250 sessions of ~4k
// tokens, 32 heads, kv 128), 54.3 / 66.5 (the same, kv 32), 184 / 224 (8 chunks of 700, 16 heads,
// kv 64); calls that leave the chip idle lose, since half as many workgroups share the work: 17.0 /
// 15.3 (32 sessions of ~1.8k tokens, 32 heads, kv 128), 15.5 / 13.6 (4 chunks of 129, 16 heads, kv
// 64).  Above kv_rank 128 O^T and Q^T of two tiles exceed 256 registers (28-60 spilled), and
// the two tiles go to two workgroups that share an L2 instead: 33.4 us against 44.3 us at 32
// heads and kv_rank 256 (41.8 us with one wave per SIMD and no spills), 30.8 us once the two
// workgroups were placed on one XCD.
template <typename T, typename Args>
hipError_t launch_tile(const Args& a, long long rows, unsigned other, hipStream_t stream) {
    constexpr bool PREFILL = std::is_same_v<Args, PrefillArgs>;
    const int ks = a.kv_rank / 32;
    const int qt = ks <= 4 && rows > 16 ? 2 : 1;
    const unsigned groups = (unsigned)((rows + 16 * qt - 1) / (16 * qt));
    const dim3 grid = PREFILL ? dim3(groups, other) : dim3((other + 7) / 8 * 8 * groups);
    if (qt == 2)
        return ks <= 2 ? launch_one<T, 2, 2>(a, grid, stream)
                       : launch_one<T, 4, 2>(a, grid, stream);
    return ks <= 2   ? launch_one<T, 2, 1>(a, grid, stream)
           : ks <= 4 ? launch_one<T, 4, 1>(a, grid, stream)
           : ks <= 8 ? launch_one<T, 8, 1>(a, grid, stream)
                     : launch_one<T, 16, 1>(a, grid, stream);
}

}  // namespace

bool attend_tile_supported(int kv_rank, int rope_dim, int page_size) {
    return page_tiled(page_size, kv_rank, rope_dim) && kv_rank <= 512 && rope_dim <= 64;
}

hipError_t launch_decode_tile(const DecodeArgs& a, int dtype, hipStream_t stream) {
    return dtype == 0 ? launch_tile<F16>(a, a.H, a.max_work, stream)
                      : launch_tile<BF16>(a, a.H, a.max_work, stream);
}

hipError_t launch_prefill_tile(const PrefillArgs& a, int max_q_len, int dtype,
                               hipStream_t stream) {
    return dtype == 0 ? launch_tile<F16>(a, (long long)max_q_len * a.H, a.B, stream)
                      : launch_tile<BF16>(a, (long long)max_q_len * a.H, a.B, stream);
}

}  // namespace mla
