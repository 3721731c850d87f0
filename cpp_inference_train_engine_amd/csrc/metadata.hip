// (a) Ragged-batch metadata and (b) paged latent append, gfx950.
//
// Batches whose page table is small are built by ONE workgroup of 1024 threads in one launch
// (build_metadata_lds_kernel).  Larger ones take two: plan_metadata_kernel, one workgroup that
// validates and scans, and fill_metadata_kernel, one workgroup per session that writes its part
// of the table, the work list and the slots.  All arithmetic is int32/int64 and bit-exact with
// the CPU builder in the oracle.
#include "mla_common.hpp"
#include "mla_internal.hpp"

#include <algorithm>
#include <climits>
#include <string>
#include <vector>

namespace mla {
namespace {

constexpr int kMetaThreads = 1024;
constexpr int kMetaWaves = kMetaThreads / 64;

// One DPP move of a 64-bit value (both halves with the same control); lanes the
// control gives no source, and rows outside row_mask, receive 0.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ long long dpp64(long long v) {
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, CTRL, ROW_MASK, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), CTRL, ROW_MASK, 0xf,
                                               true);
    return (long long)(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo);
}

// Inclusive scan over the 64 lanes of a wave on DPP moves (no LDS round trips): shifts
// of 1, 2, 4, 8 lanes within each row of 16, then lane 15 of each row broadcast into
// the next row (rows 1, 3) and lane 31 into the upper half (rows 2, 3).
__device__ __forceinline__ long long wave_scan_incl(long long v) {
    v += dpp64<0x111, 0xf>(v);  // row_shr:1
    v += dpp64<0x112, 0xf>(v);  // row_shr:2
    v += dpp64<0x114, 0xf>(v);  // row_shr:4
    v += dpp64<0x118, 0xf>(v);  // row_shr:8
    v += dpp64<0x142, 0xa>(v);  // row_bcast:15
    v += dpp64<0x143, 0xc>(v);  // row_bcast:31
    return v;
}

// Inclusive block scan of N int64 values; returns the chunk totals in tot[].
template <int N>
__device__ void block_scan(long long (&v)[N], long long (&tot)[N], long long* lds) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
#pragma unroll
    for (int k = 0; k < N; ++k) {
        v[k] = wave_scan_incl(v[k]);
        if (lane == 63)
            lds[k * kMetaWaves + wave] = v[k];
    }
    __syncthreads();
    if (wave < N) {
        const long long x = wave_scan_incl(lane < kMetaWaves ? lds[wave * kMetaWaves + lane] : 0);
        if (lane < kMetaWaves)
            lds[wave * kMetaWaves + lane] = x;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < N; ++k) {
        if (wave > 0)
            v[k] += lds[k * kMetaWaves + wave - 1];
        tot[k] = lds[k * kMetaWaves + kMetaWaves - 1];
    }
    __syncthreads();
}

// Largest b in [0, n] with a[b] <= x  (a non-decreasing, a[0] <= x).
__device__ int upper_index(const int32_t* a, int n, long long x) {
    int lo = 0, hi = n;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (a[mid] <= x)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

constexpr int kMetaLdsCap = 4096;  // sessions of build_metadata_lds_kernel

__device__ void write_error_info(const MetadataArgs& a, int session) {
    if (threadIdx.x < kInfoInts)
        a.info[threadIdx.x] = threadIdx.x == 0 ? -1 : threadIdx.x == 1 ? session : 0;
}
__device__ void write_error(const MetadataArgs& a, int session) {
    for (int w = threadIdx.x; w < a.max_work; w += kMetaThreads)
        a.work_desc[(long long)w * kWorkDescInts] = -1;
    write_error_info(a, session);
}

// ceil(x / d) for x >= 0 and d >= 1, in 32-bit arithmetic when both are below 2^31.
__device__ __forceinline__ long long ceil_div_nn(long long x, long long d) {
    if (x < 0x80000000LL && d < 0x80000000LL)
        return (long long)(((uint32_t)x + (uint32_t)(d - 1)) / (uint32_t)d);
    return (x + d - 1) / d;
}

// ------------------------------------------------------------ placement ----
// XCD placement of the work list (MetadataArgs::placement = n XCDs): every session's
// items go to one XCD so that a decode kernel's items of one session share an L2 (the
// fused split merge relies on it).  Sessions are ranked by pages read, largest first
// (ties: lower session first), and dealt to the XCDs in a snake: ranks 0..n-1 to XCDs
// 0..n-1, ranks n..2n-1 to XCDs n-1..0, and so on, so each XCD takes one session per
// round of n ranks and no two XCDs' pages differ by more than the largest session's.  A
// session's items then take its XCD's next slots: item sp of the session of round q on
// XCD x lands in slot x + n * (k + sp), k the items of that XCD's sessions of rounds < q.
// There are ceil(B / n) rounds (up to 256 when n = 1); wave x takes them 64 at a time,
// one lane per round, carrying the running item count from pass to pass.

struct Placement {
    int32_t weight[kPlaceMaxSessions], order[kPlaceMaxSessions], bin[kPlaceMaxSessions],
        k0[kPlaceMaxSessions], cnt[kPlaceMaxXcds];
};

// All threads call it (B <= kPlaceMaxSessions, 1 <= n <= kPlaceMaxXcds); q(b), ctx(b) and
// cus(b) read the session inputs and the work-item prefix.  Ends with a barrier.
template <typename Q, typename C, typename S>
__device__ void place_sessions(int B, int n, int page_size, Q q, C ctx, S cus, Placement& p) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int b = tid; b < B; b += kMetaThreads)
        p.weight[b] = q(b) > 0 ? (int32_t)ceil_div_nn((long long)ctx(b) + q(b), page_size) : 0;
    __syncthreads();
    // rank by (weight desc, session asc): tps threads per session (a power of two <= 64,
    // an aligned lane group) each count every tps-th other session, then sum in the group
    int tps = 64;
    while (tps > 1 && tps * B > kMetaThreads)
        tps >>= 1;
    {
        const int b = tid / tps, part = tid % tps;
        int r = 0, wb = 0;
        if (b < B) {
            wb = p.weight[b];
            for (int c = part; c < B; c += tps) {
                const int wc = p.weight[c];
                r += wc > wb || (wc == wb && c < b);
            }
        }
        for (int off = tps >> 1; off > 0; off >>= 1)
            r += __shfl_xor(r, off, 64);
        if (b < B && part == 0)
            p.order[r] = b;
    }
    __syncthreads();
    for (int x = wave; x < n; x += kMetaWaves) {  // lane l holds XCD x's session of round q0 + l
        long long carry = 0;  // items of XCD x's sessions of earlier passes
        for (int q0 = 0; q0 * n < B; q0 += 64) {
            const int qr = q0 + lane;
            const int r = qr * n + ((qr & 1) ? n - 1 - x : x);
            const bool real = r < B;  // rounds past the last, or the last round's gaps
            const int b = real ? p.order[r] : 0;
            const long long items = real ? cus(b + 1) - cus(b) : 0;
            const long long incl = carry + wave_scan_incl(items);
            if (real) {
                p.bin[b] = x;
                p.k0[b] = (int32_t)(incl - items);
            }
            carry = __shfl(incl, 63, 64);
        }
        if (lane == 0)
            p.cnt[x] = (int32_t)carry;
    }
    __syncthreads();
}

// Slots of the placed work list: the largest item count of one XCD, times n.
__device__ __forceinline__ long long placed_slots(const Placement& p, int n) {
    int m = 0;
    for (int i = 0; i < n; ++i)
        m = max(m, p.cnt[i]);
    return (long long)m * n;
}

// ------------------------------------------------------------- larger batches ----
// One workgroup did all of this before: filling a table of 64 K entries with a division per
// entry, and a binary search per work item and row, took 69 us at 500 sessions of up to 8,192
// tokens (16 of them with 256 new rows) and 26 us at 200 placed decode sessions.  Plan and fill take
// 9.4 and 13.5 us (two scans and, placed, the deal; latency of one workgroup), and 8.5 us for one
// session of 15,626 pages (27 by one workgroup, 42 while a session had one wave and one workgroup of
// these).  Up to kMetaSmallPt entries the single launch stays (7-13 us): with room for 14,336
// entries it took 11.2 us at 64 sessions of 188 pages, against 8.2, and 20.2 at 200 placed ones of up
// to 66, against 13.5.  A host that waits for nothing pays 2.7 us for the second launch.

// One workgroup: page-id and length checks, cu_seqlens_q / k, num_splits, cu_splits and info.  On
// an error info says so, and fill_metadata_kernel empties the work list.
__global__ __launch_bounds__(kMetaThreads) void plan_metadata_kernel(MetadataArgs a) {
    __shared__ long long lds[3 * kMetaWaves];
    __shared__ int err, bad_list, bad_id;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lo = a.cu_pages[0], hi = a.cu_pages[a.B];
    if (tid == 0) {
        err = INT_MAX;
        bad_list = bad_id = 0;
        a.cu_seqlens_q[0] = a.cu_seqlens_k[0] = a.cu_splits[0] = 0;
    }
    __syncthreads();
    // Cumulative rows and keys, and the pages that sessions with new rows read.  What the later
    // phases need of the first sessions stays in registers and LDS (the page ids pass between).
    __shared__ int32_t s_q[kPlaceMaxSessions], s_ctx[kPlaceMaxSessions];
    long long first_pages = 0, total[3] = {0, 0, 0};
    for (int base = 0; base < a.B; base += kMetaThreads) {
        const int b = base + tid;
        long long v[3] = {0, 0, 0}, tot[3];
        bool bad = false;
        if (b < a.B) {
            const long long q = a.q_len[b], ctx = a.ctx_len[b], kl = ctx + q;
            const long long npages = (long long)a.cu_pages[b + 1] - a.cu_pages[b];
            const long long need = kl < 0 ? 0 : ceil_div_nn(kl, a.page_size);
            if (npages < 0 || npages > a.max_pages)
                bad_list = 1;
            bad = q < 0 || ctx < 0 || npages < 0 || npages > a.max_pages || need > npages;
            v[0] = q;
            v[1] = kl;
            v[2] = q > 0 ? need : 0;
            if (base == 0)
                first_pages = v[2];
            if (b < kPlaceMaxSessions) {
                s_q[b] = (int32_t)q;
                s_ctx[b] = (int32_t)ctx;
            }
        }
        block_scan<3>(v, tot, lds);
        if (b < a.B) {
            const long long iq = v[0] + total[0], ik = v[1] + total[1];
            if (bad || iq > INT_MAX || ik > INT_MAX || iq > a.max_rows)
                atomicMin(&err, b);
            a.cu_seqlens_q[b + 1] = (int32_t)iq;
            a.cu_seqlens_k[b + 1] = (int32_t)ik;
        }
#pragma unroll
        for (int k = 0; k < 3; ++k)
            total[k] += tot[k];
    }
    __syncthreads();
    // Page ids: consecutive lists are adjacent, so all threads check them as one flat run, kIds loads
    // of a lane in flight (wave by session, one session of 15,626 pages took 26 us more).  Only when
    // that finds a bad id, or a list is too long or negative (then only its first max_pages ids may
    // be read), each wave walks every 16th session to name the first bad one.
    constexpr int kIds = 16;
    if (!bad_list) {
        for (int e0 = lo; e0 < hi; e0 += kMetaThreads * kIds) {
            int32_t id[kIds];
#pragma unroll
            for (int k = 0; k < kIds; ++k)
                id[k] = a.page_ids[min(e0 + kMetaThreads * k + tid, hi - 1)];
            bool bad = false;
#pragma unroll
            for (int k = 0; k < kIds; ++k)
                bad |= id[k] < 0 || id[k] >= a.num_pool_pages;
            if (bad)
                bad_id = 1;
        }
    }
    __syncthreads();
    if (bad_list || bad_id)
        for (int b = wave; b < a.B; b += kMetaWaves) {
            const int first = a.cu_pages[b], count = min(a.cu_pages[b + 1] - first, a.max_pages);
            for (int j = lane; j < count; j += 64) {
                const int32_t id = a.page_ids[first + j];
                if (id < 0 || id >= a.num_pool_pages)
                    atomicMin(&err, b);
            }
        }
    __syncthreads();
    if (err != INT_MAX) {
        write_error_info(a, err);
        return;
    }
    long long split = a.split_pages;
    if (split == 0) {
        split = (total[2] + a.target_blocks - 1) / a.target_blocks;
        if (split < 1)
            split = 1;
    }
    // Split-K work items per session.
    __shared__ int32_t s_cus[kPlaceMaxSessions + 1];  // cu_splits of a batch to be placed
    if (tid == 0)
        s_cus[0] = 0;
    long long W = 0;
    for (int base = 0; base < a.B; base += kMetaThreads) {
        const int b = base + tid;
        long long v[1] = {0}, tot[1];
        if (b < a.B) {
            const long long q = base == 0 ? 0 : a.q_len[b];
            const long long pages =
                base == 0 ? first_pages : q > 0 ? ceil_div_nn(a.ctx_len[b] + q, a.page_size) : 0;
            v[0] = ceil_div_nn(pages, split);
        }
        const long long ns = v[0];
        block_scan<1>(v, tot, lds);
        if (b < a.B) {
            if (v[0] + W > a.max_work)
                atomicMin(&err, b);
            a.num_splits[b] = (int32_t)ns;
            a.cu_splits[b + 1] = (int32_t)(v[0] + W);
            if (b < kPlaceMaxSessions)
                s_cus[b + 1] = (int32_t)(v[0] + W);
        }
        W += tot[0];
    }
    __syncthreads();
    if (err != INT_MAX) {
        write_error_info(a, err);
        return;
    }
    __shared__ Placement place;
    if (a.placement > 0) {
        place_sessions(a.B, a.placement, a.page_size, [&](int b) { return s_q[b]; },
                       [&](int b) { return s_ctx[b]; }, [&](int b) { return s_cus[b]; }, place);
        if (placed_slots(place, a.placement) > a.max_work) {
            write_error_info(a, a.B);  // max_work cannot hold the placed work list
            return;
        }
        // For fill_metadata_kernel: the first slot of session b, in the first entry of its page
        // table row, which workgroup b reads before it writes the row.  The empty slots are
        // marked here, where the XCDs' counts are.
        const int n = a.placement;
        for (int b = tid; b < a.B; b += kMetaThreads)
            a.page_table[(long long)b * a.max_pages] = place.bin[b] + n * place.k0[b];
        for (int w = tid; w < a.max_work; w += kMetaThreads)
            if (w / n >= place.cnt[w % n])
                a.work_desc[(long long)w * kWorkDescInts] = -1;
    }
    if (tid < kInfoInts)
        a.info[tid] = tid == 0   ? (int32_t)W
                      : tid == 1 ? (int32_t)split
                      : tid == 2 ? (int32_t)total[0]
                      : tid == 3 ? (int32_t)total[1]
                      : tid == kInfoPlacement ? a.placement
                                              : 0;
}

// Workgroups (b < B, y) write session b's row of the page table, its work items and its slots: one
// workgroup a session where sessions are many, more for a few long ones (fill_slices).  Workgroups
// (B .., 0) mark the empty slots of a work list in session order, kFillSlots each (all slots after
// a failed plan).
constexpr int kFillThreads = 256;
constexpr int kFillSlots = 4096;

__global__ __launch_bounds__(kFillThreads) void fill_metadata_kernel(MetadataArgs a) {
    const int tid = threadIdx.x, b = blockIdx.x, y = blockIdx.y, n = a.placement;
    const int t0 = y * kFillThreads + tid, step = gridDim.y * kFillThreads;
    const int W = a.info[0];
    if (b >= a.B) {
        if (y > 0)
            return;
        const long long w0 = (long long)(b - a.B) * kFillSlots;
        for (long long w = w0 + tid; w < min(w0 + kFillSlots, (long long)a.max_work); w += kFillThreads)
            if (W < 0 || (n == 0 && w >= W))
                a.work_desc[w * kWorkDescInts] = -1;
        return;
    }
    const int first = a.cu_pages[b], listed = min(a.cu_pages[b + 1] - first, a.max_pages);
    int32_t* row = a.page_table + (long long)b * a.max_pages;
    // placed: the session's first slot, from the plan; slice 0 writes the row's first entry, so it
    // alone reads it, and writes the items
    const bool items = n == 0 || y == 0;
    const int slot0 = n > 0 && y == 0 ? row[0] : 0;
    __syncthreads();
    for (int j = t0; j < a.max_pages; j += step)
        row[j] = j < listed ? a.page_ids[first + j] : -1;
    if (W < 0)
        return;
    const int split = a.info[1], q = a.q_len[b], ctx = a.ctx_len[b], kl = ctx + q;
    const int q0 = a.cu_seqlens_q[b], u0 = a.cu_splits[b], ns = a.cu_splits[b + 1] - u0;
    const int need = (kl + a.page_size - 1) / a.page_size;
    for (int sp = n > 0 ? tid : t0; items && sp < ns; sp += n > 0 ? kFillThreads : step) {
        const int u = u0 + sp;
        const long long w = n > 0 ? slot0 + (long long)n * sp : u;
        int32_t* d = a.work_desc + w * kWorkDescInts;
        int32_t* pg = a.work_pages + w * kWorkPages;
        const int p0 = sp * split, p1 = min(need - p0, split) + p0;  // p0 < need
        a.work_session[w] = b;
        a.work_split[w] = sp;
        d[0] = b;
        d[1] = q0;
        d[2] = kl;
        d[3] = p0;
        d[4] = p1;
        d[5] = ns;
        d[6] = u;
        d[7] = q;
#pragma unroll
        for (int j = 0; j < kWorkPages; ++j)
            pg[j] = p0 + j < p1 ? a.page_ids[first + p0 + j] : -1;
    }
    for (int i = t0; i < q; i += step) {
        const int pos = ctx + i;
        a.slot_mapping[q0 + i] = (int32_t)(a.page_ids[first + pos / a.page_size] *
                                               (long long)a.page_size +
                                           pos % a.page_size);
    }
}

// The build for batches whose session arrays and padded page table fit in LDS
// (B <= kMetaLdsCap, B * max_pages <= kMetaSmallPt).  All waves stage the inputs and the
// page ids in LDS (one load round trip each); wave 0 alone runs both scans, 64 sessions
// per pass with the running total carried between passes (a 6-step wave scan instead of
// a 1024-thread block scan, whose 64-bit shuffles and barriers cost microseconds); then
// all waves write every output, with no global store before the last barrier.  A valid batch's
// outputs are bit-identical to those of plan_metadata_kernel and fill_metadata_kernel; of a rejected
// one, info and the emptied work list are (those two also leave a page table and cumulative
// lengths, which nothing reads then).
constexpr int kMetaSmallPt = 8192;

__global__ __launch_bounds__(kMetaThreads) void build_metadata_lds_kernel(MetadataArgs a) {
    __shared__ int32_t s_cup[kMetaLdsCap + 1], s_q[kMetaLdsCap], s_ctx[kMetaLdsCap];
    __shared__ int32_t s_cuq[kMetaLdsCap + 1], s_cuk[kMetaLdsCap + 1], s_cus[kMetaLdsCap + 1];
    __shared__ int32_t s_pt[kMetaSmallPt];
    __shared__ int err;
    __shared__ long long s_tot[4];  // total_q, total_k, split, W
    const int tid = threadIdx.x, lane = tid & 63, B = a.B, mp = a.max_pages;
    const int entries = B * mp;  // <= kMetaSmallPt
    // ---- inputs to LDS ----
    for (int b = tid; b <= B; b += kMetaThreads) {
        s_cup[b] = a.cu_pages[b];
        if (b < B) {
            s_q[b] = a.q_len[b];
            s_ctx[b] = a.ctx_len[b];
        }
    }
    if (tid == 0) {
        err = INT_MAX;
        s_cuq[0] = s_cuk[0] = s_cus[0] = 0;
    }
    __syncthreads();
    // ---- padded page table in LDS; ids out of the pool name their session ----
    {
        constexpr int U = kMetaSmallPt / kMetaThreads;
        int32_t pid[U];
        int bad_b = INT_MAX;
#pragma unroll
        for (int k = 0; k < U; ++k) {
            const int e = tid + k * kMetaThreads;
            const int b = e < entries ? (int)((uint32_t)e / (uint32_t)mp) : 0;
            const int j = e - b * mp;
            const int p0 = s_cup[b], np = s_cup[b + 1] - p0;
            const bool listed = e < entries && j < np;
            pid[k] = listed ? a.page_ids[p0 + j] : -1;
            if (listed && (pid[k] < 0 || pid[k] >= a.num_pool_pages))
                bad_b = min(bad_b, b);
        }
#pragma unroll
        for (int k = 0; k < U; ++k) {
            const int e = tid + k * kMetaThreads;
            if (e < entries)
                s_pt[e] = pid[k];
        }
        if (bad_b != INT_MAX)
            atomicMin(&err, bad_b);
    }
    __syncthreads();
    // ---- wave 0: cumulative rows / keys / pages, then work items per session ----
    if (tid < 64) {
        long long cq = 0, ck = 0, cp = 0;
        int bad = INT_MAX;
        for (int base = 0; base < B; base += 64) {
            const int b = base + lane;
            long long q = 0, kl = 0, pages = 0;
            if (b < B) {
                q = s_q[b];
                const long long ctx = s_ctx[b];
                const long long npages = (long long)s_cup[b + 1] - s_cup[b];
                kl = ctx + q;
                const long long need = kl < 0 ? 0 : ceil_div_nn(kl, a.page_size);
                if (q < 0 || ctx < 0 || npages < 0 || npages > mp || need > npages)
                    bad = min(bad, b);
                pages = q > 0 ? need : 0;
            }
            const long long iq = cq + wave_scan_incl(q), ik = ck + wave_scan_incl(kl);
            const long long ip = cp + wave_scan_incl(pages);
            if (b < B) {
                if (iq > INT_MAX || ik > INT_MAX || iq > a.max_rows)
                    bad = min(bad, b);
                s_cuq[b + 1] = (int32_t)iq;
                s_cuk[b + 1] = (int32_t)ik;
            }
            cq = __shfl(iq, 63, 64);
            ck = __shfl(ik, 63, 64);
            cp = __shfl(ip, 63, 64);
        }
        long long split = a.split_pages;
        if (split == 0) {
            split = (cp + a.target_blocks - 1) / a.target_blocks;
            if (split < 1)
                split = 1;
        }
        long long cw = 0;
        for (int base = 0; base < B; base += 64) {
            const int b = base + lane;
            long long ns = 0;
            if (b < B && s_q[b] > 0)
                ns = ceil_div_nn(ceil_div_nn((long long)s_ctx[b] + s_q[b], a.page_size), split);
            const long long iw = cw + wave_scan_incl(ns);
            if (b < B) {
                if (iw > a.max_work)
                    bad = min(bad, B + b);  // reported only when the first scan found nothing
                s_cus[b + 1] = (int32_t)iw;
            }
            cw = __shfl(iw, 63, 64);
        }
        // First offending session: the row/key/page checks outrank the work-item one.
        for (int off = 32; off > 0; off >>= 1)
            bad = min(bad, __shfl_xor(bad, off, 64));
        if (lane == 0) {
            if (bad != INT_MAX)
                atomicMin(&err, bad >= B ? bad - B + (1 << 30) : bad);
            s_tot[0] = cq;
            s_tot[1] = ck;
            s_tot[2] = split;
            s_tot[3] = cw;
        }
    }
    __syncthreads();
    if (err != INT_MAX) {
        write_error(a, err >= (1 << 30) ? err - (1 << 30) : err);
        return;
    }
    const long long total_q = s_tot[0], total_k = s_tot[1], split = s_tot[2];
    const int W = (int)s_tot[3];
    __shared__ Placement place;
    if (a.placement > 0) {
        place_sessions(B, a.placement, a.page_size, [&](int b) { return s_q[b]; },
                       [&](int b) { return s_ctx[b]; }, [&](int b) { return s_cus[b]; }, place);
        if (placed_slots(place, a.placement) > a.max_work) {
            write_error(a, B);  // max_work cannot hold the placed work list
            return;
        }
    }
    // ---- outputs: global stores only from here on ----
    for (int b = tid; b <= B; b += kMetaThreads) {
        a.cu_seqlens_q[b] = s_cuq[b];
        a.cu_seqlens_k[b] = s_cuk[b];
        a.cu_splits[b] = s_cus[b];
        if (b < B)
            a.num_splits[b] = s_cus[b + 1] - s_cus[b];
    }
    for (int e = tid; e < entries; e += kMetaThreads)
        a.page_table[e] = s_pt[e];
    typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
    const int n = a.placement;
    for (int w = tid; w < a.max_work; w += kMetaThreads) {
        const bool empty = n > 0 ? w / n >= place.cnt[w % n] : w >= W;
        if (empty)
            a.work_desc[(long long)w * kWorkDescInts] = -1;
    }
    for (int u = tid; u < W; u += kMetaThreads) {
        const int b = upper_index(s_cus, B, u);
        const int sp = u - s_cus[b];
        const int w = n > 0 ? place.bin[b] + n * (place.k0[b] + sp) : u;
        const int q = s_q[b], kl = s_ctx[b] + q;
        const int need = (kl + a.page_size - 1) / a.page_size;
        const int p0 = (int)(sp * split);
        const int p1 = (int)(p0 + split < need ? p0 + split : need);
        a.work_session[w] = b;
        a.work_split[w] = sp;
        i32x4* d = reinterpret_cast<i32x4*>(a.work_desc + (long long)w * kWorkDescInts);
        d[0] = i32x4{b, s_cuq[b], kl, p0};
        d[1] = i32x4{p1, s_cus[b + 1] - s_cus[b], u, q};
        int32_t pg[kWorkPages];
#pragma unroll
        for (int j = 0; j < kWorkPages; ++j)
            pg[j] = p0 + j < p1 ? s_pt[b * mp + p0 + j] : -1;
        i32x4* dp = reinterpret_cast<i32x4*>(a.work_pages + (long long)w * kWorkPages);
        dp[0] = i32x4{pg[0], pg[1], pg[2], pg[3]};
        dp[1] = i32x4{pg[4], pg[5], pg[6], pg[7]};
    }
    for (int i = tid; i < (int)total_q; i += kMetaThreads) {
        const int b = upper_index(s_cuq, B, i);
        const int pos = s_ctx[b] + (i - s_cuq[b]);
        const int page = s_pt[b * mp + pos / a.page_size];
        a.slot_mapping[i] = (int32_t)(page * (long long)a.page_size + pos % a.page_size);
    }
    if (tid == 0) {
        a.info[0] = W;
        a.info[1] = (int32_t)split;
        a.info[2] = (int32_t)total_q;
        a.info[3] = (int32_t)total_k;
        a.info[kInfoPlacement] = n;
        for (int k = kInfoPlacement + 1; k < kInfoInts; ++k)
            a.info[k] = 0;
    }
}

// One thread per element of the appended rows; RNE rounding to 16 bits.
template <typename T>
__global__ __launch_bounds__(256) void append_kernel(AppendArgs a) {
    const int width = a.kv_rank + a.rope_dim;
    const long long total = (long long)a.T * width;
    const long long rec = (long long)a.page_size * width;
    const bool tiled = page_tiled(a.page_size, a.kv_rank, a.rope_dim);
    for (long long e = blockIdx.x * 256LL + threadIdx.x; e < total; e += 256LL * gridDim.x) {
        const int t = (int)(e / width), c = (int)(e % width);
        const int slot = a.slot_mapping[t];
        const int page = slot / a.page_size, off = slot % a.page_size;
        if (slot < 0 || page >= a.num_pool_pages)
            continue;
        uint16_t* base = a.pages + page * rec;
        if (c < a.kv_rank)
            base[latent_word(tiled, off, c, a.page_size, a.kv_rank)] =
                T::from_float(a.ckv[(long long)t * a.kv_rank + c]);
        else {
            const int j = c - a.kv_rank;
            base[rope_word(tiled, off, j, a.page_size, a.kv_rank, a.rope_dim)] =
                T::from_float(a.krope[(long long)t * a.rope_dim + j]);
        }
    }
}

}  // namespace

int metadata_launches(int B, int max_pages) {
    return B <= kMetaLdsCap && (long long)B * max_pages <= kMetaSmallPt ? 1 : 2;
}

// Workgroups of a session: about one a CU in all, with 4 rows or table entries a thread or more.
static int fill_slices(const MetadataArgs& a) {
    const int most = std::max(a.max_pages, a.max_rows) / (4 * kFillThreads) + 1;
    return std::max(1, std::min(256 / a.B, most));
}

hipError_t launch_build_metadata(const MetadataArgs& a, hipStream_t stream) {
    if (metadata_launches(a.B, a.max_pages) == 1)
        hipLaunchKernelGGL(build_metadata_lds_kernel, dim3(1), dim3(kMetaThreads), 0, stream, a);
    else {
        hipLaunchKernelGGL(plan_metadata_kernel, dim3(1), dim3(kMetaThreads), 0, stream, a);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess)
            return e;
        const int marks = (a.max_work + kFillSlots - 1) / kFillSlots;
        hipLaunchKernelGGL(fill_metadata_kernel, dim3(a.B + marks, fill_slices(a)),
                           dim3(kFillThreads), 0, stream, a);
    }
    return hipGetLastError();
}

// XCD of each workgroup of a launch (the XCC_ID hardware register), for the placement probe.
__global__ __launch_bounds__(64) void xcd_probe_kernel(int32_t* out) {
    if (threadIdx.x == 0) {
        unsigned x;
        asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID, 0, 4)" : "=s"(x));
        out[blockIdx.x] = (int32_t)x;
    }
}

int xcd_count() {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&n, hipDeviceAttributeNumberOfXccs, dev) != hipSuccess || n < 1)
        return 0;
    return n;
}

// Whether the workgroups w of a launch with one residue w % n run on one XCD, and the n
// residues on n different XCDs, on the current device: ids of 16 rounds of n workgroups,
// launched twice.  Empty string when it holds, else the reason.  (Which XCD takes
// residue 0 differs between hardware queues: each queue starts its round-robin on an XCD
// of its own, which placement does not depend on.)
std::string probe_xcd_placement() {
    const int n = xcd_count();
    if (n < 1 || n > kPlaceMaxXcds)
        return "XCD count " + std::to_string(n) + " outside 1.." + std::to_string(kPlaceMaxXcds);
    const int G = 16 * n;
    int32_t* d = nullptr;
    std::vector<int32_t> h(G);
    std::string why;
    if (hipMalloc(&d, G * sizeof(int32_t)) != hipSuccess)
        return "probe allocation failed";
    for (int rep = 0; rep < 2 && why.empty(); ++rep) {
        hipLaunchKernelGGL(xcd_probe_kernel, dim3(G), dim3(64), 0, nullptr, d);
        if (hipMemcpy(h.data(), d, G * sizeof(int32_t), hipMemcpyDeviceToHost) != hipSuccess) {
            why = "probe launch failed";
            break;
        }
        for (int w = 0; w < G && why.empty(); ++w)
            if (h[w] != h[w % n] || (w < n && std::count(h.begin(), h.begin() + n, h[w]) != 1) ||
                h[w] < 0 || h[w] > 15)
                why = "workgroup " + std::to_string(w) + " ran on XCD " + std::to_string(h[w]);
    }
    (void)hipFree(d);
    return why;
}

hipError_t launch_append(const AppendArgs& a, int dtype, hipStream_t stream) {
    const long long total = (long long)a.T * (a.kv_rank + a.rope_dim);
    if (total == 0)
        return hipSuccess;
    const int blocks = (int)((total + 255) / 256 < 4096 ? (total + 255) / 256 : 4096);
    if (dtype == 0)
        hipLaunchKernelGGL(append_kernel<F16>, dim3(blocks), dim3(256), 0, stream, a);
    else
        hipLaunchKernelGGL(append_kernel<BF16>, dim3(blocks), dim3(256), 0, stream, a);
    return hipGetLastError();
}

}  // namespace mla
