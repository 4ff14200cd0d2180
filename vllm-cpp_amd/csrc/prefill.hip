// prefill.hip -- the chunked causal prefill kernel: one workgroup per
// (query tile, chunk, kv head / head group), the work of prefill_tile
// (prefill_body.h).
#include "prefill_body.h"
#include "prefill_wide.h"
#include "profile.h"

#include <cstdlib>

namespace vcpp {

namespace {

// Workgroups are dealt to the 8 XCDs round-robin by linear id; remap so that
// each XCD walks a contiguous range of (tile, head group, chunk, kv head) ids
// and its L2 holds the K/V of the (chunk, kv head) pair it is serving.  slots: the
// workgroups one CU holds at once (a grid of at most slots per CU pairs the
// k-th heaviest tile of an XCD's share with its k-th lightest on one CU).
__device__ __forceinline__ void remap_ids(const PrefillParams& p, int slots, int& bx, int& by, int& bz) {
    bx = blockIdx.x, by = blockIdx.y, bz = blockIdx.z;
    const int nx = gridDim.x, ny = gridDim.y;
    const int total = nx * ny * gridDim.z;
    const int C = p.xcd_cus;  // CUs per XCD
    if ((total & 7) == 0) {
        const int lin = bx + nx * (by + ny * bz);
        const int per = total >> 3;  // ids per XCD
        int j = lin >> 3;            // dispatch order within the XCD
#ifndef VCPP_PF_NO_PAIRING
        // A grid that fits the GPU in one round (at most two workgroups per
        // CU): the dispatcher gives each CU of an XCD one workgroup before it
        // gives any a second, so local ids j and j + C (C CUs per XCD) share
        // a CU.  Reversing the order of the second ones puts the k-th
        // heaviest tile beside the k-th lightest of the XCD's share.
        // (Grids of several rounds keep heaviest-first order.)
        if (slots == 2 && C > 0 && per > C && per <= 2 * C && j >= C) j = per + C - 1 - j;
#endif
        // m = tile + nx (head group + HG (chunk + ny (kv head, key part))):
        // an XCD's consecutive ids are the tiles of both head groups of one
        // (chunk, kv head), which read the same K/V pages, so its L2 serves
        // them to all of its concurrently running workgroups.
        const int m = (lin & 7) * per + j;
        const int HG = p.head_groups;
        bx = m % nx;
        int r = m / nx;
        const int hg = r % HG;
        r /= HG;
        by = r % ny;
        bz = (r / ny) * HG + hg;
    }
}

// Small grids (prefill_live): workgroups placed by the chunks' real lengths,
// which the host does not know, the heaviest tiles of all an XCD's chunks
// first.  By the grid alone, chunk by chunk, the last chunk's heavy tiles
// start when the others are done, and the workgroups of tiles that short
// chunks do not have take turns on CUs: others then hold two live ones while
// some hold none, however the grid is ordered (four chunks of 32..269 rows on
// prefixes of 962..1378, 64/8 heads of 80: 46.7 us chunk by chunk, 62.3 with
// the grid's heaviest tiles first, 46.9 by real lengths).
// 5994 drawn calls against chunk by chunk: 0.972 of its time in the geometric
// mean, 8 slower by over 5 % and none by over 6.1; by the grid's heaviest
// tiles first 0.984, 24 slower by over 5 %, up to 34.  Six prompts of 9..700
// tokens (32/8 heads of 128) 34.8 us chunk by chunk, 30.5 by the grid, 27.4.

// The chunks' real lengths, one chunk per lane (at most 64): tiles of `rows`
// query rows that the grid covers (the last ceil(max_chunk_len / rows) of a
// longer chunk, a caller error), and their sum.
struct LiveChunks {
    int q0, n, prefix, tiles, incl, total;
    __device__ __forceinline__ LiveChunks(const PrefillParams& p, int rows, int lane) : q0(0), n(0), prefix(0) {
        int end = 0;
        if (lane < p.num_chunks) {
            q0 = p.q_start[lane];
            end = p.q_start[lane + 1];
            prefix = p.prefix_lens[lane];
        }
        n = end - q0;
        tiles = max(0, min((n + rows - 1) / rows, (p.max_chunk_len + rows - 1) / rows));
        incl = wave_incl_scan(tiles);
        total = __builtin_amdgcn_readlane(incl, 63);
    }
};

// Place by weight (0: the heaviest) of the j-th of an XCD's `per` workgroups
// on its C CUs.  The dispatcher gives each CU one before it gives any a second.
__device__ __forceinline__ int live_rank(const LiveChunks& c, int j, int per, int C) {
    if (per <= C || C <= 0) return j;
    if (per <= 2 * C) {  // the heaviest alone, the lightest 2 (per - C) in pairs, heavy beside light
        const int e = per - C;
        return j < e ? C - e + j : j < C ? j - e : per + C - 1 - j;
    }
    // Up to a round and a half the heaviest tile's chain is the time: the
    // second round lightest first, unless prefixes make the tiles alike.
    if (per <= 3 * C && j >= C && j < 2 * C && wave_sum(c.tiles * ((2 * c.prefix - c.n) / 32)) < 0) return 3 * C - 1 - j;
    return j;
}

// This workgroup's work by the chunks' real lengths; false: none.
template <int QT>
__device__ __forceinline__ bool live_work(const PrefillParams& p, PrefillWork& w) {
    const int lane = threadIdx.x & 63;
    const LiveChunks c(p, QT, lane);
    const int nz = p.num_kv_heads * p.head_groups;
    // grid (nz, tiles), an XCD's z ids nzx xcd .. + nzx - 1
    const int xcd = blockIdx.x & 7, nzx = nz >> 3, per = c.total * nzx;
    int q = blockIdx.y, zz = blockIdx.x >> 3;
    const int j = zz + nzx * q;  // dispatch order within the XCD
    if (j >= per) return false;
    const int rank = live_rank(c, j, per, p.xcd_cus);
    if (rank != j) {  // (a division that short calls need not wait for)
        q = rank / nzx;
        zz = rank - q * nzx;
    }
    // The q-th tile by its last key, in steps of a tile: level l holds at most
    // one tile of a chunk, its (level - l)-th from the end.  (Levels are never
    // below 0: the walk ends whatever the prefix lengths hold.)
    const int level = max((c.prefix + c.n - 1) / QT, c.tiles - 1);
    int l = wave_max0(c.tiles > 0 ? level : 0);
    uint64_t m;
    while (true) {
        m = __ballot((uint32_t)(level - l) < (uint32_t)c.tiles);
        const int cnt = __builtin_popcountll(m);
        if (q < cnt) break;
        q -= cnt;
        l = cnt > 0 ? l - 1 : wave_max0(c.tiles > 0 && level < l ? level : 0);
    }
    const int at = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
    const int by = __builtin_ctzll(__ballot((uint32_t)(level - l) < (uint32_t)c.tiles && at == q));
    const int bx = __builtin_amdgcn_readlane(level, by) - l;
    w = PrefillWork{bx, by, nzx * xcd + zz, 0, 1, __builtin_amdgcn_readlane(c.q0, by), __builtin_amdgcn_readlane(c.n, by),
                    __builtin_amdgcn_readlane(c.prefix, by)};
    return true;
}

// a / b for 0 <= a < 2^22, b > 0: a reciprocal and one correction, a third of
// the integer division's chain.
__device__ __forceinline__ int div_small(int a, int b) {
    int q = (int)((float)a * __builtin_amdgcn_rcpf((float)b));
    const int r = a - q * b;
    q += r >= b ? 1 : r < 0 ? -1 : 0;
    return q;
}

// Key parts of a split call by the chunks' real lengths: of 1 .. p.splits the
// count of least cost, at least 256 keys of the longest chunk to a part.  By
// max_chunk_len the host would count tiles that short chunks do not have, and
// so take too few parts (three chunks of 178..449 rows on prefixes up to 19757,
// 24/8 heads of 80: 432 us in two parts, 301 in three).  Lane s - 1 weighs s
// parts, and every workgroup and the merge come to the same count.
__device__ __forceinline__ int live_splits(const PrefillParams& p, const LiveChunks& c, int lane) {
    const int keys = wave_max0(c.tiles > 0 ? c.prefix + c.n : 0);
    const float work = (float)wave_sum(c.tiles * (c.prefix + c.n)) * (p.num_kv_heads * p.head_groups);
    const int last = p.num_chunks - 1;
    const int rows = __builtin_amdgcn_readlane(c.q0 + c.n, last) - __builtin_amdgcn_readlane(c.q0, 0);
    const float out_values = (float)rows * (p.num_heads * p.head_dim);
    const int items = c.total * p.num_kv_heads * p.head_groups, cus = max(8 * p.xcd_cus, 1);
    const int s = lane + 1;
    uint32_t best = ~0u;  // cost (positive: its bits are ordered), low bits the count
    if (s <= p.splits && (s == 1 || s * 256 <= keys)) {
        const float cost = prefill_split_cost(s, items, div_small(items * s, 2 * cus), (float)keys, work,
                                              out_values, cus);
        best = ((uint32_t)__float_as_int(cost) & ~15u) | lane;
    }
    static_assert(kMaxPrefillSplits == 16, "counts in four bits, of one row of lanes");
    // (rotations of the row; a shuffle's lane addresses would stay in registers)
    best = min(best, (uint32_t)__builtin_amdgcn_mov_dpp((int)best, 0x128, 0xF, 0xF, false));
    best = min(best, (uint32_t)__builtin_amdgcn_mov_dpp((int)best, 0x124, 0xF, 0xF, false));
    best = min(best, (uint32_t)__builtin_amdgcn_mov_dpp((int)best, 0x122, 0xF, 0xF, false));
    best = min(best, (uint32_t)__builtin_amdgcn_mov_dpp((int)best, 0x121, 0xF, 0xF, false));
    return (__builtin_amdgcn_readlane((int)best, 0) & 15) + 1;
}

// This workgroup's work of a split call, in `splits` parts; false: none.
template <int QT>
__device__ __forceinline__ bool live_split_work(const PrefillParams& p, PrefillWork& w) {
    const int lane = threadIdx.x & 63;
    const LiveChunks c(p, QT, lane);
    const int splits = live_splits(p, c, lane);
    const int C = p.xcd_cus, HG = p.head_groups;
    const int one = c.total * HG, total = one * p.num_kv_heads * splits, per = (total + 7) >> 3;
    int j = blockIdx.x >> 3;  // dispatch order within the XCD
    if (j >= per) return false;
    if (per > C && per <= 2 * C && j >= C) j = per + C - 1 - j;  // one round: as in remap_ids
    const int m = (int)(blockIdx.x & 7) * per + j;
    if (m >= total) return false;
    // m = tile + tiles (head group + HG (chunks before + ..)), then kv head, part
    const int y = __builtin_amdgcn_readfirstlane(div_small(m, one)), r = m - y * one;
    const int part = __builtin_amdgcn_readfirstlane(div_small(y, p.num_kv_heads));
    const int excl = c.incl - c.tiles;
    const int by = __builtin_popcountll(__ballot(lane < p.num_chunks && excl * HG <= r)) - 1;
    const int rr = r - HG * __builtin_amdgcn_readlane(excl, by);
    const int nt = __builtin_amdgcn_readlane(c.tiles, by);
    const int hg = __builtin_amdgcn_readfirstlane(div_small(rr, nt));
    w = PrefillWork{rr - hg * nt, by, (y - part * p.num_kv_heads) * HG + hg, part, splits,
                    __builtin_amdgcn_readlane(c.q0, by), __builtin_amdgcn_readlane(c.n, by),
                    __builtin_amdgcn_readlane(c.prefix, by)};
    return true;
}

// PLACE: by the grid (remap_ids), or by the chunks' real lengths, unsplit
// (live_work) or split (live_split_work).
enum { kGrid = 0, kLive = 1, kLiveSplit = 2 };

template <int KV, int D, int PLACE, int PB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
void prefill_dma_kernel(PrefillParams p) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    PrefillWork w;
    if constexpr (PLACE == kLive) {
        if (!live_work<16 * PDims<D>::RB>(p, w)) return;
    } else if constexpr (PLACE == kLiveSplit) {
        if (!live_split_work<16 * PDims<D>::RB>(p, w)) return;
    } else {
        int bx, by, bz;
        remap_ids(p, 2, bx, by, bz);
        // z: (key part, kv head, head group)
        const int zh = p.num_kv_heads * p.head_groups;
        w.bx = bx;
        w.by = by;
        w.part = bz / zh;
        w.bz = bz - w.part * zh;
        w.splits = p.splits;
        w.load_chunk(p);
    }
    w.uniform();
    prefill_tile<KV, D, false, PB>(p, w, reinterpret_cast<lds_char*>((__attribute__((address_space(3))) char*)smem));
}

// fp16 pages at head_dim 64 / 80: 128-row tiles, one wave per SIMD
// (prefill_wide_run).
template <int D>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
void prefill_wide_kernel(PrefillParams p) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    prefill_wide_run<D>(p, reinterpret_cast<lds_char*>((__attribute__((address_space(3))) char*)smem));
}

// Log-sum-exp merge of a split prefill's S parts: thread (row, head, 4 dims).
// S is a template argument so that the parts' loads are all issued before
// their first use, in exactly S registers' worth of values.
template <int S>
__global__ __launch_bounds__(256) void prefill_merge_kernel(PrefillParams p) {
    const int D4 = p.head_dim / 4;
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    int parts = S;
    bool too_long = true;  // chunks longer than max_chunk_len to look for
    if (p.live) {
        const int lane = threadIdx.x & 63;
        const LiveChunks c(p, p.tile_rows, lane);
        parts = live_splits(p, c, lane);
        if (parts <= 1) return;  // finished in place
        too_long = __any(c.n > c.tiles * p.tile_rows);
    }
    const int64_t per_row = (int64_t)p.num_heads * D4;
    const int row = (int)(idx / per_row);
    if (row >= p.q_start[p.num_chunks]) return;
    // Rows of a chunk longer than max_chunk_len (a caller error) that no
    // query tile of the grid covered are left unwritten, as the unsplit
    // kernel leaves them: the grid covers each chunk's last
    // ceil(max_chunk_len / tile_rows) tiles.
    if (too_long) {
        int lo = 0, hi = p.num_chunks - 1;  // chunk of the row: last c with q_start[c] <= row
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (p.q_start[mid] <= row) lo = mid;
            else hi = mid - 1;
        }
        const int q0 = p.q_start[lo], n = p.q_start[lo + 1] - q0;
        const int ntile = (n + p.tile_rows - 1) / p.tile_rows;
        const int first = ntile - (p.max_chunk_len + p.tile_rows - 1) / p.tile_rows;
        if (first > 0 && row - q0 < first * p.tile_rows) return;
    }
    const int rem = (int)(idx - row * per_row);
    const int head = rem / D4, d4 = rem - head * D4;
    float2 ml[S];
    float4 v[S];
    float M = -__builtin_inff();
#pragma unroll
    for (int s = 0; s < S; ++s) {
        // (parts past the count are not there: part 0 again, with weight 0)
        const int64_t rh = ((int64_t)(s < parts ? s : 0) * p.rows_cap + row) * p.num_heads + head;
        ml[s] = p.ws_ml[rh];
        if (s >= parts) ml[s].y = 0.f;
        v[s] = reinterpret_cast<const float4*>(p.ws_o + rh * p.head_dim)[d4];
    }
#pragma unroll
    for (int s = 0; s < S; ++s)
        if (ml[s].y > 0.f) M = fmaxf(M, ml[s].x);  // parts with no visible key (sum 0) weigh 0
    float L = 0.f;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int s = 0; s < S; ++s) {
        if (ml[s].y > 0.f) {
            const float w = exp2f(ml[s].x - M);
            L += w * ml[s].y;
            acc.x += w * v[s].x;
            acc.y += w * v[s].y;
            acc.z += w * v[s].z;
            acc.w += w * v[s].w;
        }
    }
    const float inv = 1.0f / (L + 1e-9f);
    reinterpret_cast<float4*>(p.out + ((int64_t)row * p.num_heads + head) * p.head_dim)[d4] =
        make_float4(acc.x * inv, acc.y * inv, acc.z * inv, acc.w * inv);
}

template <int S>
hipError_t launch_merge_s(const PrefillParams& p, hipStream_t stream) {
    if (p.splits != S) return launch_merge_s<S - 1>(p, stream);
    const int64_t threads = (int64_t)p.rows_cap * p.num_heads * (p.head_dim / 4);
    hipLaunchKernelGGL(prefill_merge_kernel<S>, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, stream, p);
    return hipGetLastError();
}
template <>
hipError_t launch_merge_s<1>(const PrefillParams&, hipStream_t) { return hipErrorInvalidValue; }

// VCPP_PF_WIDE=1: fp16 pages at head_dim 64 / 80 (power-of-two block size)
// run prefill_wide_kernel instead of prefill_dma_kernel.  Opt-in: on MI355X
// it measured about 10 % slower on config 3 (read at every launch, so a
// process can switch).
bool wide_requested() {
    const char* e = std::getenv("VCPP_PF_WIDE");
    return e && e[0] == '1';
}

template <int KV, int D>
constexpr bool use_wide_t() { return KV == VCPP_KV_F16 && wide_prefill_ok<D>(); }

bool pow2(int x) { return x > 0 && (x & (x - 1)) == 0; }

// Whether a call of prefill_dma_kernel places its workgroups by the chunks'
// real lengths (live_work): grids of up to three rounds of two workgroups per
// CU, with more than one tile to a chunk and more than one chunk or head group
// to an XCD.  In longer grids the balance matters less and the L2 more: 8
// chunks of up to 2048 tokens on prefixes up to 4000 (int8) 720 us chunk by
// chunk, 801 heaviest first.
bool prefill_live(const PrefillParams& p) {
    if (p.splits > 1 || p.num_chunks > 64 || prefill_uses_wide(p.kv_dtype, p.head_dim, p.block_size)) return false;
    const int QT = prefill_tile_rows(p.kv_dtype, p.head_dim, p.block_size);
    const int64_t nz = (int64_t)p.num_kv_heads * p.head_groups;
    const int64_t total = (p.max_chunk_len + QT - 1) / QT * nz * p.num_chunks;
    return (p.num_chunks > 1 || nz > 8) && p.max_chunk_len > QT && p.xcd_cus > 0 && nz % 8 == 0 && total <= 8 * 6 * p.xcd_cus;
}

// Whether the four-stage fp16 ring (head_dim 128) takes two key blocks per
// barrier after all: a grid of at most one workgroup per CU, over more than
// 1024 keys to a part as far as the tables bound them.  A workgroup alone has
// no other to cover its barriers: 35 rows on a prefix of 2800 (64/8 heads) 65.0
// us in pairs, 67.8 one by one, 3 x 16 rows on 16000 341.5 against 363.7; but
// 61 rows on 600 22.4 against 21.8.
bool prefill_pairs(const PrefillParams& p, int64_t workgroups) {
    return workgroups <= 8 * (int64_t)p.xcd_cus &&
           (int64_t)p.max_blocks * p.block_size > 1024 * (int64_t)std::max(p.splits, 1);
}

// Raises a kernel's dynamic LDS limit on this device only when a launch needs
// more than `set` last held there (the attribute call is a host round trip;
// the limit is per device).
hipError_t raise_lds(const void* fn, size_t (&set)[64], size_t lds) {
    int dev = 0;
    const bool known = hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < 64;
    if (!known || lds > std::max<size_t>(set[dev], 65536)) {
        const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
        if (known) set[dev] = lds;
    }
    return hipSuccess;
}

template <int KV, int D, int PLACE, int PB>
hipError_t launch_ring(const PrefillParams& p, dim3 grid, size_t lds, hipStream_t stream) {
    static size_t attr_lds[64] = {};
    const hipError_t e = raise_lds((const void*)prefill_dma_kernel<KV, D, PLACE, PB>, attr_lds, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((prefill_dma_kernel<KV, D, PLACE, PB>), grid, dim3(256), lds, stream, p);
    return hipGetLastError();
}

template <int KV, int D>
hipError_t launch_dma(const PrefillParams& p, hipStream_t stream) {
    const bool wide = prefill_uses_wide(KV, D, p.block_size);
    const int QT = prefill_tile_rows(KV, D, p.block_size);
    dim3 grid((p.max_chunk_len + QT - 1) / QT, p.num_chunks,
              p.num_kv_heads * p.head_groups * max(p.splits, 1));
    size_t lds = (wide ? (size_t)WDims<D>::STAGES * DmaDims<D>::STAGE + 1024 : prefill_ring_bytes(KV, D)) +
                 (size_t)p.max_blocks * 4;
#ifdef VCPP_PREFILL_LDS_PAD
    lds = std::max<size_t>(lds, VCPP_PREFILL_LDS_PAD);
#endif
    const int64_t total = (int64_t)grid.x * grid.y * grid.z;
    if constexpr (use_wide_t<KV, D>()) {
        if (wide) {
            // A 1-D grid of all tiles (ordered by wide_tile_ids).
            static size_t attr_lds[64] = {};
            const hipError_t e = raise_lds((const void*)prefill_wide_kernel<D>, attr_lds, lds);
            if (e != hipSuccess) return e;
            hipLaunchKernelGGL((prefill_wide_kernel<D>), dim3((unsigned)total), dim3(256), lds, stream, p);
            return hipGetLastError();
        }
    }
    constexpr int PB = DmaDims<D>::PER_BARRIER;
    if (p.live) return launch_ring<KV, D, kLiveSplit, PB>(p, dim3((unsigned)((total + 7) / 8 * 8)), lds, stream);
    const bool live = prefill_live(p);
    if (live) grid = dim3(grid.z, grid.x * grid.y);
    if constexpr (KV == VCPP_KV_F16 && PB == 1) {
        if (prefill_pairs(p, total))
            return live ? launch_ring<KV, D, kLive, 2>(p, grid, lds, stream)
                        : launch_ring<KV, D, kGrid, 2>(p, grid, lds, stream);
    }
    return live ? launch_ring<KV, D, kLive, PB>(p, grid, lds, stream)
                : launch_ring<KV, D, kGrid, PB>(p, grid, lds, stream);
}

}  // namespace

bool prefill_uses_wide(int kv_dtype, int head_dim, int block_size) {
    return kv_dtype == VCPP_KV_F16 && (head_dim == 64 || head_dim == 80) && pow2(block_size) && wide_requested();
}

int prefill_tile_rows(int kv_dtype, int head_dim, int block_size) {
    if (prefill_uses_wide(kv_dtype, head_dim, block_size)) return WDims<80>::QT;
    switch (head_dim) {
        case 64: return 16 * PDims<64>::RB;
        case 80: return 16 * PDims<80>::RB;
        default: return 16 * PDims<128>::RB;
    }
}

int prefill_head_groups(int group) { return (group + kHeadsPerGroup - 1) / kHeadsPerGroup; }

// LDS of the ring of prefill_dma_kernel.
size_t prefill_ring_bytes(int kv_dtype, int head_dim) {
    auto ring = [&](auto d) -> size_t {
        constexpr int D = decltype(d)::value;
        if (kv_dtype == VCPP_KV_I8)
            return (size_t)ByteDims<D, true>::STAGES * ByteDims<D, true>::STAGE + 2 * (size_t)DmaDims<D>::STAGE;
        if (kv_dtype == VCPP_KV_FP8)
            return (size_t)ByteDims<D, false>::STAGES * ByteDims<D, false>::STAGE + 2 * (size_t)DmaDims<D>::STAGE;
        return (size_t)DmaDims<D>::STAGES * DmaDims<D>::STAGE;
    };
    switch (head_dim) {
        case 64: return ring(std::integral_constant<int, 64>{});
        case 80: return ring(std::integral_constant<int, 80>{});
        case 128: return ring(std::integral_constant<int, 128>{});
        default: return 0;
    }
}

size_t prefill_lds_bytes(int kv_dtype, int head_dim, int max_blocks) {
    size_t r = prefill_ring_bytes(kv_dtype, head_dim);
    if (r == 0) return 0;
    if (kv_dtype == VCPP_KV_F16 && head_dim == 64)
        r = std::max<size_t>(r, (size_t)WDims<64>::STAGES * DmaDims<64>::STAGE + 1024);
    if (kv_dtype == VCPP_KV_F16 && head_dim == 80)
        r = std::max<size_t>(r, (size_t)WDims<80>::STAGES * DmaDims<80>::STAGE + 1024);
    return r + (size_t)max_blocks * 4;
}

hipError_t launch_prefill(const PrefillParams& p, hipStream_t stream) {
    if (p.num_chunks == 0 || p.max_chunk_len == 0) return hipSuccess;
    const bool prof = prof_enabled();
    if (prof) prof_begin(kKernelPrefill, stream);
    hipError_t err = hipErrorInvalidValue;
#define VCPP_PF_D(KVT)                                      \
    switch (p.head_dim) {                                   \
        case 64: err = launch_dma<KVT, 64>(p, stream); break;   \
        case 80: err = launch_dma<KVT, 80>(p, stream); break;   \
        case 128: err = launch_dma<KVT, 128>(p, stream); break; \
        default: return hipErrorInvalidValue;               \
    }
    if (p.kv_dtype == VCPP_KV_F16) {
        VCPP_PF_D(VCPP_KV_F16)
    } else if (p.kv_dtype == VCPP_KV_FP8) {
        VCPP_PF_D(VCPP_KV_FP8)
    } else {
        VCPP_PF_D(VCPP_KV_I8)
    }
#undef VCPP_PF_D
    if (err != hipSuccess) return err;
    if (p.splits > 1) {
        if (p.splits > kMaxPrefillSplits) return hipErrorInvalidValue;
        PrefillParams pm = p;
        pm.tile_rows = prefill_tile_rows(p.kv_dtype, p.head_dim, p.block_size);
        err = launch_merge_s<kMaxPrefillSplits>(pm, stream);
        if (err != hipSuccess) return err;
    }
    if (prof) prof_end(kKernelPrefill, stream);
    return hipSuccess;
}

size_t prefill_split_bytes(int splits, int rows_cap, int num_heads, int head_dim) {
    if (splits <= 1) return 0;
    const size_t rows = (size_t)splits * rows_cap * num_heads;
    return ((rows * head_dim * sizeof(float) + 255) & ~size_t(255)) + rows * sizeof(float2);
}

}  // namespace vcpp

#ifdef VCPP_PF_TIMING
// Timing builds only: reads and clears the wide prefill's segment sums.
extern "C" int vcpp_pf_timing_read(unsigned long long* out) {
    if (hipMemcpyFromSymbol(out, HIP_SYMBOL(vcpp::g_pf_timing), 16 * sizeof(unsigned long long)) != hipSuccess)
        return -1;
    unsigned long long z[16] = {};
    return hipMemcpyToSymbol(HIP_SYMBOL(vcpp::g_pf_timing), z, sizeof(z)) == hipSuccess ? 0 : -1;
}
#endif
