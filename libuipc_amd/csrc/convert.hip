// Triplet -> sorted upper-triangular 3x3 BCOO + BSR row offsets on gfx950,
// plus the full (both triangles) BSR the SpMV streams.
//
// Replaces MatrixConverter<Float,3>::convert_sym
// (algorithm/details/matrix_converter.inl:1549-1699) and the segmented reduce
// it calls (algorithm/fast_segmental_reduce.h:33-103).  Same contract:
//   keep (row >= 0 && row <= col), key = row * B + col, stable sort on
//   bit_width(B*B - 1) bits (matrix_converter.inl:726-735), run-length encode,
//   sum each run of equal keys.
// Differences by design:
//   * the sort is a hand-written LSD radix sort (8-bit digits, wave64 ballot
//     ranking, LDS-staged stable scatter) instead of CUB;
//   * duplicates are summed sequentially in ascending source order by one
//     thread per entry of the output block, so the values are deterministic
//     (the reference sums in atomic arrival order,
//     fast_segmental_reduce.h:23-26);
//   * values land in 9 SoA planes (see BsrMatrix);
//   * two host read-backs: the largest col - row, which chooses the sort key, and
//     the unique count, which sizes the outputs;
//   * the upper BCOO is then transposed (a stable radix sort of the off-diagonal
//     blocks by column alone: they come in row order) and laid out for the SpMV,
//     as a full BSR, a pure row gather without atomics, or in windows.
#include "linsys.hpp"
#include "segtile.hpp"

namespace mi
{
namespace
{
constexpr int kThreads   = 256;
constexpr int kItems     = 16;
constexpr int kTileItems = kItems;
constexpr int kTile      = kThreads * kItems;  // 4096 keys per tile
constexpr int kWaves     = kThreads / kWave;

// kept entries and their sort keys.  Mode 0: the triplet filter of
// matrix_converter.inl:142 (plus a bound on col, which the reference leaves
// to its producers), key (row, col).  Mode 1: the off-diagonal blocks of the
// upper BCOO, key (col, row) (the transpose).
template <int MODE>
__device__ __forceinline__ bool keep_entry(int32_t r, int32_t c, int32_t B)
{
    if constexpr(MODE == 0)
        return r >= 0 && r <= c && c < B;
    else
        return r != c;
}
template <int MODE>
__device__ __forceinline__ uint64_t entry_key(int32_t r, int32_t c, const KeyCodec& kc)
{
    if constexpr(MODE == 0)
        return kc.up(r, c);
    else
        return kc.lo(r, c);
}

// ---- 1. count kept entries per tile
// (and, with d_band, the largest col - row of the kept entries)
template <int MODE>
__global__ __launch_bounds__(kThreads) void cv_count_kernel(int64_t        T,
                                                           const int32_t* rows,
                                                           const int32_t* cols,
                                                           int32_t        B,
                                                           uint32_t*      tile_cnt,
                                                           int32_t*       d_band)
{
    __shared__ uint32_t lds[kWaves];
    __shared__ int32_t  bmax[kWaves];
    const int64_t       base = (int64_t)blockIdx.x * kTile;
    uint32_t            c    = 0;
    int32_t             band = 0;
#pragma unroll
    for(int k = 0; k < kItems; ++k)
    {
        int64_t i = base + (int64_t)k * kThreads + threadIdx.x;
        if(i < T)
        {
            const int32_t r = rows[i], cc = cols[i];
            if(keep_entry<MODE>(r, cc, B))
            {
                ++c;
                band = max(band, cc - r);
            }
        }
    }
    uint32_t s = block_sum<kThreads>(c, lds);
    if(threadIdx.x == 0)
        tile_cnt[blockIdx.x] = s;
    if(d_band)
    {
#pragma unroll
        for(int o = kWave / 2; o > 0; o >>= 1)
            band = max(band, __shfl_xor(band, o, kWave));
        if(threadIdx.x % kWave == 0)
            bmax[threadIdx.x / kWave] = band;
        __syncthreads();
        if(threadIdx.x == 0)
        {
            int32_t m = bmax[0];
            for(int w = 1; w < kWaves; ++w)
                m = max(m, bmax[w]);
            atomicMax(d_band, m);
        }
    }
}

// Exclusive scan of n consecutive values by one workgroup of NT threads, in
// place, rounds of 16 NT values: consecutive lanes move consecutive values
// between memory and LDS, a thread sums 16 consecutive ones (padded by one
// word in 16, so that they lie in different banks).  Returns the total.
constexpr int kScanItems = 16;
template <int NT>
__device__ __forceinline__ uint32_t scan_span(uint32_t* data, int64_t n, uint32_t* sv, uint32_t* lds)
{
    uint32_t carry = 0;
    for(int64_t base = 0; base < n; base += NT * kScanItems)
    {
#pragma unroll
        for(int k = 0; k < kScanItems; ++k)
        {
            const int t       = k * NT + (int)threadIdx.x;
            sv[t + (t >> 4)] = base + t < n ? data[base + t] : 0u;
        }
        __syncthreads();
        const int first = (int)threadIdx.x * (kScanItems + 1);
        uint32_t  sum   = 0;
#pragma unroll
        for(int k = 0; k < kScanItems; ++k)
            sum += sv[first + k];
        uint32_t tot;
        uint32_t e = carry + block_exclusive_scan<NT>(sum, lds, &tot);
#pragma unroll
        for(int k = 0; k < kScanItems; ++k)
        {
            const uint32_t v = sv[first + k];
            sv[first + k]    = e;
            e += v;
        }
        carry += tot;
        __syncthreads();
#pragma unroll
        for(int k = 0; k < kScanItems; ++k)
        {
            const int t = k * NT + (int)threadIdx.x;
            if(base + t < n)
                data[base + t] = sv[t + (t >> 4)];
        }
        __syncthreads();
    }
    return carry;
}

// ---- single-workgroup exclusive scan (n up to 64k), total -> *total (one
// value per thread and round took 24 us for 36k values)
__global__ __launch_bounds__(1024) void scan_small_kernel(uint32_t* data, int64_t n, int64_t* total)
{
    __shared__ uint32_t sv[1024 * (kScanItems + 1)];
    __shared__ uint32_t lds[1024 / kWave + 1];
    const uint32_t      tot = scan_span<1024>(data, n, sv, lds);
    if(threadIdx.x == 0 && total)
        *total = (int64_t)tot;
}

// ---- large exclusive scan: per-chunk sums, scan of sums, down-sweep
constexpr int kScanChunk = kThreads * kItems;
__global__ __launch_bounds__(kThreads) void scan_reduce_kernel(const uint32_t* data, int64_t n, uint32_t* sums)
{
    __shared__ uint32_t lds[kWaves];
    const int64_t       base = (int64_t)blockIdx.x * kScanChunk;
    uint32_t            s    = 0;
#pragma unroll
    for(int k = 0; k < kItems; ++k)
    {
        int64_t i = base + (int64_t)k * kThreads + threadIdx.x;
        if(i < n)
            s += data[i];
    }
    s = block_sum<kThreads>(s, lds);
    if(threadIdx.x == 0)
        sums[blockIdx.x] = s;
}
__global__ __launch_bounds__(kThreads) void scan_down_kernel(uint32_t* data, int64_t n, const uint32_t* sums)
{
    __shared__ uint32_t sv[kScanChunk];
    __shared__ uint32_t lds[kWaves + 1];
    const int64_t       base = (int64_t)blockIdx.x * kScanChunk;
#pragma unroll
    for(int k = 0; k < kItems; ++k)
    {
        int     t = k * kThreads + threadIdx.x;
        int64_t i = base + t;
        sv[t]     = i < n ? data[i] : 0u;
    }
    __syncthreads();
    const int first = threadIdx.x * kItems;
    uint32_t  c     = 0;
#pragma unroll
    for(int k = 0; k < kItems; ++k)
        c += sv[first + k];
    uint32_t o = block_exclusive_scan<kThreads>(c, lds, (uint32_t*)nullptr) + sums[blockIdx.x];
#pragma unroll
    for(int k = 0; k < kItems; ++k)
    {
        uint32_t v      = sv[first + k];
        sv[first + k] = o;
        o += v;
    }
    __syncthreads();
#pragma unroll
    for(int k = 0; k < kItems; ++k)
    {
        int     t = k * kThreads + threadIdx.x;
        int64_t i = base + t;
        if(i < n)
            data[i] = sv[t];
    }
}

// ---- radix sort inputs.  PairSource: the (key, source) pairs of the last
// pass, m of them.  TripletSource: the first pass straight from the
// triplets' (row, col) -- entries that keep_entry drops are skipped and the
// key is built on the fly, so the compaction writes no pairs of its own (a
// stable pass over the kept entries in index order, as compacting first
// would give).
template <typename KeyT>
struct PairSource
{
    const int64_t* d_m;
    const KeyT*    keys;
    const int32_t* srcs;
    __device__ int64_t count() const { return *d_m; }
    __device__ bool    key_at(int64_t i, int64_t m, KeyT& k) const
    {
        if(i >= m)
            return false;
        k = keys[i];
        return true;
    }
    __device__ bool pair_at(int64_t i, int64_t m, KeyT& k, int32_t& v) const
    {
        if(i >= m)
            return false;
        k = keys[i];
        v = srcs[i];
        return true;
    }
};
template <int MODE, typename KeyT>
struct TripletSource
{
    const int32_t* rows;
    const int32_t* cols;
    int64_t        n;
    int32_t        B;
    KeyCodec       kc;
    __device__ int64_t count() const { return n; }
    __device__ bool    key_at(int64_t i, int64_t m, KeyT& k) const
    {
        if(i >= m)
            return false;
        const int32_t r = rows[i], c = cols[i];
        if(!keep_entry<MODE>(r, c, B))
            return false;
        k = (KeyT)entry_key<MODE>(r, c, kc);
        return true;
    }
    __device__ bool pair_at(int64_t i, int64_t m, KeyT& k, int32_t& v) const
    {
        v = (int32_t)i;
        return key_at(i, m, k);
    }
};

// ---- radix sort: the digit counts of every tile and where each tile's runs
// start.  Many tiles: hist[d * ntiles + tile], each digit's row scanned over
// the tiles by a workgroup of its own (rs_rows_kernel), the digits' totals
// scanned by every scatter workgroup: three launches per pass (a general scan
// of the 256 ntiles counts took three by itself, or one of up to 24 us).  Up to
// kFewKeys keys, where a pass is little more than its launches and its tiles'
// serial rounds, tiles of 1,024 keys and hist[tile * 256 + d], which every
// scatter workgroup sums over the tiles by itself: two launches.
// (Counting the next pass's digits in the scatter, by global atomics at the
// keys' new places, was slower: 81k keys' assembly 239 -> 368 us, the keys of
// a run meet in a few counters.)
constexpr int     kFewItems = 4;
constexpr int     kFewTile  = kThreads * kFewItems;
constexpr int64_t kFewKeys  = 128 * kFewTile;

template <typename KeyT, typename Src, bool kFew>
__global__ __launch_bounds__(kThreads) void rs_hist_kernel(Src           src,
                                                          int           shift,
                                                          uint32_t      dmask,
                                                          uint32_t*     hist,
                                                          int           ntiles)
{
    constexpr int kItems = kFew ? kFewItems : kTileItems;
    constexpr int kTile  = kThreads * kItems;
    __shared__ uint32_t h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    const int64_t m    = src.count();
    const int64_t base = (int64_t)blockIdx.x * kTile;
#pragma unroll
    for(int k = 0; k < kItems; ++k)
    {
        const int64_t i = base + (int64_t)k * kThreads + threadIdx.x;
        KeyT          key;
        if(src.key_at(i, m, key))
            atomicAdd(&h[(uint32_t)(key >> shift) & dmask], 1u);
    }
    __syncthreads();
    if constexpr(kFew)
        hist[(int64_t)blockIdx.x * 256 + threadIdx.x] = h[threadIdx.x];
    else
        hist[(int64_t)threadIdx.x * ntiles + blockIdx.x] = h[threadIdx.x];
}

// exclusive scan of digit blockIdx.x's counts over the tiles, in place; its
// total -> totals[digit]
__global__ __launch_bounds__(kThreads) void rs_rows_kernel(uint32_t* hist, int ntiles, uint32_t* totals)
{
    __shared__ uint32_t sv[kThreads * (kScanItems + 1)];
    __shared__ uint32_t lds[kWaves + 1];
    const uint32_t      tot = scan_span<kThreads>(hist + (int64_t)blockIdx.x * ntiles, ntiles, sv, lds);
    if(threadIdx.x == 0)
        totals[blockIdx.x] = tot;
}

__device__ __forceinline__ uint64_t lanemask_lt64()
{
    return (1ull << __lane_id()) - 1ull;
}

// ---- radix sort: stable scatter of one tile.  Wave w ranks the 64-key rounds
// of its contiguous quarter of the tile in order (ballot-matched peers +
// per-wave digit counters), the tile is reordered by digit in LDS, then each
// digit run is written out contiguously.
// (Counting by returning LDS atomics, so that no round waits for the one
// before: 142 -> 160 us per pass of the 64^3 + 2M system; the other waves hide
// that chain.)
// totals: the digits' totals (many tiles).
template <typename KeyT, typename Src, bool kFew>
__global__ __launch_bounds__(kThreads) void rs_scatter_kernel(Src             src,
                                                             KeyT*           kout,
                                                             int32_t*        vout,
                                                             int             shift,
                                                             uint32_t        dmask,
                                                             const uint32_t* __restrict__ hist,
                                                             int             ntiles,
                                                             const uint32_t* __restrict__ totals)
{
    constexpr int       kItems = kFew ? kFewItems : kTileItems;
    constexpr int       kTile  = kThreads * kItems;
    __shared__ KeyT     sk[kTile];
    __shared__ int32_t  sv[kTile];
    __shared__ uint32_t wcnt[kWaves][256];
    __shared__ uint32_t dstart[256];
    __shared__ uint32_t gbase[256];
    __shared__ uint32_t lds[kWaves + 1];

    const int64_t m    = src.count();
    const int64_t base = (int64_t)blockIdx.x * kTile;
    if(base >= m)
        return;  // uniform per block
    const int w    = threadIdx.x / kWave;
    const int lane = threadIdx.x % kWave;
#pragma unroll
    for(int q = 0; q < kWaves; ++q)
        wcnt[q][threadIdx.x] = 0;
    // this digit's count in all tiles and in the tiles before this one
    uint32_t dtotal = 0, dbefore = 0;
    if constexpr(kFew)
    {
#pragma unroll 16
        for(int t = 0; t < ntiles; ++t)
        {
            const uint32_t c = hist[t * 256 + (int)threadIdx.x];
            dtotal += c;
            dbefore += t < (int)blockIdx.x ? c : 0u;
        }
    }
    else
    {
        dtotal  = totals[threadIdx.x];
        dbefore = hist[(int64_t)threadIdx.x * ntiles + blockIdx.x];
    }
    __syncthreads();

    KeyT           key[kItems];
    int32_t        val[kItems];
    uint32_t       rank[kItems];
    uint32_t       dig[kItems];
    const uint64_t lt = lanemask_lt64();
#pragma unroll
    for(int k = 0; k < kItems; ++k)
    {
        int64_t  i     = base + (int64_t)w * (kWave * kItems) + (int64_t)k * kWave + lane;
        key[k]         = KeyT(0);
        val[k]         = 0;
        const bool valid = src.pair_at(i, m, key[k], val[k]);
        uint32_t d     = valid ? ((uint32_t)(key[k] >> shift) & dmask) : 0u;
        dig[k]         = valid ? d : 0xFFFFFFFFu;
        uint64_t peers = __ballot(valid);
#pragma unroll
        for(int b = 0; b < 8; ++b)
        {
            uint64_t bm = __ballot((d >> b) & 1u);
            peers &= ((d >> b) & 1u) ? bm : ~bm;
        }
        uint32_t r = 0;
        if(valid)
        {
            uint32_t cnt = wcnt[w][d];
            r            = cnt + (uint32_t)__popcll(peers & lt);
            int leader   = 63 - __clzll(peers);
            if(lane == leader)
                wcnt[w][d] = cnt + (uint32_t)__popcll(peers);
        }
        rank[k] = r;
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    // per digit: wave prefixes (in place) and the tile total
    uint32_t tile_total;  // the tile's kept entries
    {
        const int d   = threadIdx.x;
        uint32_t  acc = 0;
#pragma unroll
        for(int q = 0; q < kWaves; ++q)
        {
            uint32_t c = wcnt[q][d];
            wcnt[q][d] = acc;
            acc += c;
        }
        uint32_t e = block_exclusive_scan<kThreads>(acc, lds, &tile_total);
        dstart[d]  = e;
        gbase[d]   = block_exclusive_scan<kThreads>(dtotal, lds, (uint32_t*)nullptr) + dbefore;
    }
    __syncthreads();
#pragma unroll
    for(int k = 0; k < kItems; ++k)
        if(dig[k] != 0xFFFFFFFFu)
        {
            uint32_t pos = dstart[dig[k]] + wcnt[w][dig[k]] + rank[k];
            sk[pos]      = key[k];
            sv[pos]      = val[k];
        }
    __syncthreads();
    const int64_t cnt = tile_total;
#pragma unroll
    for(int k = 0; k < kItems; ++k)
    {
        int i = k * kThreads + threadIdx.x;
        if(i < cnt)
        {
            KeyT     kk  = sk[i];
            uint32_t d   = (uint32_t)(kk >> shift) & dmask;
            uint32_t out = gbase[d] + ((uint32_t)i - dstart[d]);
            kout[out]    = kk;
            vout[out]    = sv[i];
        }
    }
}

// stage one tile of sorted keys into LDS (plus the key before the tile)
template <typename KeyT>
__device__ __forceinline__ void stage_keys(const KeyT* keys, int64_t m, int64_t base, KeyT* sk)
{
#pragma unroll
    for(int k = 0; k < kItems; ++k)
    {
        int     t = k * kThreads + threadIdx.x;
        int64_t i = base + t;
        sk[t + 1] = i < m ? keys[i] : ~KeyT(0);
    }
    if(threadIdx.x == 0)
        sk[0] = base > 0 ? keys[base - 1] : ~KeyT(0);
    __syncthreads();
}

// ---- run-length encode: heads per tile
template <typename KeyT>
__global__ __launch_bounds__(kThreads) void rle_count_kernel(const int64_t* d_m, const KeyT* keys, uint32_t* tile_cnt)
{
    __shared__ uint32_t lds[kWaves];
    const int64_t       m    = *d_m;
    const int64_t       base = (int64_t)blockIdx.x * kTile;
    uint32_t            c    = 0;
#pragma unroll
    for(int k = 0; k < kItems; ++k)
    {
        int64_t i = base + (int64_t)k * kThreads + threadIdx.x;
        if(i < m && (i == 0 || keys[i] != keys[i - 1]))
            ++c;
    }
    uint32_t s = block_sum<kThreads>(c, lds);
    if(threadIdx.x == 0)
        tile_cnt[blockIdx.x] = s;
}

template <typename KeyT>
__global__ __launch_bounds__(kThreads) void rle_write_kernel(const int64_t*  d_m,
                                                            const KeyT*     keys,
                                                            const uint32_t* tile_off,
                                                            KeyCodec        kc,
                                                            int32_t*        out_rows,
                                                            int32_t*        out_cols,
                                                            int32_t*        seg_start,
                                                            uint32_t*       seg_tile)
{
    __shared__ KeyT     sk[kTile + 1];
    __shared__ int32_t  hp[kTile];
    __shared__ uint32_t lds[kWaves + 1];
    const int64_t       m    = *d_m;
    const int64_t       base = (int64_t)blockIdx.x * kTile;
    stage_keys(keys, m, base, sk);
    const int first = threadIdx.x * kItems;
    uint32_t  flags = 0, c = 0;
    KeyT      kk[kItems];
#pragma unroll
    for(int k = 0; k < kItems; ++k)
    {
        int64_t i = base + first + k;
        kk[k]     = sk[first + k + 1];
        if(i < m && (i == 0 || kk[k] != sk[first + k]))
        {
            flags |= 1u << k;
            ++c;
        }
    }
    uint32_t       heads = 0;
    uint32_t       o     = block_exclusive_scan<kThreads>(c, lds, &heads);  // its barriers end every read of sk
    const uint32_t g     = tile_off[blockIdx.x];
    // the heads before every segment tile of the reduce
    if(first % kSegTile == 0)
        seg_tile[(base + first) / kSegTile] = g + o;
    // the heads' keys (in place, in order) and positions, then written out by
    // consecutive lanes
#pragma unroll
    for(int k = 0; k < kItems; ++k)
        if(flags & (1u << k))
        {
            sk[o] = kk[k];
            hp[o] = first + k;
            ++o;
        }
    __syncthreads();
    for(uint32_t i = threadIdx.x; i < heads; i += kThreads)
    {
        int32_t r, c;
        kc.up_rc((uint64_t)sk[i], r, c);
        out_rows[g + i]    = r;
        out_cols[g + i]    = c;
        seg_start[g + i]   = (int32_t)(base + hp[i]);
    }
}

// ---- segmented reduce: duplicates summed in FP64 in ascending source order
// (bit-identical to a sequential left fold of the values as doubles).  Bound
// by the random gathers of whole records (72 or 36 bytes, m of them).
//
// A workgroup takes tiles of 256 sorted entries.  It owns the blocks whose
// first entry lies in the tile and stages the tile's records, and those of the
// next kSegTail entries (where its last block ends), in LDS: nine consecutive
// lanes load one record, so a load instruction touches about as many cache lines
// as it has records, and the records of one element that meet in a row of
// the matrix come from the same lines at the same time.  One thread per
// scalar of a block sums from LDS and writes consecutive
// doubles.  The next tile's values are in flight (in registers) while a tile
// is summed, and the sources and block starts of the one after it.
// 32.8M triplets of the 64^3 + 2M contact system: 1.62 -> 0.78 ms (2.36 GB of
// records; one thread per block gathering its records one by one before),
// FP32 33^3 + 150k 91 -> 63 us, 11^3 + 3k 21 -> 8 us.  Tails of 64, 32 and 16
// entries: 0.92, 1.21 and 1.45 ms (a diagonal block has about 50 entries and
// runs past them), 128: 0.78; 4 or 8 workgroups per CU 0.78, 16 0.90.  Giving
// each XCD consecutive tiles changed nothing.
template <typename TV>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4))) void seg_reduce_kernel(int64_t        U,
                                                             const int64_t* d_m,
                                                             const int32_t* __restrict__ seg_start,
                                                             const uint32_t* __restrict__ seg_tile,
                                                             const int32_t* __restrict__ srcs,
                                                             const TV* __restrict__ vals,
                                                             double* out)
{
    constexpr int kCap  = kSegTile + kSegTail;
    constexpr int kLoad = (9 * kCap + kThreads - 1) / kThreads;
    static_assert(kSegTile == kThreads && kSegTail <= kThreads, "one entry and one block start per thread");
    __shared__ TV      sv[9 * kCap];
    __shared__ int32_t ss[2][kCap];
    __shared__ int32_t sb[2][kSegTile + 1];
    const uint32_t m   = (uint32_t)*d_m;
    const int32_t  nt  = (int32_t)seg_tiles(m);
    const int      tid = threadIdx.x;
    auto tile_of = [&](int64_t k) -> int32_t {  // the workgroup's k-th tile (nt: none)
        const int64_t t = k * gridDim.x + blockIdx.x;
        return t < nt ? (int32_t)t : nt;
    };
    // indices of a tile: its entries' sources, its blocks' starts
    int32_t  i_src = 0, i_tail = 0, i_sb = 0, i_end = 0;
    uint32_t hu0 = 0, hu1 = 0;
    auto heads = [&](int32_t t) {
        hu0 = t < nt ? seg_tile[t] : 0;
        hu1 = t < nt ? (t + 1 < nt ? seg_tile[t + 1] : (uint32_t)U) : 0;
    };
    auto index_load = [&](int32_t t) {  // uses hu0, hu1 of t
        const uint32_t e = seg_entry((uint32_t)t, tid), et = seg_entry((uint32_t)t, kSegTile + tid);
        i_src  = e < m ? srcs[e] : 0;
        i_tail = tid < kSegTail && et < m ? srcs[et] : 0;
        i_sb   = hu0 + tid < hu1 ? seg_start[hu0 + tid] : (int32_t)m;
        i_end  = hu1 < U ? seg_start[hu1] : (int32_t)m;
    };
    auto index_store = [&](int s, int nb) {
        ss[s][tid] = i_src;
        if(tid < kSegTail)
            ss[s][kSegTile + tid] = i_tail;
        if(tid < nb)
            sb[s][tid] = i_sb;
        if(tid == 0)
            sb[s][nb] = i_end;
    };
    TV v[kLoad];
    auto vals_load = [&](int s, int32_t c0, int nb) {
        const int f0 = nb ? 9 * (sb[s][0] - c0) : 0;
        const int f1 = nb ? 9 * min(sb[s][nb] - c0, kCap) : 0;
#pragma unroll
        for(int k = 0; k < kLoad; ++k)
        {
            const int f = k * kThreads + tid;
            if(f >= f0 && f < f1)
            {
                const int r = f / 9;
                v[k]        = vals[9 * (int64_t)ss[s][r] + (f - 9 * r)];
            }
        }
    };
    int32_t t0 = tile_of(0);
    if(t0 >= nt)
        return;
    heads(t0);
    uint32_t u0 = hu0;  // the current tile's blocks [u0, u0 + nb)
    int      nb = (int)(hu1 - hu0);
    index_load(t0);
    index_store(0, nb);
    int32_t t1 = tile_of(1);
    heads(t1);
    uint32_t n_u0 = hu0;
    int      n_nb = (int)(hu1 - hu0);
    index_load(t1);
    __syncthreads();
    vals_load(0, t0 * kSegTile, nb);
    index_store(1, n_nb);
    int32_t t2 = tile_of(2);
    heads(t2);
    __syncthreads();
    for(int k = 0;; ++k)
    {
        const int     cur = k & 1;
        const int32_t c0  = t0 * kSegTile;
#pragma unroll
        for(int q = 0; q < kLoad; ++q)
        {
            const int f = q * kThreads + tid;
            if(f < 9 * kCap)
                sv[f] = v[q];
        }
        __syncthreads();
        // the next tile's values, and the indices of the one after it
        if(t1 < nt)
            vals_load(cur ^ 1, t1 * kSegTile, n_nb);
        const uint32_t nn_u0 = hu0;
        const int      nn_nb = (int)(hu1 - hu0);
        if(t2 < nt)
            index_load(t2);
        const int32_t t3 = tile_of(k + 3);
        heads(t3);
        for(int i = tid; i < 9 * nb; i += kThreads)
        {
            const int     j = i / 9, q = i - 9 * j;
            int           e  = sb[cur][j] - c0;
            const int     e1 = sb[cur][j + 1] - c0, el = min(e1, kCap);
            double acc = (double)sv[9 * e++ + q];
            for(; e + 4 <= el; e += 4)
            {
                const double w0 = (double)sv[9 * e + q], w1 = (double)sv[9 * e + 9 + q],
                             w2 = (double)sv[9 * e + 18 + q], w3 = (double)sv[9 * e + 27 + q];
                acc = acc + w0;
                acc = acc + w1;
                acc = acc + w2;
                acc = acc + w3;
            }
            for(; e < el; ++e)
                acc = acc + (double)sv[9 * e + q];
            // a block running past the staged entries
            for(; e + 8 <= e1; e += 8)
            {
                TV w[8];
#pragma unroll
                for(int h = 0; h < 8; ++h)
                    w[h] = vals[9 * (int64_t)srcs[c0 + e + h] + q];
#pragma unroll
                for(int h = 0; h < 8; ++h)
                    acc = acc + (double)w[h];
            }
            for(; e < e1; ++e)
                acc = acc + (double)vals[9 * (int64_t)srcs[c0 + e] + q];
            out[upper_at(u0 + j, q)] = acc;
        }
        if(t1 >= nt)
            break;
        __syncthreads();
        if(t2 < nt)
            index_store(cur, nn_nb);
        t0   = t1;
        t1   = t2;
        t2   = t3;
        u0   = n_u0;
        nb   = n_nb;
        n_u0 = nn_u0;
        n_nb = nn_nb;
    }
}

// ---- BSR row offsets from sorted rows: row_ptr[r] = first u with rows[u] >= r
__global__ __launch_bounds__(kThreads) void row_ptr_kernel(int64_t U, const int32_t* rows, int32_t* row_ptr, int32_t B)
{
    for(int64_t u = (int64_t)blockIdx.x * kThreads + threadIdx.x; u <= U; u += (int64_t)gridDim.x * kThreads)
    {
        int32_t prev = (u == 0) ? -1 : rows[u - 1];
        int32_t cur  = (u == U) ? B : rows[u];
        for(int32_t r = prev + 1; r <= cur; ++r)
            row_ptr[r] = (int32_t)u;
    }
}

// the same for the lower entries, from their sorted keys
template <typename KeyT>
__global__ __launch_bounds__(kThreads) void lower_ptr_kernel(const int64_t* d_n, const KeyT* __restrict__ keys,
                                                            KeyCodec kc, int32_t* lower_ptr, int32_t B)
{
    const int64_t n = *d_n;
    for(int64_t k = (int64_t)blockIdx.x * kThreads + threadIdx.x; k <= n; k += (int64_t)gridDim.x * kThreads)
    {
        int32_t prev = -1, cur = B, lc;
        if(k > 0)
            kc.lo_rc((uint64_t)keys[k - 1], prev, lc);
        if(k < n)
            kc.lo_rc((uint64_t)keys[k], cur, lc);
        for(int32_t r = prev + 1; r <= cur; ++r)
            lower_ptr[r] = (int32_t)k;
    }
}

// ---- full BSR: lower part (transposed upper blocks, sorted by (col, row)) then
// upper part of each row

// chunk_row[c] = the first row whose first full-BSR block is at or after
// c kChunkStep (binary search in full_ptr); chunk_row[nchunks] = B
__global__ void chunk_row_kernel(const int32_t* __restrict__ fptr, int32_t B, int32_t nchunks, int32_t* chunk_row)
{
    for(int32_t c = blockIdx.x * blockDim.x + threadIdx.x; c <= nchunks; c += gridDim.x * blockDim.x)
    {
        if(c == nchunks)
        {
            chunk_row[c] = B;
            continue;
        }
        const int64_t target = (int64_t)c * kChunkStep;
        int32_t       lo = 0, hi = B;  // answer in [0, B]
        while(lo < hi)
        {
            const int32_t mid = lo + (hi - lo) / 2;
            if((int64_t)fptr[mid] >= target)
                hi = mid;
            else
                lo = mid + 1;
        }
        chunk_row[c] = lo;
    }
}

// blocks per full-BSR row (lower + upper; an empty row gets one zero diagonal
// block, so every row holds at least one), scanned into full_ptr afterwards
__global__ void full_count_kernel(const int32_t* lower_ptr, const int32_t* upper_ptr, uint32_t* cnt, int32_t B)
{
    for(int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i <= B; i += (int64_t)gridDim.x * blockDim.x)
    {
        if(i == B)
        {
            cnt[i] = 0;
            continue;
        }
        const int32_t c = (lower_ptr[i + 1] - lower_ptr[i]) + (upper_ptr[i + 1] - upper_ptr[i]);
        cnt[i]          = c > 0 ? (uint32_t)c : 1u;
    }
}

// A layout's blocks are written in two steps: a kernel that knows the layout
// gives every output block its index word and its source (the upper block, bit
// 31 where it is stored transposed; kNoBlock for a zero block), and
// fill_values_kernel moves the values.  One lane per upper block writing nine
// planes at its own places cost more than the bytes: its stores were pieces of
// a row's length (64^3 + 2M contacts, window layout: 276 us for the upper and 205 for
// the lower blocks, now 48 us for words and sources and 188 for the values).
constexpr uint32_t kTransposed = 0x80000000u;
constexpr uint32_t kNoBlock    = 0xffffffffu;

template <typename KeyT>
__global__ void full_place_kernel(int64_t        U,
                                  const int64_t* d_n,
                                  const KeyT* __restrict__ keys,
                                  KeyCodec       kc,
                                  const int32_t* __restrict__ src,
                                  const int32_t* __restrict__ rows,
                                  const int32_t* __restrict__ cols,
                                  const int32_t* __restrict__ upper_ptr,
                                  const int32_t* __restrict__ lower_ptr,
                                  const int32_t* __restrict__ full_ptr,
                                  int32_t        B,
                                  int32_t* __restrict__ fcols,
                                  uint32_t* __restrict__ from)
{
    const int64_t t0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, step = (int64_t)gridDim.x * blockDim.x;
    const int64_t n = *d_n;
    for(int64_t u = t0; u < U; u += step)
    {
        const int32_t i = rows[u];
        const int64_t d = (int64_t)full_ptr[i] + (lower_ptr[i + 1] - lower_ptr[i]) + (u - upper_ptr[i]);
        fcols[d]        = cols[u];
        from[d]         = (uint32_t)u;
    }
    for(int64_t k = t0; k < n; k += step)
    {
        int32_t i, j;  // lower row = upper col, lower col = upper row
        kc.lo_rc((uint64_t)keys[k], i, j);
        const int64_t d = (int64_t)full_ptr[i] + (k - lower_ptr[i]);
        fcols[d]        = j;
        from[d]         = (uint32_t)src[k] | kTransposed;
    }
    for(int64_t i = t0; i < B; i += step)
        if(lower_ptr[i + 1] == lower_ptr[i] && upper_ptr[i + 1] == upper_ptr[i])
        {
            fcols[full_ptr[i]] = (int32_t)i;
            from[full_ptr[i]]  = kNoBlock;
        }
}

// the nine planes of *d_n blocks from their sources: memory bound.  A block's nine
// scalars are read by nine consecutive lanes (72 B at a time, nine loads in
// flight per lane), turned in LDS where they are stored transposed, and
// written by plane, 256 consecutive blocks at a time.
template <typename VT>
__global__ __launch_bounds__(kThreads) void fill_values_kernel(const int32_t* d_n,
                                                              const uint32_t* __restrict__ from,
                                                              const double* __restrict__ uvals,
                                                              VT* __restrict__ planes,
                                                              int64_t        stride)
{
    __shared__ uint32_t sf[kThreads];
    __shared__ double   sv[9 * kThreads];
    const int64_t       n = *d_n;
    for(int64_t d0 = (int64_t)blockIdx.x * kThreads; d0 < n; d0 += (int64_t)gridDim.x * kThreads)
    {
        const int nb = (int)min((int64_t)kThreads, n - d0);
        __syncthreads();  // the last tile's blocks are read
        if((int)threadIdx.x < nb)
            sf[threadIdx.x] = from[d0 + threadIdx.x];
        __syncthreads();
        double v[9];
#pragma unroll
        for(int k = 0; k < 9; ++k)
        {
            const int      f = k * kThreads + threadIdx.x, j = f / 9, q = f - 9 * j;
            const uint32_t w = j < nb ? sf[j] : kNoBlock;
            v[k] = w == kNoBlock ? 0.0 : uvals[upper_at((int64_t)(w & ~kTransposed), q)];
        }
#pragma unroll
        for(int k = 0; k < 9; ++k)
        {
            const int f = k * kThreads + threadIdx.x, j = f / 9, q = f - 9 * j;
            if(j < nb)
                sv[9 * j + ((sf[j] & kTransposed) ? 3 * (q % 3) + q / 3 : q)] = v[k];
        }
        __syncthreads();
        if((int)threadIdx.x < nb)
#pragma unroll
            for(int q = 0; q < 9; ++q)
                planes[q * stride + d0 + threadIdx.x] = (VT)sv[9 * threadIdx.x + q];
    }
}

// ---- window layout (BsrMatrix::w*): blocks per row position; a row holds its
// upper blocks and the lower blocks whose other row is in another window.
// 16 lanes per row walk the row's lower entries together (coalesced reads of
// the transposed keys; one lane per row read them 16 times over).
constexpr int kRowLanes = 16;

template <typename KeyT>
__global__ __launch_bounds__(kThreads) void win_count_kernel(int32_t        B,
                                                            int            shift,
                                                            const int32_t* __restrict__ pos,
                                                            const int32_t* __restrict__ real,
                                                            const int32_t* __restrict__ row_ptr,
                                                            const int32_t* __restrict__ lower_ptr,
                                                            const KeyT* __restrict__ lkeys,
                                                            KeyCodec       kc,
                                                            uint32_t*      cnt)
{
    const int64_t groups = (int64_t)gridDim.x * (kThreads / kRowLanes);
    const int     lane   = threadIdx.x % kRowLanes;
    for(int64_t p = ((int64_t)blockIdx.x * kThreads + threadIdx.x) / kRowLanes; p <= B; p += groups)
    {
        if(p == B)
        {
            if(lane == 0)
                cnt[p] = 0;
            continue;
        }
        const int32_t v  = real[p];
        const int32_t ch = (int32_t)p >> shift;
        uint32_t      c  = 0;
        for(int32_t k = lower_ptr[v] + lane; k < lower_ptr[v + 1]; k += kRowLanes)
        {
            int32_t lr, i;  // i: the upper row
            kc.lo_rc((uint64_t)lkeys[k], lr, i);
            c += (pos[i] >> shift) != ch ? 1u : 0u;
        }
#pragma unroll
        for(int o = kRowLanes / 2; o > 0; o >>= 1)
            c += __shfl_xor(c, o, kWave);
        if(lane == 0)
            cnt[p] = c + (uint32_t)(row_ptr[v + 1] - row_ptr[v]);
    }
}

__host__ __device__ __forceinline__ int32_t win_inner_word(int32_t li, int32_t lj)
{
    return (int32_t)(0x80000000u | ((uint32_t)li << 15) | (uint32_t)lj);
}

// words and sources of the window layout's blocks: 16 lanes per row, its upper
// blocks and then the lower ones of other windows
template <typename KeyT>
__global__ __launch_bounds__(kThreads) void win_place_kernel(int32_t        B,
                                                            int            shift,
                                                            const int32_t* __restrict__ pos,
                                                            const int32_t* __restrict__ real,
                                                            const int32_t* __restrict__ row_ptr,
                                                            const int32_t* __restrict__ cols,
                                                            const int32_t* __restrict__ lower_ptr,
                                                            const KeyT* __restrict__ lkeys,
                                                            KeyCodec       kc,
                                                            const int32_t* __restrict__ lsrc,
                                                            const int32_t* __restrict__ wptr,
                                                            int32_t* __restrict__ words,
                                                            uint32_t* __restrict__ from)
{
    const int32_t mask   = (1 << shift) - 1;
    const int64_t groups = (int64_t)gridDim.x * (kThreads / kRowLanes);
    const int     lane   = threadIdx.x % kRowLanes;
    const int     gsh    = (int)(threadIdx.x % kWave) & ~(kRowLanes - 1);  // the group's first lane in the wave
    // the group's rows run in lockstep: every group of a wave takes the same
    // number of rounds (the wave-wide ballots below need all 64 lanes)
    const int64_t first  = ((int64_t)blockIdx.x * kThreads + threadIdx.x) / kRowLanes;
    const int64_t rounds = (B + groups - 1) / groups;
    for(int64_t it = 0; it < rounds; ++it)
    {
        const int64_t p    = first + it * groups;
        const bool    live = p < B;
        const int32_t v    = live ? real[p] : 0;
        const int32_t ch   = (int32_t)p >> shift;
        const int32_t lo = live ? lower_ptr[v] : 0, hi = live ? lower_ptr[v + 1] : 0;
        int64_t       d  = live ? (int64_t)wptr[p] : 0;
        if(live)
        {
            const int32_t u0 = row_ptr[v], u1 = row_ptr[v + 1];
            for(int32_t u = u0 + lane; u < u1; u += kRowLanes)
            {
                const int32_t pj    = pos[cols[u]];
                words[d + (u - u0)] = (pj >> shift) == ch ? win_inner_word((int32_t)p & mask, pj & mask) : pj;
                from[d + (u - u0)]  = (uint32_t)u;
            }
            d += u1 - u0;
        }
        // the wave's longest lower list bounds its rounds
        int32_t len = hi - lo;
#pragma unroll
        for(int o = kWave / 2; o > 0; o >>= 1)
            len = max(len, __shfl_xor(len, o, kWave));
        for(int32_t b = 0; b < len; b += kRowLanes)
        {
            const int32_t k   = lo + b + lane;
            int32_t       i   = 0, pi = 0;
            bool          out = false;
            if(k < hi)
            {
                int32_t lr;
                kc.lo_rc((uint64_t)lkeys[k], lr, i);
                pi  = pos[i];
                out = (pi >> shift) != ch;  // an inner block is stored once, with row i
            }
            const uint64_t  bal  = __ballot(out);
            const uint32_t  mine = (uint32_t)(bal >> gsh) & ((1u << kRowLanes) - 1u);
            if(out)
            {
                const int64_t dk = d + __popc(mine & ((1u << lane) - 1u));
                words[dk]        = pi;
                from[dk]         = (uint32_t)lsrc[k] | kTransposed;
            }
            d += __popc(mine);
        }
    }
}

// lowest row and highest row + 1 of every window (batched solves skip the
// windows that hold no row of a running system): one workgroup per window
__global__ __launch_bounds__(kThreads) void win_range_kernel(int32_t B, int shift, int32_t nchunks,
                                                            const int32_t* __restrict__ real, int32_t* lo,
                                                            int32_t* hi)
{
    __shared__ int32_t smin[kThreads / kWave], smax[kThreads / kWave];
    for(int32_t c = blockIdx.x; c < nchunks; c += gridDim.x)
    {
        const int32_t p0 = c << shift, p1 = (int32_t)std::min<int64_t>((int64_t)(c + 1) << shift, B);
        int32_t       a = B, b = -1;
        for(int32_t p = p0 + (int32_t)threadIdx.x; p < p1; p += kThreads)
        {
            a = std::min(a, real[p]);
            b = std::max(b, real[p]);
        }
#pragma unroll
        for(int o = kWave / 2; o > 0; o >>= 1)
        {
            a = std::min(a, __shfl_xor(a, o, kWave));
            b = std::max(b, __shfl_xor(b, o, kWave));
        }
        if(threadIdx.x % kWave == 0)
        {
            smin[threadIdx.x / kWave] = a;
            smax[threadIdx.x / kWave] = b;
        }
        __syncthreads();
        if(threadIdx.x == 0)
        {
            for(int w = 1; w < kThreads / kWave; ++w)
            {
                a = std::min(a, smin[w]);
                b = std::max(b, smax[w]);
            }
            lo[c] = a;
            hi[c] = b + 1;
        }
        __syncthreads();
    }
}

int key_bits_for(uint64_t max_key)
{
    int bits = 0;
    while(max_key > 0)
    {
        ++bits;
        max_key >>= 1;
    }
    return bits > 0 ? bits : 1;
}

void scan_exclusive(uint32_t* data, int64_t n, DBuf<uint32_t>& chunk, int64_t* total, hipStream_t s)
{
    if(n <= 64 * 1024)
    {
        scan_small_kernel<<<1, 1024, 0, s>>>(data, n, total);
        return;
    }
    int nch = ceil_div(n, kScanChunk);
    chunk.resize((size_t)nch + 1);
    scan_reduce_kernel<<<nch, kThreads, 0, s>>>(data, n, chunk.data());
    scan_small_kernel<<<1, 1024, 0, s>>>(chunk.data(), nch, total);
    scan_down_kernel<<<nch, kThreads, 0, s>>>(data, n, chunk.data());
}

int grid_of(int64_t n)
{
    return std::max(1, std::min(ceil_div(n, kThreads), device_cu_count() * 16));
}

// fill_values_kernel: its LDS allows eight workgroups per CU
int fill_grid(int64_t n)
{
    return (int)std::max<int64_t>(1, std::min<int64_t>((n + kThreads - 1) / kThreads, (int64_t)device_cu_count() * 8));
}
}  // namespace

MatrixConverter::~MatrixConverter()
{
    if(pinned_)
        (void)hipHostFree(pinned_);
}

template <typename KeyT, typename First>
int radix_sort_from(First           first,
                    KeyT*           k0,
                    int32_t*        v0,
                    KeyT*           k1,
                    int32_t*        v1,
                    const int64_t*  d_n,
                    int64_t         nmax,
                    int             low,
                    int             bits,
                    DBuf<uint32_t>& hist,
                    hipStream_t     s);

// compaction + stable radix sort of (key, source) pairs; returns the buffer
// index holding the result, *d_count = number of kept entries (device)
template <int MODE, typename KeyT>
int MatrixConverter::compact_sort(int64_t        n,
                                  const int32_t* rows,
                                  const int32_t* cols,
                                  int32_t        B,
                                  int64_t*       d_count,
                                  double         ratio,
                                  hipStream_t    s)
{
    const int ntiles = ceil_div(n, kTile);
    tile_cnt_.resize((size_t)ntiles + 1, ratio);
    keys_[0].resize((size_t)n, ratio);
    keys_[1].resize((size_t)n, ratio);
    srcs_[0].resize((size_t)n, ratio);
    srcs_[1].resize((size_t)n, ratio);
    hist_.resize((size_t)256 * (std::max(ntiles, (int)(kFewKeys / kFewTile)) + 1), ratio);
    if(!(MODE == 0 && counted_))
        cv_count_kernel<MODE><<<ntiles, kThreads, 0, s>>>(n, rows, cols, B, tile_cnt_.data(), nullptr);
    counted_ = false;
    scan_exclusive(tile_cnt_.data(), ntiles, chunk_, d_count, s);
    KeyT* k0 = reinterpret_cast<KeyT*>(keys_[0].data());
    KeyT* k1 = reinterpret_cast<KeyT*>(keys_[1].data());
    // compaction (the kept count, *d_count, from the tile counts) and a stable
    // LSD radix sort (matrix_converter.inl:1579-1616) on the key's bits, whose
    // first pass reads the triplets' (row, col) and skips the dropped entries
    // (mode 1: the upper blocks come in row order, so a stable sort by column
    // alone gives (column, row))
    TripletSource<MODE, KeyT> first{rows, cols, n, B, codec_};
    const int                 low  = MODE == 1 ? codec_.lo_shift() : 0;
    const int                 bits = MODE == 1 ? low + key_bits_for((uint64_t)std::max(B - 1, 1)) : key_bits_;
    return radix_sort_from<KeyT>(first, k0, srcs_[0].data(), k1, srcs_[1].data(), d_count, n, low, bits, hist_, s);
}

void MatrixConverter::build_window(BsrMatrix& A, int shape, bool want32, double ratio, hipStream_t s)
{
    MI_REQUIRE(shape >= 0 && shape < spmv_shape_count(), MI_ERR_ARG, "window layout: unknown kernel shape");
    const int shift = spmv_shape_shift(shape);
    MI_REQUIRE(shift >= 4 && shift <= kWinShiftMax, MI_ERR_ARG, "window layout: window size out of range");
    A.wshape = shape;
    const int32_t B = A.B;
    MI_REQUIRE(A.wpos.data() && A.wreal.data() && A.wpos.size() >= (size_t)B && A.wreal.size() >= (size_t)B,
               MI_ERR_STATE, "window layout: no row order");
    A.wshift   = shift;
    A.wnchunks = (int32_t)(((int64_t)B + (1 << shift) - 1) >> shift);
    A.wptr.resize((size_t)B + 1, ratio);
    A.wchunk_lo.resize((size_t)std::max(1, A.wnchunks), ratio);
    A.wchunk_hi.resize((size_t)std::max(1, A.wnchunks), ratio);
    A.has_win = false;
    if(B == 0)
    {
        A.wblocks = 0;
        A.has_win = true;
        return;
    }
    const int64_t U = A.U;
    uint32_t*     cnt = reinterpret_cast<uint32_t*>(A.wptr.data());  // scanned in place
    const bool narrow = codec_.bb > 0;
    if(narrow)
        win_count_kernel<uint32_t><<<grid_of(((int64_t)B + 1) * kRowLanes), kThreads, 0, s>>>(
            B, shift, A.wpos.data(), A.wreal.data(), A.row_ptr.data(), lower_ptr_.data(),
            U > 0 ? key_ptr<uint32_t>(tcur_) : nullptr, codec(), cnt);
    else
        win_count_kernel<uint64_t><<<grid_of(((int64_t)B + 1) * kRowLanes), kThreads, 0, s>>>(
            B, shift, A.wpos.data(), A.wreal.data(), A.row_ptr.data(), lower_ptr_.data(),
            U > 0 ? key_ptr<uint64_t>(tcur_) : nullptr, codec(), cnt);
    scan_exclusive(cnt, (int64_t)B + 1, chunk_, counts_.data() + 4, s);
    win_range_kernel<<<std::max(1, std::min(A.wnchunks, device_cu_count() * 8)), kThreads, 0, s>>>(
        B, shift, A.wnchunks, A.wreal.data(), A.wchunk_lo.data(), A.wchunk_hi.data());
    // the window layout holds at most the full BSR's 2U blocks; four blocks of
    // padding past the last, and a plane stride that is a multiple of 4 (the
    // SpMV reads up to four consecutive blocks per load)
    const int64_t wmax = 2 * U;
    A.wwords.resize((size_t)wmax + 4, ratio);
    A.wstride = ((int64_t)A.wwords.cap + 3) & ~(int64_t)3;
    if(want32)
        A.wvals32.resize((size_t)9 * A.wstride);
    else
        A.wvals.resize((size_t)9 * A.wstride);
    if(U > 0)
    {
        from_.resize((size_t)wmax, ratio);
        if(narrow)
            win_place_kernel<uint32_t><<<grid_of((int64_t)B * kRowLanes), kThreads, 0, s>>>(
                B, shift, A.wpos.data(), A.wreal.data(), A.row_ptr.data(), A.cols.data(), lower_ptr_.data(),
                key_ptr<uint32_t>(tcur_), codec(), srcs_[tcur_].data(), A.wptr.data(), A.wwords.data(), from_.data());
        else
            win_place_kernel<uint64_t><<<grid_of((int64_t)B * kRowLanes), kThreads, 0, s>>>(
                B, shift, A.wpos.data(), A.wreal.data(), A.row_ptr.data(), A.cols.data(), lower_ptr_.data(),
                key_ptr<uint64_t>(tcur_), codec(), srcs_[tcur_].data(), A.wptr.data(), A.wwords.data(), from_.data());
        if(want32)
            fill_values_kernel<float><<<fill_grid(wmax), kThreads, 0, s>>>(A.wptr.data() + B, from_.data(),
                                                                           A.vals.data(), A.wvals32.data(), A.wstride);
        else
            fill_values_kernel<double><<<fill_grid(wmax), kThreads, 0, s>>>(A.wptr.data() + B, from_.data(),
                                                                            A.vals.data(), A.wvals.data(), A.wstride);
    }
    MI_HIP(hipGetLastError());
    A.wblocks = -1;  // read back lazily (window_blocks)
    A.has_win = true;
}

// stable LSD passes of 8 bits over the key bits [low, bits); the first reads `first` (pairs or triplets),
// the rest ping-pong between the buffers; returns the buffer holding the result
template <typename KeyT, typename First>
int radix_sort_from(First           first,
                    KeyT*           k0,
                    int32_t*        v0,
                    KeyT*           k1,
                    int32_t*        v1,
                    const int64_t*  d_n,
                    int64_t         nmax,
                    int             low,
                    int             bits,
                    DBuf<uint32_t>& hist,
                    hipStream_t     s)
{
    const bool few    = nmax <= kFewKeys;
    const int  ntiles = ceil_div(nmax, few ? kFewTile : kTile);
    if(ntiles == 0)
        return 0;
    hist.resize((size_t)256 * (ntiles + 1));  // the counts, the digits' totals
    uint32_t* totals = hist.data() + (size_t)256 * ntiles;
    KeyT*     kb[2]  = {k0, k1};
    int32_t*  vb[2]  = {v0, v1};
    int       cur    = 0;
    for(int shift = low; shift < bits; shift += 8)
    {
        const uint32_t dmask = (1u << std::min(8, bits - shift)) - 1u;
        auto           pass  = [&](auto src) {
            using Src = decltype(src);
            auto go   = [&](auto tag) {
                constexpr bool kFew = decltype(tag)::value;
                rs_hist_kernel<KeyT, Src, kFew><<<ntiles, kThreads, 0, s>>>(src, shift, dmask, hist.data(), ntiles);
                if(!kFew)
                    rs_rows_kernel<<<256, kThreads, 0, s>>>(hist.data(), ntiles, totals);
                rs_scatter_kernel<KeyT, Src, kFew><<<ntiles, kThreads, 0, s>>>(src, kb[cur ^ 1], vb[cur ^ 1], shift,
                                                                               dmask, hist.data(), ntiles, totals);
            };
            if(few)
                go(std::true_type{});
            else
                go(std::false_type{});
        };
        if(shift == low)
            pass(first);
        else
            pass(PairSource<KeyT>{d_n, kb[cur], vb[cur]});
        cur ^= 1;
    }
    return cur;
}

template <typename KeyT>
int radix_sort_pairs_t(KeyT*           k0,
                       int32_t*        v0,
                       KeyT*           k1,
                       int32_t*        v1,
                       const int64_t*  d_n,
                       int64_t         nmax,
                       int             bits,
                       DBuf<uint32_t>& hist,
                       hipStream_t     s)
{
    return radix_sort_from<KeyT>(PairSource<KeyT>{d_n, k0, v0}, k0, v0, k1, v1, d_n, nmax, 0, bits, hist, s);
}

int radix_sort_pairs(uint64_t*       k0,
                     int32_t*        v0,
                     uint64_t*       k1,
                     int32_t*        v1,
                     const int64_t*  d_n,
                     int64_t         nmax,
                     int             bits,
                     DBuf<uint32_t>& hist,
                     hipStream_t     s)
{
    return radix_sort_pairs_t<uint64_t>(k0, v0, k1, v1, d_n, nmax, bits, hist, s);
}

void exclusive_scan_u32(uint32_t* data, int64_t n, DBuf<uint32_t>& chunk, int64_t* d_total, hipStream_t s)
{
    scan_exclusive(data, n, chunk, d_total, s);
}

int radix_key_bits(uint64_t max_key)
{
    return key_bits_for(max_key);
}

void MatrixConverter::convert(int32_t        B,
                              int64_t        T,
                              const int32_t* rows,
                              const int32_t* cols,
                              const void*    vals,
                              bool           vals32,
                              BsrMatrix&     out,
                              bool           want32,
                              bool           build_full,
                              double         ratio,
                              hipStream_t    s)
{
    MI_REQUIRE(B >= 0 && T >= 0, MI_ERR_ARG, "convert_sym: negative size");
    MI_REQUIRE(T < ((int64_t)1 << 31), MI_ERR_ARG, "convert_sym: more than 2^31-1 triplets");
    MI_REQUIRE(T == 0 || (rows && cols && vals), MI_ERR_ARG, "convert_sym: null triplet arrays");
    out.B = B;
    out.row_ptr.resize((size_t)B + 1, ratio);
    out.full_ptr.resize((size_t)B + 1, ratio);
    out.has32 = want32;
    if(!pinned_)
        MI_HIP(hipHostMalloc((void**)&pinned_, 8 * sizeof(int64_t)));
    counts_.resize(6);
    MI_HIP(hipMemsetAsync(counts_.data(), 0, 6 * sizeof(int64_t), s));
    codec_ = KeyCodec{(uint64_t)std::max(B, 1), 0, 0};
    out.has_win  = false;
    out.has_full = false;
    if(T == 0 || B == 0)
    {
        out.U = 0;
        MI_HIP(hipMemsetAsync(out.row_ptr.data(), 0, sizeof(int32_t) * ((size_t)B + 1), s));
        MI_HIP(hipMemsetAsync(out.full_ptr.data(), 0, sizeof(int32_t) * ((size_t)B + 1), s));
        lower_ptr_.resize((size_t)B + 1, ratio);
        MI_HIP(hipMemsetAsync(lower_ptr_.data(), 0, sizeof(int32_t) * ((size_t)B + 1), s));
        return;
    }
    int64_t* d_m   = counts_.data();      // kept triplets
    int64_t* d_u   = counts_.data() + 1;  // unique upper blocks
    int64_t* d_off = counts_.data() + 2;  // off-diagonal upper blocks

    // 1. count the kept triplets and their largest col - row; one host read
    // of the band chooses the key (narrow 32-bit keys when they fit)
    const int ntiles = ceil_div(T, kTile);
    {
        tile_cnt_.resize((size_t)ntiles + 1, ratio);
        int32_t* d_band = reinterpret_cast<int32_t*>(counts_.data() + 5);
        cv_count_kernel<0><<<ntiles, kThreads, 0, s>>>(T, rows, cols, B, tile_cnt_.data(), d_band);
        MI_HIP(hipMemcpyAsync(pinned_ + 5, counts_.data() + 5, sizeof(int64_t), hipMemcpyDeviceToHost, s));
        MI_HIP(hipStreamSynchronize(s));
        const int32_t band  = (int32_t)(pinned_[5] & 0x7fffffff);
        const int     bb    = key_bits_for((uint64_t)std::max(band, 1));
        const int     nbits = key_bits_for(((uint64_t)(B - 1) << bb) | (uint64_t)band);
        static const bool wide_only = [] {
            const char* e = std::getenv("MI_SORT_KEY");
            return e && std::string(e) == "wide";
        }();
        if(!wide_only && nbits <= 32)
        {
            codec_    = KeyCodec{(uint64_t)B, bb, band};
            key_bits_ = nbits;
        }
        else
        {
            codec_    = KeyCodec{(uint64_t)B, 0, 0};
            key_bits_ = key_bits_for((uint64_t)B * (uint64_t)B - 1ull);
        }
        counted_ = true;
    }
    const bool narrow = codec_.bb > 0;
    // 2-4. scan, compact, stable radix sort (matrix_converter.inl:1579-1616)
    const int cur = narrow ? compact_sort<0, uint32_t>(T, rows, cols, B, d_m, ratio, s)
                           : compact_sort<0, uint64_t>(T, rows, cols, B, d_m, ratio, s);

    // 5-6. run-length encode (1626-1650); the one host read-back sizes the outputs
    if(narrow)
        rle_count_kernel<uint32_t><<<ntiles, kThreads, 0, s>>>(d_m, key_ptr<uint32_t>(cur), tile_cnt_.data());
    else
        rle_count_kernel<uint64_t><<<ntiles, kThreads, 0, s>>>(d_m, key_ptr<uint64_t>(cur), tile_cnt_.data());
    scan_exclusive(tile_cnt_.data(), ntiles, chunk_, d_u, s);
    MI_HIP(hipMemcpyAsync(pinned_, counts_.data(), 2 * sizeof(int64_t), hipMemcpyDeviceToHost, s));
    MI_HIP(hipStreamSynchronize(s));
    const int64_t U = pinned_[1];
    out.U           = U;
    out.rows.resize((size_t)(U > 0 ? U : 1), ratio);
    out.cols.resize((size_t)(U > 0 ? U : 1), ratio);
    out.vals.resize((size_t)9 * out.rows.cap);
    seg_start_.resize((size_t)(U > 0 ? U : 1), ratio);
    seg_tile_.resize((size_t)ntiles * (kTile / kSegTile), ratio);
    if(narrow)
        rle_write_kernel<uint32_t><<<ntiles, kThreads, 0, s>>>(d_m, key_ptr<uint32_t>(cur), tile_cnt_.data(),
                                                               codec(), out.rows.data(), out.cols.data(),
                                                               seg_start_.data(), seg_tile_.data());
    else
        rle_write_kernel<uint64_t><<<ntiles, kThreads, 0, s>>>(d_m, key_ptr<uint64_t>(cur), tile_cnt_.data(),
                                                               codec(), out.rows.data(), out.cols.data(),
                                                               seg_start_.data(), seg_tile_.data());

    // 7-8. segmented reduce over the sorted permutation (1652-1698)
    if(U > 0)
    {
        // as many workgroups as are resident at once (4 per CU)
        const int  nseg   = std::min(ceil_div(T, kSegTile), device_cu_count() * 4);
        const auto reduce = [&](auto* v) {
            seg_reduce_kernel<<<nseg, kThreads, 0, s>>>(U, d_m, seg_start_.data(), seg_tile_.data(),
                                                        srcs_[cur].data(), v, out.vals.data());
        };
        if(vals32)
            reduce(static_cast<const float*>(vals));
        else
            reduce(static_cast<const double*>(vals));
    }
    row_ptr_kernel<<<grid_of(U + 1), kThreads, 0, s>>>(U, out.rows.data(), out.row_ptr.data(), B);

    // the transpose of the off-diagonal upper blocks (the lower triangle)
    const int tcur = narrow ? compact_sort<1, uint32_t>(U, out.rows.data(), out.cols.data(), B, d_off, ratio, s)
                            : compact_sort<1, uint64_t>(U, out.rows.data(), out.cols.data(), B, d_off, ratio, s);
    tcur_          = tcur;
    lower_ptr_.resize((size_t)B + 1, ratio);
    if(narrow)
        lower_ptr_kernel<uint32_t><<<grid_of(U + 1), kThreads, 0, s>>>(d_off, key_ptr<uint32_t>(tcur), codec(),
                                                                       lower_ptr_.data(), B);
    else
        lower_ptr_kernel<uint64_t><<<grid_of(U + 1), kThreads, 0, s>>>(d_off, key_ptr<uint64_t>(tcur), codec(),
                                                                       lower_ptr_.data(), B);
    out.has_win  = false;
    out.has_full = false;
    if(build_full)
        this->build_full(out, want32, ratio, s);
    MI_HIP(hipGetLastError());
}

// the full BSR (both triangles) of the last conversion, from its upper BCOO
// and its sorted lower keys (both kept until the next conversion)
void MatrixConverter::build_full(BsrMatrix& out, bool want32, double ratio, hipStream_t s)
{
    const int32_t B      = out.B;
    const int64_t U      = out.U;
    const bool    narrow = codec_.bb > 0;
    const int     tcur   = tcur_;
    int64_t*      d_off  = counts_.data() + 2;
    if(B == 0)
        return;
    {
        uint32_t* cnt = reinterpret_cast<uint32_t*>(out.full_ptr.data());  // scanned in place
        full_count_kernel<<<grid_of(B + 1), kThreads, 0, s>>>(lower_ptr_.data(), out.row_ptr.data(), cnt, B);
        scan_exclusive(cnt, (int64_t)B + 1, chunk_, counts_.data() + 3, s);
    }
    // SpMV chunks over the full rows (the full BSR has at most 2U + B blocks)
    const int64_t fmax = 2 * U + B;
    out.nchunks = (int32_t)std::max<int64_t>(1, (fmax + kChunkStep - 1) / kChunkStep);
    out.chunk_row.resize((size_t)out.nchunks + 1, ratio);
    chunk_row_kernel<<<grid_of(out.nchunks + 1), kThreads, 0, s>>>(out.full_ptr.data(), B, out.nchunks,
                                                                   out.chunk_row.data());
    // two blocks past the end: the FP32 SpMV reads blocks in aligned pairs;
    // an even plane stride keeps every pair 8-byte aligned
    out.fcols.resize((size_t)fmax + 2, ratio);
    out.fstride = ((int64_t)out.fcols.cap + 1) & ~(int64_t)1;
    from_.resize((size_t)fmax, ratio);
    if(narrow)
        full_place_kernel<uint32_t><<<grid_of(std::max(U, (int64_t)B)), kThreads, 0, s>>>(
            U, d_off, key_ptr<uint32_t>(tcur), codec(), srcs_[tcur].data(), out.rows.data(), out.cols.data(),
            out.row_ptr.data(), lower_ptr_.data(), out.full_ptr.data(), B, out.fcols.data(), from_.data());
    else
        full_place_kernel<uint64_t><<<grid_of(std::max(U, (int64_t)B)), kThreads, 0, s>>>(
            U, d_off, key_ptr<uint64_t>(tcur), codec(), srcs_[tcur].data(), out.rows.data(), out.cols.data(),
            out.row_ptr.data(), lower_ptr_.data(), out.full_ptr.data(), B, out.fcols.data(), from_.data());
    if(want32)
    {
        out.fvals32.resize((size_t)9 * out.fstride);
        fill_values_kernel<float><<<fill_grid(fmax), kThreads, 0, s>>>(out.full_ptr.data() + B, from_.data(),
                                                                       out.vals.data(), out.fvals32.data(), out.fstride);
    }
    else
    {
        out.fvals.resize((size_t)9 * out.fstride);
        fill_values_kernel<double><<<fill_grid(fmax), kThreads, 0, s>>>(out.full_ptr.data() + B, from_.data(),
                                                                        out.vals.data(), out.fvals.data(), out.fstride);
    }
    out.has_full = true;
    MI_HIP(hipGetLastError());
}
}  // namespace mi
