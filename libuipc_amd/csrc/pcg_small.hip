// The PCG iterations of a small system in one cooperative launch.
//
// Replaces, for systems of at most kSmallRows slots on the full BSR,
// LinearFusedPCG::run_iteration (linear_system/linear_fused_pcg.cu:1374-1594)
// and the captured blocks of it: same recurrences, preconditioners and stopping
// rule, other summation orders.
//
// Bound by latency: five dependent launches per MAS iteration took 4.6-5.4 us
// each (three with 3x3 block Jacobi), whatever the size, where the data of an
// iteration fits the registers.  So one workgroup of 1,024 threads per CU
// keeps 64 rows (four MAS clusters) for the whole solve:
//   * its blocks in registers (three per thread, rows' blocks end to end over
//     the threads), the MAS inverses of its clusters in registers (12 entries of
//     one row per thread; threads 768.. hold one coarse cluster's);
//   * x, r, p, z of its rows and p of every column it meets in LDS: a column's p
//     is updated by its readers, p = z + beta p, so that only z travels;
//   * workgroups meet at exchanges (two per iteration with 3x3 block Jacobi,
//     three with MAS levels: p.Ap and the restricted Ap; the coarse Z; r.z and
//     r.r).
//
// An exchange: every workgroup stores an epoch and its partial sums, then
// polls every other's; each adds them in the same order, so all take the
// same decisions.  All data that passes between workgroups is stored and
// loaded by relaxed agent-scope atomics: they go to the point of coherence of
// the XCDs' L2s, so no L2 is written back or invalidated (an agent-scope
// release and acquire per exchange cost 6 us at 64 workgroups and 20 at 256,
// against 1.8 and 2.6).  Such a store has reached that point when its wave's
// vmcnt counts it done; every wave waits for that, then the workgroup's barrier,
// before the workgroup's words are stored.  A partial sum is halved over two
// 64-bit words that each carry the epoch, so a word is never read half new;
// words alternate between two buffers: a workgroup that stores epoch e + 2 has
// seen all of epoch e + 1, which every workgroup stores after it has read all
// of epoch e.
//
// The cooperative launch guarantees that all workgroups are resident, within one
// process; a wait ends after a time (4 s) all the same, and the caller then solves
// again from its start by launches.
//
// Rows are split by their count, not by their blocks, so one workgroup may hold
// what all others wait for.  A launch whose heaviest workgroup is past the limits
// below gives up before its first iteration (unfit), and the caller takes the
// launches, whose SpMV is split by blocks.  us per iteration against theirs, by a
// workgroup's blocks:
//   2,048 columns or fewer: 7,455 blocks (12^3 + 200k contacts) 30 against 33, 5,726
//     (8^3 + 100k) 24 (33); 7,649 random ones of 2,048 rows 6.9 (5.5);
//   more columns: 2,741 blocks (random rows) 7.4 (9.2); 3,223, eight rows of 319
//     among them, 21.0 (16.5); 16 rows of 2,000 and more together 110 to 1,230
//     (33 to 117), 64 of 13,000 4,887 (136);
//   one long row, which is as serial in the launches: of 4,000 blocks 43 to 49
//     (42 to 57), of 13,000 86 to 102 (108 to 125), two of 1,500 31 (25).
#include <algorithm>

#include "linsys.hpp"

namespace mi
{
namespace
{
constexpr int      kNT        = 1024;
constexpr int      kRows      = 64;             // slots per workgroup
constexpr int      kOwn       = 3 * kRows;      // their scalars, one per thread
constexpr int      kPer       = 3;              // blocks per thread in registers
constexpr int      kStage     = kPer * kNT;     // blocks per stage
constexpr int      kCols      = 2048;           // columns whose p is kept in LDS
constexpr int      kMaxWg     = kSmallRows / kRows;
constexpr int      kFitNear   = 7500;           // blocks of a workgroup whose columns are all in LDS
constexpr int      kFitLong   = 2048;           // ... beside its longest row, where they are not
constexpr int      kBitWords  = kSmallRows / 32;
constexpr int      kLvl       = 5;              // coarse levels
constexpr int      kBank      = 16;
constexpr int      kSym       = 136;
static_assert(kMaxWg <= 256, "one polled workgroup per thread of four waves");

__device__ __forceinline__ void put(double* p, double v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double get(const double* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void put(uint64_t* p, uint64_t v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t get(const uint64_t* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// the sum over the lane's quad, in every lane of it
__device__ __forceinline__ double quad_sum(double v)
{
    v += dpp_f64<kDppQuadXor1>(v);
    v += dpp_f64<kDppQuadXor2>(v);
    return v;
}

// a value the compiler must take as new: what is derived from it in a loop is
// computed there, not kept in registers over the whole loop
template <typename T>
__device__ __forceinline__ void renew(T& v)
{
    asm volatile("" : "+v"(v));
}

struct Exchange
{
    uint64_t* words;  // 2 buffers of kMaxWg x 4
    uint32_t  epoch = 0;
    int       wgs, me;
    int64_t   wait_ticks;  // of the 100 MHz clock; 0: a wait ends at its first look
    double (*red)[4][2];   // LDS, by epoch parity
    int* failed;          // LDS

    // NV values summed over the workgroups in their order; false when a wait
    // has run out.  A workgroup's value k is the sum of part[k][0 .. waves), LDS
    // that its waves have written.  All threads call it; what any of them stored
    // with put() before is seen by the others' get() after.
    template <int NV, int kParts = 1>
    __device__ __forceinline__ bool run(const double (*part)[kNT / kWave], double& v0, double& v1)
    {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        ++epoch;
        constexpr int  kWords = NV == 0 ? 1 : 2 * NV;
        int            t      = threadIdx.x;
        renew(t);
        const int      par    = epoch & 1u;
        uint64_t*      buf    = words + (size_t)par * kMaxWg * 4;
        const uint64_t tag    = (uint64_t)epoch << 32;
        if(t < kWords)
        {
            uint64_t b = 0ull;
            if constexpr(NV > 0)
            {
                double s = part[t / 2][0];
#pragma unroll
                for(int k = 1; k < kParts; ++k)
                    s += part[t / 2][k];
                b = __builtin_bit_cast(uint64_t, s);
            }
            put(buf + 4 * me + t, tag | (NV == 0 ? 0ull : (t & 1) ? b >> 32 : b & 0xffffffffull));
        }
        if(t < kMaxWg)
        {
            const bool     mine  = t < wgs;
            uint64_t       w[kWords];
            const uint64_t start = wall_clock64();
            for(uint32_t spin = 0;; ++spin)
            {
                bool ok = true;
                if(mine)
#pragma unroll
                    for(int k = 0; k < kWords; ++k)
                    {
                        w[k] = get(buf + 4 * t + k);
                        ok   = ok && (uint32_t)(w[k] >> 32) == epoch;
                    }
                if(__all(ok))
                    break;
                if(wait_ticks == 0 || ((spin & 255u) == 255u && wall_clock64() - start > (uint64_t)wait_ticks))
                {
                    *failed = 1;
                    break;
                }
            }
            if constexpr(NV > 0)
            {
                double s = mine ? __builtin_bit_cast(double, (w[1] << 32) | (w[0] & 0xffffffffull)) : 0.0;
                s        = wave_total(s);
                double q = 0.0;
                if constexpr(NV > 1)
                {
                    q = mine ? __builtin_bit_cast(double, (w[3] << 32) | (w[2] & 0xffffffffull)) : 0.0;
                    q = wave_total(q);
                }
                if(t % kWave == 0)
                {
                    red[par][t / kWave][0] = s;
                    red[par][t / kWave][1] = q;
                }
            }
        }
        __syncthreads();
        if constexpr(NV > 0)
            v0 = (red[par][0][0] + red[par][1][0]) + (red[par][2][0] + red[par][3][0]);
        if constexpr(NV > 1)
            v1 = (red[par][0][1] + red[par][1][1]) + (red[par][2][1] + red[par][3][1]);
        return *failed == 0;
    }
};

// clears the exchange words and the restricted r and Ap (nodes no vertex feeds
// stay 0); copies x to x0 where a solve that starts from it may have to start again
__global__ void pcg_small_clear_kernel(uint64_t* words, int64_t nwords, double* R, int64_t nr, const double* x,
                                       double* x0, int64_t n)
{
    const int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, st = (int64_t)gridDim.x * blockDim.x;
    for(int64_t i = i0; i < nwords; i += st)
        words[i] = 0ull;
    for(int64_t i = i0; i < nr; i += st)
        R[i] = 0.0;
    if(x0)
        for(int64_t i = i0; i < n; i += st)
            x0[i] = x[i];
}

// VT: the matrix values; IT: the MAS inverses; MAS: else 3x3 block Jacobi on
// [blk_off, blk_off + blk_cnt) (D) and the identity elsewhere
template <typename VT, typename IT, bool MAS>
__global__ __launch_bounds__(kNT) void pcg_small_kernel(SmallPcg a)
{
    __shared__ double   w[3][kStage];
    __shared__ double   pj[3 * kCols];
    __shared__ double   sx[kOwn], sr[kOwn], sp[kOwn], sz[kOwn], sy[kOwn];
    __shared__ uint32_t bits[kBitWords], rank[kBitWords];
    __shared__ int32_t  glob[kCols];
    __shared__ int32_t  rs[kRows + 1], rb[kRows], row_v[kRows];
    __shared__ int32_t  sib[kRows], par_node[kRows], anc[kLvl][kRows];
    __shared__ double   sC[3 * kBank], sD[kNT / kWave][3];
    __shared__ double   wred[2][2][kNT / kWave];
    __shared__ double   xred[2][4][2];
    __shared__ uint32_t lds[kNT / kWave + 1];
    __shared__ int      failed;

    const int t  = threadIdx.x;
    const int wg = blockIdx.x;
    // ---- the workgroup's rows, their blocks end to end: row i's at [rs[i], rs[i + 1])
    if(t == 0)
        failed = 0;
    if(t < kRows)
    {
        const int32_t slot = wg * kRows + t;
        int32_t       v    = -1;
        if(slot < a.slots)
            v = MAS ? a.slot_vec[slot] : slot;
        const int32_t b0 = v >= 0 ? a.fptr[v] : 0;
        const int32_t c  = v >= 0 ? a.fptr[v + 1] - b0 : 0;
        row_v[t]         = v;
        rb[t]            = b0;
        int32_t inc      = c;
#pragma unroll
        for(int o = 1; o < kRows; o <<= 1)
        {
            const int32_t y = __shfl_up(inc, o, kWave);
            if(t >= o)
                inc += y;
        }
        rs[t + 1] = inc;
        if(t == 0)
            rs[0] = 0;
        if constexpr(MAS)
        {
            sib[t]      = v >= 0 ? a.sib[slot] : 0;
            par_node[t] = v >= 0 ? a.parent[slot] : 0;
            for(int l = 1; l < a.levels; ++l)
                anc[l - 1][t] = v >= 0 ? a.anc_slot[(int64_t)(l - 1) * a.slots + slot] : 0;
        }
    }
    if(t < kBitWords)
        bits[t] = 0u;
    __syncthreads();
    const int nb      = rs[kRows];
    int       longest = 0;  // row
    {
        int l = t < kRows ? rs[t + 1] - rs[t] : 0;
        if(t < kRows)
        {
#pragma unroll
            for(int o = kRows / 2; o > 0; o >>= 1)
                l = max(l, __shfl_xor(l, o, kWave));
            if(t == 0)
                lds[0] = (uint32_t)l;
        }
        __syncthreads();
        longest = (int)lds[0];
        __syncthreads();
    }
    // unfit whatever its columns (they need not be looked at then)
    bool unfit = nb > kFitNear && nb - longest > kFitLong;
    auto      row_of  = [&](int i) {
        int lo = 0;
#pragma unroll
        for(int h = kRows / 2; h > 0; h >>= 1)
            lo += rs[lo + h] <= i ? h : 0;
        return lo;
    };
    // ---- the columns it meets: a bit each, numbered in ascending order
    for(int i = t; i < nb && !unfit; i += kNT)
    {
        const int     row = row_of(i);
        const int32_t j   = a.fcols[rb[row] + (i - rs[row])];
        atomicOr(&bits[j >> 5], 1u << (j & 31));
    }
    __syncthreads();
    uint32_t ncols;
    {
        const uint32_t c = t < kBitWords ? (uint32_t)__popc(bits[t]) : 0u;
        uint32_t       e = block_exclusive_scan<kNT>(c, lds, &ncols);
        if(t < kBitWords)
        {
            rank[t] = e;
            for(uint32_t m = bits[t]; m; m &= m - 1u, ++e)
                if(e < (uint32_t)kCols)
                    glob[e] = 32 * t + __ffs((int)m) - 1;
        }
    }
    __syncthreads();
    unfit = unfit || (ncols > (uint32_t)kCols && nb > kStage && nb - longest > kFitLong);
    const int nl = 3 * (int)(ncols < (uint32_t)kCols ? ncols : (uint32_t)kCols);
    // a column's place in pj, or ~column past the ones kept there
    auto local_of = [&](int32_t j) -> int32_t {
        const uint32_t l = rank[j >> 5] + (uint32_t)__popc(bits[j >> 5] & ((1u << (j & 31)) - 1u));
        return l < (uint32_t)kCols ? (int32_t)(3u * l) : ~j;
    };
    // ---- the blocks in registers
    const VT* vals = static_cast<const VT*>(a.fvals);
    VT        A[kPer][9];
    int32_t   lj[kPer];
#pragma unroll
    for(int m = 0; m < kPer; ++m)
    {
        const int i = m * kNT + t;
        lj[m]       = 0;
#pragma unroll
        for(int q = 0; q < 9; ++q)
            A[m][q] = VT(0);
        if(i < nb)
        {
            const int     row = row_of(i);
            const int64_t k   = rb[row] + (i - rs[row]);
            lj[m]             = local_of(a.fcols[k]);
#pragma unroll
            for(int q = 0; q < 9; ++q)
                A[m][q] = vals[q * a.fstride + k];
        }
    }
    // ---- the preconditioner in registers.  MAS: thread t < 768 holds entries
    // [12 part, 12 part + 12) of row i of the inverse of cluster t / 192 (i =
    // t % 192 / 4, part = t % 4), threads 768 .. 959 of this workgroup's coarse
    // cluster.  Block Jacobi: a row of the 3x3 inverse.
    constexpr int kInv = MAS ? 12 : 3;
    IT            inv[kInv];
    const bool    coarse_wg = MAS && wg < a.coarse && a.levels > 1;
#pragma unroll
    for(int j = 0; j < kInv; ++j)
        inv[j] = IT(0);
    if constexpr(MAS)
    {
        const int ui = t % kOwn >> 2, upart = t & 3, uq = t / kOwn;
        int64_t   k = -1;
        if(uq < kRows / kBank)
        {
            k = (int64_t)wg * (kRows / kBank) + uq;
            if(k * kBank >= a.slots)
                k = -1;
        }
        else if(uq == kRows / kBank && coarse_wg)
            k = a.c_first + wg;
        if(k >= 0)
        {
            const IT* M = static_cast<const IT*>(a.inv) + k * (9 * kSym);
#pragma unroll
            for(int j = 0; j < 12; ++j)
            {
                const int col = 12 * upart + j;
                const int ra = ui / 3, rc = ui % 3, ca = col / 3, cc = col % 3;
                // the upper block (lo, hi): its entry, or the transposed one below the diagonal
                const int lo = ra < ca ? ra : ca, hi = ra < ca ? ca : ra;
                const int blk = kBank * lo - lo * (lo + 1) / 2 + hi;
                const int q   = ra <= ca ? rc + 3 * cc : cc + 3 * rc;
                inv[j]        = M[q * kSym + blk];
            }
        }
    }
    // ---- state: thread t < 192 owns scalar t % 3 of row t / 3
    auto owned = [&](int t, int32_t& v) {
        v = t < kOwn ? row_v[t / 3] : -1;
        return v >= 0;
    };
    {
        int32_t       v;
        const bool    live = owned(t, v);
        const int64_t oi   = 3 * (int64_t)v + t % 3;
        if(t < kOwn)
        {
            sx[t] = live ? a.x[oi] : 0.0;
            sr[t] = live ? a.r[oi] : 0.0;
            sp[t] = live ? a.p[oi] : 0.0;
            sz[t] = sy[t] = 0.0;
        }
        if constexpr(!MAS)
        {
            const int64_t lb  = (int64_t)v - a.blk_off;
            const bool    jac = live && a.D && lb >= 0 && lb < a.blk_cnt;
#pragma unroll
            for(int q = 0; q < 3; ++q)
                inv[q] = jac ? a.D[9 * lb + t % 3 + 3 * q] : q == t % 3 ? 1.0 : 0.0;
        }
    }
    const double rz_tol = a.sc->rz_tol, rr_tol = a.sc->rr_tol;
    const int    crit   = a.sc->criterion;
    const int    it0    = a.sc->iter;
    double       rz = a.sc->rz_pending, rz_old = rz, pap = 0.0, alpha = 0.0, beta = 0.0, rr = a.sc->rr;
    bool         conv = false;
    int          it   = 0;
    __syncthreads();
    Exchange ex{a.words, 0u, (int)gridDim.x, wg, a.wait_ticks, xred, &failed};
    // waves that share a node of this workgroup's coarse cluster, above level 1: 2^wsh
    // (one wave per node summed the top cluster's single node in 14 serial rounds,
    // 21.4 us per iteration on 24^3 + 60k against 15.9)
    int wsh = 0;
    if constexpr(MAS)
        if(coarse_wg && a.c_first + wg >= a.c_desc)
        {
            const int64_t q    = (a.c_first + wg - a.c_desc) * kBank;
            int           live = 1;
            for(int i = 1; i < kBank; ++i)
                live = a.desc_ptr[q + i + 1] > a.desc_ptr[q + i] ? i + 1 : live;
            while((live << (wsh + 1)) <= kBank)
                ++wsh;
        }
    // level 1's share of a vector in LDS: the sum over the slots that share a
    // parent, stored by the lowest of them (threads 768 .. 959)
    auto restrict1 = [&](int t, const double* v, double* R) {
        const int     s = t % kOwn / 3, c = t % 3;
        const int32_t m = sib[s];
        if(m & 0x10000)
        {
            const double* b   = v + 3 * (s & ~(kBank - 1)) + c;
            double        acc = 0.0;
#pragma unroll
            for(int q = 0; q < kBank; ++q)
            {
                const double e = b[3 * q];
                acc += (m >> q) & 1 ? e : 0.0;
            }
            put(&R[3 * (int64_t)par_node[s] + c], acc);
        }
    };
    // this workgroup's coarse cluster: its nodes' r += f times what R holds for
    // them (level 1's own entries, or the sums of their descendants')
    auto coarse_r = [&](int t, const double* R, double f) {
        const int64_t k = a.c_first + wg;
        if(k < a.c_desc)
        {
            if(t < 3 * kBank)
                sC[t] += f * get(&R[3 * kBank * k + t]);
            return;
        }
        const int     node = t / kWave >> wsh, part = (t / kWave) & ((1 << wsh) - 1);
        const int64_t q    = (k - a.c_desc) * kBank + node;
        double        s[3] = {0.0, 0.0, 0.0};
#pragma unroll 2
        for(int32_t e = a.desc_ptr[q] + part * kWave + t % kWave; e < a.desc_ptr[q + 1]; e += kWave << wsh)
        {
            const double* y = &R[3 * (int64_t)a.desc_idx[e]];
#pragma unroll
            for(int c = 0; c < 3; ++c)
                s[c] += get(y + c);
        }
#pragma unroll
        for(int c = 0; c < 3; ++c)
        {
            s[c] = wave_total(s[c]);
            if(t % kWave == 0)
                sD[t / kWave][c] = s[c];
        }
        __syncthreads();
        if(t < 3 * kBank && t / 3 < kBank >> wsh)
        {
            double acc = 0.0;
            for(int h = 0; h < 1 << wsh; ++h)
                acc += sD[(t / 3 << wsh) + h][t % 3];
            sC[t] += f * acc;
        }
    };
    double d0 = 0.0, d1 = 0.0;
    if(t == 0)
        wred[0][0][0] = unfit ? 1.0 : 0.0;
    if constexpr(MAS)
    {
        if(t < 3 * kBank)
            sC[t] = 0.0;
        if(a.levels > 1 && t / kOwn == kRows / kBank)
            restrict1(t, sr, a.R);
    }
    bool go = ex.run<1, 1>(wred[0], d0, d1);
    if(go && d0 != 0.0)
    {
        if(wg == 0 && t == 0)
            a.sc->stalled = kPcgUnfit;
        return;
    }
    if constexpr(MAS)
        if(go && coarse_wg)
            coarse_r(t, a.R, 1.0);
    while(go && it < a.max_it)
    {
        int t = threadIdx.x;
        renew(t);
        if constexpr(sizeof(VT) == 4)
#pragma unroll
            for(int m = 0; m < kPer; ++m)
#pragma unroll
                for(int q = 0; q < 9; ++q)
                    renew(A[m][q]);
        if constexpr(sizeof(IT) == 4)
#pragma unroll
            for(int j = 0; j < kInv; ++j)
                renew(inv[j]);
        int32_t       ov;
        const bool    live = owned(t, ov);
        const int64_t oi   = 3 * (int64_t)ov + t % 3;
        const int     ui = t % kOwn >> 2, upart = t & 3, uq = t / kOwn;  // MAS: cluster row, part, cluster
        const bool    first = it == 0;
        double*    pout  = a.pb + (size_t)(it & 1) * 3 * (size_t)a.B;
        double*    pold  = a.pb + (size_t)(~it & 1) * 3 * (size_t)a.B;
        // ---- p = z + beta p: of the own rows, and of the columns in LDS
        if(live)
        {
            if(!first)
                sp[t] = sz[t] + beta * sp[t];
            put(&pout[oi], sp[t]);  // for columns past a workgroup's kCols
        }
        for(int f = t; f < nl; f += kNT)
        {
            const int     l = f / 3;
            const int64_t g = 3 * (int64_t)glob[l] + (f - 3 * l);
            pj[f]           = first ? a.p[g] : get(&a.z[g]) + beta * pj[f];
        }
        __syncthreads();
        // ---- Ap: products staged in LDS, 16 lanes per row sum them in a fixed order
        auto row_sums = [&](int base, bool add) {
            __syncthreads();
            const int row = t >> 4, lane = t & 15;
            const int lo = max(rs[row], base) - base, hi = min(rs[row + 1], base + kStage) - base;
            double    s0 = 0.0, s1 = 0.0, s2 = 0.0;
            for(int i = lo + lane; i < hi; i += 16)
            {
                s0 += w[0][i];
                s1 += w[1][i];
                s2 += w[2][i];
            }
            s0 = row16_sum(s0);
            s1 = row16_sum(s1);
            s2 = row16_sum(s2);
            double pap = 0.0;
            if(lane == 0)
            {
                if(add)
                {
                    s0 += sy[3 * row];
                    s1 += sy[3 * row + 1];
                    s2 += sy[3 * row + 2];
                }
                sy[3 * row]     = s0;
                sy[3 * row + 1] = s1;
                sy[3 * row + 2] = s2;
                pap             = sp[3 * row] * s0 + sp[3 * row + 1] * s1 + sp[3 * row + 2] * s2;
            }
            pap = wave_total(pap);
            if(t % kWave == 0)
                wred[0][0][t / kWave] = pap;
        };
#pragma unroll
        for(int m = 0; m < kPer; ++m)
        {
            const int i = m * kNT + t;
            if(i < nb)
            {
                const int    l  = lj[m] >= 0 ? lj[m] : 0;
                const double q0 = pj[l], q1 = pj[l + 1], q2 = pj[l + 2];
#pragma unroll
                for(int c = 0; c < 3; ++c)
                    w[c][i] = lj[m] >= 0 ? (double)A[m][c] * q0 + (double)A[m][3 + c] * q1 + (double)A[m][6 + c] * q2
                                         : 0.0;
            }
        }
        row_sums(0, false);
        // blocks past the registers, and those whose column's p is not in LDS, from memory
        for(int base = ncols > (uint32_t)kCols ? 0 : kStage; base < nb; base += kStage)
        {
            __syncthreads();  // the last stage's products have been summed
#pragma unroll 1
            for(int i = base + t; i < min(nb, base + kStage); i += kNT)
            {
                const int     row = row_of(i);
                const int64_t k   = rb[row] + (i - rs[row]);
                const int32_t j   = a.fcols[k], l = local_of(j);
                if(i < kStage && l >= 0)
                {
                    w[0][i] = w[1][i] = w[2][i] = 0.0;
                    continue;
                }
                double q[3];
#pragma unroll
                for(int c = 0; c < 3; ++c)
                {
                    const int64_t g = 3 * (int64_t)j + c;
                    q[c] = l >= 0 ? pj[l + c] : first ? a.p[g] : get(&a.z[g]) + beta * get(&pold[g]);
                }
#pragma unroll
                for(int c = 0; c < 3; ++c)
                    w[c][i - base] = (double)vals[c * a.fstride + k] * q[0] + (double)vals[(3 + c) * a.fstride + k] * q[1]
                                     + (double)vals[(6 + c) * a.fstride + k] * q[2];
            }
            row_sums(base, true);
        }
        if constexpr(MAS)
            if(a.levels > 1)
            {
                // the restriction is linear: Ap's goes out with p.Ap, and r's
                // follows from it with alpha, as r does
                __syncthreads();
                if(t / kOwn == kRows / kBank)
                    restrict1(t, sy, a.RA);
            }
        if(!ex.run<1, kNT / kWave>(wred[0], d0, d1))
            break;
        pap   = d0;
        alpha = rz / pap;
        // ---- x, r
        if(live)
        {
            sx[t] += alpha * sp[t];
            sr[t] -= alpha * sy[t];
        }
        __syncthreads();
        // ---- z
        double z = 0.0;
        if constexpr(MAS)
        {
            if(t < kRows / kBank * kOwn)
            {
                double acc = 0.0;
#pragma unroll
                for(int j = 0; j < 12; ++j)
                    acc += (double)inv[j] * sr[3 * kBank * uq + 12 * upart + j];
                acc = quad_sum(acc);
                if(upart == 0)
                    sz[3 * kBank * uq + ui] = acc;
            }
            if(a.levels > 1)
            {
                if(coarse_wg)
                {
                    coarse_r(t, a.RA, -alpha);
                    __syncthreads();
                    if(uq == kRows / kBank)
                    {
                        double acc = 0.0;
#pragma unroll
                        for(int j = 0; j < 12; ++j)
                            acc += (double)inv[j] * sC[12 * upart + j];
                        acc = quad_sum(acc);
                        if(upart == 0)
                            put(&a.Z[3 * kBank * (a.c_first + wg) + ui], acc);
                    }
                }
                if(!ex.run<0>(wred[0], d0, d1))
                    break;
            }
            else
                __syncthreads();
            if(live)
            {
                z = sz[t];
                double zl[kLvl];
#pragma unroll
                for(int l = 0; l < kLvl; ++l)
                    zl[l] = l + 1 < a.levels ? get(&a.Z[3 * (int64_t)anc[l][t / 3] + t % 3]) : 0.0;
#pragma unroll
                for(int l = 0; l < kLvl; ++l)
                    z += zl[l];
            }
        }
        else if(live)
            z = inv[0] * sr[t - t % 3] + inv[1] * sr[t - t % 3 + 1] + inv[2] * sr[t - t % 3 + 2];
        if(live)
        {
            sz[t] = z;
            put(&a.z[oi], z);
        }
        if(t < kOwn)  // three whole waves
        {
            const double ro = live ? sr[t] : 0.0;
            const double v0 = wave_total(ro * z), v1 = wave_total(ro * ro);
            if(t % kWave == 0)
            {
                wred[1][0][t / kWave] = v0;
                wred[1][1][t / kWave] = v1;
            }
        }
        if(!ex.run<2, kOwn / kWave>(wred[1], d0, d1))
            break;
        // ---- convergence, beta (as pcg_update_p)
        ++it;
        rr               = d1;
        const bool fin   = isfinite(d0) && isfinite(rr);
        conv             = fin && (crit == 0 ? fabs(d0) <= rz_tol : rr <= rr_tol);
        beta             = d0 / rz;
        rz_old           = rz;
        rz               = d0;
        if(conv || !fin)
            break;
    }
    if(failed)
    {
        if(t == 0)
            a.sc->stalled = kPcgStalled;
        return;
    }
    int32_t v;
    if(owned(t, v))
    {
        const int64_t oi = 3 * (int64_t)v + t % 3;
        a.x[oi]          = sx[t];
        a.r[oi]          = sr[t];
        if(!conv)
            a.p[oi] = sz[t] + beta * sp[t];
    }
    if(wg == 0 && t == 0)
    {
        a.sc->rz         = rz_old;
        a.sc->pAp        = pap;
        a.sc->alpha      = alpha;
        a.sc->beta       = beta;
        a.sc->rz_new     = rz;
        a.sc->rz_pending = rz;
        a.sc->rr         = rr;
        a.sc->iter       = it0 + it;
        if(conv)
        {
            a.sc->converged = 1;
            a.sc->conv_iter = it0 + it;
        }
    }
}

const void* small_kernel(const SmallPcg& a)
{
    if(!a.slot_vec)
        return a.use32 ? (const void*)pcg_small_kernel<float, double, false>
                       : (const void*)pcg_small_kernel<double, double, false>;
    if(a.use32)
        return a.inv32 ? (const void*)pcg_small_kernel<float, float, true>
                       : (const void*)pcg_small_kernel<float, double, true>;
    return a.inv32 ? (const void*)pcg_small_kernel<double, float, true>
                   : (const void*)pcg_small_kernel<double, double, true>;
}
}  // namespace

bool pcg_small_launch(SmallPcg& a, SmallPcgScratch& scr, int64_t max_it, bool keep_x, hipStream_t s)
{
    const int     wgs = (a.slots + kRows - 1) / kRows;
    const int64_t n   = 3 * (int64_t)a.B;
    if(wgs < 1 || wgs > kMaxWg || wgs > device_cu_count() || a.B > kSmallRows || a.coarse > wgs || a.levels > kLvl + 1)
        return false;
    scr.words.resize(2 * kMaxWg * 4);
    scr.z.resize((size_t)n);
    scr.pb.resize((size_t)2 * n);
    scr.R.resize((size_t)std::max<int64_t>(1, 6 * a.nodes));
    scr.Z.resize((size_t)std::max<int64_t>(1, 3 * a.nodes));
    a.words  = scr.words.data();
    a.z      = scr.z.data();
    a.pb     = scr.pb.data();
    a.R      = scr.R.data();
    a.RA     = a.R + 3 * a.nodes;
    a.Z      = scr.Z.data();
    a.max_it = (int32_t)std::min<int64_t>(max_it, 512);
    if(keep_x)
        scr.x0.resize((size_t)n);
    pcg_small_clear_kernel<<<32, 256, 0, s>>>(a.words, 2 * kMaxWg * 4, a.R, a.slot_vec ? 6 * a.nodes : 0, a.x,
                                              keep_x ? scr.x0.data() : nullptr, n);
    void*            args[] = {&a};
    const hipError_t e      = hipLaunchCooperativeKernel(small_kernel(a), dim3(wgs), dim3(kNT), args, 0, s);
    if(e != hipSuccess)
    {
        (void)hipGetLastError();
        return false;
    }
    return true;
}
}  // namespace mi
