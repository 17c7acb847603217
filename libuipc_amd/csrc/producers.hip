// Hessian producers on gfx950: the step before the solve, writing triplets
// straight into the triplet buffer in the reference's layout.
//
//   kinetic  m_i I per vertex (finite_element/bdf/finite_element_bdf1_kinetic.cu:60-70)
//   SNH      per tet, V dt^2 times the PSD projection of the stable Neo-Hookean
//            Hessian, Psi = mu/2 (tr F^T F - 3) + lambda/2 (J - alpha)^2,
//            alpha = 1 + mu / lambda (finite_element/constitutions/
//            stable_neo_hookean_3d.cu:100-264), projected through its analytic
//            eigensystem: in the SVD frame F = U S V^T the Hessian splits into
//            three scaling modes (eigenvectors of a 3x3 matrix in the singular
//            values) and, per pair (i, j) with k the third index, a twist mode
//            (antisymmetric, mu + lambda (J - alpha) s_k) and a flip mode
//            (symmetric, mu - lambda (J - alpha) s_k); negative eigenvalues
//            are clamped to 0
//   contact  dt^2 kappa g g^T per vertex-triangle stencil (the synthetic
//            stand-in for contact_system/simplex_normal_contact.cu:74-161)
// and, for the line search after the solve, the kinetic and SNH energies
// (each reduced in a fixed order: per-workgroup partials, then one workgroup)
// and the trial step x = x0 + alpha dx.
//
// Each 4-node stencil writes its 10 upper blocks as the reference's half-block
// writer does (utils/matrix_assembler.h:312-437): slot (a, b), a <= b, in the
// order a = 0..3, b = a..3; the block is written at (min, max) of the two
// global vertex ids, transposed when the stencil order is reversed.
// All arithmetic in FP64.
#include "linsys.hpp"

namespace mi
{
namespace
{
constexpr int kThreads = 256;

int grid_of(int64_t n)
{
    return std::max(1, std::min(ceil_div(n, kThreads), device_cu_count() * 16));
}

__device__ __forceinline__ double det3(const double m[9])  // column-major
{
    return m[0] * (m[4] * m[8] - m[7] * m[5]) - m[3] * (m[1] * m[8] - m[7] * m[2])
           + m[6] * (m[1] * m[5] - m[4] * m[2]);
}

__device__ __forceinline__ void inv3(const double m[9], double o[9])
{
    const double id = 1.0 / det3(m);
    o[0]            = (m[4] * m[8] - m[7] * m[5]) * id;
    o[3]            = -(m[3] * m[8] - m[6] * m[5]) * id;
    o[6]            = (m[3] * m[7] - m[6] * m[4]) * id;
    o[1]            = -(m[1] * m[8] - m[7] * m[2]) * id;
    o[4]            = (m[0] * m[8] - m[6] * m[2]) * id;
    o[7]            = -(m[0] * m[7] - m[6] * m[1]) * id;
    o[2]            = (m[1] * m[5] - m[4] * m[2]) * id;
    o[5]            = -(m[0] * m[5] - m[3] * m[2]) * id;
    o[8]            = (m[0] * m[4] - m[3] * m[1]) * id;
}

// cyclic Jacobi eigen-decomposition of a symmetric 3x3 matrix (row-major a):
// a -> diag(w), eigenvectors in the columns of q (row-major)
__device__ void jacobi3(double a[3][3], double w[3], double q[3][3])
{
    for(int i = 0; i < 3; ++i)
        for(int j = 0; j < 3; ++j)
            q[i][j] = i == j ? 1.0 : 0.0;
    for(int sweep = 0; sweep < 20; ++sweep)
    {
        const double off = a[0][1] * a[0][1] + a[0][2] * a[0][2] + a[1][2] * a[1][2];
        const double dia = a[0][0] * a[0][0] + a[1][1] * a[1][1] + a[2][2] * a[2][2];
        if(off <= 1e-32 * dia || off == 0.0)
            break;
        for(int p = 0; p < 2; ++p)
            for(int r = p + 1; r < 3; ++r)
            {
                const double apr = a[p][r];
                if(apr == 0.0)
                    continue;
                const double theta = (a[r][r] - a[p][p]) / (2.0 * apr);
                const double t     = (theta >= 0.0 ? 1.0 : -1.0) / (fabs(theta) + sqrt(theta * theta + 1.0));
                const double c     = 1.0 / sqrt(t * t + 1.0);
                const double s     = t * c;
                for(int k = 0; k < 3; ++k)
                {
                    const double akp = a[k][p], akr = a[k][r];
                    a[k][p]          = c * akp - s * akr;
                    a[k][r]          = s * akp + c * akr;
                }
                for(int k = 0; k < 3; ++k)
                {
                    const double apk = a[p][k], ark = a[r][k];
                    a[p][k]          = c * apk - s * ark;
                    a[r][k]          = s * apk + c * ark;
                }
                for(int k = 0; k < 3; ++k)
                {
                    const double qkp = q[k][p], qkr = q[k][r];
                    q[k][p]          = c * qkp - s * qkr;
                    q[k][r]          = s * qkp + c * qkr;
                }
            }
    }
    for(int i = 0; i < 3; ++i)
        w[i] = a[i][i];
}

// F = U diag(S) V^T with U, V rotations (S[2] carries the sign of det F);
// F, U, V column-major
__device__ void svd3(const double F[9], double U[9], double S[3], double V[9])
{
    double C[3][3], w[3], q[3][3];
    for(int i = 0; i < 3; ++i)
        for(int j = 0; j < 3; ++j)
            C[i][j] = F[3 * i] * F[3 * j] + F[3 * i + 1] * F[3 * j + 1] + F[3 * i + 2] * F[3 * j + 2];
    jacobi3(C, w, q);
    // descending singular values
    int o[3] = {0, 1, 2};
    for(int i = 0; i < 2; ++i)
        for(int j = i + 1; j < 3; ++j)
            if(w[o[j]] > w[o[i]])
            {
                const int t = o[i];
                o[i]        = o[j];
                o[j]        = t;
            }
    for(int c = 0; c < 3; ++c)
        for(int r = 0; r < 3; ++r)
            V[r + 3 * c] = q[r][o[c]];
    // V a rotation
    const double dv = det3(V);
    if(dv < 0.0)
        for(int r = 0; r < 3; ++r)
            V[r + 6] = -V[r + 6];
    // u_c = F v_c / s_c for the two largest; u_2 = u_0 x u_1
    double Fv[3][3];
    for(int c = 0; c < 3; ++c)
        for(int r = 0; r < 3; ++r)
            Fv[c][r] = F[r] * V[3 * c] + F[r + 3] * V[3 * c + 1] + F[r + 6] * V[3 * c + 2];
    double n0 = sqrt(Fv[0][0] * Fv[0][0] + Fv[0][1] * Fv[0][1] + Fv[0][2] * Fv[0][2]);
    for(int r = 0; r < 3; ++r)
        U[r] = Fv[0][r] / n0;
    double d01 = U[0] * Fv[1][0] + U[1] * Fv[1][1] + U[2] * Fv[1][2];
    double u1[3];
    for(int r = 0; r < 3; ++r)
        u1[r] = Fv[1][r] - d01 * U[r];
    double n1 = sqrt(u1[0] * u1[0] + u1[1] * u1[1] + u1[2] * u1[2]);
    for(int r = 0; r < 3; ++r)
        U[3 + r] = u1[r] / n1;
    U[6] = U[1] * U[5] - U[2] * U[4];
    U[7] = U[2] * U[3] - U[0] * U[5];
    U[8] = U[0] * U[4] - U[1] * U[3];
    S[0] = n0;
    S[1] = U[3] * Fv[1][0] + U[4] * Fv[1][1] + U[5] * Fv[1][2];
    S[2] = U[6] * Fv[2][0] + U[7] * Fv[2][1] + U[8] * Fv[2][2];
}

// The triplets of 4-node stencils, written by consecutive lanes: a stencil's 10
// blocks are 720 consecutive bytes, which one lane per stencil writes in 90
// stores that each touch 64 cache lines per wave.  Instead a wave's 64 stencils
// pass each slot's blocks through LDS and nine lanes write a block
// (StencilOut), or every lane computes the consecutive entries it writes
// (contact_kernel).
constexpr int kSlots = 10;
// slot s = (a, b), a <= b: two bits per slot
__device__ __forceinline__ constexpr int slot_a(int s)
{
    return (0xE9500 >> (2 * s)) & 3;  // 0 0 0 0 1 1 1 2 2 3
}
__device__ __forceinline__ constexpr int slot_b(int s)
{
    return (0xFB9E4 >> (2 * s)) & 3;  // 0 1 2 3 1 2 3 2 3 3
}

// rows and cols of n stencils (ids: LDS, 4 per stencil), by NT threads:
// (min, max) of the slot's two ids
template <int NT>
__device__ __forceinline__ void put_ids(const int32_t (*ids)[4], int n, int t, int32_t* rows, int32_t* cols)
{
    for(int e = t; e < kSlots * n; e += NT)
    {
        const int     i = e / kSlots, s = e - kSlots * i;
        const int32_t x = ids[i][slot_a(s)], y = ids[i][slot_b(s)];
        rows[e]         = x < y ? x : y;
        cols[e]         = x < y ? y : x;
    }
}

// orders a wave's LDS accesses before it against those after it
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// one wave's stencils, a lane each: blocks of one slot at a time
struct StencilOut
{
    double (*st)[9];       // LDS, one block per lane
    int32_t (*ids)[4];     // LDS, the stencils' global ids
    double* vals;          // of the wave's first stencil
    int     n;             // its stencils
    int     lane;
    // K_ab row-major; written transposed when the stencil order is reversed
    __device__ __forceinline__ void put(int s, const double K[3][3])
    {
        const bool swap = ids[lane][slot_a(s)] > ids[lane][slot_b(s)];
#pragma unroll
        for(int c = 0; c < 3; ++c)
#pragma unroll
            for(int r = 0; r < 3; ++r)
                st[lane][r + 3 * c] = swap ? K[c][r] : K[r][c];
        wave_lds_fence();
#pragma unroll 1  // (unrolled, its addresses take 60 registers over the whole kernel)
        for(int k = 0; k < 9; ++k)
        {
            const int e = k * kWave + lane, i = e / 9, q = e - 9 * i;
            if(i < n)
                vals[9 * (kSlots * i + s) + q] = st[i][q];
        }
        wave_lds_fence();  // st is rewritten by the next slot
    }
};

// one thread per entry: consecutive lanes write consecutive doubles
__global__ __launch_bounds__(kThreads) void kinetic_kernel(int32_t V,
                                                          const double* __restrict__ mass,
                                                          int32_t  vert_offset,
                                                          int32_t* rows,
                                                          int32_t* cols,
                                                          double*  vals)
{
    const int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (int64_t)gridDim.x * blockDim.x;
    for(int64_t i = i0; i < 9 * (int64_t)V; i += stride)
    {
        const int64_t v = i / 9;
        const int     q = (int)(i - 9 * v);
        vals[i]         = q % 4 == 0 ? mass[v] : 0.0;
    }
    for(int64_t v = i0; v < V; v += stride)
    {
        rows[v] = (int32_t)v + vert_offset;
        cols[v] = (int32_t)v + vert_offset;
    }
}

// Bound by the registers of its FP64 arithmetic (two SVD-sized Jacobi sweeps)
// and by the writes: 149k tets of a 32^3 grid 82 -> 51 us (119 MB written) with
// three waves per SIMD (four: 128 registers and 146 us of spills; one, of 256: 63).
__global__ __launch_bounds__(kThreads, 3) void snh_kernel(int64_t n_tets,
                                                      const int32_t* __restrict__ tets,
                                                      const double* __restrict__ X,
                                                      const double* __restrict__ x,
                                                      double   mu,
                                                      double   lambda,
                                                      double   dt2,
                                                      int32_t  vert_offset,
                                                      int32_t* rows,
                                                      int32_t* cols,
                                                      double*  vals)
{
    __shared__ double  st[kThreads][9];
    __shared__ int32_t ids[kThreads][4];
    const int          lane = threadIdx.x % kWave, w0 = threadIdx.x - lane;
    // a wave's 64 tets in a row; lanes past the last repeat it and write nothing
    for(int64_t t0 = (int64_t)blockIdx.x * kThreads + w0; t0 < n_tets; t0 += (int64_t)gridDim.x * kThreads)
    {
        const int     n = n_tets - t0 < kWave ? (int)(n_tets - t0) : kWave;
        const int64_t t = t0 + (lane < n ? lane : n - 1);
        int32_t       q[4];
#pragma unroll
        for(int c = 0; c < 4; ++c)
        {
            q[c]                 = tets[4 * t + c];
            ids[threadIdx.x][c] = q[c] + vert_offset;
        }
        wave_lds_fence();
        put_ids<kWave>(&ids[w0], n, lane, rows + kSlots * t0, cols + kSlots * t0);
        StencilOut out{&st[w0], &ids[w0], vals + 9 * kSlots * t0, n, lane};
        double     Dm[9], Ds[9], Dmi[9], F[9];
#pragma unroll
        for(int c = 0; c < 3; ++c)
#pragma unroll
            for(int r = 0; r < 3; ++r)
            {
                Dm[r + 3 * c] = X[3 * (int64_t)q[c + 1] + r] - X[3 * (int64_t)q[0] + r];
                Ds[r + 3 * c] = x[3 * (int64_t)q[c + 1] + r] - x[3 * (int64_t)q[0] + r];
            }
        const double vol = fabs(det3(Dm)) / 6.0;
        inv3(Dm, Dmi);
#pragma unroll
        for(int c = 0; c < 3; ++c)
#pragma unroll
            for(int r = 0; r < 3; ++r)
                F[r + 3 * c] = Ds[r] * Dmi[3 * c] + Ds[r + 3] * Dmi[1 + 3 * c] + Ds[r + 6] * Dmi[2 + 3 * c];
        // shape gradients: dN_i = row (i - 1) of Dm^-1, dN_0 = -(dN_1 + dN_2 + dN_3)
        double gN[4][3];
#pragma unroll
        for(int i = 1; i < 4; ++i)
#pragma unroll
            for(int c = 0; c < 3; ++c)
                gN[i][c] = Dmi[(i - 1) + 3 * c];
#pragma unroll
        for(int c = 0; c < 3; ++c)
            gN[0][c] = -(gN[1][c] + gN[2][c] + gN[3][c]);

        double U[9], S[3], Vm[9];
        svd3(F, U, S, Vm);
        const double J     = S[0] * S[1] * S[2];
        const double alpha = 1.0 + mu / lambda;
        const double s     = lambda * (J - alpha);
        const double scale = vol * dt2;
        // sa[i][k] = V_k . dN_i
        double sa[4][3];
#pragma unroll
        for(int i = 0; i < 4; ++i)
#pragma unroll
            for(int k = 0; k < 3; ++k)
                sa[i][k] = Vm[3 * k] * gN[i][0] + Vm[3 * k + 1] * gN[i][1] + Vm[3 * k + 2] * gN[i][2];
        // scaling modes: the 3x3 Hessian of Psi in the singular values
        double A[3][3], ew[3], ev[3][3];
        A[0][0] = mu + lambda * (S[1] * S[2]) * (S[1] * S[2]);
        A[1][1] = mu + lambda * (S[0] * S[2]) * (S[0] * S[2]);
        A[2][2] = mu + lambda * (S[0] * S[1]) * (S[0] * S[1]);
        const double c2 = lambda * (2.0 * J - alpha);
        A[0][1] = A[1][0] = c2 * S[2];
        A[0][2] = A[2][0] = c2 * S[1];
        A[1][2] = A[2][1] = c2 * S[0];
        jacobi3(A, ew, ev);
        // The 10 upper blocks, K_ab = U T_ab U^T with T_ab in the frame of the
        // singular vectors: the scaling modes' projected Hessian P couples sa_i
        // and sb_j, the twist and flip modes of a pair (i, j) (eigenvalues lt, lf
        // with the vectors (U_i s_j -/+ U_j s_i) / sqrt 2) give (lt + lf) / 2 on
        // the diagonal and (lf - lt) / 2 off it.  (Summing lam w_a w_b^T over
        // the nine modes is five times the arithmetic.)
        double P[3][3], ht[3], hd[3];
#pragma unroll
        for(int i = 0; i < 3; ++i)
#pragma unroll
            for(int j = i; j < 3; ++j)
            {
                double acc = 0.0;
#pragma unroll
                for(int m = 0; m < 3; ++m)
                    acc += fmax(ew[m], 0.0) * (ev[i][m] * ev[j][m]);
                P[i][j] = P[j][i] = scale * acc;
            }
#pragma unroll
        for(int k = 0; k < 3; ++k)
        {
            const double lt = fmax(mu + s * S[k], 0.0), lf = fmax(mu - s * S[k], 0.0);
            ht[k]           = 0.5 * scale * (lt + lf);
            hd[k]           = 0.5 * scale * (lf - lt);
        }
        int slot = 0;
#pragma unroll
        for(int a = 0; a < 4; ++a)
#pragma unroll
            for(int b = a; b < 4; ++b)
            {
                double pr[3][3];  // sa_i sb_j
#pragma unroll
                for(int i = 0; i < 3; ++i)
#pragma unroll
                    for(int j = 0; j < 3; ++j)
                        pr[i][j] = sa[a][i] * sa[b][j];
                double T[3][3];
#pragma unroll
                for(int i = 0; i < 3; ++i)
#pragma unroll
                    for(int j = 0; j < 3; ++j)
                        if(i == j)
                        {
                            const int u = (i + 1) % 3, v = (i + 2) % 3;  // pairs (i, u) and (i, v): third indices v, u
                            T[i][i] = P[i][i] * pr[i][i] + ht[v] * pr[u][u] + ht[u] * pr[v][v];
                        }
                        else
                            T[i][j] = P[i][j] * pr[i][j] + hd[3 - i - j] * pr[j][i];
                double UT[3][3], K[3][3];
#pragma unroll
                for(int r = 0; r < 3; ++r)
#pragma unroll
                    for(int j = 0; j < 3; ++j)
                        UT[r][j] = U[r] * T[0][j] + U[r + 3] * T[1][j] + U[r + 6] * T[2][j];
#pragma unroll
                for(int r = 0; r < 3; ++r)
#pragma unroll
                    for(int c = 0; c < 3; ++c)
                        if(a == b && c < r)
                            K[r][c] = K[c][r];  // a diagonal block is symmetric to the bit
                        else
                            K[r][c] = UT[r][0] * U[c] + UT[r][1] * U[c + 3] + UT[r][2] * U[c + 6];
                out.put(slot++, K);
            }
    }
}

// A workgroup takes 64 stencils at a time: their g, kappa and ids staged in LDS,
// then every lane computes the consecutive entries it writes.  Bound by them:
// 200k stencils (160 MB written, 21 MB read) 76 -> 42 us, 4.3 TB/s.
__global__ __launch_bounds__(kThreads) void contact_kernel(int64_t n,
                                                          const int32_t* __restrict__ cidx,
                                                          const double* __restrict__ g,
                                                          const double* __restrict__ kappa,
                                                          double   dt2,
                                                          int32_t  vert_offset,
                                                          int32_t* rows,
                                                          int32_t* cols,
                                                          double*  vals)
{
    constexpr int      kN = 64;
    __shared__ double  sg[kN][12], sk[kN];
    __shared__ int32_t ids[kN][4];
    const int          tid = threadIdx.x;
    for(int64_t s0 = (int64_t)blockIdx.x * kN; s0 < n; s0 += (int64_t)gridDim.x * kN)
    {
        const int m = n - s0 < kN ? (int)(n - s0) : kN;
        for(int e = tid; e < 12 * m; e += kThreads)
            (&sg[0][0])[e] = g[12 * s0 + e];
        if(tid < 4 * m)
            (&ids[0][0])[tid] = cidx[4 * s0 + tid] + vert_offset;
        if(tid < m)
            sk[tid] = dt2 * kappa[s0 + tid];
        __syncthreads();
        put_ids<kThreads>(ids, m, tid, rows + kSlots * s0, cols + kSlots * s0);
        for(int e = tid; e < 9 * kSlots * m; e += kThreads)
        {
            const int i = e / (9 * kSlots), f = e - 9 * kSlots * i, s = f / 9, q = f - 9 * s;
            const int a = slot_a(s), b = slot_b(s);
            // the block in its written orientation (L, R) = (a, b) or (b, a),
            // each entry k g_(L, r) g_(R, c) as one product chain
            const bool swap                = ids[i][a] > ids[i][b];
            const int  L = swap ? b : a, R = swap ? a : b, c = q / 3, r = q - 3 * c;
            vals[9 * kSlots * s0 + e]      = sk[i] * sg[i][3 * L + r] * sg[i][3 * R + c];
        }
        __syncthreads();
    }
}
// ---- line-search side: energies and the trial step
constexpr int kEnergyBlocks = 1024;

int energy_grid(int64_t n)
{
    return (int)std::max<int64_t>(1, std::min<int64_t>(ceil_div(n, kThreads), kEnergyBlocks));
}

// FiniteElementBDF1Kinetic_do_compute_energy_kernel: 1/2 m |x - x_tilde|^2
__global__ __launch_bounds__(kThreads) void kinetic_energy_kernel(int32_t V,
                                                                 const double* __restrict__ x,
                                                                 const double* __restrict__ xt,
                                                                 const double* __restrict__ m,
                                                                 double* part)
{
    __shared__ double lds[kThreads / kWave];
    double            acc = 0.0;
    for(int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < V; v += (int64_t)gridDim.x * blockDim.x)
    {
        const double d0 = x[3 * v] - xt[3 * v], d1 = x[3 * v + 1] - xt[3 * v + 1], d2 = x[3 * v + 2] - xt[3 * v + 2];
        acc += 0.5 * m[v] * (d0 * d0 + d1 * d1 + d2 * d2);
    }
    acc = block_sum<kThreads>(acc, lds);
    if(threadIdx.x == 0)
        part[blockIdx.x] = acc;
}

// StableNeoHookean3D_do_compute_energy_kernel: dt^2 V_rest Psi(F),
// Psi = 1/2 (mu (|F|^2 - 3) + lambda (J - 1 - mu / lambda)^2), J = det F
__global__ __launch_bounds__(kThreads) void snh_energy_kernel(int64_t n_tets,
                                                             const int32_t* __restrict__ tets,
                                                             const double* __restrict__ X,
                                                             const double* __restrict__ x,
                                                             double  mu,
                                                             double  lambda,
                                                             double  dt2,
                                                             double* part)
{
    __shared__ double lds[kThreads / kWave];
    double            acc = 0.0;
    for(int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n_tets; t += (int64_t)gridDim.x * blockDim.x)
    {
        int32_t q[4];
#pragma unroll
        for(int c = 0; c < 4; ++c)
            q[c] = tets[4 * t + c];
        double Dm[9], Ds[9], Dmi[9], F[9];
#pragma unroll
        for(int c = 0; c < 3; ++c)
#pragma unroll
            for(int r = 0; r < 3; ++r)
            {
                Dm[r + 3 * c] = X[3 * (int64_t)q[c + 1] + r] - X[3 * (int64_t)q[0] + r];
                Ds[r + 3 * c] = x[3 * (int64_t)q[c + 1] + r] - x[3 * (int64_t)q[0] + r];
            }
        const double vol = fabs(det3(Dm)) / 6.0;
        inv3(Dm, Dmi);
        double Ic = 0.0;
#pragma unroll
        for(int c = 0; c < 3; ++c)
#pragma unroll
            for(int r = 0; r < 3; ++r)
            {
                F[r + 3 * c] = Ds[r] * Dmi[3 * c] + Ds[r + 3] * Dmi[1 + 3 * c] + Ds[r + 6] * Dmi[2 + 3 * c];
                Ic += F[r + 3 * c] * F[r + 3 * c];
            }
        const double Jm = det3(F) - 1.0 - mu / lambda;
        acc += 0.5 * (mu * (Ic - 3.0) + lambda * Jm * Jm) * dt2 * vol;
    }
    acc = block_sum<kThreads>(acc, lds);
    if(threadIdx.x == 0)
        part[blockIdx.x] = acc;
}

// the partials in a fixed order (one workgroup), so the total is reproducible
__global__ __launch_bounds__(kThreads) void energy_total_kernel(const double* __restrict__ part, int n, double* out)
{
    __shared__ double lds[kThreads / kWave];
    double            acc = 0.0;
    for(int i = threadIdx.x; i < n; i += kThreads)
        acc += part[i];
    acc = block_sum<kThreads>(acc, lds);
    if(threadIdx.x == 0)
        *out = acc;
}

__global__ __launch_bounds__(kThreads) void step_forward_kernel(const double* __restrict__ x0,
                                                               const double* __restrict__ dx,
                                                               double  alpha,
                                                               double* x,
                                                               int64_t n)
{
    for(int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        x[i] = x0[i] + alpha * dx[i];
}
}  // namespace

void energy_kinetic(int32_t V, const double* x, const double* xt, const double* m, double* energy,
                    DBuf<double>& part, hipStream_t s)
{
    const int g = energy_grid(V);
    part.resize(kEnergyBlocks);
    kinetic_energy_kernel<<<g, kThreads, 0, s>>>(V, x, xt, m, part.data());
    energy_total_kernel<<<1, kThreads, 0, s>>>(part.data(), g, energy);
    MI_HIP(hipGetLastError());
}

void energy_snh(int64_t        n_tets,
                const int32_t* tets,
                const double*  X,
                const double*  x,
                double         mu,
                double         lambda,
                double         dt,
                double*        energy,
                DBuf<double>&  part,
                hipStream_t    s)
{
    const int g = energy_grid(n_tets);
    part.resize(kEnergyBlocks);
    snh_energy_kernel<<<g, kThreads, 0, s>>>(n_tets, tets, X, x, mu, lambda, dt * dt, part.data());
    energy_total_kernel<<<1, kThreads, 0, s>>>(part.data(), g, energy);
    MI_HIP(hipGetLastError());
}

void step_forward(const double* x0, const double* dx, double alpha, double* x, int64_t n, hipStream_t s)
{
    if(n > 0)
        step_forward_kernel<<<grid_of(n), kThreads, 0, s>>>(x0, dx, alpha, x, n);
    MI_HIP(hipGetLastError());
}

void produce_kinetic(int32_t V, const double* mass, int32_t vert_offset, int32_t* rows, int32_t* cols, double* vals,
                     hipStream_t s)
{
    if(V > 0)
        kinetic_kernel<<<grid_of(9 * (int64_t)V), kThreads, 0, s>>>(V, mass, vert_offset, rows, cols, vals);
    MI_HIP(hipGetLastError());
}

void produce_snh(int64_t        n_tets,
                 const int32_t* tets,
                 const double*  X,
                 const double*  x,
                 double         mu,
                 double         lambda,
                 double         dt,
                 int32_t        vert_offset,
                 int32_t*       rows,
                 int32_t*       cols,
                 double*        vals,
                 hipStream_t    s)
{
    if(n_tets > 0)
        snh_kernel<<<grid_of(n_tets), kThreads, 0, s>>>(n_tets, tets, X, x, mu, lambda, dt * dt, vert_offset, rows,
                                                        cols, vals);
    MI_HIP(hipGetLastError());
}

void produce_contact(int64_t        n,
                     const int32_t* stencils,
                     const double*  g,
                     const double*  kappa,
                     double         dt,
                     int32_t        vert_offset,
                     int32_t*       rows,
                     int32_t*       cols,
                     double*        vals,
                     hipStream_t    s)
{
    if(n > 0)
        contact_kernel<<<grid_of(4 * n), kThreads, 0, s>>>(n, stencils, g, kappa, dt * dt, vert_offset, rows, cols, vals);
    MI_HIP(hipGetLastError());
}
}  // namespace mi
