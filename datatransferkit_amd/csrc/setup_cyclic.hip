// Fused MLS setup with a cyclic symmetric Jacobi eigen-solver: the fast
// FP64 path (DTKX_SOLVER_CYCLIC_JACOBI).
//
// One target system per lane (per lane pair for the quadratic basis, see
// setup_cyclic_kernel). The moment matrix A = P^T Phi P is symmetric
// positive semi-definite, so A^+ e_0 = V Lambda^+ V^T e_0 with A = V Lambda
// V^T; the pseudo-inverse is the same as the reference's two-sided SVD
// (DTK_DetailsSVDImpl.hpp) up to rounding. Every (p, q) index is a
// compile-time constant (fully unrolled sweeps), so A (upper triangle) and
// V stay in registers: no LDS, no barriers, no divergence except the
// per-wave sweep count. Rotations use the Rutishauser form (t = sgn(theta)
// / (|theta| + sqrt(theta^2 + 1)), c = 1/sqrt(1 + t^2), tau = s/(1 + c)).
// Each system sweeps until its off-diagonal mass is below (DBL_EPSILON/8)^2
// of its diagonal mass, or to the sweep cap (a converged system idles while
// the rest of its wave finishes, so its bits do not depend on its wave).
// Truncation keeps the reference's semantics: eigenvalues with |l| >=
// DBL_EPSILON (or rcond * max|l|) contribute. Rows listed by the Cholesky
// setup (systems it could not certify) whose eigenvalues all pass are
// solved again by Cholesky (setup_fast.hip).
// Neighbour data is re-gathered from L2 in three passes (radius, moments,
// coefficients) instead of being staged.
#include "cyclic_device.hpp"
#include "setup.hpp"

#include <algorithm>
#include <type_traits>

namespace dtkx
{
namespace
{

using namespace cyc;
constexpr int kBlock = 64;

// One listed or ranged row's neighbour list, target and radius (row_reach).
struct SystemRow
{
    int64_t rbeg;
    int kk;
    int32_t const *nbr;
    double4 tp;
    double radius;
};

template <int M, bool F32>
__device__ __forceinline__ SystemRow
    system_row( bool valid, int64_t slot, double4 const *__restrict__ src,
                double4 const *__restrict__ tgt,
                int32_t const *__restrict__ indices,
                int32_t const *__restrict__ order,
                int64_t const *__restrict__ row_off, int kk_uniform,
                int geometry, bool by_distance )
{
    int64_t const t = valid ? ( order ? order[slot] : slot ) : 0;
    int64_t const rbeg =
        valid ? ( row_off ? row_off[slot] : slot * kk_uniform ) : 0;
    int const kk =
        valid ? ( row_off ? (int)( row_off[slot + 1] - rbeg ) : kk_uniform )
              : 0;
    int32_t const *nbr = indices + rbeg;
    double4 const tp = valid ? tgt[t] : double4{0, 0, 0, 0};

    double const dmax = row_reach<M, F32>( geometry, by_distance, src, nbr, kk, tp );
    double const radius = F32 ? (double)( 1.1f * (float)dmax ) : 1.1 * dmax;
    return SystemRow{rbeg, kk, nbr, tp, radius};
}

// A row with its moments (upper triangle) written to A. Shared by the
// kernels below, so all form the same bits.
template <int M, bool F32>
__device__ __forceinline__ SystemRow
    system_moments( bool valid, int64_t slot, double4 const *__restrict__ src,
                    double4 const *__restrict__ tgt,
                    int32_t const *__restrict__ indices,
                    int32_t const *__restrict__ order,
                    int64_t const *__restrict__ row_off, int kk_uniform,
                    int rbf, int geometry, bool by_distance,
                    double *A )
{
    using S = SymIdx<M>;
    SystemRow const sr =
        system_row<M, F32>( valid, slot, src, tgt, indices, order, row_off,
                            kk_uniform, geometry, by_distance );

#pragma unroll
    for ( int e = 0; e < S::size; ++e )
        A[e] = 0.0;
    if ( valid )
        for ( int l = 0; l < sr.kk; ++l )
        {
            double P[M];
            double const phi = nbr_row<M, F32>( geometry, rbf, sr.radius,
                                                src[sr.nbr[l]], sr.tp, P );
#pragma unroll
            for ( int r = 0; r < M; ++r )
            {
                double const pr = P[r] * phi;
#pragma unroll
                for ( int c = r; c < M; ++c )
                    A[S::at( r, c )] = fma( pr, P[c], A[S::at( r, c )] );
            }
        }
    return sr;
}

// Truncation threshold of a system's eigenvalues (DBL_EPSILON, or rcond
// times the largest |eigenvalue|) and whether any falls below it.
template <int M>
__device__ __forceinline__ bool truncated( double const *A, int truncation,
                                           double rcond, double &thr )
{
    using S = SymIdx<M>;
    thr = DBL_EPSILON;
    if ( truncation == DTKX_TRUNCATION_RELATIVE )
    {
        double lmax = 0.;
#pragma unroll
        for ( int k = 0; k < M; ++k )
            lmax = fmax( lmax, fabs( A[S::at( k, k )] ) );
        thr = rcond * lmax;
    }
    bool under = false;
#pragma unroll
    for ( int k = 0; k < M; ++k )
        under = under || !( fabs( A[S::at( k, k )] ) >= thr );
    return under;
}

// H lanes per system (H = 1, or 2 for M = 10 so A and half of V fit the
// 256 VGPRs): every lane of the pair keeps the whole moment matrix and runs
// the same rotations on it (identical values, so both agree), and owns
// R = M / H rows of V.
template <int M, int H, bool F32, bool STORE>
__device__ __forceinline__ void
    cyclic_system( int64_t const li, double4 const *__restrict__ src,
                         double4 const *__restrict__ tgt, int64_t n_tgt,
                         int32_t const *__restrict__ indices,
                         int32_t const *__restrict__ order, int64_t row0,
                         int64_t const *__restrict__ row_off,
                         int32_t const *__restrict__ rows,
                         int32_t const *__restrict__ n_rows, int kk_uniform,
                         int rbf,
                         int geometry, int truncation, double rcond,
                         int max_sweeps, double *__restrict__ coeffs,
                         float *__restrict__ coeffs32,
                         double *__restrict__ pinv_out,
                         unsigned long long *__restrict__ counters,
                         bool by_distance,
                         bool screened )
{
    using S = SymIdx<M>;
    constexpr int R = M / H;
    int const h = threadIdx.x % H;
    bool valid;
    int64_t slot;
    if ( rows )
    {
        valid = li < *n_rows;
        slot = valid ? rows[li] : 0;
    }
    else
    {
        slot = row0 + li;
        valid = slot < n_tgt;
    }
    double A[S::size];
    SystemRow const sr =
        system_moments<M, F32>( valid, slot, src, tgt, indices, order, row_off,
                                kk_uniform, rbf, geometry, by_distance, A );
    int const kk = sr.kk;
    int64_t const rbeg = sr.rbeg;
    int32_t const *nbr = sr.nbr;
    double4 const tp = sr.tp;
    double const radius = sr.radius;

    // cyclic Jacobi; this lane owns rows h*R .. h*R + R - 1 of V
    double V[R * M];
#pragma unroll
    for ( int e = 0; e < R * M; ++e )
        V[e] = ( h * R + e / M == e % M ) ? 1.0 : 0.0;
    // each system stops at its own convergence, so its result does not
    // depend on which systems share its wave
    int sweeps = 0;
    bool done = !valid || converged<M>( A );
    for ( int pass = 0; !__all( done ) && pass < max_sweeps; ++pass )
    {
        sweep_all<M, R>( A, V, done );
        sweeps += done ? 0 : 1;
        done = done || converged<M>( A );
    }

    // x = A^+ e_0 = sum_k [|l_k| >= thr] V(0,k) V(:,k) / l_k
    double thr = DBL_EPSILON;
    if ( truncation == DTKX_TRUNCATION_RELATIVE )
    {
        double lmax = 0.;
#pragma unroll
        for ( int k = 0; k < M; ++k )
            lmax = fmax( lmax, fabs( A[S::at( k, k )] ) );
        thr = rcond * lmax;
    }
    double w[M];
    bool under = false;
#pragma unroll
    for ( int k = 0; k < M; ++k )
    {
        double const lk = A[S::at( k, k )];
        bool const keep = fabs( lk ) >= thr;
        under = under || !keep;
        // V(0, k) lives in the lane owning row 0 (h == 0)
        double v0k = V[k];
        if ( H > 1 )
            v0k = __shfl( v0k, ( threadIdx.x / H ) * H, kBlock );
        w[k] = keep ? v0k / lk : 0.0;
    }
    double x[M];
#pragma unroll
    for ( int r = 0; r < R; ++r )
    {
        double acc = 0.0;
#pragma unroll
        for ( int k = 0; k < M; ++k )
            acc = fma( w[k], V[r * M + k], acc );
        x[r] = acc;
    }
    if ( H > 1 )
    {
        // gather the partner's rows: x[R..M) from lane h^1 (H == 2)
        double xo[R];
#pragma unroll
        for ( int r = 0; r < R; ++r )
            xo[r] = __shfl_xor( x[r], 1, kBlock );
#pragma unroll
        for ( int r = 0; r < R; ++r )
        {
            double const mine = x[r];
            x[h * R + r] = mine;
            x[( 1 - h ) * R + r] = xo[r];
        }
    }

    if constexpr ( STORE )
    {
        // the whole pseudo-inverse V diag(w) V^T, packed upper triangle;
        // each lane writes the rows it owns, with the partner's V rows
        // fetched by shuffles (H == 2)
        double wk[M];
#pragma unroll
        for ( int k = 0; k < M; ++k )
        {
            double const lk = A[S::at( k, k )];
            wk[k] = fabs( lk ) >= thr ? 1.0 / lk : 0.0;
        }
#pragma unroll
        for ( int jr = 0; jr < M; ++jr )
        {
            // row jr of V, from the lane that owns it
            double vj[M];
#pragma unroll
            for ( int k = 0; k < M; ++k )
            {
                double const mine = V[( jr % R ) * M + k];
                double const other =
                    H > 1 ? __shfl_xor( mine, 1, kBlock ) : mine;
                vj[k] = ( jr / R == h ) ? mine : other;
            }
#pragma unroll
            for ( int r = 0; r < R; ++r )
            {
                int const i = h * R + r;
                if ( valid && i <= jr )
                {
                    double acc = 0.0;
#pragma unroll
                    for ( int k = 0; k < M; ++k )
                        acc = fma( V[r * M + k] * wk[k], vj[k], acc );
                    pinv_out[slot * S::size + S::at( i, jr )] = acc;
                }
            }
        }
    }
    if ( !valid )
        return;
    // coefficients c_l = phi_l (P_l . x), neighbours split over the H lanes
    for ( int l = h; l < kk; l += H )
    {
        double P[M];
        double const phi =
            nbr_row<M, F32>( geometry, rbf, radius, src[nbr[l]], tp, P );
        if constexpr ( F32 )
        {
            // the float basis row and weight are exact in double: the short
            // dot product with x (large cancelling terms, the monomials span
            // several scales) is formed in double and rounded once
            double acc = 0.0;
#pragma unroll
            for ( int j = 0; j < M; ++j )
                acc = fma( x[j], P[j], acc );
            coeffs32[rbeg + l] = (float)( acc * phi );
        }
        else
        {
            double acc = 0.0;
#pragma unroll
            for ( int j = 0; j < M; ++j )
                acc = fma( x[j], P[j], acc );
            coeffs[rbeg + l] = acc * phi;
        }
    }
    // (a screened list's untruncated rows had their sweeps counted by the
    // screen)
    if ( counters && h == 0 )
    {
        if ( under )
            atomicAdd( counters + 0, 1ull );
        if ( !screened || under )
        {
            if ( !done )
                atomicAdd( counters + 1, 1ull );
            atomicAdd( counters + 2, (unsigned long long)sweeps );
        }
    }
}

// Row-list mode (a device-side list of rows, its length known only on the
// device) runs a bounded grid that strides over the list, so an empty list
// costs a few thousand empty blocks, not one per row of the operator.
constexpr int kListBlocks = 2048;

template <int M, int H, bool F32, bool STORE, bool LIST>
__global__ void __launch_bounds__( kBlock )
    setup_cyclic_kernel( double4 const *__restrict__ src,
                         double4 const *__restrict__ tgt, int64_t n_tgt,
                         int32_t const *__restrict__ indices,
                         int32_t const *__restrict__ order, int64_t row0,
                         int64_t const *__restrict__ row_off,
                         int32_t const *__restrict__ rows,
                         int32_t const *__restrict__ n_rows, int kk_uniform,
                         int rbf, int geometry, int truncation, double rcond,
                         int max_sweeps, double *__restrict__ coeffs,
                         float *__restrict__ coeffs32,
                         double *__restrict__ pinv_out,
                         unsigned long long *__restrict__ counters,
                         bool by_distance,
                         bool screened )
{
    constexpr int SPB = kBlock / H;
    auto one = [&]( int64_t tile ) {
        cyclic_system<M, H, F32, STORE>(
            tile * SPB + threadIdx.x / H, src, tgt, n_tgt, indices, order, row0,
            row_off, rows, n_rows, kk_uniform, rbf, geometry, truncation, rcond,
            max_sweeps, coeffs, coeffs32, pinv_out, counters, by_distance,
            screened );
    };
    if constexpr ( LIST )
    {
        // the trip count is uniform over the block (the pair shuffles and
        // the wave-wide convergence vote need every lane); the loop costs
        // registers, so the whole-operator form below has none
        // (a list's rows sit in its first tiles and are scattered over the
        // operator: tiles in dispatch order spread them over the XCDs)
        int64_t const n = *n_rows;
        for ( int64_t tile = blockIdx.x; tile * SPB < n; tile += gridDim.x )
            one( tile );
    }
    else
        one( xcd_tile() );
}

template <int M, int H>
void launch_cyclic( double4 const *src, double4 const *tgt, int64_t n_tgt,
                    int32_t const *indices, int32_t const *order,
                    SetupParams const &p, double *coeffs, float *coeffs32,
                    double *pinv, unsigned long long *counters, hipStream_t s )
{
    int const sweeps = p.max_rot > 0 ? static_cast<int>( p.max_rot ) : 30;
    bool const strided = p.rows != nullptr;
    int64_t blocks = ceil_div( n_tgt - p.row0, kBlock / H );
    if ( strided )
        blocks = blocks < kListBlocks ? blocks : kListBlocks;
    dim3 const grid( blocks ), block( kBlock );
    auto run = [&]( auto f32, auto store ) {
        auto kernel = strided ? setup_cyclic_kernel<M, H, decltype( f32 )::value,
                                                    decltype( store )::value, true>
                              : setup_cyclic_kernel<M, H, decltype( f32 )::value,
                                                    decltype( store )::value, false>;
        kernel<<<grid, block, 0, s>>>( src, tgt, n_tgt, indices, order, p.row0,
                                     p.row_off, p.rows, p.n_rows, p.kk,
                                     p.rbf, p.geometry, p.truncation, p.rcond,
                                     sweeps, coeffs, coeffs32, pinv, counters,
                                     p.by_distance, p.screened );
    };
    using T = std::true_type;
    using F = std::false_type;
    if ( coeffs32 )
        pinv ? run( T{}, T{} ) : run( T{}, F{} );
    else
        pinv ? run( F{}, T{} ) : run( F{}, F{} );
    DTKX_HIP( hipGetLastError() );
}

// Listed rows, one lane each: the cyclic Jacobi of cyclic_system on A, whose
// rotations never read V. Rows whose eigenvalues all pass the truncation test
// go to refine_rows (solved again by Cholesky). For the others V is formed
// afterwards, in the registers that A leaves, from the rotations' tangents
// (kept for each wave and sweep; the last region takes all later sweeps,
// which are not read). The operations are cyclic_system's and a converged system's
// rotations exact no-ops whatever its wave, so all results are its bit for
// bit. A wave with few truncated rows, or a row that took more sweeps than
// are kept, leaves those to a second pass (listed_rest_kernel), where the
// waves are full and ten regions kept; what still needs more there, or holds
// a value that is not finite, goes to full_rows (cyclic_system, from their
// start).
//
// Bound by the FP64 of the rotations (a division chain and 64 fused
// operations on A, 45 a sweep). A and V together (155 doubles) took two lanes
// a system that both rotated A, at one wave a SIMD, after a first pass over
// the list for the eigenvalues: a transfer with 300,000 such rows of 32 (a
// shell) 2.26 ms, now 1.45. Measured on the way: the stores of the tangents
// cost nothing beside the rotations; tiles from a queue instead of a stride
// 797 -> 688 us of the kernel, as 4,688 tiles over 2,048 blocks leave some
// with a third; gathers four neighbours at a time gave nothing.
// The full grid's blocks have seven regions each, for six sweeps: the shell's
// rows take 4.3 on average, and at its size seven regions measure as ten do
// (setup 1.04-1.06 ms), at 330 MB of scratch instead of 472. A smaller grid's
// blocks share as many, up to ten each: there a few rows' second pass is a
// tenth of the setup.
constexpr int kKeptSweeps = 7;
constexpr int kKeptAgain = 10;
// A block whose rows need more takes one of these further shares, of three
// regions, if any is left: one wave with a seventh sweep would otherwise add
// the second pass's whole latency (a shell of 130k rows 0.85 -> 1.04 ms).
constexpr int kSpares = 128;
constexpr int kSpareRegions = 3;
// Where the list is longer than a tile a block, a wave with less than a
// quarter of its rows truncated leaves them to the second pass. Rows of 10
// with the quadratic basis, of which half are listed and 5 % of those
// truncated, 3 or 4 a wave, whose V nearly every wave formed: setup of 1M rows
// (3.8 tiles a block) 1.46 -> 1.22 ms, of 300k (1.1) 590 -> 565 us; of 250k
// (0.95) the second pass's own latency would cost 20 us. Where every row is
// truncated (a shell) it would only repeat the sweeps. A share of 1/8 left
// 1.27 ms, 1/2 as 1/4.
// two waves a SIMD at this kernel's registers (one: 1.21 ms)
constexpr int kListedBlocks = 2048;

int64_t listed_blocks( int64_t rows )
{
    return std::min<int64_t>( ceil_div( rows, kBlock ), kListedBlocks );
}

// regions of each block of the first pass
int kept_regions( int64_t rows )
{
    return static_cast<int>( std::min<int64_t>(
        kListedBlocks * kKeptSweeps / listed_blocks( rows ), kKeptAgain ) );
}

// blocks of the second pass that take truncated rows: their ten regions
// within the first pass's scratch
int64_t again_blocks( int64_t rows )
{
    return std::max<int64_t>(
        listed_blocks( rows ) * kept_regions( rows ) / kKeptAgain, 1 );
}

// regions of the first pass, or of the second
int64_t listed_regions( int64_t rows )
{
    return std::max<int64_t>( listed_blocks( rows ) * kept_regions( rows ),
                              again_blocks( rows ) * kKeptAgain );
}

struct Listed
{
    double4 const *src, *tgt;
    int32_t const *indices, *order;
    int64_t const *row_off;
    int32_t const *rows, *n_rows;
    int kk, rbf, geometry, truncation;
    double rcond;
    int max_sweeps;
    bool by_distance;
    double *coeffs;
    float *coeffs32;
    double *tangents, *spares;
    int kept;
    unsigned long long *counters;
    // rows for Cholesky from the front of refine_rows, rows for the second
    // pass from its end (both together are at most the listed rows)
    int32_t *refine_rows, *n_refine, *n_later;
    int64_t refine_end;
    int32_t *full_rows, *n_full, *queue, *refine_queue, *n_spares;
};

// the coefficients of a row whose a0 is x
template <int M, bool F32>
__device__ __forceinline__ void listed_coefficients( Listed const &a,
                                                     double const *x,
                                                     SystemRow const &sr )
{
    for ( int l = 0; l < sr.kk; ++l )
    {
        double P[M];
        double const phi = nbr_row<M, F32>( a.geometry, a.rbf, sr.radius,
                                            a.src[sr.nbr[l]], sr.tp, P );
        double acc = 0.0;
#pragma unroll
        for ( int j = 0; j < M; ++j )
            acc = fma( x[j], P[j], acc );
        if constexpr ( F32 )
            a.coeffs32[sr.rbeg + l] = (float)( acc * phi );
        else
            a.coeffs[sr.rbeg + l] = acc * phi;
    }
}

// a block's spare share: its number, none asked for yet, or none left
constexpr int kNoSpare = -1;
constexpr int kSparesGone = -2;

// one row (every lane of the wave has to call: the vote); AGAIN: the second
// pass, whose rows are all truncated; sparse: waves with few truncated rows
// leave them to it
template <int M, bool F32, bool AGAIN>
__device__ __forceinline__ void listed_row( Listed const &a, bool valid,
                                            int64_t slot, double *mine,
                                            bool sparse, int &spare )
{
    using S = SymIdx<M>;
    constexpr int kStride = rotations<M> * kLanes;
    int const kept = AGAIN ? kKeptAgain : a.kept;
    // where a sweep's tangents are (sweeps beyond the kept ones: the spare
    // share if the block has one, else over the last region)
    auto region = [&]( int pass ) {
        int const last = ( !AGAIN && spare >= 0 ? kSpareRegions : 0 ) + kept - 1;
        int const p = pass < last ? pass : last;
        return p < kept ? mine + p * kStride
                        : a.spares + threadIdx.x +
                              ( (int64_t)spare * kSpareRegions + p - kept ) *
                                  kStride;
    };
    double A[S::size];
    (void)system_moments<M, F32>( valid, slot, a.src, a.tgt, a.indices,
                                  a.order, a.row_off, a.kk, a.rbf, a.geometry,
                                  a.by_distance, A );
    double no_v[1];
    int sweeps = 0, pass = 0;
    bool done = !valid || converged<M>( A );
    for ( ; !__all( done ) && pass < a.max_sweeps; ++pass )
    {
        if constexpr ( !AGAIN )
            if ( pass == kept && spare == kNoSpare )
            {
                int taken = 0;
                if ( threadIdx.x == 0 )
                    taken = atomicAdd( a.n_spares, 1 );
                taken = __builtin_amdgcn_readfirstlane( taken );
                spare = taken < kSpares ? taken : kSparesGone;
            }
        sweep_all<M, 0, true>( A, no_v, done, region( pass ) );
        sweeps += done ? 0 : 1;
        done = done || converged<M>( A );
    }
    double thr;
    bool const under = valid && truncated<M>( A, a.truncation, a.rcond, thr );
    bool finite = true;
#pragma unroll
    for ( int k = 0; k < M; ++k )
        finite = finite && fabs( A[S::at( k, k )] ) <= DBL_MAX;
    // a sweep is kept if no later one was written over it
    int const readable =
        kept + ( !AGAIN && spare >= 0 ? kSpareRegions : 0 );
    bool here =
        under && finite && ( sweeps < readable || pass <= readable );
    if constexpr ( !AGAIN )
    {
        int const formed = __popcll( __ballot( here ) );
        int const rows = __popcll( __ballot( valid ) );
        here = here && ( !sparse || 4 * formed >= rows );
        if ( valid && !under )
            a.refine_rows[atomicAdd( a.n_refine, 1 )] = (int32_t)slot;
        if ( under && finite && !here )
            a.refine_rows[a.refine_end - atomicAdd( a.n_later, 1 )] =
                (int32_t)slot;
    }
    if ( under && !here && ( AGAIN || !finite ) )
        a.full_rows[atomicAdd( a.n_full, 1 )] = (int32_t)slot;
    if ( a.counters && valid && ( here || !under ) )
    {
        if ( under )
            atomicAdd( a.counters + 0, 1ull );
        if ( !done )
            atomicAdd( a.counters + 1, 1ull );
        atomicAdd( a.counters + 2, (unsigned long long)sweeps );
    }
    if ( !here )
        return;
    double lambda[M], x[M];
#pragma unroll
    for ( int k = 0; k < M; ++k )
        lambda[k] = A[S::at( k, k )];
    {
        double V[M * M];
#pragma unroll
        for ( int e = 0; e < M * M; ++e )
            V[e] = e / M == e % M ? 1.0 : 0.0;
        for ( int p = 0; p < sweeps; ++p )
            sweep_vectors<M>( V, region( p ) );
#pragma unroll
        for ( int r = 0; r < M; ++r )
            x[r] = 0.0;
#pragma unroll
        for ( int k = 0; k < M; ++k )
        {
            double const w = fabs( lambda[k] ) >= thr ? V[k] / lambda[k] : 0.0;
#pragma unroll
            for ( int r = 0; r < M; ++r )
                x[r] = fma( w, V[r * M + k], x[r] );
        }
    }
    // the row read again instead of held through the sweeps (its 14 registers
    // were spilled there: 4.60 -> 4.48 ms for the 2M rows of a shell); the
    // empty statement hides from the compiler that it is the same row
    int32_t again = (int32_t)slot;
    asm volatile( "" : "+v"( again ) );
    listed_coefficients<M, F32>(
        a, x,
        system_row<M, F32>( true, again, a.src, a.tgt, a.indices, a.order,
                            a.row_off, a.kk, a.geometry, a.by_distance ) );
}

template <int M, bool F32>
__global__ void __launch_bounds__( kBlock, 2 ) eigen_listed_kernel( Listed a )
{
    double *const mine =
        a.tangents + (int64_t)blockIdx.x * a.kept * rotations<M> * kLanes +
        threadIdx.x;
    // tiles in dispatch order spread the list's first tiles over the XCDs; a
    // block's next one comes from the queue (uniform over the block: the
    // wave-wide vote needs every lane), which ends with the list
    int64_t const n = *a.n_rows;
    bool const sparse = n > (int64_t)gridDim.x * kBlock;
    int spare = kNoSpare;
    auto next = [&]() {
        int t = 0;
        if ( threadIdx.x == 0 )
            t = atomicAdd( a.queue, 1 );
        return (int64_t)gridDim.x + __builtin_amdgcn_readfirstlane( t );
    };
    for ( int64_t tile = blockIdx.x; tile * kBlock < n; tile = next() )
    {
        int64_t const li = tile * kBlock + threadIdx.x;
        bool const valid = li < n;
        listed_row<M, F32, false>( a, valid, valid ? a.rows[li] : 0, mine,
                                   sparse, spare );
    }
}

// The untruncated rows again by Cholesky, one lane a row: the moments, their
// inverse factor and the row's coefficients. A non-positive pivot sends the
// row to full_rows.
template <int M, bool F32>
__device__ __forceinline__ void refine_row( Listed const &a, int64_t slot )
{
    using S = SymIdx<M>;
    double A[S::size];
    SystemRow const sr = system_moments<M, F32>(
        true, slot, a.src, a.tgt, a.indices, a.order, a.row_off, a.kk, a.rbf,
        a.geometry, a.by_distance, A );
    if ( !cholesky_factor_inverse<M>( A ) )
    {
        a.full_rows[atomicAdd( a.n_full, 1 )] = (int32_t)slot;
        return;
    }
    double x[M];
#pragma unroll
    for ( int i = 0; i < M; ++i )
    {
        double acc = 0.0;
#pragma unroll
        for ( int k = i; k < M; ++k )
            acc = fma( A[S::at( i, k )], A[S::at( 0, k )], acc );
        x[i] = acc;
    }
    listed_coefficients<M, F32>( a, x, sr );
}

// What the first pass left: its truncated rows, packed into full waves, over
// the first n_again blocks, and the Cholesky rows beside them, tiles from a
// queue that the blocks without truncated rows start on at once.
template <int M, bool F32>
__global__ void __launch_bounds__( kBlock, 2 )
    listed_rest_kernel( Listed a, int n_again )
{
    int64_t const n_later = *a.n_later;
    if ( (int)blockIdx.x < n_again )
    {
        double *const mine =
            a.tangents +
            (int64_t)blockIdx.x * kKeptAgain * rotations<M> * kLanes +
            threadIdx.x;
        int none = kSparesGone;
        for ( int64_t tile = blockIdx.x; tile * kBlock < n_later;
              tile += n_again )
        {
            int64_t const li = tile * kBlock + threadIdx.x;
            bool const valid = li < n_later;
            listed_row<M, F32, true>(
                a, valid, valid ? a.refine_rows[a.refine_end - li] : 0, mine,
                false, none );
        }
    }
    // a block's first tile is its own (one atomic a block on a single word cost
    // a short list 15 us), counted from the first block without truncated
    // rows; later ones come from the queue
    int64_t const n = *a.n_refine;
    int64_t const tiles = ( n_later + kBlock - 1 ) / kBlock;
    int64_t const busy = tiles < n_again ? tiles : n_again;
    auto next = [&]() {
        int t = 0;
        if ( threadIdx.x == 0 )
            t = atomicAdd( a.refine_queue, 1 );
        return (int64_t)gridDim.x + __builtin_amdgcn_readfirstlane( t );
    };
    int64_t const first =
        blockIdx.x + ( blockIdx.x < busy ? (int64_t)gridDim.x : 0 ) - busy;
    for ( int64_t tile = first; tile * kBlock < n; tile = next() )
    {
        int64_t const li = tile * kBlock + threadIdx.x;
        if ( li < n )
            refine_row<M, F32>( a, a.refine_rows[li] );
    }
}

} // namespace

std::size_t setup_listed_scratch( int m, int64_t rows )
{
    int const n = m == 10 ? rotations<10> : ( m == 4 ? rotations<4> : 0 );
    if ( rows <= 0 )
        return 0;
    int64_t const regions = listed_regions( rows );
    return static_cast<std::size_t>( regions + kSpares * kSpareRegions ) * n *
           kLanes;
}

void setup_listed( double4 const *src, double4 const *tgt, int64_t n_tgt,
                   int32_t const *indices, int32_t const *order,
                   SetupParams const &p, double *coeffs, float *coeffs32,
                   int32_t *full_rows, int32_t *n_full, int32_t *counts,
                   unsigned long long *counters, hipStream_t s )
{
    DTKX_REQUIRE( p.rows && p.n_rows, DTKX_ERR_INVALID_ARGUMENT );
    if ( n_tgt <= p.row0 )
        return;
    int64_t const n = n_tgt - p.row0, blocks = listed_blocks( n );
    DeviceBuffer<int32_t> rlist( n, s );
    DeviceBuffer<double> owned;
    double *tangents = p.tangents;
    if ( !tangents )
    {
        owned.resize( std::max<std::size_t>( setup_listed_scratch( p.m, n ), 1 ),
                      s );
        tangents = owned.get();
    }
    int const sweeps = p.max_rot > 0 ? static_cast<int>( p.max_rot ) : 30;
    Listed const a{ src, tgt, indices, order, p.row_off, p.rows, p.n_rows, p.kk,
                    p.rbf, p.geometry, p.truncation, p.rcond, sweeps,
                    p.by_distance, coeffs, coeffs32, tangents,
                    tangents + listed_regions( n ) * p.m * ( p.m - 1 ) / 2 * kLanes,
                    kept_regions( n ), counters,
                    rlist.get(), counts, counts + 1, n - 1,
                    full_rows, n_full, counts + 2, counts + 3, counts + 4 };
    auto run = [&]( auto m, auto f32 ) {
        constexpr int kM = decltype( m )::value;
        constexpr bool kF32 = decltype( f32 )::value;
        eigen_listed_kernel<kM, kF32><<<blocks, kBlock, 0, s>>>( a );
        listed_rest_kernel<kM, kF32><<<blocks, kBlock, 0, s>>>(
            a, static_cast<int>( again_blocks( n ) ) );
    };
    using T = std::true_type;
    using F = std::false_type;
    using M1 = std::integral_constant<int, 1>;
    using M4 = std::integral_constant<int, 4>;
    using M10 = std::integral_constant<int, 10>;
    if ( p.m == 1 )
        coeffs32 ? run( M1{}, T{} ) : run( M1{}, F{} );
    else if ( p.m == 4 )
        coeffs32 ? run( M4{}, T{} ) : run( M4{}, F{} );
    else if ( p.m == 10 )
        coeffs32 ? run( M10{}, T{} ) : run( M10{}, F{} );
    else
        DTKX_REQUIRE( p.m == 1 || p.m == 4 || p.m == 10,
                      DTKX_ERR_INVALID_ARGUMENT );
    DTKX_HIP( hipGetLastError() );
}

void setup_cyclic( double4 const *src, double4 const *tgt, int64_t n_tgt,
                   int32_t const *indices, int32_t const *order,
                   SetupParams const &p, double *coeffs, float *coeffs32,
                   double *pinv, unsigned long long *counters, hipStream_t s )
{
    if ( n_tgt <= p.row0 )
        return;
    switch ( p.m )
    {
    case 1:
        launch_cyclic<1, 1>( src, tgt, n_tgt, indices, order, p, coeffs,
                                 coeffs32, pinv, counters, s );
        return;
    case 4:
        launch_cyclic<4, 1>( src, tgt, n_tgt, indices, order, p, coeffs,
                                 coeffs32, pinv, counters, s );
        return;
    case 10:
        launch_cyclic<10, 2>( src, tgt, n_tgt, indices, order, p, coeffs,
                                 coeffs32, pinv, counters, s );
        return;
    }
    DTKX_REQUIRE( p.m == 1 || p.m == 4 || p.m == 10, DTKX_ERR_INVALID_ARGUMENT );
}

} // namespace dtkx
