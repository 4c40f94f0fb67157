// Scene box, curve codes and both sorts of a small search in one launch.
//
// A search of up to kSmallSort sources and targets spends its time on
// launches, not on work: the scene box (two), the codes (one) and eight radix
// passes of a tile or two took 95 us for 1000 points, most of it waiting for
// the launch before. Here one block of 16 waves sorts the sources and another
// the targets (each forms the scene box for itself): the keys stay in
// registers, a pass ranks them as radix_sort.hpp does (per wave and slot,
// lanes with the same digit found by ballots) and moves them through LDS.
// 1000 points take 26 us. One CU does the ranking of all keys, so the time
// grows with them: search of 2000 / 4000 / 8000 points, k = 4, 0.074 / 0.095 /
// 0.150 ms, and 0.202 ms for 8200 with the passes' launches; at 12 keys a
// thread this lost (0.32 ms against 0.22 at 12,000).
#ifndef DTKX_KNN_SMALL_HPP
#define DTKX_KNN_SMALL_HPP

namespace dtkx
{
namespace
{

constexpr int kSmallThreads = 1024;
constexpr int kSmallWaves = kSmallThreads / 64;
constexpr int kSmallSort = 8 * kSmallThreads;

template <typename T, typename V>
struct SmallSortArgs
{
    V const *src = nullptr, *tgt = nullptr;
    int n_src = 0, n_tgt = 0;
    T *box = nullptr;          // the scene box, lower then upper corner
    uint64_t *codes = nullptr; // the sources' codes, sorted
    int32_t *src_ids = nullptr, *src_pos = nullptr; // src_pos nullable
    int32_t *tgt_ids = nullptr, *tgt_pos = nullptr; // tgt_pos nullable
    V *src_sorted = nullptr;
    double4 const *src4 = nullptr; // nullable, with src4_sorted
    double4 *src4_sorted = nullptr;
};

// Block 0 takes the sources, block 1 the targets; ITEMS keys a thread.
template <typename T, typename V, int ITEMS>
__global__ void __launch_bounds__( kSmallThreads )
    small_sort_kernel( SmallSortArgs<T, V> const g )
{
    constexpr int kDigits = rsort::kDigits;
    __shared__ uint64_t skeys[ITEMS * kSmallThreads];
    __shared__ uint16_t svals[ITEMS * kSmallThreads];
    __shared__ uint32_t whist[kSmallWaves][kDigits];
    __shared__ uint32_t start[kDigits];
    __shared__ uint32_t scan[kDigits / 64];
    __shared__ T corner[kSmallWaves][6];
    int const t = threadIdx.x, lane = t & 63, w = t >> 6;
    bool const is_src = blockIdx.x == 0;

    // the sources' box (min and max are exact in any order)
    T b[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    for ( int i = t; i < g.n_src; i += kSmallThreads )
    {
        V const p = g.src[i];
        b[0] = fmin( b[0], p.x );
        b[1] = fmin( b[1], p.y );
        b[2] = fmin( b[2], p.z );
        b[3] = fmax( b[3], p.x );
        b[4] = fmax( b[4], p.y );
        b[5] = fmax( b[5], p.z );
    }
    for ( int o = 32; o > 0; o >>= 1 )
        for ( int d = 0; d < 3; ++d )
        {
            b[d] = fmin( b[d], __shfl_xor( b[d], o, 64 ) );
            b[3 + d] = fmax( b[3 + d], __shfl_xor( b[3 + d], o, 64 ) );
        }
    if ( lane == 0 )
        for ( int d = 0; d < 6; ++d )
            corner[w][d] = b[d];
    __syncthreads();
    for ( int v = 0; v < kSmallWaves; ++v )
        for ( int d = 0; d < 3; ++d )
        {
            b[d] = fmin( b[d], corner[v][d] );
            b[3 + d] = fmax( b[3 + d], corner[v][3 + d] );
        }
    if ( is_src && t == 0 )
        for ( int d = 0; d < 6; ++d )
            g.box[d] = b[d];
    CurveFrame const frame = curve_frame( b );

    V const *const pts = is_src ? g.src : g.tgt;
    int const n = is_src ? g.n_src : g.n_tgt;
    int const bits = is_src ? kSrcKeyBits : kTgtKeyBits;
    int const w0 = w * ( 64 * ITEMS );
    uint64_t key[ITEMS];
    uint32_t val[ITEMS], rank[ITEMS];
#pragma unroll
    for ( int s = 0; s < ITEMS; ++s )
    {
        int const i = w0 + s * 64 + lane;
        key[s] = 0;
        val[s] = i;
        if ( i < n )
        {
            uint32_t q[3];
            curve_cell( pts[i], frame, q );
            key[s] = is_src ? hilbert_code<21>( q )
                            : target_key( pts[i], frame );
        }
    }
    for ( int shift = 0; shift < bits; shift += 8 )
    {
        int const nbits = min( 8, bits - shift );
        uint32_t const mask = ( 1u << nbits ) - 1u;
        for ( int i = lane; i < kDigits; i += 64 )
            whist[w][i] = 0;
        rsort::wave_lds_order();
#pragma unroll
        for ( int s = 0; s < ITEMS; ++s )
        {
            bool const ok = w0 + s * 64 + lane < n;
            uint32_t const d = (uint32_t)( key[s] >> shift ) & mask;
            // (bits past nbits are 0 in every digit)
            uint64_t const m = rsort::same_digit( d, __ballot( ok ) );
            uint32_t const below = rsort::lanes_below( m );
            uint32_t prior = 0;
            if ( ok )
                prior = whist[w][d];
            rsort::wave_lds_order();
            if ( ok && below == 0 )
                whist[w][d] = prior + (uint32_t)__popcll( m );
            rsort::wave_lds_order();
            rank[s] = prior + below;
        }
        __syncthreads();
        // thread t < 256: digit t's offset in each wave and its total
        uint32_t total = 0;
        if ( t < kDigits )
        {
#pragma unroll
            for ( int v = 0; v < kSmallWaves; ++v )
            {
                uint32_t const c = whist[v][t];
                whist[v][t] = total;
                total += c;
            }
        }
        uint32_t const sum = rsort::wave_inclusive_scan( total );
        if ( t < kDigits && lane == 63 )
            scan[w] = sum;
        __syncthreads();
        if ( t < kDigits )
        {
            uint32_t before = sum - total;
            for ( int v = 0; v < w; ++v )
                before += scan[v];
            start[t] = before;
        }
        __syncthreads();
#pragma unroll
        for ( int s = 0; s < ITEMS; ++s )
            if ( w0 + s * 64 + lane < n )
            {
                uint32_t const d = (uint32_t)( key[s] >> shift ) & mask;
                uint32_t const at = start[d] + whist[w][d] + rank[s];
                skeys[at] = key[s];
                svals[at] = (uint16_t)val[s];
            }
        __syncthreads();
#pragma unroll
        for ( int s = 0; s < ITEMS; ++s )
        {
            int const i = w0 + s * 64 + lane;
            if ( i < n )
            {
                key[s] = skeys[i];
                val[s] = svals[i];
            }
        }
    }
#pragma unroll
    for ( int s = 0; s < ITEMS; ++s )
    {
        int const i = w0 + s * 64 + lane;
        if ( i >= n )
            continue;
        int32_t const id = (int32_t)val[s];
        if ( is_src )
        {
            g.codes[i] = key[s];
            g.src_ids[i] = id;
            if ( g.src_pos )
                g.src_pos[id] = i;
            g.src_sorted[i] = g.src[id];
            if ( g.src4_sorted )
                g.src4_sorted[i] = g.src4[id];
        }
        else
        {
            g.tgt_ids[i] = id;
            if ( g.tgt_pos )
                g.tgt_pos[id] = i;
        }
    }
}

template <typename T, typename V>
void small_sort( SmallSortArgs<T, V> const &g, hipStream_t s )
{
    int const n = std::max( g.n_src, g.n_tgt );
    dim3 const grid( g.n_tgt > 0 ? 2 : 1 ), block( kSmallThreads );
    if ( n <= 2 * kSmallThreads )
        small_sort_kernel<T, V, 2><<<grid, block, 0, s>>>( g );
    else if ( n <= 4 * kSmallThreads )
        small_sort_kernel<T, V, 4><<<grid, block, 0, s>>>( g );
    else
        small_sort_kernel<T, V, 8><<<grid, block, 0, s>>>( g );
    DTKX_HIP( hipGetLastError() );
}

} // namespace
} // namespace dtkx

#endif
