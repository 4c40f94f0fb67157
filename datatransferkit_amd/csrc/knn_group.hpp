// Neighbour search by groups of targets, for gfx950 wave64.
//
// The sources are sorted along a Hilbert curve, so any run of consecutive
// sources is spatially compact: eight consecutive sources form a block,
// eight blocks a node, and so on up, each with its exact box (an implicit
// eight-way tree; no links). The targets are sorted along the same curve,
// and a wave takes a group of consecutive targets:
//   1. gather: the nodes and blocks whose box lies within a radius R of the
//      group's box are found level by level, 64 box tests at a time, then
//      the points of those blocks within R of the group's box. Every source
//      within R of any of the group's targets is among them. They are held
//      in registers, one a lane and chunk of 64.
//   2. select: for each target, whose coordinates are uniform over the wave,
//      every lane forms the squared distance of its candidates, and a
//      threshold t with between kk and S candidates at or below it is found
//      by counting (a ballot and a population count a chunk). The target is
//      done if t (with the margin of the rounded root below) does not reach
//      past R; else the group's unfinished targets are gathered again with
//      the larger radius that the count names. Where distances are tied the
//      counts may jump from below kk to above S (on a lattice 7 and 19 around
//      a node, 8 and 32 around a cell's centre): then the kk-th distance
//      itself is found, and at it the lowest source indices.
//   3. sort: the selected candidates of 16 targets are sorted together, four
//      lanes a row, and the first kk of each row written.
// R starts from the size of the 64-point node nearest the wave's first
// group, and then from the radii that the wave's last group needed.
//
// Why this and not one traversal per lane: a lane that walks a tree by
// itself spends about 30 vector instructions a node and 35 a list insertion
// with most lanes of its wave masked off, some 40,000 a target at k = 32.
// Here a target costs about 16 a chunk of 64 candidates (four to five chunks
// at k = 32), a sixteenth of the group's gather and of the sort. 1M x 1M
// uniform points, the query alone: k = 32 0.59 ms against 1.82 ms, k = 10
// 0.43 against 0.69, k = 1 0.27 against 0.32 (whose hierarchies took another
// 0.08 to build); 9e4 x 1e5 with k = 64 0.23 against 0.57. What bounds it now
// is instruction issue (7,450 vector and 4,950 scalar instructions a wave
// of 32 targets at k = 32, four waves a SIMD): no HBM figure is near.
//
// Exactness: distances are formed in the operation order of box_sq, box
// distances per axis from the same rounded differences, and rounding is
// monotonic, so no source with a squared distance <= R^2 is dropped by the
// gather. Rows are ordered by (rounded root, source index): the sort's
// 32-bit keys hold the squared distance in steps of t 2^-25 or finer, and
// any two neighbours of a row closer than the root's rounding send the
// rows through a second sort by the full (distance, index) keys.
#ifndef DTKX_KNN_GROUP_HPP
#define DTKX_KNN_GROUP_HPP

#include <type_traits>
#include <utility>

namespace dtkx
{
namespace
{

// Levels up to the first of at most 64 nodes (at least two), and the node
// count of each.
inline int box_levels( int64_t n, int64_t *count )
{
    int l = 0;
    int64_t nodes = n;
    do
    {
        nodes = ( nodes + 7 ) / 8;
        count[l] = nodes;
        ++l;
    } while ( ( nodes > 64 || l < 2 ) && l < kMaxBoxLevels );
    return l;
}

template <typename T>
__device__ inline T shfl_xor( T v, int o )
{
    return __shfl_xor( v, o, 64 );
}

// Three levels of boxes above n inputs (points, or the boxes of the level
// below), 512 inputs a block, one a thread. ids (nullable): the points are
// read through it and also written in order to out_pts.
template <typename T, typename V, bool POINTS>
__global__ void __launch_bounds__( 512 )
    box_levels_kernel( V const *pts, int32_t const *ids, V *out_pts,
                       CurveBox<T> const *in, int64_t n, CurveBox<T> *l0,
                       CurveBox<T> *l1, CurveBox<T> *l2 )
{
    __shared__ T sh[8][6];
    int64_t const i = blockIdx.x * (int64_t)512 + threadIdx.x;
    T b[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    if ( i < n )
    {
        if constexpr ( POINTS )
        {
            V const p = ids ? pts[ids[i]] : pts[i];
            if ( ids )
                out_pts[i] = p;
            b[0] = b[3] = p.x;
            b[1] = b[4] = p.y;
            b[2] = b[5] = p.z;
        }
        else
        {
            CurveBox<T> const c = in[i];
#pragma unroll
            for ( int d = 0; d < 3; ++d )
            {
                b[d] = c.lo[d];
                b[3 + d] = c.hi[d];
            }
        }
    }
    auto store = [&]( CurveBox<T> *out, int64_t j ) {
        CurveBox<T> c;
#pragma unroll
        for ( int d = 0; d < 3; ++d )
        {
            c.lo[d] = b[d];
            c.hi[d] = b[3 + d];
        }
        c.lo[3] = c.hi[3] = T( 0 );
        out[j] = c;
    };
#pragma unroll
    for ( int o = 1; o < 64; o <<= 1 )
    {
#pragma unroll
        for ( int d = 0; d < 3; ++d )
        {
            b[d] = fmin( b[d], shfl_xor( b[d], o ) );
            b[3 + d] = fmax( b[3 + d], shfl_xor( b[3 + d], o ) );
        }
        if ( o == 4 && ( threadIdx.x & 7 ) == 0 && i < n )
            store( l0, i / 8 );
    }
    int const w = threadIdx.x / 64;
    if ( ( threadIdx.x & 63 ) == 0 )
    {
        if ( l1 && i < n )
            store( l1, i / 64 );
#pragma unroll
        for ( int d = 0; d < 6; ++d )
            sh[w][d] = b[d];
    }
    __syncthreads();
    if ( l2 && threadIdx.x == 0 )
    {
        for ( int v = 1; v < 8; ++v )
            for ( int d = 0; d < 3; ++d )
            {
                b[d] = fmin( b[d], sh[v][d] );
                b[3 + d] = fmax( b[3 + d], sh[v][3 + d] );
            }
        store( l2, blockIdx.x );
    }
}

// -------------------------------------------------------- wave helpers
// Lane permutations within groups of 8 by DPP (no LDS traffic).
constexpr int kDppXor1 = 0xB1;       // quad_perm 1,0,3,2
constexpr int kDppXor2 = 0x4E;       // quad_perm 2,3,0,1
constexpr int kDppXor3 = 0x1B;       // quad_perm 3,2,1,0
constexpr int kDppHalfMirror = 0x141; // lane ^ 7
constexpr int kDppMirror = 0x140;    // lane ^ 15

template <int CTRL>
__device__ inline uint32_t dpp( uint32_t v )
{
    return (uint32_t)__builtin_amdgcn_mov_dpp( (int)v, CTRL, 0xf, 0xf, true );
}
template <int CTRL>
__device__ inline float dpp( float v )
{
    return __uint_as_float( dpp<CTRL>( __float_as_uint( v ) ) );
}
template <int CTRL>
__device__ inline uint64_t dpp( uint64_t v )
{
    return ( (uint64_t)dpp<CTRL>( (uint32_t)( v >> 32 ) ) << 32 ) |
           dpp<CTRL>( (uint32_t)v );
}
template <int CTRL>
__device__ inline double dpp( double v )
{
    return __longlong_as_double(
        (long long)dpp<CTRL>( (uint64_t)__double_as_longlong( v ) ) );
}
template <int CTRL>
__device__ inline DKey dpp( DKey k )
{
    return {dpp<CTRL>( k.d ), (int32_t)dpp<CTRL>( (uint32_t)k.id )};
}

__device__ inline float lane_value( float v, int lane )
{
    return __uint_as_float(
        (uint32_t)__builtin_amdgcn_readlane( (int)__float_as_uint( v ), lane ) );
}
__device__ inline double lane_value( double v, int lane )
{
    long long const b = __double_as_longlong( v );
    uint32_t const lo =
        (uint32_t)__builtin_amdgcn_readlane( (int)( b & 0xffffffff ), lane );
    uint32_t const hi =
        (uint32_t)__builtin_amdgcn_readlane( (int)( b >> 32 ), lane );
    return __longlong_as_double( (long long)( ( (uint64_t)hi << 32 ) | lo ) );
}
template <typename T>
__device__ inline T uniform( T v )
{
    return lane_value( v, 0 );
}
__device__ inline int uniform( int v )
{
    return __builtin_amdgcn_readfirstlane( v );
}
__device__ inline uint64_t uniform( uint64_t v )
{
    uint32_t const lo = (uint32_t)__builtin_amdgcn_readfirstlane( (int)v );
    uint32_t const hi =
        (uint32_t)__builtin_amdgcn_readfirstlane( (int)( v >> 32 ) );
    return ( (uint64_t)hi << 32 ) | lo;
}

// min / max over the wave, uniform. Floats as integers of the same order
// (the sign's complement of the other bits), whose last step is scalar.
__device__ inline int ordered( float v )
{
    int const b = (int)__float_as_uint( v );
    return b ^ ( ( b >> 31 ) & 0x7fffffff );
}
__device__ inline float from_ordered( int b )
{
    return __uint_as_float( (uint32_t)( b ^ ( ( b >> 31 ) & 0x7fffffff ) ) );
}
template <int CTRL>
__device__ inline int dpp( int v )
{
    return __builtin_amdgcn_mov_dpp( v, CTRL, 0xf, 0xf, true );
}
__device__ inline int wave_min_int( int v )
{
    v = min( v, dpp<kDppXor1>( v ) );
    v = min( v, dpp<kDppXor2>( v ) );
    v = min( v, dpp<kDppHalfMirror>( v ) );
    v = min( v, dpp<kDppMirror>( v ) );
    return min( min( __builtin_amdgcn_readlane( v, 0 ),
                     __builtin_amdgcn_readlane( v, 16 ) ),
                min( __builtin_amdgcn_readlane( v, 32 ),
                     __builtin_amdgcn_readlane( v, 48 ) ) );
}
__device__ inline float wave_min( float v )
{
    return from_ordered( wave_min_int( ordered( v ) ) );
}
__device__ inline float wave_max( float v )
{
    return from_ordered( ~wave_min_int( ~ordered( v ) ) );
}
__device__ inline double wave_min( double v )
{
    v = fmin( v, dpp<kDppXor1>( v ) );
    v = fmin( v, dpp<kDppXor2>( v ) );
    v = fmin( v, dpp<kDppHalfMirror>( v ) );
    v = fmin( v, dpp<kDppMirror>( v ) );
    return uniform( fmin( fmin( lane_value( v, 0 ), lane_value( v, 16 ) ),
                          fmin( lane_value( v, 32 ), lane_value( v, 48 ) ) ) );
}
__device__ inline double wave_max( double v ) { return -wave_min( -v ); }
__device__ inline uint32_t wave_min_u32( uint32_t v )
{
    v = min( v, dpp<kDppXor1>( v ) );
    v = min( v, dpp<kDppXor2>( v ) );
    v = min( v, dpp<kDppHalfMirror>( v ) );
    v = min( v, dpp<kDppMirror>( v ) );
    uint32_t const a = (uint32_t)__builtin_amdgcn_readlane( (int)v, 0 );
    uint32_t const b = (uint32_t)__builtin_amdgcn_readlane( (int)v, 16 );
    uint32_t const c = (uint32_t)__builtin_amdgcn_readlane( (int)v, 32 );
    uint32_t const d = (uint32_t)__builtin_amdgcn_readlane( (int)v, 48 );
    return min( min( a, b ), min( c, d ) );
}

// The wave's lane, opaque to the compiler: what a loop derives from it is
// formed in the loop instead of being held in registers over all of it.
__device__ inline int opaque_lane()
{
    int l = threadIdx.x;
    asm volatile( "" : "+v"( l ) );
    return l;
}

// ------------------------------------------------------------ row sort
__device__ inline bool row_less( uint32_t a, uint32_t b ) { return a < b; }
__device__ inline bool row_less( uint64_t a, uint64_t b ) { return a < b; }
__device__ inline bool row_less( DKey const &a, DKey const &b )
{
    return key_less( a, b );
}
template <typename Key>
__device__ inline void row_exchange( Key &a, Key &b )
{
    bool const s = row_less( b, a );
    Key const x = a, y = b;
    a = key_pick( s, y, x );
    b = key_pick( s, x, y );
}
template <>
__device__ inline void row_exchange<uint32_t>( uint32_t &a, uint32_t &b )
{
    uint32_t const x = a, y = b;
    a = min( x, y );
    b = max( x, y );
}
// the smaller (hi false) or the larger of the lane's key and another lane's
template <typename Key>
__device__ inline Key row_keep( Key k, Key o, bool hi )
{
    bool const mine = row_less( k, o );
    return key_pick( mine != hi, k, o );
}
template <>
__device__ inline uint32_t row_keep<uint32_t>( uint32_t k, uint32_t o, bool hi )
{
    uint32_t const a = min( k, o ), b = max( k, o );
    return hi ? b : a;
}

// Each key against the other lane's key of the same place, or (REVERSE) of
// the mirrored place, taken in pairs so that no copy of the keys is held.
template <int CTRL, bool REVERSE, int E, typename Key>
__device__ inline void cross_lane( Key ( &k )[E], bool hi )
{
#pragma unroll
    for ( int e = 0; e < E; ++e )
    {
        if ( REVERSE && e < E / 2 )
        {
            Key const a = k[e], b = k[E - 1 - e];
            k[e] = row_keep( a, dpp<CTRL>( b ), hi );
            k[E - 1 - e] = row_keep( b, dpp<CTRL>( a ), hi );
        }
        else if ( !REVERSE )
            k[e] = row_keep( k[e], dpp<CTRL>( k[e] ), hi );
    }
}

// Compare-exchanges (lower, upper) of Batcher's odd-even merge sort of N
// keys, in order: a list, so that every index is a compile-time constant
// whatever the compiler's unrolling limits.
template <int N>
struct OddEven
{
    int lower[N * N] = {}, upper[N * N] = {};
    int count = 0;
    constexpr OddEven()
    {
        for ( int p = 1; p < N; p <<= 1 )
            for ( int q = p; q >= 1; q >>= 1 )
                for ( int j = q % p; j + q < N; j += 2 * q )
                    for ( int i = 0; i < q && i + j + q < N; ++i )
                        if ( ( i + j ) / ( 2 * p ) == ( i + j + q ) / ( 2 * p ) )
                        {
                            lower[count] = i + j;
                            upper[count] = i + j + q;
                            ++count;
                        }
    }
};
template <int N>
struct OddEvenCount
{
    static constexpr OddEven<N> kNet{};
    static constexpr int kCount = kNet.count;
};

template <int E, typename Key, std::size_t... I>
__device__ inline void odd_even_sort( Key ( &k )[E],
                                      std::index_sequence<I...> )
{
    ( row_exchange( k[std::integral_constant<
                          int, OddEven<E>{}.lower[I]>::value],
                    k[std::integral_constant<
                          int, OddEven<E>{}.upper[I]>::value] ),
      ... );
}

// Rows of W E keys, lane sub of a row's W lanes holding keys sub E ..
// sub E + E - 1, sorted ascending: each lane's keys by Batcher's odd-even
// merge sort, then runs of w lanes merged into runs of 2 w by a mirrored
// first step and half-cleaners.
template <int W, int E, typename Key>
__device__ inline void sort_rows( Key ( &k )[E], int sub )
{
    odd_even_sort( k, std::make_index_sequence<OddEvenCount<E>::kCount>{} );
    auto clean = [&]() {
#pragma unroll
        for ( int d = E / 2; d >= 1; d >>= 1 )
#pragma unroll
            for ( int e = 0; e < E; ++e )
                if ( !( e & d ) )
                    row_exchange( k[e], k[e + d] );
    };
    if constexpr ( W >= 2 )
    {
        cross_lane<kDppXor1, true>( k, sub & 1 );
        clean();
    }
    if constexpr ( W >= 4 )
    {
        cross_lane<kDppXor3, true>( k, sub & 2 );
        cross_lane<kDppXor1, false>( k, sub & 1 );
        clean();
    }
    if constexpr ( W >= 8 )
    {
        cross_lane<kDppHalfMirror, true>( k, sub & 4 );
        cross_lane<kDppXor2, false>( k, sub & 2 );
        cross_lane<kDppXor1, false>( k, sub & 1 );
        clean();
    }
}

// The key of the lane whose number is o different in its bits.
__device__ inline uint64_t lane_xor( uint64_t k, int o )
{
    return ( (uint64_t)(uint32_t)__shfl_xor( (int)( k >> 32 ), o, 64 ) << 32 ) |
           (uint32_t)__shfl_xor( (int)(uint32_t)k, o, 64 );
}
__device__ inline DKey lane_xor( DKey k, int o )
{
    return {__shfl_xor( k.d, o, 64 ), __shfl_xor( k.id, o, 64 )};
}

// N P keys over the first N lanes of the wave, P (1 or 2) a lane, sorted
// ascending (bitonic, as sort_rows' merges).
template <int P, int N, typename Key>
__device__ inline void sort_wave( Key ( &k )[P], int lane )
{
    static_assert( P == 1 || P == 2, "keys a lane" );
    if constexpr ( P == 2 )
        row_exchange( k[0], k[1] );
    for ( int w = 1; w < N; w <<= 1 )
        for ( int o = 2 * w - 1; o; o = ( o == 2 * w - 1 ? w : o ) >> 1 )
        {
            bool const mirror = o == 2 * w - 1;
            bool const hi = lane & ( mirror ? w : o );
            Key other[P];
#pragma unroll
            for ( int e = 0; e < P; ++e )
                other[e] = lane_xor( k[e], o );
#pragma unroll
            for ( int e = 0; e < P; ++e )
                k[e] = row_keep(
                    k[e], P == 2 && mirror ? other[P - 1 - e] : other[e], hi );
            if ( P == 2 && o == 1 && ( w == 1 || !mirror ) )
                row_exchange( k[0], k[P - 1] );
        }
}

// ----------------------------------------------------------- the search
// Squared distance from p to the box [lo, hi] in box_sq's order of
// operations: per axis at most the rounded |q - p| of any q in the box.
template <typename T>
__device__ inline T gap_sq( T const *plo, T const *phi, T const *lo, T const *hi )
{
#pragma clang fp contract( off )
    T s = 0;
#pragma unroll
    for ( int d = 0; d < 3; ++d )
    {
        T const tmp = fmax( fmax( plo[d] - hi[d], lo[d] - phi[d] ), T( 0 ) );
        s += tmp * tmp;
    }
    return s;
}

// box_sq of a point: the same operations
template <typename T>
__device__ inline T point_sq( T const *q, T const *b )
{
#pragma clang fp contract( off )
    T s = 0;
#pragma unroll
    for ( int d = 0; d < 3; ++d )
    {
        T const tmp = b[d] - q[d];
        s += tmp * tmp;
    }
    return s;
}

__device__ inline float reciprocal( float v ) { return __builtin_amdgcn_rcpf( v ); }
__device__ inline double reciprocal( double v )
{
    return (double)__builtin_amdgcn_rcpf( (float)v );
}

template <typename T>
struct GroupArgs
{
    QueryArgs<T> a;
    BoxLevels<T> boxes;
    typename Vec4<T>::type const *pts = nullptr; // sources in sorted order
    int32_t const *ids = nullptr;                // sorted position -> source
    T const *scene = nullptr; // the sources' box, six values a problem
    int per_wave = 64; // targets a wave
    int group = 16;    // targets gathered together, at most
    float spacing = 1.f; // source spacing over the k-th distance, k^(-1/3)
    float root_k = 1.f;  // k^(-1/2)
};

// Row slots S of a search for kk results: room for the count to land in
// [kk, S] after one or two tries (a count that must hit a narrow window
// takes more), at least one and a half times kk. (k = 8 takes 32: with 16,
// the counts 7 and 19 around a lattice's node leave every row to the kk-th
// distance itself, 1.80 ms of query against 0.68 at 1M nodes; uniform points
// 0.42 either way.) The nearest source alone needs no row.
constexpr int group_slots( int kk )
{
    return kk <= 1 ? 1 : kk <= 7 ? 16 : ( kk <= 20 ? 32 : ( kk <= 42 ? 64 : 128 ) );
}

template <typename T>
constexpr T type_max()
{
    return sizeof( T ) == 4 ? (T)3.4028234663852886e38 : (T)1.7976931348623157e308;
}

template <typename T, int S>
struct GroupShape
{
    // lanes a row in the sort (k = 1 needs none: any target of the wave can
    // be in one gather)
    static constexpr int kLanes = S == 128 ? 8 : ( S == 1 ? 1 : 4 );
    static constexpr int kKeys = S / kLanes;
    static constexpr int kRows = 64 / kLanes;       // rows a sort
    static constexpr int kChunks = sizeof( T ) == 4 ? 8 : 6;
    static constexpr int kCand = 64 * kChunks;
    static constexpr int kQueue = 224; // nodes of a level
    static constexpr int kPitch = S + 4; // row pitch in words: rows on other banks
    // low bits of a sort key: the row slot; the rest the squared distance
    static constexpr int kSlotBits = S == 128 ? 7 : ( S == 64 ? 6 : ( S == 32 ? 5 : 4 ) );
    static constexpr int kDistBits = 32 - kSlotBits < 26 ? 32 - kSlotBits : 26;
};

// Gathers of a wave that finish no target before its rows are left over:
// kGroupTries where kManyLeft rows of its part of the list are left already
// (the tree search has work then), kMaxTries where not (the hierarchy and the
// longest descent of a few rows take 400 us).
constexpr int kGroupTries = 8, kMaxTries = 96, kManyLeft = 512;
// Targets this many expected k-th distances outside the sources' box are
// left over at once where half of a wave of kFarWave or more are: a few such
// targets are found sooner than the tree is built, and a wave a target finds
// 3000 of them 2 box sides away in a third of the tree search's time.
constexpr float kFar = 4.f;
constexpr int kFarWave = 4;
// counts of a target on the way to a threshold (one or two find it on evenly
// spread points), before its kk-th distance itself is looked for
constexpr int kSteps = 8;

// Radius expected to hold the part `part` of a box's points (sides x, y, z),
// read as an evenly filled volume, or as a surface or curve where those give
// the larger radius.
__device__ inline float even_radius( float x, float y, float z, float part )
{
    float const e0 = fmaxf( fmaxf( x, y ), z ), e2 = fminf( fminf( x, y ), z ),
                e1 = __builtin_amdgcn_fmed3f( x, y, z );
    return fmaxf(
        __builtin_amdgcn_exp2f(
            0.33333334f *
            __builtin_amdgcn_logf( 0.23873f * e0 * e1 * e2 * part ) ),
        fmaxf( 0.95f * __builtin_amdgcn_sqrtf( 0.31831f * e0 * e1 * part ),
               0.45f * e0 * part ) );
}

// Squared radius expected to hold kk sources around q (uniform): from the
// boxes of the 64- and 512-point nodes that hold q (or of the nearest node,
// and then the distance to it too), read as evenly filled (even_radius); the
// smallest of the nodes' radii (a run's box may have corners that the run
// does not fill), and a tenth more. One round of 64 boxes a level: the children of up
// to 8 nodes.
template <typename T>
__device__ inline T first_radius_sq( BoxLevels<T> const &boxes, int64_t beg,
                                     int64_t end, int top, T const *q, int kk,
                                     float root_k, int32_t *queue )
{
    int const lane = opaque_lane();
    int n_in = 64;
    float rad = INFINITY, gap = 0.f;
    for ( int l = top; l >= 1; --l )
    {
        int const sh = 3 * l + 3;
        int const i0 = (int)( beg >> sh ), i1 = (int)( ( end - 1 ) >> sh );
        int const i = l == top ? i0 + lane
                               : queue[lane >> 3] * 8 + ( lane & 7 );
        bool const ok =
            i >= i0 && i <= i1 && ( l == top || lane < 8 * n_in );
        float s = INFINITY, r = INFINITY;
        if ( ok )
        {
            CurveBox<T> const b = boxes.level[l][i];
            s = (float)gap_sq( q, q, b.lo, b.hi );
            r = even_radius( (float)( b.hi[0] - b.lo[0] ),
                             (float)( b.hi[1] - b.lo[1] ),
                             (float)( b.hi[2] - b.lo[2] ),
                             (float)kk *
                                 __builtin_amdgcn_rcpf( (float)(
                                     min( end, (int64_t)( i + 1 ) << sh ) -
                                     max( beg, (int64_t)i << sh ) ) ) );
        }
        uint64_t hits = __ballot( s <= 0.f );
        gap = 0.f;
        if ( hits == 0 )
        {
            uint32_t const key = wave_min_u32(
                ok ? ( __float_as_uint( s ) & ~63u ) | (uint32_t)lane : ~0u );
            hits = 1ull << ( key & 63u );
            gap = lane_value( s, (int)( key & 63u ) );
        }
        int const at = (int)rsort::lanes_below( hits );
        bool const mine = ( ( hits >> lane ) & 1 ) && at < 8;
        if ( l <= 2 )
            rad = fminf( rad, wave_min( mine ? r : INFINITY ) );
        rsort::wave_lds_order();
        if ( mine )
            queue[at] = i;
        rsort::wave_lds_order();
        n_in = min( __popcll( hits ), 8 );
    }
    T const w = (T)( __builtin_amdgcn_sqrtf( gap ) +
                     ( 1.1f + 0.5f * root_k ) * rad );
    return uniform( w * w );
}

template <typename T, int S>
__global__ void __launch_bounds__( 64 )
    __attribute__( ( amdgpu_waves_per_eu( sizeof( T ) == 4 ? 4 : 3 ) ) )
    knn_group_kernel( GroupArgs<T> const g )
{
    using Sh = GroupShape<T, S>;
    using V = typename Vec4<T>::type;
    using SK = SortKey<T>;
    constexpr int W = Sh::kLanes, E = Sh::kKeys, C = Sh::kChunks;
    // the gather's candidates and queues, then (once the candidates are in
    // registers) the rows
    constexpr int kCandBytes = Sh::kCand * (int)( 3 * sizeof( T ) + 4 );
    constexpr int kGatherBytes = kCandBytes + 2 * Sh::kQueue * 4;
    constexpr int kRowBytes = Sh::kRows * Sh::kPitch * 8;
    __shared__ alignas( 16 ) unsigned char
        sm[kGatherBytes > kRowBytes ? kGatherBytes : kRowBytes];
    T *const cx = reinterpret_cast<T *>( sm );
    T *const cy = cx + Sh::kCand;
    T *const cz = cy + Sh::kCand;
    int32_t *const cpos = reinterpret_cast<int32_t *>( cz + Sh::kCand );
    int32_t *const queue = cpos + Sh::kCand;
    uint32_t *const rkey = reinterpret_cast<uint32_t *>( sm );
    int32_t *const rpos =
        reinterpret_cast<int32_t *>( sm ) + Sh::kRows * Sh::kPitch;

    QueryArgs<T> const &a = g.a;
    int const lane = threadIdx.x;
    int64_t const first_row = xcd_tile<0>() * g.per_wave;
    int const n_here =
        (int)min<int64_t>( g.per_wave, a.n_rows - first_row );
    if ( n_here <= 0 )
        return;
    int64_t const my_row = a.row0 + first_row + lane;
    int32_t my_t = 0, my_prob = 0;
    T q[3] = {0, 0, 0};
    if ( lane < n_here )
    {
        my_t = a.order[my_row];
        V const qp = a.tgt[my_t];
        q[0] = qp.x;
        q[1] = qp.y;
        q[2] = qp.z;
        if ( a.src_off )
            my_prob = a.tgt_prob[my_t];
    }

    uint64_t todo = n_here == 64 ? ~0ull : ( 1ull << n_here ) - 1;
    auto leave = [&]( uint64_t which ) {
        // rows that this search does not finish: the tree search's
        if ( ( which >> lane ) & 1 )
            leave_row( a, my_row );
    };
    {
        // Far outside the sources' box a sphere around a target that holds kk
        // sources holds many more a little further on: no radius serves.
        T box[6];
        float part;
        if ( a.src_off )
        {
#pragma unroll
            for ( int d = 0; d < 6; ++d )
                box[d] = g.scene[6 * my_prob + d];
            part = (float)a.kk_prob[my_prob] *
                   __builtin_amdgcn_rcpf( (float)( a.src_off[my_prob + 1] -
                                                   a.src_off[my_prob] ) );
        }
        else
        {
#pragma unroll
            for ( int d = 0; d < 6; ++d )
                box[d] = g.scene[d];
            part = (float)a.kk * __builtin_amdgcn_rcpf( (float)a.n_src );
        }
        float const gap = (float)gap_sq( q, q, box, box + 3 );
        uint64_t out = uniform( (uint64_t)( todo & __ballot( gap > 0.f ) ) );
        if ( out )
        {
            float const r =
                kFar * even_radius( (float)( box[3] - box[0] ),
                                    (float)( box[4] - box[1] ),
                                    (float)( box[5] - box[2] ), part );
            out = uniform( (uint64_t)( out & __ballot( gap > r * r ) ) );
            if ( g.per_wave >= kFarWave && 2 * __popcll( out ) >= g.per_wave )
            {
                leave( out );
                todo &= ~out;
            }
        }
    }
    int group = g.group; // at most kRows: a group's rows are sorted together
    T r2 = T( -1 );    // squared gather radius, negative: not known
    T t_last = T( 0 ); // the last target's threshold
    bool guessed = false; // R is an estimate
    // for a target gathered alone: squared radii that held too few sources
    // and too many
    T r2_few = T( 0 ), r2_full = type_max<T>();
    int last_prob = -1, tries = 0, shrinks = 0;
    int steps = kSteps; // counts of a target: one after a group of ties
    int kk = a.kk;
    // the next group's R^2 over this one's largest: the k-th distances' spread
    // grows as k falls (1M uniform points, k = 10 / 32 / 64: 1.2 + 0.4 k^-1/2
    // 431 / 596 / 1175 us, 1.08 + 0.4 k^-1/2 435 / 589 / 1202, 1 + 0.4 k^-1/2
    // 446 / 599 / 1237)
    float const slack = 1.14f + 0.4f * g.root_k;
    int64_t beg = 0, end = a.n_src;
    // counts grow with the 3/2 power of the squared distance; logarithms of
    // kk and of the count that a first threshold aims at, times 2/3
    constexpr float kPower = 0.6666667f;
    float log_kk = 0.f, to_aim = 1.f, log_aim = 0.f;
    auto set_k = [&]() {
        log_kk = kPower * __builtin_amdgcn_logf( (float)kk );
        log_aim = kPower *
                  __builtin_amdgcn_logf( (float)kk + 0.375f * (float)( S - kk ) );
        to_aim = __builtin_amdgcn_exp2f( log_aim - log_kk );
    };
    set_k();

    // (the search's state is the same in every lane: saying so where it
    // enters a loop keeps its control flow scalar)
    while ( ( todo = uniform( todo ) ) != 0 )
    {
        r2 = uniform( r2 );
        t_last = uniform( t_last );
        group = uniform( group );
        last_prob = uniform( last_prob );
        shrinks = uniform( shrinks );
        steps = uniform( steps );
        guessed = uniform( (int)guessed ) != 0;
        tries = uniform( tries );
        if ( tries > kGroupTries &&
             ( tries > kMaxTries ||
               uniform( __hip_atomic_load(
                   a.left_count + blockIdx.x % kListParts * kListPad,
                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT ) ) > kManyLeft ) )
        {
            leave( todo );
            break;
        }
        int const first = __builtin_ctzll( todo );
        uint64_t sub = todo;
        if ( a.src_off )
        {
            int const pb = __builtin_amdgcn_readlane( my_prob, first );
            sub &= __ballot( my_prob == pb );
            if ( pb != last_prob )
            {
                last_prob = pb;
                beg = uniform( (int)a.src_off[pb] );
                end = uniform( (int)a.src_off[pb + 1] );
                kk = uniform( (int)a.kk_prob[pb] );
                set_k();
                r2 = T( -1 );
                group = g.group;
                t_last = T( 0 );
            }
        }
        beg = (int64_t)uniform( (uint64_t)beg );
        end = (int64_t)uniform( (uint64_t)end );
        kk = uniform( kk );
        int const np = (int)( end - beg );
        bool const all = np <= Sh::kCand / 2;
        T const q0[3] = {lane_value( q[0], first ), lane_value( q[1], first ),
                         lane_value( q[2], first )};
        // the level at which the sources' range spans at most 64 nodes
        int top = 1;
        while ( ( ( end - 1 ) >> ( 3 * top + 3 ) ) - ( beg >> ( 3 * top + 3 ) ) >=
                    64 &&
                top + 1 < g.boxes.n_levels )
            ++top;
        if ( all )
            r2 = type_max<T>();
        else
        {
            if ( r2 < T( 0 ) )
            {
                r2 = first_radius_sq( g.boxes, beg, end, top, q0, kk,
                                      g.root_k, queue );
                guessed = true;
            }
            // the targets near the first: within 2 R and three source
            // spacings (R holds about kk sources)
            T const b[3] = {q[0], q[1], q[2]};
            T const reach = T( 2 ) + T( 4.8 ) * T( g.spacing );
            sub &= __ballot( point_sq( q0, b ) <= r2 * reach * reach );
            sub |= 1ull << first;
        }
        // at most `group` of them
        if ( __popcll( sub ) > group )
            sub = __ballot( ( ( sub >> lane ) & 1 ) &&
                            (int)rsort::lanes_below( sub ) < group );
        sub = uniform( sub );
        bool const in_sub = ( sub >> lane ) & 1;
        T lo[3], hi[3];
#pragma unroll
        for ( int d = 0; d < 3; ++d )
        {
            lo[d] = wave_min( in_sub ? q[d] : T( INFINITY ) );
            hi[d] = wave_max( in_sub ? q[d] : T( -INFINITY ) );
        }

        r2 = uniform( r2 );

        // 1. gather
        int const gl = opaque_lane();
        int n_cand = 0;
        bool full = false;
        if ( all )
        {
            // few sources: every one is a candidate
            for ( int i = gl; i < np; i += 64 )
            {
                V const p = g.pts[beg + i];
                cx[i] = p.x;
                cy[i] = p.y;
                cz[i] = p.z;
                cpos[i] = (int32_t)beg + i;
            }
            n_cand = np;
        }
        else
        {
            // nodes within R, level by level
            int64_t const f0 = beg >> ( 3 * top + 3 );
            int64_t const f1 = ( end - 1 ) >> ( 3 * top + 3 );
            int n_in = 0;
            {
                int64_t const i = f0 + gl;
                bool hit = false;
                if ( i <= f1 )
                {
                    CurveBox<T> const b = g.boxes.level[top][i];
                    hit = gap_sq( lo, hi, b.lo, b.hi ) <= r2;
                }
                uint64_t const m = __ballot( hit );
                if ( hit )
                    queue[rsort::lanes_below( m )] = (int32_t)i;
                n_in = __popcll( m );
            }
            rsort::wave_lds_order();
            int cur = 0;
            for ( int l = top - 1; l >= 0 && !full; --l )
            {
                n_in = uniform( n_in );
                int const c0 = (int)( beg >> ( 3 * l + 3 ) );
                int const c1 = (int)( ( end - 1 ) >> ( 3 * l + 3 ) );
                CurveBox<T> const *const lev = g.boxes.level[l];
                int n_out = 0;
                for ( int j = 0; j < 8 * n_in; j += 64 )
                {
                    int const jj = j + gl;
                    bool hit = false;
                    int child = 0;
                    if ( jj < 8 * n_in )
                    {
                        child = queue[cur + ( jj >> 3 )] * 8 + ( jj & 7 );
                        if ( child >= c0 && child <= c1 )
                        {
                            CurveBox<T> const b = lev[child];
                            hit = gap_sq( lo, hi, b.lo, b.hi ) <= r2;
                        }
                    }
                    uint64_t const m = __ballot( hit );
                    int const nm = __popcll( m );
                    if ( n_out + nm > Sh::kQueue )
                    {
                        full = true;
                        break;
                    }
                    if ( hit )
                        queue[Sh::kQueue - cur + n_out +
                              rsort::lanes_below( m )] = child;
                    n_out += nm;
                }
                rsort::wave_lds_order();
                cur = Sh::kQueue - cur;
                n_in = n_out;
            }
            // the blocks' points within R
            n_in = uniform( n_in );
            for ( int j = 0; j < 8 * n_in && !full; j += 64 )
            {
                int const jj = j + gl;
                bool hit = false;
                T p[3] = {0, 0, 0};
                int32_t pos = 0;
                if ( jj < 8 * n_in )
                {
                    pos = queue[cur + ( jj >> 3 )] * 8 + ( jj & 7 );
                    if ( pos >= beg && pos < end )
                    {
                        V const s = g.pts[pos];
                        p[0] = s.x;
                        p[1] = s.y;
                        p[2] = s.z;
                        hit = gap_sq( lo, hi, p, p ) <= r2;
                    }
                }
                uint64_t const m = __ballot( hit );
                int const nm = __popcll( m );
                if ( n_cand + nm > Sh::kCand )
                {
                    full = true;
                    break;
                }
                if ( hit )
                {
                    int const at = n_cand + (int)rsort::lanes_below( m );
                    cx[at] = p[0];
                    cy[at] = p[1];
                    cz[at] = p[2];
                    cpos[at] = pos;
                }
                n_cand += nm;
            }
        }
        full = uniform( (int)full ) != 0;
        n_cand = uniform( n_cand );
        if ( full )
        {
            // too many: a smaller radius where it is an estimate, fewer
            // targets at once where they need it; for one target, a radius
            // between one that held too few and this one
            int const n_sub = __popcll( sub );
            if ( guessed && ++shrinks <= 3 )
                r2 *= T( 0.6 );
            else if ( n_sub > 1 )
            {
                group = ( n_sub + 1 ) / 2;
                // (targets much sparser than the sources)
                if ( 8 * group <= g.group && __popcll( todo ) > 8 )
                    tries = max( tries, kGroupTries );
            }
            else
            {
                r2_full = r2;
                r2 = T( 0.5 ) * ( r2_few + r2_full );
                if ( !( r2 > r2_few && r2 < r2_full ) )
                {
                    leave( sub );
                    todo &= ~sub;
                    r2 = T( -1 );
                    r2_few = T( 0 );
                    r2_full = type_max<T>();
                }
            }
            ++tries;
            rsort::wave_lds_order();
            continue;
        }
        rsort::wave_lds_order();
        T px[C], py[C], pz[C];
        int32_t pp[C];
        int const chunks = ( n_cand + 63 ) / 64;
#pragma unroll
        for ( int c = 0; c < C; ++c )
        {
            px[c] = py[c] = pz[c] = T( INFINITY );
            pp[c] = 0;
            int const i = c * 64 + gl;
            if ( i < n_cand )
            {
                px[c] = cx[i];
                py[c] = cy[i];
                pz[c] = cz[i];
                pp[c] = cpos[i];
            }
        }
        rsort::wave_lds_order();

        // 2. select. t_max: the largest threshold whose margin ends within R
        constexpr T kMargin =
            sizeof( T ) == 4 ? (T)1.0000019073486328 : (T)( 1.0 + 1e-14 );
        T const t_max = all ? type_max<T>() * T( 0.9999 )
                            : r2 * ( sizeof( T ) == 4 ? (T)0.99999618530273
                                                      : (T)( 1.0 - 2e-14 ) );
        uint64_t done = 0, lost = 0, hard = 0;
        T need = T( 0 ), widest = T( 0 );
        int n_rows = 0;
        int row_lane = first; // the wave's lane of the target of this lane's row
        auto distances = [&]( int i, T ( &d2 )[C] ) {
            T const qt[3] = {lane_value( q[0], i ), lane_value( q[1], i ),
                             lane_value( q[2], i )};
#pragma unroll
            for ( int c = 0; c < C; ++c )
            {
                if ( c >= chunks )
                    break;
                T const b[3] = {px[c], py[c], pz[c]};
                d2[c] = point_sq( qt, b );
            }
        };
        auto count_to = [&]( T const ( &d )[C], T t ) {
            int n = 0;
#pragma unroll
            for ( int c = 0; c < C; ++c )
            {
                if ( c >= chunks )
                    break;
                n += __popcll( __ballot( d[c] <= t ) );
            }
            return n;
        };
        // target i's candidates with d <= t into row n_rows; how many. The
        // sort key is d in steps of t 2^-kDistBits (a reciprocal to one unit:
        // 64 steps of room), then the slot
        auto fill_row = [&]( T const ( &d )[C], T t ) {
            T const scale = t > T( 1e-30 )
                                ? (T)( ( 1u << Sh::kDistBits ) - 64u ) *
                                      reciprocal( t )
                                : T( 0 );
            for ( int s = lane; s < S; s += 64 )
                rkey[n_rows * Sh::kPitch + s] = ~0u;
            rsort::wave_lds_order();
            int at = 0;
#pragma unroll
            for ( int c = 0; c < C; ++c )
            {
                if ( c >= chunks )
                    break;
                bool const in = d[c] <= t;
                uint64_t const m = __ballot( in );
                // (past the row's end: its padding)
                uint32_t const slot =
                    min( __builtin_amdgcn_mbcnt_hi(
                             (uint32_t)( m >> 32 ),
                             __builtin_amdgcn_mbcnt_lo( (uint32_t)m, at ) ),
                         (uint32_t)( Sh::kPitch - 1 ) );
                if ( in )
                {
                    rkey[n_rows * Sh::kPitch + slot] =
                        ( (uint32_t)( d[c] * scale ) << Sh::kSlotBits ) | slot;
                    rpos[n_rows * Sh::kPitch + slot] = pp[c];
                }
                at += __popcll( m );
            }
            return at;
        };
        // target i's row is filled, its kk-th squared distance about w
        auto keep_row = [&]( int i, T w ) {
            done |= 1ull << i;
            row_lane = lane / W == n_rows ? i : row_lane;
            widest = widest > w ? widest : w;
            // the next target's first threshold aims at the window's middle
            t_last = uniform( w * (T)to_aim );
            ++n_rows;
        };
        // R^2 of the next gather where this one held too few and no candidate
        // says how far the rest is
        auto wider = [&]() {
            if ( __popcll( sub ) > 1 )
                return r2 * T( 2.25 );
            r2_few = r2;
            return r2_full < type_max<T>() ? T( 0.5 ) * ( r2_few + r2_full )
                                           : r2 * T( 2.25 );
        };
        // The nearest source of each target: the least squared distance, and
        // among those that the rounded root may tie the lowest index. Without
        // rows a gather serves all 64 targets of a wave: 1M x 1M uniform points
        // 357 -> 274 us, 3000 sources and 400,000 targets 109 -> 69.
        if constexpr ( S == 1 )
        {
            int32_t my_pos = 0;
            for ( uint64_t left = sub; left; left &= left - 1 )
            {
                left = uniform( left );
                int const i = __builtin_ctzll( left );
                T d2[C];
                distances( i, d2 );
                T m = T( INFINITY );
#pragma unroll
                for ( int c = 0; c < C; ++c )
                {
                    if ( c >= chunks )
                        break;
                    m = fmin( m, d2[c] );
                }
                m = uniform( wave_min( m ) );
                if ( uniform( (int)!( m <= t_max ) ) )
                {
                    T const u = m < type_max<T>() ? m : wider();
                    need = need > u ? need : u;
                    lost |= 1ull << i;
                    continue;
                }
                T const limit = m * kMargin;
                int n = 0;
                int32_t v = -1;
#pragma unroll
                for ( int c = 0; c < C; ++c )
                {
                    if ( c >= chunks )
                        break;
                    bool const in = d2[c] <= limit;
                    v = in ? pp[c] : v;
                    n += __popcll( __ballot( in ) );
                }
                uint64_t who = __ballot( v >= 0 );
                if ( uniform( n ) > 1 )
                {
                    T const root = sqrt_rn( m );
                    int32_t id = INT32_MAX;
#pragma unroll
                    for ( int c = 0; c < C; ++c )
                    {
                        if ( c >= chunks )
                            break;
                        if ( d2[c] <= limit && sqrt_rn( d2[c] ) == root )
                        {
                            int32_t const o = g.ids[pp[c]];
                            v = o < id ? pp[c] : v;
                            id = o < id ? o : id;
                        }
                    }
                    who = __ballot( id == wave_min_int( id ) );
                }
                int32_t const pos = __builtin_amdgcn_readlane(
                    v, __builtin_ctzll( uniform( who ) ) );
                my_pos = lane == i ? pos : my_pos;
                done |= 1ull << i;
                widest = widest > m ? widest : m;
            }
            if ( ( done >> lane ) & 1 )
            {
                int64_t const at = a.row_off ? a.row_off[my_row]
                                             : ( a.src_pos ? my_row : (int64_t)my_t );
                a.out_idx[at] = a.src_pos ? my_pos : g.ids[my_pos];
                if ( a.out_dist )
                {
                    V const p = g.pts[my_pos];
                    T const b[3] = {p.x, p.y, p.z};
                    a.out_dist[at] = (double)sqrt_rn( point_sq( q, b ) );
                }
            }
        }
        // The k nearest.
        if constexpr ( S > 1 )
        for ( uint64_t left = sub; left; left &= left - 1 )
        {
            left = uniform( left );
            n_rows = uniform( n_rows );
            int const i = __builtin_ctzll( left );
            T d2[C];
            distances( i, d2 );
            // a threshold with kk to S candidates at or below it
            T below = T( -1 ), above = type_max<T>();
            T limit = t_max;
            T t = t_last > T( 0 ) ? t_last : ( all ? T( 1 ) : t_max );
            t = uniform( t < t_max ? t : t_max );
            bool found = false, beyond = false;
            int n = 0;
            for ( int it = 0; it < steps; ++it )
            {
                t = uniform( t );
                n = uniform( count_to( d2, t ) );
                if ( n >= kk && n <= S )
                {
                    found = true;
                    break;
                }
                if ( n < kk )
                {
                    if ( uniform( (int)( t >= limit ) ) )
                    {
                        // more needed than R holds: how much more, among
                        // the candidates at hand
                        if ( beyond || n_cand < kk )
                            break;
                        beyond = true;
                        limit = type_max<T>();
                        it -= 2 * kSteps;
                    }
                    below = t;
                }
                else
                    above = t;
                float const f = __builtin_amdgcn_exp2f(
                    log_aim - kPower * __builtin_amdgcn_logf( (float)n + 0.5f ) );
                T u = t * (T)f;
                if ( !( u > below && u < above ) )
                    u = above < type_max<T>()
                            ? T( 0.5 ) * ( below > T( 0 ) ? below : T( 0 ) ) +
                                  T( 0.5 ) * above
                            : ( below > T( 0 ) ? below * T( 2 ) : T( 1 ) );
                u = u < limit ? u : limit;
                u = uniform( u );
                if ( uniform( (int)!( u > below && u < above ) ) )
                    break;
                t = u;
            }
            if ( uniform( (int)( found && !beyond ) ) )
            {
                // squared distances whose root may round as the kk-th's
                // stay in
                n = uniform( n );
                if ( uniform( fill_row( d2, t * kMargin ) ) <= S )
                    keep_row( i, t * (T)__builtin_amdgcn_exp2f(
                                         log_kk - kPower * __builtin_amdgcn_logf(
                                                               (float)n ) ) );
                else
                    hard |= 1ull << i;
                continue;
            }
            above = uniform( above );
            if ( uniform( (int)!( found || beyond ||
                                  above < type_max<T>() ) ) )
                // no step came above: does R hold enough?
                beyond = uniform( count_to( d2, t_max ) ) < kk;
            if ( uniform( (int)!beyond ) )
            {
                hard |= 1ull << i;
                continue;
            }
            T u = found ? t : above;
            if ( !( u < type_max<T>() ) )
                u = wider();
            need = need > u ? need : u;
            lost |= 1ull << i;
        }
        // Targets that R serves but no threshold does (distances tied on a
        // lattice or among copies of a point: the counts jump over the
        // window): the kk-th distance itself, from the rounded roots and
        // without margins, and at it the lowest indices.
        for ( uint64_t left = S > 1 ? hard : 0; left; left &= left - 1 )
        {
            left = uniform( left );
            n_rows = uniform( n_rows );
            int const i = __builtin_ctzll( left );
            T const qt[3] = {lane_value( q[0], i ), lane_value( q[1], i ),
                             lane_value( q[2], i )};
            // (past the candidates: infinite)
            T r[C];
#pragma unroll
            for ( int c = 0; c < C; ++c )
            {
                T const b[3] = {px[c], py[c], pz[c]};
                r[c] = sqrt_rn( point_sq( qt, b ) );
                // (one root at a time: their temporaries are many)
                __builtin_amdgcn_sched_barrier( 0 );
            }
            auto count_roots = [&]( T t ) {
                int m = 0;
#pragma unroll
                for ( int c = 0; c < C; ++c )
                    m += __popcll( __ballot( r[c] <= t ) );
                return m;
            };
            // a root with kk to S candidates at or below it, or the kk-th
            // itself: lo < root <= hi, narrowed between the candidates' own
            // values, so that each count rules one out
            T lo = T( -1 ), hi = uniform( sqrt_rn( t_max ) ), root = hi;
            int n = 0;
            bool tied = false;
            while ( !tied )
            {
                lo = uniform( lo );
                hi = uniform( hi );
                T v_min = T( INFINITY ), v_max = T( -1 );
#pragma unroll
                for ( int c = 0; c < C; ++c )
                {
                    bool const in = r[c] > lo && r[c] <= hi;
                    v_min = fmin( v_min, in ? r[c] : T( INFINITY ) );
                    v_max = fmax( v_max, in ? r[c] : T( -1 ) );
                }
                v_min = uniform( wave_min( v_min ) );
                v_max = uniform( wave_max( v_max ) );
                tied = uniform( (int)!( v_min < v_max ) ) != 0;
                T m = v_max > T( 4 ) * v_min ? sqrt_rn( v_min * v_max )
                                             : v_min + T( 0.5 ) * ( v_max - v_min );
                m = tied ? v_max : ( m > v_min && m < v_max ? m : v_min );
                root = m = uniform( m );
                n = uniform( count_roots( m ) );
                if ( n < kk )
                    lo = m;
                else if ( n <= S )
                    break;
                else
                    hi = m;
            }
            if ( n > S )
            {
                // more at the kk-th distance than fit: of the lowest indices
                // (they are distinct: some cut leaves just kk)
                auto id = [&]( int c ) {
                    return r[c] == root ? g.ids[pp[c]] : INT32_MAX;
                };
                auto count_ids = [&]( int cut ) {
                    int m = 0;
#pragma unroll
                    for ( int c = 0; c < C; ++c )
                        m += __popcll( __ballot( r[c] < root || id( c ) <= cut ) );
                    return m;
                };
                int lo_id = INT32_MAX, hi_id = INT32_MAX;
#pragma unroll
                for ( int c = 0; c < C; ++c )
                {
                    int const v = id( c );
                    lo_id = min( lo_id, v );
                    hi_id = min( hi_id, v < INT32_MAX ? ~v : INT32_MAX );
                }
                lo_id = uniform( wave_min_int( lo_id ) ) - 1;
                hi_id = ~uniform( wave_min_int( hi_id ) );
                while ( hi_id - lo_id > 1 )
                {
                    int const m = lo_id + ( hi_id - lo_id ) / 2;
                    n = uniform( count_ids( m ) );
                    if ( n < kk )
                        lo_id = uniform( m );
                    else
                        hi_id = uniform( m );
                    if ( n >= kk && n <= S )
                        break;
                }
#pragma unroll
                for ( int c = 0; c < C; ++c )
                    if ( r[c] == root && id( c ) > hi_id )
                        r[c] = T( INFINITY );
            }
            fill_row( r, root );
            keep_row( i, root * root );
        }

        // 3. sort
        if ( S > 1 && n_rows )
        {
            rsort::wave_lds_order();
            int const ol = opaque_lane();
            int const row = ol / W, sl = ol % W;
            bool const valid = row < n_rows;
            uint32_t key[E];
#pragma unroll
            for ( int e = 0; e < E; ++e )
                key[e] = valid ? rkey[row * Sh::kPitch + sl * E + e] : ~0u;
            int64_t const r = a.row0 + first_row + row_lane;
            int32_t const rt = __shfl( my_t, row_lane, 64 );
            int64_t const base = a.row_off ? a.row_off[r]
                                           : ( a.src_pos ? r : (int64_t)rt ) *
                                                 (int64_t)kk;
            int32_t *const out = a.out_idx + base + sl * E;
            // results of this lane's keys
            int mine = ( valid ? kk : 0 ) - sl * E;
            sort_rows<W, E>( key, sl );
            // neighbours of a row within the root's rounding (or the key's
            // step), the one past the last result included
            constexpr uint32_t kNear =
                ( sizeof( T ) == 4 ? ( ( 1u << ( Sh::kDistBits - 22 ) ) + 8u )
                                   : 3u )
                << Sh::kSlotBits;
            bool close = false;
            uint32_t const after = (uint32_t)__builtin_amdgcn_mov_dpp(
                (int)key[0], 0x101, 0xf, 0xf, true ); // the next lane's
#pragma unroll
            for ( int e = 0; e < E; ++e )
            {
                uint32_t const nx = e + 1 < E ? key[e + 1] : after;
                bool const pair = e < mine && ( e + 1 < E || sl + 1 < W );
                close |= pair && nx - key[e] < kNear;
            }
            // (every lane of a row learns of its row's)
            uint64_t const closes = __ballot( close );
            uint64_t const row_bits = ( ( 1ull << W ) - 1 ) << ( row * W );
            if ( closes & row_bits )
                mine = 0;
            int32_t pos[E];
#pragma unroll
            for ( int e = 0; e < E; ++e )
            {
                pos[e] = rpos[row * Sh::kPitch + ( key[e] & ( S - 1 ) )];
                if ( e >= mine )
                    pos[e] = (int32_t)beg;
            }
            if ( a.out_dist )
            {
                V const tq = a.tgt[rt];
                T const qq[3] = {tq.x, tq.y, tq.z};
#pragma unroll
                for ( int e = 0; e < E; ++e )
                {
                    V const p = g.pts[pos[e]];
                    T const b[3] = {p.x, p.y, p.z};
                    T const d = sqrt_rn( point_sq( qq, b ) );
                    if ( e < mine )
                        a.out_dist[base + sl * E + e] = (double)d;
                    if ( e % 4 == 3 )
                        __builtin_amdgcn_sched_barrier( 0 );
                }
            }
            if ( !a.src_pos )
            {
#pragma unroll
                for ( int e = 0; e < E; ++e )
                    pos[e] = g.ids[pos[e]];
            }
#pragma unroll
            for ( int e = 0; e < E; ++e )
                if ( e < mine )
                    out[e] = pos[e];

            // the close rows by the full (distance, index) keys: a few in a
            // thousand rows of scattered points, one row at a time over the
            // wave; every row of a lattice, all rows together where their
            // keys fit the registers
            bool together = false;
            if constexpr ( S <= 32 )
            {
                together = __popcll( closes ) > 4;
                if ( together )
                {
                    V const tq = a.tgt[rt];
                    T const qq[3] = {tq.x, tq.y, tq.z};
                    typename SK::type fk[E];
#pragma unroll
                    for ( int e = 0; e < E; ++e )
                    {
                        int const at = row * Sh::kPitch + sl * E + e;
                        fk[e] = SK::none();
                        if ( valid && rkey[at] != ~0u )
                        {
                            int32_t const ps = rpos[at];
                            V const p = g.pts[ps];
                            T const b[3] = {p.x, p.y, p.z};
                            fk[e] = SK::make( sqrt_rn( point_sq( qq, b ) ),
                                              g.ids[ps] );
                        }
                    }
                    sort_rows<W, E>( fk, sl );
#pragma unroll
                    for ( int e = 0; e < E; ++e )
                        if ( valid && sl * E + e < kk )
                        {
                            int32_t const id = SK::index( fk[e] );
                            out[e] = a.src_pos ? a.src_pos[id] : id;
                            if ( a.out_dist )
                                a.out_dist[base + sl * E + e] =
                                    SK::distance( fk[e] );
                        }
                    // (tied counts do not follow the power law that estimated
                    // the kk-th distances: the next group's R from the rows)
                    T w = T( 0 );
#pragma unroll
                    for ( int e = 0; e < E; ++e )
                        if ( valid && sl * E + e == kk - 1 )
                            w = (T)SK::distance( fk[e] );
                    w = uniform( wave_max( w ) );
                    widest = widest > w * w ? widest : w * w;
                }
            }
            for ( uint64_t left = together ? 0 : closes; left; )
            {
                int const fl = __builtin_ctzll( left );
                int const cr = fl / W;
                left &= ~( ( ( 1ull << W ) - 1 ) << ( cr * W ) );
                int const ti = __builtin_amdgcn_readlane( row_lane, fl );
                T const qt[3] = {lane_value( q[0], ti ), lane_value( q[1], ti ),
                                 lane_value( q[2], ti )};
                constexpr int kPer = S > 64 ? S / 64 : 1;
                typename SK::type fk[kPer];
#pragma unroll
                for ( int e = 0; e < kPer; ++e )
                {
                    int const at = cr * Sh::kPitch + ol * kPer + e;
                    fk[e] = SK::none();
                    if ( ol * kPer + e < S && rkey[at] != ~0u )
                    {
                        int32_t const ps = rpos[at];
                        V const p = g.pts[ps];
                        T const b[3] = {p.x, p.y, p.z};
                        fk[e] =
                            SK::make( sqrt_rn( point_sq( qt, b ) ), g.ids[ps] );
                    }
                }
                sort_wave<kPer, ( S < 64 ? S : 64 )>( fk, ol );
                int64_t const cr_row = a.row0 + first_row + ti;
                int64_t const cr_base =
                    a.row_off
                        ? a.row_off[cr_row]
                        : ( a.src_pos ? cr_row
                                      : (int64_t)__builtin_amdgcn_readlane(
                                            my_t, ti ) ) *
                              (int64_t)kk;
#pragma unroll
                for ( int e = 0; e < kPer; ++e )
                {
                    int const j = ol * kPer + e;
                    if ( j < kk )
                    {
                        int32_t const id = SK::index( fk[e] );
                        a.out_idx[cr_base + j] = a.src_pos ? a.src_pos[id] : id;
                        if ( a.out_dist )
                            a.out_dist[cr_base + j] = SK::distance( fk[e] );
                    }
                }
            }
        }
        todo &= ~done;
        tries += done ? 0 : 1;
        if ( done )
        {
            steps = hard ? 1 : kSteps;
            r2_few = T( 0 );
            r2_full = type_max<T>();
            shrinks = 0;
        }
        if ( lost )
        {
            // the first lost targets again, with what they asked for
            guessed = false;
            r2 = uniform( need * T( 1.0001 ) );
            if ( !( r2 < type_max<T>() ) )
            {
                leave( lost );
                todo &= ~lost;
                r2 = T( -1 );
            }
        }
        else if ( !all )
        {
            guessed = true;
            // (so small a gather gains nothing from a smaller R: 1M points on a line,
            // k = 1 355 -> 285 us)
            T const next = widest * T( slack );
            r2 = uniform( n_cand <= 32 && r2 > next ? r2 : next );
            if ( 5 * n_cand < 2 * Sh::kCand )
                group = min( 2 * group, g.group );
            if ( !( r2 > T( 0 ) ) )
                r2 = T( -1 );
        }
        rsort::wave_lds_order();
    }
}

} // namespace
} // namespace dtkx

#endif
