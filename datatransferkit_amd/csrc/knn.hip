// k-nearest-neighbour search for gfx950.
//
// Build: scene box -> 63-bit Hilbert codes (21 bits per axis) with every
// radix pass's digit counts -> the hand-written radix sort of (code, index)
// (radix_sort.hpp; the targets' 48-bit codes sort in the same launches, and
// the last pass writes both inverse permutations and the points in sorted
// order) -> the boxes of 8, 64, 512, ... consecutive sources.
// Query: groups of targets that are consecutive on the curve (knn_group.hpp).
// The exact k smallest (distance, index) pairs of each target, as brute force
// gives. 1M x 1M uniform points, build and query: k = 32 0.84 ms, k = 10
// 0.69 ms, k = 1 0.54 ms (one tree traversal a lane over the hierarchy below
// took 2.11, 1.00 and 0.64).
//
// The rows that the groups leave (targets far outside the sources' box or in
// the middle of a hollow cloud, where a sphere that holds k sources holds
// hundreds a little further on), and searches with fewer than 64 sources,
// go to a tree search: a Karras hierarchy over the sorted codes (duplicate
// codes split by index), in which each internal node also writes both child
// boxes: exact for small children, the curve cell of the child's common
// prefix, cut to the boxes of the runs that hold its points, for large ones.
// One lane per target; a per-lane stack in LDS, its deeper entries in global
// memory; for small k the best candidates stay sorted in registers as 64-bit
// keys (float distance bits << 32 | index), so the ordering is (distance,
// index) with one integer compare, for larger k a second traversal collects
// them. Pruning uses squared distances against a threshold slightly above
// the square of the current k-th distance, which never drops a candidate
// that could tie or beat it. 1M x 1M, k = 10, build and query: targets 2 box
// sides away 1.52 ms (9.4 by groups alone), in a box 3 times as wide 1.59
// (8.9).
#include "knn.hpp"
#include "radix_sort.hpp"


#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstring>
#include <vector>

namespace dtkx
{
namespace
{

template <typename T>
struct Vec4;
template <>
struct Vec4<float>
{
    using type = float4;
};
template <>
struct Vec4<double>
{
    using type = double4;
};

// Child code c >= 0: internal node c; c < 0: leaf holding source index ~c.
template <typename T>
struct alignas( 16 ) Node
{
    T lo[2][3];
    T hi[2][3];
    int32_t child[2];
};

// A node's box; entry 3 of each corner is unused (two 16-byte loads).
template <typename T>
struct alignas( 16 ) CurveBox
{
    T lo[4];
    T hi[4];
};

// Boxes of the sorted sources: node i of level l covers the sources
// [i 8^(l+1), (i + 1) 8^(l+1)).
constexpr int kMaxBoxLevels = 10;
template <typename T>
struct BoxLevels
{
    CurveBox<T> *level[kMaxBoxLevels] = {};
    int n_levels = 0;
};

constexpr int kBlock = 256;

// ------------------------------------------------------------- scene box
// Also clears zero[0, n_zero): counters that later kernels of the same
// build accumulate into.
template <typename T, typename V>
__global__ void __launch_bounds__( kBlock )
    bbox_partial( V const *pts, int64_t n, T *partial, uint4 *zero,
                  int64_t n_zero )
{
    for ( int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < n_zero;
          i += (int64_t)gridDim.x * kBlock )
        zero[i] = make_uint4( 0u, 0u, 0u, 0u );
    T lo[3] = {INFINITY, INFINITY, INFINITY};
    T hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for ( int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < n;
          i += (int64_t)gridDim.x * kBlock )
    {
        V p = pts[i];
        lo[0] = fmin( lo[0], p.x );
        lo[1] = fmin( lo[1], p.y );
        lo[2] = fmin( lo[2], p.z );
        hi[0] = fmax( hi[0], p.x );
        hi[1] = fmax( hi[1], p.y );
        hi[2] = fmax( hi[2], p.z );
    }
    __shared__ T sh[6][kBlock];
    for ( int d = 0; d < 3; ++d )
    {
        sh[d][threadIdx.x] = lo[d];
        sh[3 + d][threadIdx.x] = hi[d];
    }
    __syncthreads();
    for ( int off = kBlock / 2; off > 0; off >>= 1 )
    {
        if ( threadIdx.x < off )
            for ( int d = 0; d < 3; ++d )
            {
                sh[d][threadIdx.x] =
                    fmin( sh[d][threadIdx.x], sh[d][threadIdx.x + off] );
                sh[3 + d][threadIdx.x] = fmax(
                    sh[3 + d][threadIdx.x], sh[3 + d][threadIdx.x + off] );
            }
        __syncthreads();
    }
    if ( threadIdx.x == 0 )
        for ( int d = 0; d < 6; ++d )
            partial[blockIdx.x * 6 + d] = sh[d][0];
}

template <typename T>
__global__ void __launch_bounds__( kBlock )
    bbox_final( T const *partial, int nparts, T *box )
{
    __shared__ T sh[6][kBlock];
    T v[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    for ( int i = threadIdx.x; i < nparts; i += kBlock )
        for ( int d = 0; d < 3; ++d )
        {
            v[d] = fmin( v[d], partial[i * 6 + d] );
            v[3 + d] = fmax( v[3 + d], partial[i * 6 + 3 + d] );
        }
    for ( int d = 0; d < 6; ++d )
        sh[d][threadIdx.x] = v[d];
    __syncthreads();
    for ( int off = kBlock / 2; off > 0; off >>= 1 )
    {
        if ( threadIdx.x < off )
            for ( int d = 0; d < 3; ++d )
            {
                sh[d][threadIdx.x] =
                    fmin( sh[d][threadIdx.x], sh[d][threadIdx.x + off] );
                sh[3 + d][threadIdx.x] = fmax(
                    sh[3 + d][threadIdx.x], sh[3 + d][threadIdx.x + off] );
            }
        __syncthreads();
    }
    if ( threadIdx.x == 0 )
        for ( int d = 0; d < 6; ++d )
            box[d] = sh[d][0];
}

// ----------------------------------------------------------- curve codes
// Bits 0..20 of v spread to every third bit.
__device__ inline uint64_t expand21( uint32_t v )
{
    uint64_t x = v & 0x1fffffu;
    x = ( x | x << 32 ) & 0x1f00000000ffffull;
    x = ( x | x << 16 ) & 0x1f0000ff0000ffull;
    x = ( x | x << 8 ) & 0x100f00f00f00f00full;
    x = ( x | x << 4 ) & 0x10c30c30c30c30c3ull;
    x = ( x | x << 2 ) & 0x1249249249249249ull;
    return x;
}

// The largest extent of a scene box (box[0..2] = lower corner, box[3..5] =
// upper corner).
template <typename T>
__device__ inline double scene_extent( T const *box )
{
    double e = 0;
    for ( int d = 0; d < 3; ++d )
        e = fmax( e, (double)box[3 + d] - (double)box[d] );
    return e;
}

// The 2^21 grid of a scene box, of cubic cells over its largest extent: cell
// = (p - lo) scale. One division a box, not a point. (With the grid stretched
// over each extent, 64 consecutive points of a box of 1 x 0.01 x 0.0001 lay
// within 0.04 x 0.0004 x 4e-6: k = 32 for 1M points took 41 ms with the group
// search and 11.5 with a tree search a lane.)
struct CurveFrame
{
    double lo[3], scale;
};
template <typename T>
__device__ inline CurveFrame curve_frame( T const *box )
{
    double const ext = scene_extent( box );
    return {{(double)box[0], (double)box[1], (double)box[2]},
            ext > 0 ? 2097151.0 / ext : 0.0};
}

// Cell of p on the grid of f.
template <typename V>
__device__ inline void curve_cell( V p, CurveFrame const &f, uint32_t *q )
{
    double const c[3] = {(double)p.x, (double)p.y, (double)p.z};
    for ( int d = 0; d < 3; ++d )
    {
        double u = ( c[d] - f.lo[d] ) * f.scale;
        u = u < 0 ? 0 : ( u > 2097151.0 ? 2097151.0 : u );
        q[d] = (uint32_t)u;
    }
}

// Place on the Hilbert curve of the cell q of a 2^BITS grid (3 BITS bits),
// by Skilling's transform (AIP Conf. Proc. 707, 2004): from the top bit
// down, an axis' bit inverts or exchanges the lower bits of the first axis;
// then a Gray decode across the axes. The code of q >> s is the code of q
// without its last 3 s bits, so a prefix of 3 L bits names an octree cell,
// one further bit a half and two a quarter of one. Consecutive cells share
// a face: a run of consecutive points, unlike one in Morton order, never
// jumps, and its box stays small (the sources within the k-th distance of
// 16 consecutive targets number 223 against 360, the 8-point blocks they
// lie in 55 against 102: uniform points, k = 32).
template <int BITS>
__device__ inline uint64_t hilbert_code( uint32_t const *q )
{
    uint32_t x = q[0], y = q[1], z = q[2];
#pragma unroll
    for ( int b = BITS - 1; b >= 1; --b )
    {
        uint32_t const Q = 1u << b, P = Q - 1u;
        x ^= x & Q ? P : 0u;
        uint32_t const ty = ( x ^ y ) & P;
        uint32_t const iy = y & Q ? P : ty;
        y ^= y & Q ? 0u : ty;
        x ^= iy;
        uint32_t const tz = ( x ^ z ) & P;
        uint32_t const iz = z & Q ? P : tz;
        z ^= z & Q ? 0u : tz;
        x ^= iz;
    }
    y ^= x;
    z ^= y;
    uint32_t t = z >> 1;
    t ^= t >> 1;
    t ^= t >> 2;
    t ^= t >> 4;
    t ^= t >> 8;
    t ^= t >> 16;
    return ( expand21( x ^ t ) << 2 ) | ( expand21( y ^ t ) << 1 ) |
           expand21( z ^ t );
}

// Radix passes of the two key kinds: the sources' 63-bit codes and the
// targets' top 48 bits (a cell of 1.5e-5 of the scene: a group of targets
// must be close together in terms of the sources around it. With 30 bits,
// cells of 1e-3, the targets inside a cluster of that size were in no order,
// and half of the rows of 1M points in 200 such clusters were left over. 39
// bits, one pass less: 1M x 1M nearest 471 -> 465 us, but in clusters of 1e-4
// k = 10 took 1.69 ms instead of 1.15).
constexpr int kSrcKeyBits = 63, kTgtLevels = 16, kTgtKeyBits = 3 * kTgtLevels;
constexpr int kSrcPasses = ( kSrcKeyBits + 7 ) / 8;
constexpr int kTgtPasses = ( kTgtKeyBits + 7 ) / 8;
constexpr int kHistWords = ( kSrcPasses + kTgtPasses ) * rsort::kDigits;

// Key of a target (kTgtKeyBits bits). Outside the grid: by the side or corner
// of the grid that it lies beyond, then the code of its mirror image inside (a
// coarser one), so that consecutive targets are close in all three directions.
// Inside: after all those (a wave of a few scattered targets is done while the
// others run; as the last one it made the query of 1M uniform targets 20 us
// longer), the top bits of its code. (Clamped to the
// grid, targets 2 to 3 box sides away followed each other at random depths, in
// the order in which the curve visits the face: tree search of 1M x 1M such
// points, k = 10, 1.06 ms.)
template <typename V>
__device__ inline uint64_t target_key( V p, CurveFrame const &f )
{
    constexpr double kMax = 2097151.0;
    double const c[3] = {(double)p.x, (double)p.y, (double)p.z};
    uint32_t q[3];
    uint32_t image = 0;
    for ( int d = 0; d < 3; ++d )
    {
        double u = ( c[d] - f.lo[d] ) * f.scale;
        uint32_t const side = u < 0 ? 1u : ( u > kMax ? 2u : 0u );
        image = image * 3u + side;
        if ( side )
        {
            double const x = fabs( u ) * ( 1.0 / kMax );
            double const y = x - 2.0 * floor( 0.5 * x ); // [0, 2)
            u = kMax * ( y > 1.0 ? 2.0 - y : y );
            u = u >= 0 && u <= kMax ? u : 0.0; // (not finite)
        }
        q[d] = (uint32_t)u;
    }
    constexpr int kOuter = kTgtLevels - 2; // 1 + 5 bits name the image
    int const cut = image ? 21 - kOuter : 21 - kTgtLevels;
    uint32_t const top[3] = {q[0] >> cut, q[1] >> cut, q[2] >> cut};
    uint64_t const code = hilbert_code<kTgtLevels>( top );
    return image ? ( (uint64_t)image << ( 3 * kOuter ) ) | code
                 : ( 1ull << ( kTgtKeyBits - 1 ) ) | code >> 1;
}

// Hilbert codes of the sources (63-bit) and keys of the targets in one launch, one sort tile of points a block (blocks [0, src_blocks) take
// the sources), with the digit counts of every radix pass added into hist
// (sources' passes first, zero on entry). src_prob / tgt_prob (nullable, a batch):
// each point's problem, whose scene box is box + 6 problem.
template <typename T, typename V>
__global__ void __launch_bounds__( rsort::kThreads )
    curve_hist_kernel( V const *src, int64_t n_src, V const *tgt,
                        int64_t n_tgt, T const *box, int32_t const *src_prob,
                        int32_t const *tgt_prob, int src_blocks,
                        uint64_t *scodes, uint64_t *tcodes, uint32_t *hist )
{
    __shared__ uint32_t h[kSrcPasses * rsort::kDigits];
    bool const is_src = static_cast<int>( blockIdx.x ) < src_blocks;
    int const words = ( is_src ? kSrcPasses : kTgtPasses ) * rsort::kDigits;
    for ( int i = threadIdx.x; i < words; i += rsort::kThreads )
        h[i] = 0;
    __syncthreads();
    int64_t const c0 =
        (int64_t)( is_src ? blockIdx.x : blockIdx.x - src_blocks ) *
        rsort::kTile;
    int64_t const n = is_src ? n_src : n_tgt;
    V const *pts = is_src ? src : tgt;
    int32_t const *prob = is_src ? src_prob : tgt_prob;
    CurveFrame frame = curve_frame( box );
    for ( int s = 0; s < rsort::kItems; ++s )
    {
        int64_t const i = c0 + s * rsort::kThreads + threadIdx.x;
        if ( i >= n )
            break;
        if ( prob )
            frame = curve_frame( box + 6 * prob[i] );
        if ( is_src )
        {
            uint32_t q[3];
            curve_cell( pts[i], frame, q );
            uint64_t const code = hilbert_code<21>( q );
            scodes[i] = code;
#pragma unroll
            for ( int p = 0; p < kSrcPasses; ++p )
                atomicAdd( &h[p * rsort::kDigits + ( ( code >> ( 8 * p ) ) & 255 )],
                           1u );
        }
        else
        {
            uint64_t const c = target_key( pts[i], frame );
            tcodes[i] = c;
#pragma unroll
            for ( int p = 0; p < kTgtPasses; ++p )
                atomicAdd( &h[p * rsort::kDigits + ( ( c >> ( 8 * p ) ) & 255 )],
                           1u );
        }
    }
    __syncthreads();
    uint32_t *g = hist + ( is_src ? 0 : kSrcPasses * rsort::kDigits );
    for ( int i = threadIdx.x; i < words; i += rsort::kThreads )
    {
        uint32_t const v = h[i];
        if ( v )
            atomicAdd( g + i, v );
    }
}

} // namespace
} // namespace dtkx

#include "knn_small.hpp"

namespace dtkx
{
namespace
{

// The rows that a search leaves to the tree search are listed in eight parts,
// by the XCD that leaves them, their counts kListPad apart: an atomic on one
// counter takes some 10 ns, which 31,000 waves that each leave rows wait for
// one after the other.
constexpr int kListParts = 8, kListPad = 32;
__device__ inline int left_total( int32_t const *count )
{
    int n = 0;
#pragma unroll
    for ( int p = 0; p < kListParts; ++p )
        n += count[p * kListPad];
    return n;
}

// ------------------------------------------------------ Karras hierarchy
// delta(i, j): common prefix length of keys i and j, with the index used
// to break ties between equal codes; -1 outside [0, n).
__device__ inline int prefix_delta( uint64_t const *codes, int64_t n,
                                    int64_t i, int64_t j )
{
    if ( j < 0 || j >= n )
        return -1;
    uint64_t a = codes[i], b = codes[j];
    if ( a != b )
        return __clzll( a ^ b );
    return 64 + __clz( (uint32_t)i ^ (uint32_t)j );
}

__device__ inline float round_down( double v ) { return __double2float_rd( v ); }
__device__ inline float round_up( double v ) { return __double2float_ru( v ); }

// Conservative box of the points between two points of the curve order
// whose cells are qb and qe (qm: a point between them) and whose codes share
// the first `delta` bits (bit 63 is always 0): the octree cell of the
// prefix's whole digits, cut to the two octants that it then holds when the
// prefix ends two bits into a digit (those of qb and qe), and to their half
// of the cell when it ends one bit in and the three points show two of the
// half's axes. (The curve enters and leaves a half through octants that
// differ in one axis only, so its middle names the other.) Mapped back to
// world coordinates with a margin and outward rounding, so it contains the
// points whatever the rounding of the forward quantisation (curve_cell).
template <typename T>
__device__ inline void cell_box( uint32_t const *qb, uint32_t const *qm,
                                 uint32_t const *qe, int delta, T const *scene,
                                 T *lo, T *hi )
{
    int const nb = delta >= 64 ? 63 : ( delta - 1 ); // known bits below 63
    int const digits = nb > 0 ? nb / 3 : 0, part = nb > 0 ? nb % 3 : 0;
    int const sh = 21 - digits;
    uint32_t diff[3];
    int n_diff = 0;
    for ( int d = 0; d < 3; ++d )
    {
        uint32_t const x = ( qb[d] ^ qe[d] ) | ( qb[d] ^ qm[d] );
        diff[d] = part ? ( x >> ( sh - 1 ) ) & 1u : 1u;
        n_diff += (int)diff[d];
    }
    bool const cut = part == 2 || ( part == 1 && n_diff == 2 );
    double const ext = scene_extent( scene );
    double const h = ext / 2097151.0;
    double const margin = 1e-9 * ext + 1e-300;
    for ( int d = 0; d < 3; ++d )
    {
        int const s = cut && !diff[d] ? sh - 1 : sh;
        uint32_t const qmin = ( qb[d] >> s ) << s;
        double const s0 = scene[d];
        double l = s0 + qmin * h - margin;
        double u = s0 + ( (double)qmin + (double)( 1u << s ) ) * h + margin;
        if ( sizeof( T ) == 4 )
        {
            lo[d] = (T)round_down( l );
            hi[d] = (T)round_up( u );
        }
        else
        {
            lo[d] = (T)l;
            hi[d] = (T)u;
        }
    }
}

// Children of internal node i: ranges, codes, parents and child boxes.
// A child that is a leaf gets its point as a degenerate box and the code
// ~source_index; an internal child covering at most kTight points gets its
// exact box, a larger one the curve cell of its common prefix, cut to the
// boxes of the group search where there are any (without them 1M x 1M searches
// of targets 20 box sides away took 2.1 ms at k = 10, with them 1.4).
#ifndef DTKX_KNN_TIGHT
#define DTKX_KNN_TIGHT 16
#endif
constexpr int kTight = DTKX_KNN_TIGHT;

// Problem owning internal node i of a batch: the largest p with
// src_off[p] - p <= i (problem p's internal nodes are
// [src_off[p] - p, src_off[p + 1] - p - 1), empty for one source).
__device__ inline int node_problem( int32_t const *src_off, int n_prob,
                                    int64_t i )
{
    int lo = 0, hi = n_prob - 1;
    while ( lo < hi )
    {
        int const mid = ( lo + hi + 1 ) >> 1;
        if ( src_off[mid] - mid <= i )
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

// One problem (src_off null): n points, internal nodes [0, n - 1).
// left_count (nullable): nothing is built if all parts are empty (no row left to the
// hierarchy). Batch: n_int internal nodes in all; node i belongs to problem p, whose
// sorted points are [src_off[p], src_off[p + 1]) with scene box scene + 6 p;
// the hierarchy of each problem is built over its own range (child node
// indices and leaf codes are global).
template <typename T, typename V>
__global__ void __launch_bounds__( kBlock )
    karras_kernel( uint64_t const *codes_all, int32_t const *sorted_all,
                   V const *pts, V const *sorted_pts_all, int64_t n_int,
                   T const *scenes, BoxLevels<T> const boxes,
                   int32_t const *src_off, int n_prob, Node<T> *nodes, int32_t *sizes, int32_t const *left_count )
{
    if ( left_count && left_total( left_count ) == 0 )
        return;
    int64_t const gi = blockIdx.x * (int64_t)kBlock + threadIdx.x;
    if ( gi >= n_int )
        return;
    int64_t so = 0, io = 0, n = n_int + 1;
    T const *scene = scenes;
    if ( src_off )
    {
        int const pb = node_problem( src_off, n_prob, gi );
        so = src_off[pb];
        n = src_off[pb + 1] - so;
        io = so - pb;
        scene = scenes + 6 * pb;
    }
    uint64_t const *codes = codes_all + so;
    int32_t const *sorted_ids = sorted_all + so;
    // the points in sorted order: a copy when given, else through the ids
    V const *sorted_pts = sorted_pts_all ? sorted_pts_all + so : nullptr;
    auto point = [&]( int64_t q ) {
        return sorted_pts ? sorted_pts[q] : pts[sorted_ids[q]];
    };
    int64_t const i = gi - io;
    int d = ( prefix_delta( codes, n, i, i + 1 ) -
              prefix_delta( codes, n, i, i - 1 ) ) >= 0
                ? 1
                : -1;
    int dmin = prefix_delta( codes, n, i, i - d );
    int64_t lmax = 2;
    while ( prefix_delta( codes, n, i, i + lmax * d ) > dmin )
        lmax <<= 1;
    int64_t l = 0;
    for ( int64_t t = lmax >> 1; t >= 1; t >>= 1 )
        if ( prefix_delta( codes, n, i, i + ( l + t ) * d ) > dmin )
            l += t;
    int64_t j = i + l * d;
    int dnode = prefix_delta( codes, n, i, j );
    int64_t s = 0, t = l;
    do
    {
        t = ( t + 1 ) >> 1;
        if ( prefix_delta( codes, n, i, i + ( s + t ) * d ) > dnode )
            s += t;
    } while ( t > 1 );
    int64_t const gamma = i + s * d + ( d < 0 ? -1 : 0 );
    int64_t const first = i < j ? i : j, last = i < j ? j : i;
    sizes[gi] = (int32_t)( last - first + 1 );
    int64_t const rb[2] = {first, gamma + 1};
    int64_t const re[2] = {gamma, last};
    Node<T> nd;
    for ( int c = 0; c < 2; ++c )
    {
        int64_t const b = rb[c], e = re[c];
        if ( b == e )
        {
            int32_t const orig = sorted_ids[b];
            V const p = point( b );
            nd.lo[c][0] = nd.hi[c][0] = p.x;
            nd.lo[c][1] = nd.hi[c][1] = p.y;
            nd.lo[c][2] = nd.hi[c][2] = p.z;
            nd.child[c] = ~orig;
            continue;
        }
        int64_t const child = io + ( c == 0 ? gamma : gamma + 1 );
        nd.child[c] = (int32_t)child;
        if ( e - b + 1 <= kTight )
        {
            T lo[3] = {INFINITY, INFINITY, INFINITY};
            T hi[3] = {-INFINITY, -INFINITY, -INFINITY};
            for ( int64_t q = b; q <= e; ++q )
            {
                V const p = point( q );
                lo[0] = fmin( lo[0], p.x );
                lo[1] = fmin( lo[1], p.y );
                lo[2] = fmin( lo[2], p.z );
                hi[0] = fmax( hi[0], p.x );
                hi[1] = fmax( hi[1], p.y );
                hi[2] = fmax( hi[2], p.z );
            }
            for ( int q = 0; q < 3; ++q )
            {
                nd.lo[c][q] = lo[q];
                nd.hi[c][q] = hi[q];
            }
        }
        else
        {
            CurveFrame const frame = curve_frame( scene );
            uint32_t qb[3], qm[3], qe[3];
            curve_cell( point( b ), frame, qb );
            curve_cell( point( ( b + e ) / 2 ), frame, qm );
            curve_cell( point( e ), frame, qe );
            cell_box<T>( qb, qm, qe, prefix_delta( codes, n, b, e ), scene,
                         nd.lo[c], nd.hi[c] );
            if ( boxes.n_levels > 0 )
            {
                // and the boxes of the (at most 12) runs that hold the points
                int l = 0;
                while ( ( ( so + e ) >> ( 3 * l + 3 ) ) -
                                ( ( so + b ) >> ( 3 * l + 3 ) ) >=
                            12 &&
                        l + 1 < boxes.n_levels )
                    ++l;
                T lo[3] = {INFINITY, INFINITY, INFINITY};
                T hi[3] = {-INFINITY, -INFINITY, -INFINITY};
                for ( int64_t q = ( so + b ) >> ( 3 * l + 3 );
                      q <= ( so + e ) >> ( 3 * l + 3 ); ++q )
                {
                    CurveBox<T> const r = boxes.level[l][q];
                    for ( int x = 0; x < 3; ++x )
                    {
                        lo[x] = fmin( lo[x], r.lo[x] );
                        hi[x] = fmax( hi[x], r.hi[x] );
                    }
                }
                for ( int x = 0; x < 3; ++x )
                {
                    nd.lo[c][x] = fmax( nd.lo[c][x], lo[x] );
                    nd.hi[c][x] = fmin( nd.hi[c][x], hi[x] );
                }
            }
        }
    }
    nodes[gi] = nd;
}

// --------------------------------------------------------- k-best lists
template <int K>
struct KBestF
{
    uint64_t key[K];
    __device__ void init()
    {
#pragma unroll
        for ( int j = 0; j < K; ++j )
            key[j] = ~0ull;
    }
    // squared-distance threshold above which nothing can enter
    // every slot a candidate at distance w with an index above any source
    // (kept out of the results as long as kk sources lie within w)
    __device__ void seed( float w )
    {
        uint64_t const v = ( (uint64_t)__float_as_uint( w ) << 32 ) | 0xffffffffu;
#pragma unroll
        for ( int j = 0; j < K; ++j )
            key[j] = v;
    }
    __device__ float threshold() const
    {
        if ( key[K - 1] == ~0ull )
            return INFINITY;
        float w = __uint_as_float( (uint32_t)( key[K - 1] >> 32 ) );
        return w * w * 1.00000095367431640625f; // (1 + 2^-20)
    }
    __device__ void insert( float d, int32_t id )
    {
        uint64_t c = ( (uint64_t)__float_as_uint( d ) << 32 ) | (uint32_t)id;
        if ( c < key[K - 1] )
        {
#pragma unroll
            for ( int j = K - 1; j > 0; --j )
            {
                uint64_t prev = key[j - 1], cur = key[j];
                key[j] = c < prev ? prev : ( c < cur ? c : cur );
            }
            key[0] = c < key[0] ? c : key[0];
        }
    }
    __device__ int32_t index( int j ) const
    {
        return (int32_t)( key[j] & 0xffffffffu );
    }
    __device__ double distance( int j ) const
    {
        return (double)__uint_as_float( (uint32_t)( key[j] >> 32 ) );
    }
};

template <int K>
struct KBestD
{
    double dk[K];
    int32_t ik[K];
    __device__ void init()
    {
#pragma unroll
        for ( int j = 0; j < K; ++j )
        {
            dk[j] = INFINITY;
            ik[j] = INT32_MAX;
        }
    }
    __device__ void seed( double w )
    {
#pragma unroll
        for ( int j = 0; j < K; ++j )
        {
            dk[j] = w;
            ik[j] = INT32_MAX;
        }
    }
    __device__ double threshold() const
    {
        if ( ik[K - 1] == INT32_MAX && dk[K - 1] == INFINITY )
            return INFINITY;
        double w = dk[K - 1];
        return w * w * 1.0000000000000009; // (1 + 2^-50)
    }
    __device__ static bool less( double a, int32_t ia, double b, int32_t ib )
    {
        return a < b || ( a == b && ia < ib );
    }
    __device__ void insert( double d, int32_t id )
    {
        if ( less( d, id, dk[K - 1], ik[K - 1] ) )
        {
#pragma unroll
            for ( int j = K - 1; j > 0; --j )
            {
                bool lp = less( d, id, dk[j - 1], ik[j - 1] );
                bool lc = less( d, id, dk[j], ik[j] );
                double nd = lp ? dk[j - 1] : ( lc ? d : dk[j] );
                int32_t ni = lp ? ik[j - 1] : ( lc ? id : ik[j] );
                dk[j] = nd;
                ik[j] = ni;
            }
            if ( less( d, id, dk[0], ik[0] ) )
            {
                dk[0] = d;
                ik[0] = id;
            }
        }
    }
    __device__ int32_t index( int j ) const { return ik[j]; }
    __device__ double distance( int j ) const { return dk[j]; }
};

template <typename T, int K>
struct KBest;
template <int K>
struct KBest<float, K>
{
    using type = KBestF<K>;
};
template <int K>
struct KBest<double, K>
{
    using type = KBestD<K>;
};

// q clamped to [lo, hi] (lo <= hi): one median-of-three for float, a max
// and a min for double, the values of q < lo ? lo : (q > hi ? hi : q) (a
// signed-zero difference between the forms squares to the same zero).
__device__ inline float clamp_to( float q, float lo, float hi )
{
    return __builtin_amdgcn_fmed3f( q, lo, hi );
}
__device__ inline double clamp_to( double q, double lo, double hi )
{
    return fmin( fmax( q, lo ), hi );
}

// Squared distance from q to its projection onto [lo, hi]: the operation
// sequence of the point distance (tmp = b - a; s += tmp * tmp), so for a
// degenerate box it is that distance exactly and otherwise a lower bound.
template <typename T>
__device__ inline T box_sq( T const *q, T const *lo, T const *hi )
{
#pragma clang fp contract( off )
    T s = 0;
#pragma unroll
    for ( int d = 0; d < 3; ++d )
    {
        T tmp = clamp_to( q[d], lo[d], hi[d] ) - q[d];
        s += tmp * tmp;
    }
    return s;
}

// Squared distance from q to the farthest corner of [lo, hi], in
// box_sq's operations: per axis the larger of the two rounded differences
// q - lo and hi - q. Rounding is monotonic, so for every point p of the
// box the rounded |p - q| is at most that axis term, and the sum bounds
// box_sq(q, p, p) from above.
template <typename T>
__device__ inline T far_sq( T const *q, T const *lo, T const *hi )
{
#pragma clang fp contract( off )
    T s = 0;
#pragma unroll
    for ( int d = 0; d < 3; ++d )
    {
        T const tmp = fmax( q[d] - lo[d], hi[d] - q[d] );
        s += tmp * tmp;
    }
    return s;
}

// Seed of a search for kk neighbours below internal node `root` (whose
// subtree holds at least kk sources): follow the query's nearer child down
// to the deepest node still holding kk sources and return far_sq of its
// box, an upper bound of the kk-th squared distance as the traversal
// computes it. sizes: sources under each internal node.
template <typename T>
__device__ inline T seed_far_sq( Node<T> const *nodes, int32_t const *sizes,
                                 int32_t root, T const *q, int kk )
{
    Node<T> nd = nodes[root];
    T lo[3], hi[3];
#pragma unroll
    for ( int d = 0; d < 3; ++d )
    {
        lo[d] = fmin( nd.lo[0][d], nd.lo[1][d] );
        hi[d] = fmax( nd.hi[0][d], nd.hi[1][d] );
    }
    while ( true )
    {
        int const c =
            box_sq( q, nd.lo[1], nd.hi[1] ) < box_sq( q, nd.lo[0], nd.hi[0] ) ? 1
                                                                              : 0;
        int32_t const ch = nd.child[c];
        if ( ch < 0 || sizes[ch] < kk )
            break;
#pragma unroll
        for ( int d = 0; d < 3; ++d )
        {
            lo[d] = nd.lo[c][d];
            hi[d] = nd.hi[c][d];
        }
        nd = nodes[ch];
    }
    return far_sq( q, lo, hi );
}

// Correctly rounded square roots: llvm.sqrt without fast-math flags (the
// library is built with -fhip-fp32-correctly-rounded-divide-sqrt). HIP's
// __fsqrt_rn maps to the native 1-ulp instruction and must not be used.
__device__ inline float sqrt_rn( float s ) { return __builtin_sqrtf( s ); }
__device__ inline double sqrt_rn( double s ) { return __builtin_sqrt( s ); }

constexpr int kQueryBlock = 64;

// Seed the k-th distance from the deepest node on the query's path holding
// k sources.
#ifndef DTKX_KNN_SEED
#define DTKX_KNN_SEED 1
#endif
constexpr bool kSeed = DTKX_KNN_SEED != 0;

// A lane's traversal stack holds its first kLdsStack entries in LDS (14 waves
// per CU). With the seeded k-th distance (seed_far_sq) a descent pushes only
// far children inside the seed's bound, so shallow stacks almost always
// suffice. Deeper entries go to global memory where rows come from a list;
// a launch over all rows lists the rare row that needs them.
// Every level of the hierarchy lengthens the common prefix of the node's
// keys (63 curve bits, then 32 index bits for equal codes), so no path
// from the root has more than 96 internal levels.
#ifndef DTKX_KNN_LDS_STACK
#define DTKX_KNN_LDS_STACK 22
#endif
constexpr int kLdsStack = DTKX_KNN_LDS_STACK;
constexpr int kMaxDepth = 97;
// stack entries of the fixed-radius pass of a two-pass search when its row
// is collected in the LDS stack's other slots (its radius is final, so it
// descends far less deep than the first pass)
constexpr int kPass2Stack = 12;
// global stack entries a lane
constexpr int kSpill = kMaxDepth - kPass2Stack;
// the largest K whose two-pass rows are sorted by their own lane
constexpr int kFusedSortK = 32;
// The smallest K searched in two passes (below). 1M uniform sources and
// targets, one pass against two: float coordinates 1.54 / 1.75 ms at k = 24,
// 2.21 / 2.12 at k = 32; double coordinates, whose (distance, index)
// comparisons cost three operations, 4.2 / 3.2 at k = 16, 11.9 / 5.1 at 32.
template <typename T>
constexpr int two_pass_k()
{
    return sizeof( T ) == 4 ? 32 : 16;
}

// Arguments of a query launch. One problem: rows [row0, row0 + n_rows) of
// the Hilbert-ordered targets against n_src sources, kk results per row.
// Batch (src_off set): target t belongs to problem tgt_prob[t], whose
// sources are [src_off[p], src_off[p + 1]), whose hierarchy is rooted at
// internal node src_off[p] - p and whose rows hold kk_prob[p] results at
// CSR offset row_off[r].
template <typename T>
struct QueryArgs
{
    Node<T> const *nodes = nullptr;
    // nullable: points under each internal node (seeds the k-th distance)
    int32_t const *node_size = nullptr;
    typename Vec4<T>::type const *src = nullptr, *tgt = nullptr;
    int32_t const *order = nullptr; // row -> target
    int64_t row0 = 0, n_rows = 0;
    int64_t n_src = 0;
    int kk = 0;
    int32_t const *src_off = nullptr, *tgt_prob = nullptr,
                  *kk_prob = nullptr;
    int64_t const *row_off = nullptr;
    int32_t *out_idx = nullptr;
    double *out_dist = nullptr;
    // curve layout: row r written at row r with indices as positions
    int32_t const *src_pos = nullptr;
    // rows left over: part p's are left_rows[p left_cap + i] for i <
    // left_count[p kListPad]
    int32_t *left_rows = nullptr, *left_count = nullptr;
    int64_t left_cap = 0;
    // launch over those rows: the tiles taken of each part (as left_count,
    // zero before), the nodes of kSpill deeper stack entries per lane laid
    // out [level][lane] (stride gstride)
    int32_t *taken = nullptr;
    // nullable: the list's length is added here (one lane)
    int32_t *n_rows_total = nullptr;
    int32_t *gstack = nullptr;
    int64_t gstride = 0;
};

template <typename T>
__device__ inline void leave_row( QueryArgs<T> const &a, int64_t r )
{
    int const p = blockIdx.x % kListParts;
    a.left_rows[p * a.left_cap + atomicAdd( a.left_count + p * kListPad, 1 )] =
        (int32_t)r;
}

// One row of a one-pass search: row r, st_node and st_d the block's LDS
// stack, spill the lane's slot in global memory. LIST: deeper entries go
// there (nodes only: they are tested again when taken); else a row that needs
// them is listed. Whether the row is written.
template <typename T, int K, bool LIST>
__device__ inline bool query_row( QueryArgs<T> const &a, int64_t const spill,
                                 int64_t const r, int32_t *st_node, T *st_d )
{
    int32_t const t = a.order[r];
    int64_t so = 0, np = a.n_src;
    int32_t root = 0;
    int kk = a.kk;
    if ( a.src_off )
    {
        int const pb = a.tgt_prob[t];
        so = a.src_off[pb];
        np = a.src_off[pb + 1] - so;
        root = (int32_t)( so - pb );
        kk = a.kk_prob[pb];
    }
    typename Vec4<T>::type qp = a.tgt[t];
    T const q[3] = {qp.x, qp.y, qp.z};
    typename KBest<T, K>::type best;
    best.init();
    if ( a.node_size && np > 1 )
        best.seed(
            sqrt_rn( seed_far_sq( a.nodes, a.node_size, root, q, kk ) ) );
    T thr = best.threshold();

    if ( np == 1 )
    {
        // single source: the tree has no internal node
        typename Vec4<T>::type sp0 = a.src[so];
        T const b[3] = {sp0.x, sp0.y, sp0.z};
        best.insert( sqrt_rn( box_sq( q, b, b ) ), (int32_t)so );
    }
    else
    {
        int sp = 0;
        int32_t node = root;
        while ( node >= 0 )
        {
            Node<T> const nd = a.nodes[node];
            T s0 = box_sq( q, nd.lo[0], nd.hi[0] );
            T s1 = box_sq( q, nd.lo[1], nd.hi[1] );
            int32_t c0 = nd.child[0], c1 = nd.child[1];
            if ( c0 < 0 && s0 <= thr )
            {
                best.insert( sqrt_rn( s0 ), ~c0 );
                thr = best.threshold();
            }
            if ( c1 < 0 && s1 <= thr )
            {
                best.insert( sqrt_rn( s1 ), ~c1 );
                thr = best.threshold();
            }
            bool g0 = c0 >= 0 && s0 <= thr;
            bool g1 = c1 >= 0 && s1 <= thr;
            int32_t next = -1;
            if ( g0 && g1 )
            {
                bool near0 = s0 <= s1;
                int32_t far = near0 ? c1 : c0;
                T fs = near0 ? s1 : s0;
                next = near0 ? c0 : c1;
                if ( sp < kLdsStack )
                {
                    st_node[sp * kQueryBlock + threadIdx.x] = far;
                    st_d[sp * kQueryBlock + threadIdx.x] = fs;
                }
                else if ( LIST )
                    a.gstack[( sp - kLdsStack ) * a.gstride + spill] = far;
                else
                {
                    leave_row( a, r );
                    return false;
                }
                ++sp;
            }
            else if ( g0 )
                next = c0;
            else if ( g1 )
                next = c1;
            else
            {
                while ( sp > 0 )
                {
                    --sp;
                    if ( LIST && sp >= kLdsStack )
                    {
                        next = a.gstack[( sp - kLdsStack ) * a.gstride + spill];
                        break;
                    }
                    if ( st_d[sp * kQueryBlock + threadIdx.x] <= thr )
                    {
                        next = st_node[sp * kQueryBlock + threadIdx.x];
                        break;
                    }
                }
            }
            node = next;
        }
    }
    // compile-time indices keep the k-best list in registers (a loop bounded
    // by the runtime kk would index it dynamically and move it to scratch)
    int64_t const base =
        a.row_off ? a.row_off[r] : ( a.src_pos ? r : (int64_t)t ) * kk;
#pragma unroll
    for ( int j = 0; j < K; ++j )
        if ( j < kk )
        {
            int32_t const id = best.index( j );
            a.out_idx[base + j] = a.src_pos ? a.src_pos[id] : id;
            if ( a.out_dist )
                a.out_dist[base + j] = best.distance( j );
        }
    return true;
}

// ------------------------------------------------- two-pass k-best search
// For larger k the sorted (distance, index) list costs five operations per
// slot for every candidate, and a wave runs it whenever any of its lanes
// meets one. Two traversals do the same work with fewer operations:
// pass 1 keeps only the k smallest SQUARED distances, a sorted register
// array updated with one median-of-three per slot; its last entry s_k gives
// the k-th distance d_k = sqrt(s_k) (a correctly rounded square root is
// monotone, so it maps order statistics to order statistics). Exactly the
// pass-1 entries whose root is below d_k are sources at distance < d_k, say
// c_lt of them. Pass 2 is a fixed-radius traversal that writes those c_lt
// sources and the k - c_lt smallest indices among the sources at distance
// == d_k to the row; the row is then sorted by (distance, index) in
// registers. The result is the set and order the sorted list gives.
template <typename T>
__device__ inline T med3( T a, T b, T c );
template <>
__device__ inline float med3( float a, float b, float c )
{
    return __builtin_amdgcn_fmed3f( a, b, c );
}
template <>
__device__ inline double med3( double a, double b, double c )
{
    return fmin( c, fmax( a, b ) ); // a <= c
}

// The k smallest squared distances, ascending. Slots below K - kk hold -1,
// so the last slot is the kk-th smallest for any kk <= K.
template <typename T, int K>
struct KthList
{
    T d[K];
    __device__ void init( int kk )
    {
#pragma unroll
        for ( int j = 0; j < K; ++j )
            d[j] = j < K - kk ? T( -1 ) : T( INFINITY );
    }
    // new d[j] = clamp(s, d[j - 1], d[j]): the j-th of the sorted union
    __device__ void insert( T s )
    {
#pragma unroll
        for ( int j = K - 1; j > 0; --j )
            d[j] = med3( d[j - 1], s, d[j] );
        d[0] = fmin( d[0], s );
    }
    __device__ T last() const { return d[K - 1]; }
    // kk entries of value b (padding stays -1): b acts as kk candidates
    // at squared distance b, so the list ends at the true kk-th value
    // whenever at least kk sources lie at or below b
    __device__ void seed( int kk, T b )
    {
#pragma unroll
        for ( int j = 0; j < K; ++j )
            if ( j >= K - kk )
                d[j] = b;
    }
};

// A squared-distance bound above every s whose rounded root is <= w.
__device__ inline float root_bound( float w )
{
    return w * w * 1.00000095367431640625f; // (1 + 2^-20)
}
__device__ inline double root_bound( double w )
{
    return w * w * 1.0000000000000009; // (1 + 2^-50)
}

// (distance, index) keys
template <typename T>
struct SortKey;
template <>
struct SortKey<float>
{
    using type = uint64_t;
    __device__ static type make( float d, int32_t id )
    {
        return ( (uint64_t)__float_as_uint( d ) << 32 ) | (uint32_t)id;
    }
    __device__ static type none() { return ~0ull; }
    __device__ static bool less( type a, type b ) { return a < b; }
    __device__ static int32_t index( type a ) { return (int32_t)( a & 0xffffffffu ); }
    __device__ static double distance( type a )
    {
        return (double)__uint_as_float( (uint32_t)( a >> 32 ) );
    }
};
struct DKey
{
    double d;
    int32_t id;
};
template <>
struct SortKey<double>
{
    using type = DKey;
    __device__ static type make( double d, int32_t id ) { return {d, id}; }
    __device__ static type none() { return {INFINITY, INT32_MAX}; }
    __device__ static bool less( type a, type b )
    {
        return a.d < b.d || ( a.d == b.d && a.id < b.id );
    }
    __device__ static int32_t index( type a ) { return a.id; }
    __device__ static double distance( type a ) { return a.d; }
};

constexpr int pow2_at_least( int k )
{
    int n = 1;
    while ( n < k )
        n <<= 1;
    return n;
}

// ascending bitonic sorting network, all indices compile-time constants
template <typename T, int N>
__device__ inline void bitonic_sort( typename SortKey<T>::type ( &a )[N] )
{
    using SK = SortKey<T>;
#pragma unroll
    for ( int k = 2; k <= N; k <<= 1 )
#pragma unroll
        for ( int j = k >> 1; j > 0; j >>= 1 )
#pragma unroll
            for ( int i = 0; i < N; ++i )
            {
                int const l = i ^ j;
                if ( l > i )
                {
                    bool const up = ( i & k ) == 0;
                    auto const x = a[i], y = a[l];
                    bool const swap = up ? SK::less( y, x ) : SK::less( x, y );
                    a[i] = swap ? y : x;
                    a[l] = swap ? x : y;
                }
            }
}

// One row of a two-pass search (query_row's arguments). Rows of K >
// kFusedSortK are written unordered, as source indices.
template <typename T, int K, bool LIST>
__device__ inline bool query2_row( QueryArgs<T> const &a, int64_t const spill,
                                  int64_t const r, int32_t *st_node, T *st_d )
{
    using SK = SortKey<T>;
    int32_t const t = a.order[r];
    int64_t so = 0, np = a.n_src;
    int32_t root = 0;
    int kk = a.kk;
    if ( a.src_off )
    {
        int const pb = a.tgt_prob[t];
        so = a.src_off[pb];
        np = a.src_off[pb + 1] - so;
        root = (int32_t)( so - pb );
        kk = a.kk_prob[pb];
    }
    typename Vec4<T>::type qp = a.tgt[t];
    T const q[3] = {qp.x, qp.y, qp.z};
    int64_t const base =
        a.row_off ? a.row_off[r] : ( a.src_pos ? r : (int64_t)t ) * kk;
    int32_t *row = a.out_idx + base;

    // pass 1: the kk-th smallest squared distance
    KthList<T, K> list;
    list.init( kk );
    if ( a.node_size && np > 1 )
        // pruning starts at the seed, so the descent pushes no far child
        // beyond it
        list.seed( kk, root_bound( sqrt_rn(
                           seed_far_sq( a.nodes, a.node_size, root, q, kk ) ) ) );
    if ( np == 1 )
    {
        typename Vec4<T>::type sp0 = a.src[so];
        T const b[3] = {sp0.x, sp0.y, sp0.z};
        list.insert( box_sq( q, b, b ) );
    }
    else
    {
        T thr = list.last();
        int sp = 0;
        int32_t node = root;
        while ( node >= 0 )
        {
            Node<T> const nd = a.nodes[node];
            T const s0 = box_sq( q, nd.lo[0], nd.hi[0] );
            T const s1 = box_sq( q, nd.lo[1], nd.hi[1] );
            int32_t const c0 = nd.child[0], c1 = nd.child[1];
            // an entry equal to the bound leaves the list's values unchanged
            if ( c0 < 0 && s0 < thr )
            {
                list.insert( s0 );
                thr = list.last();
            }
            if ( c1 < 0 && s1 < thr )
            {
                list.insert( s1 );
                thr = list.last();
            }
            bool const g0 = c0 >= 0 && s0 < thr;
            bool const g1 = c1 >= 0 && s1 < thr;
            int32_t next = -1;
            if ( g0 && g1 )
            {
                bool const near0 = s0 <= s1;
                int32_t const far = near0 ? c1 : c0;
                T const fs = near0 ? s1 : s0;
                next = near0 ? c0 : c1;
                if ( sp < kLdsStack )
                {
                    st_node[sp * kQueryBlock + threadIdx.x] = far;
                    st_d[sp * kQueryBlock + threadIdx.x] = fs;
                }
                else if ( LIST )
                    a.gstack[( sp - kLdsStack ) * a.gstride + spill] = far;
                else
                {
                    leave_row( a, r );
                    return false;
                }
                ++sp;
            }
            else if ( g0 )
                next = c0;
            else if ( g1 )
                next = c1;
            else
            {
                while ( sp > 0 )
                {
                    --sp;
                    if ( LIST && sp >= kLdsStack )
                    {
                        next = a.gstack[( sp - kLdsStack ) * a.gstride + spill];
                        break;
                    }
                    if ( st_d[sp * kQueryBlock + threadIdx.x] < thr )
                    {
                        next = st_node[sp * kQueryBlock + threadIdx.x];
                        break;
                    }
                }
            }
            node = next;
        }
    }

    // pass 2: the sources at distance < d_k, and the smallest indices among
    // those at distance == d_k, written to the row unordered
    T const dk = sqrt_rn( list.last() );
    int c_lt = 0;
#pragma unroll
    for ( int j = 0; j < K; ++j )
        c_lt += ( list.d[j] >= 0 && sqrt_rn( list.d[j] ) < dk ) ? 1 : 0;
    T const s_hi = root_bound( dk );
    // The row is collected in LDS when it fits beside pass 2's stack (whose
    // pass-1 distances are dead): the stack keeps the first kPass2Stack node
    // slots, the row takes the distance slots (as ints) and the node slots
    // above. Scattered 4-byte stores to the row in global memory, spread
    // over the traversal, would leave partly written lines for the L2 to
    // evict (8 times the row's bytes, measured).
    constexpr int kDistSlots = kLdsStack * (int)( sizeof( T ) / 4 );
    constexpr bool kRowLds = K <= kFusedSortK &&
                             K <= kDistSlots + kLdsStack - kPass2Stack;
    constexpr int kStack2 = kRowLds ? kPass2Stack : kLdsStack;
    int32_t *const ids_d = reinterpret_cast<int32_t *>( st_d );
    auto slot = [&]( int j ) -> int32_t & {
        if constexpr ( kRowLds )
        {
            if ( j < kDistSlots )
                return ids_d[j * kQueryBlock + threadIdx.x];
            return st_node[( kPass2Stack + j - kDistSlots ) * kQueryBlock +
                           threadIdx.x];
        }
        else
            return row[j];
    };
    int n_lt = 0, n_eq = 0;
    auto take = [&]( T s, int32_t id ) {
        T const d = sqrt_rn( s );
        if ( d < dk )
        {
            if ( n_lt < c_lt )
                slot( n_lt++ ) = id;
        }
        else if ( d == dk )
        {
            if ( c_lt + n_eq < kk )
                slot( c_lt + n_eq++ ) = id;
            else
            {
                // all tie slots taken: replace the largest index if larger
                int jm = c_lt;
                for ( int j = c_lt + 1; j < kk; ++j )
                    jm = slot( j ) > slot( jm ) ? j : jm;
                if ( id < slot( jm ) )
                    slot( jm ) = id;
            }
        }
    };
    if ( np == 1 )
    {
        typename Vec4<T>::type sp0 = a.src[so];
        T const b[3] = {sp0.x, sp0.y, sp0.z};
        take( box_sq( q, b, b ), (int32_t)so );
    }
    else
    {
        int sp = 0;
        int32_t node = root;
        while ( node >= 0 )
        {
            Node<T> const nd = a.nodes[node];
            T const s0 = box_sq( q, nd.lo[0], nd.hi[0] );
            T const s1 = box_sq( q, nd.lo[1], nd.hi[1] );
            int32_t const c0 = nd.child[0], c1 = nd.child[1];
            if ( c0 < 0 && s0 <= s_hi )
                take( s0, ~c0 );
            if ( c1 < 0 && s1 <= s_hi )
                take( s1, ~c1 );
            bool const g0 = c0 >= 0 && s0 <= s_hi;
            bool const g1 = c1 >= 0 && s1 <= s_hi;
            int32_t next = -1;
            if ( g0 && g1 )
            {
                next = c0;
                if ( sp < kStack2 )
                    st_node[sp * kQueryBlock + threadIdx.x] = c1;
                else if ( LIST )
                    a.gstack[( sp - kStack2 ) * a.gstride + spill] = c1;
                else
                {
                    leave_row( a, r );
                    return false;
                }
                ++sp;
            }
            else if ( g0 )
                next = c0;
            else if ( g1 )
                next = c1;
            else if ( sp > 0 )
            {
                --sp;
                next = sp < kStack2
                           ? st_node[sp * kQueryBlock + threadIdx.x]
                           : a.gstack[( sp - kStack2 ) * a.gstride + spill];
            }
            node = next;
        }
    }
    if constexpr ( K <= kFusedSortK )
    {
        constexpr int N = pow2_at_least( K );
        typename SK::type key[N];
#pragma unroll
        for ( int j = 0; j < N; ++j )
        {
            key[j] = SK::none();
            if ( j < kk )
            {
                int32_t const id = slot( j );
                typename Vec4<T>::type const p = a.src[id];
                T const b[3] = {p.x, p.y, p.z};
                key[j] = SK::make( sqrt_rn( box_sq( q, b, b ) ), id );
            }
        }
        bitonic_sort<T, N>( key );
#pragma unroll
        for ( int j = 0; j < K; ++j )
            if ( j < kk )
            {
                int32_t const id = SK::index( key[j] );
                row[j] = a.src_pos ? a.src_pos[id] : id;
                if ( a.out_dist )
                    a.out_dist[base + j] = SK::distance( key[j] );
            }
    }
    return true;
}

// a < b and (c ? a : b) field by field, without short-circuit branches
__device__ inline bool key_less( DKey const &a, DKey const &b )
{
    return ( a.d < b.d ) | ( ( a.d == b.d ) & ( a.id < b.id ) );
}
__device__ inline uint64_t key_pick( bool c, uint64_t a, uint64_t b )
{
    return c ? a : b;
}
__device__ inline DKey key_pick( bool c, DKey const &a, DKey const &b )
{
    return {c ? a.d : b.d, c ? a.id : b.id};
}

} // namespace
} // namespace dtkx

#include "knn_group.hpp"

namespace dtkx
{
namespace
{

// The unordered rows of a wave's lanes (K > kFusedSortK; has: the lane has
// one, row r) sorted by (distance, index), a row at a time over the wave.
template <typename T>
__device__ inline void sort_lane_rows( QueryArgs<T> const &a, int64_t r, bool has )
{
    using SK = SortKey<T>;
    int const lane = threadIdx.x;
    __threadfence_block(); // the lanes' rows are read by other lanes
    for ( uint64_t left = __ballot( has ); left; left &= left - 1 )
    {
        int const l = __builtin_ctzll( left );
        int64_t const rr = a.row0 + __builtin_amdgcn_readlane(
                                        (int)( r - a.row0 ), l );
        int32_t const t = a.order[rr];
        int const kk = a.src_off ? a.kk_prob[a.tgt_prob[t]] : a.kk;
        int64_t const base =
            a.row_off ? a.row_off[rr] : ( a.src_pos ? rr : (int64_t)t ) * kk;
        typename SK::type key[1] = {SK::none()};
        if ( lane < kk )
        {
            typename Vec4<T>::type const qp = a.tgt[t];
            T const q[3] = {qp.x, qp.y, qp.z};
            int32_t const id = a.out_idx[base + lane];
            typename Vec4<T>::type const p = a.src[id];
            T const b[3] = {p.x, p.y, p.z};
            key[0] = SK::make( sqrt_rn( box_sq( q, b, b ) ), id );
        }
        sort_wave<1, 64>( key, lane );
        if ( lane < kk )
        {
            int32_t const id = SK::index( key[0] );
            a.out_idx[base + lane] = a.src_pos ? a.src_pos[id] : id;
            if ( a.out_dist )
                a.out_dist[base + lane] = SK::distance( key[0] );
        }
    }
}

// The tree search, one row a lane. LIST: the listed rows, whose number only
// the device knows; else rows [row0, row0 + n_rows), a block each 64.
template <typename T, int K, bool LIST>
__global__ void __launch_bounds__( kQueryBlock )
    knn_query_kernel( QueryArgs<T> const a )
{
    __shared__ int32_t st_node[kLdsStack * kQueryBlock];
    __shared__ T st_d[kLdsStack * kQueryBlock];
    auto tile = [&]( int64_t r, bool has ) {
        constexpr bool kTwo = K >= two_pass_k<T>();
        int64_t const spill = blockIdx.x * (int64_t)kQueryBlock + threadIdx.x;
        if ( has )
        {
            if constexpr ( kTwo )
                has = query2_row<T, K, LIST>( a, spill, r, st_node, st_d );
            else
                has = query_row<T, K, LIST>( a, spill, r, st_node, st_d );
        }
        if constexpr ( kTwo && K > kFusedSortK )
            sort_lane_rows( a, r, has );
    };
    if constexpr ( LIST )
    {
        int const total = left_total( a.left_count );
        if ( total == 0 )
            return;
        if ( a.n_rows_total && blockIdx.x == 0 && threadIdx.x == 0 )
            atomicAdd( a.n_rows_total, total );
        // A block takes tiles of the part that its XCD left (consecutive on
        // the curve: its L2 then holds their subtrees), and then of the
        // others: a queue each, which every block sees empty before it ends.
        for ( int j = 0; j < kListParts; ++j )
        {
            int const p = ( blockIdx.x + j ) % kListParts;
            int const n = a.left_count[p * kListPad];
            while ( n > 0 )
            {
                int i = 0;
                if ( threadIdx.x == 0 )
                    i = atomicAdd( a.taken + p * kListPad, 1 );
                i = __builtin_amdgcn_readfirstlane( i ) * kQueryBlock;
                if ( i >= n )
                    break;
                i += threadIdx.x;
                tile( i < n ? a.left_rows[p * a.left_cap + i] : 0, i < n );
            }
        }
    }
    else
    {
        int64_t const i = xcd_tile<0>() * kQueryBlock + threadIdx.x;
        tile( a.row0 + i, i < a.n_rows );
    }
}

template <typename T>
struct QueryLauncher
{
    // k: the largest number of results of a row in this launch
    static void dispatch( int k, bool list, int64_t blocks,
                          QueryArgs<T> const &a, hipStream_t s )
    {
        if ( blocks == 0 )
            return;
        dim3 const grid( blocks ), block( kQueryBlock );
#define DTKX_KNN_CASE( KV )                                                    \
    if ( k <= KV )                                                             \
    {                                                                          \
        if ( list )                                                            \
            knn_query_kernel<T, KV, true><<<grid, block, 0, s>>>( a );         \
        else                                                                   \
            knn_query_kernel<T, KV, false><<<grid, block, 0, s>>>( a );        \
        DTKX_HIP( hipGetLastError() );                                         \
        return;                                                                \
    }
        DTKX_KNN_CASE( 1 )
        DTKX_KNN_CASE( 4 )
        DTKX_KNN_CASE( 8 )
        DTKX_KNN_CASE( 10 )
        DTKX_KNN_CASE( 16 )
        DTKX_KNN_CASE( 24 )
        DTKX_KNN_CASE( 32 )
        DTKX_KNN_CASE( 48 )
        DTKX_KNN_CASE( 64 )
#undef DTKX_KNN_CASE
        DTKX_REQUIRE( k <= knn_max_k, DTKX_ERR_UNSUPPORTED );
    }
};

// Targets a group and a wave (per_target sources a target). Groups of as
// many rows as a sort takes, fewer where so many sources lie within the k-th
// distance of a group (estimated for evenly spread points) that a wave's
// registers would not hold them. 64 targets a wave, half of that from
// k = 17, where a wave works long enough for the last ones to show (1M x 1M,
// search with build: k = 32 0.939 ms against 0.961, k = 10 0.749 against
// 0.726), and fewer where the launch would have less than 8192 waves (1e5 x
// 1e5, k = 32: 0.310 ms against 0.332 with 2048 waves at least).
template <typename T, int S>
void plan_groups( double per_target, int64_t n_rows, int kk, GroupArgs<T> &g )
{
    double const reach = 2.2 * std::cbrt( 0.2387 * kk );
    auto candidates = [&]( int n ) {
        double const e = std::cbrt( n * per_target ) + reach;
        return e * e * e;
    };
    using Shape = GroupShape<T, S>;
    g.group = Shape::kRows;
    while ( g.group > 1 &&
            candidates( g.group ) > 0.7 * Shape::kCand )
        g.group /= 2;
    g.per_wave = kk > 16 ? 32 : 64;
    while ( g.per_wave > 1 && n_rows / g.per_wave < 8192 )
        g.per_wave /= 2;
    g.group = std::min( g.group, g.per_wave );
    g.spacing = (float)( 1.0 / std::cbrt( (double)kk ) );
    g.root_k = (float)( 1.0 / std::sqrt( (double)kk ) );
}

template <typename T, int S>
void launch_group( GroupArgs<T> g, double per_target, int kk, hipStream_t s )
{
    plan_groups<T, S>( per_target, g.a.n_rows, kk, g );
    knn_group_kernel<T, S>
        <<<ceil_div( g.a.n_rows, g.per_wave ), 64, 0, s>>>( g );
    DTKX_HIP( hipGetLastError() );
}

// Boxes of the n sorted sources, level by level (box_levels launches of
// three levels each). ids (nullable): pts are read through it, and copied
// in order to sorted.
template <typename T, typename V>
void build_boxes( V const *pts, int32_t const *ids, V *sorted, int64_t n,
                  DeviceBuffer<CurveBox<T>> &buf, BoxLevels<T> &out,
                  hipStream_t s )
{
    int64_t count[kMaxBoxLevels] = {};
    out.n_levels = box_levels( n, count );
    int64_t total = 0;
    for ( int l = 0; l < out.n_levels; ++l )
        total += count[l];
    buf.resize( total, s );
    CurveBox<T> *p = buf.get();
    for ( int l = 0; l < out.n_levels; ++l )
    {
        out.level[l] = p;
        p += count[l];
    }
    auto level = [&]( int l ) {
        return l < out.n_levels ? out.level[l] : nullptr;
    };
    box_levels_kernel<T, V, true><<<ceil_div( n, 512 ), 512, 0, s>>>(
        pts, ids, sorted, nullptr, n, level( 0 ), level( 1 ), level( 2 ) );
    DTKX_HIP( hipGetLastError() );
    for ( int l = 3; l < out.n_levels; l += 3 )
    {
        box_levels_kernel<T, V, false>
            <<<ceil_div( count[l - 1], 512 ), 512, 0, s>>>(
                nullptr, nullptr, nullptr, level( l - 1 ), count[l - 1],
                level( l ), level( l + 1 ), level( l + 2 ) );
        DTKX_HIP( hipGetLastError() );
    }
}

// the smallest source set searched by groups: one 64-point node
constexpr int64_t kGroupSources = 64;

// Blocks of the launch over the rows left over: 14 a CU, as their LDS stacks
// allow (float coordinates; 78 MB of deeper stack entries at most).
constexpr int64_t kListBlocks = 3584;

// The queries of a search, in launches of rows with up to kmax results.
// With boxes, rows are searched by groups of targets (knn_group.hpp);
// without, the tree search with its LDS stack runs over every row. Rows that
// either leaves are run by the tree search over a list, with deeper stacks in
// global memory. After the groups the hierarchy is built only if there
// are such rows: the device decides, the launch returns at once otherwise
// (5 us, where the hierarchy of 1M sources takes 80).
// build_tree( left_count ): launches karras_kernel, for rows left if given.
template <typename T, typename BuildTree>
void run_queries( std::vector<KnnBatch::Launch> const &launches,
                  QueryArgs<T> qa, int64_t n_tgt, double per_target,
                  BoxLevels<T> const *boxes, typename Vec4<T>::type const *pts,
                  int32_t const *ids, T const *scene, BuildTree &&build_tree,
                  KnnInfo *info, hipStream_t s )
{
    if ( n_tgt == 0 )
        return;
    // the rows left over (a part's blocks hold an eighth of each launch's
    // rows and a block or two more), their counts and the tiles taken
    qa.left_cap = 0;
    for ( auto const &l : launches )
        qa.left_cap += ( l.end - l.begin ) / kListParts + 2 * kQueryBlock;
    DeviceBuffer<int32_t> rows( kListParts * qa.left_cap, s );
    constexpr int kCounts = kListParts * kListPad;
    DeviceBuffer<int32_t> count( 2 * kCounts, s );
    zero_async( count.get(), 2 * kCounts * sizeof( int32_t ), s );
    qa.left_rows = rows.get();
    qa.left_count = count.get();
    qa.taken = count.get() + kCounts;
    int kmax = 1;
    for ( auto const &l : launches )
        kmax = std::max( kmax, l.kmax );
    if ( boxes )
    {
        for ( auto const &l : launches )
        {
            GroupArgs<T> g;
            g.a = qa;
            g.a.row0 = l.begin;
            g.a.n_rows = l.end - l.begin;
            g.boxes = *boxes;
            g.pts = pts;
            g.ids = ids;
            g.scene = scene;
            if ( g.a.n_rows == 0 )
                continue;
            switch ( group_slots( l.kmax ) )
            {
            case 1:
                launch_group<T, 1>( g, per_target, l.kmax, s );
                break;
            case 16:
                launch_group<T, 16>( g, per_target, l.kmax, s );
                break;
            case 32:
                launch_group<T, 32>( g, per_target, l.kmax, s );
                break;
            case 64:
                launch_group<T, 64>( g, per_target, l.kmax, s );
                break;
            default:
                launch_group<T, 128>( g, per_target, l.kmax, s );
            }
        }
        build_tree( static_cast<int32_t const *>( count.get() ) );
    }
    else
    {
        build_tree( nullptr );
        for ( auto const &l : launches )
        {
            qa.row0 = l.begin;
            qa.n_rows = l.end - l.begin;
            QueryLauncher<T>::dispatch( l.kmax, false,
                                        ceil_div( qa.n_rows, kQueryBlock ), qa,
                                        s );
        }
    }
    // The launch over the list is made without reading its length back (a
    // stream synchronisation, 60 us of idle GPU at 1M x 1M): a bounded grid
    // whose blocks stride over the list, each lane with its own deeper stack.
    // Almost always the list is empty and the launch costs a few us.
    int64_t const blocks =
        std::min<int64_t>( ceil_div( n_tgt, kQueryBlock ), kListBlocks );
    DeviceBuffer<int32_t> gstack(
        static_cast<std::size_t>( kSpill ) * blocks * kQueryBlock, s );
    QueryArgs<T> ra = qa;
    ra.row0 = 0;
    ra.gstack = gstack.get();
    ra.gstride = blocks * kQueryBlock;
    if ( info && info->n_overflow_dev )
        ra.n_rows_total = info->n_overflow_dev;
    QueryLauncher<T>::dispatch( kmax, true, blocks, ra, s );
    if ( info && !info->n_overflow_dev )
    {
        int32_t left[kCounts];
        DTKX_HIP( hipMemcpyAsync( left, count.get(), sizeof( left ),
                                  hipMemcpyDeviceToHost, s ) );
        DTKX_HIP( hipStreamSynchronize( s ) );
        int32_t n_over = 0;
        for ( int p = 0; p < kListParts; ++p )
            n_over += left[p * kListPad];
        info->n_overflow += n_over;
    }
}

template <typename T>
void knn_impl( void const *src_v, int64_t n_src, void const *tgt_v,
               int64_t n_tgt, int k, KnnOutput const &out, KnnInfo *info,
               hipStream_t s )
{
    using V = typename Vec4<T>::type;
    V const *src = static_cast<V const *>( src_v );
    V const *tgt = static_cast<V const *>( tgt_v );
    int const kk = static_cast<int>( k < n_src ? k : n_src );

    // outputs of the sort: the permutations, their inverses, the points in
    // sorted order (the hierarchy's copy, and the caller's double4 copy,
    // one buffer when they coincide)
    DeviceBuffer<int32_t> ids_sorted_buf, pos_buf, order_buf;
    int32_t *ids_sorted = out.src_perm;
    if ( !ids_sorted )
    {
        ids_sorted_buf.resize( n_src, s );
        ids_sorted = ids_sorted_buf.get();
    }
    int32_t *src_pos = out.src_pos;
    if ( out.morton_layout && !src_pos )
    {
        pos_buf.resize( n_src, s );
        src_pos = pos_buf.get();
    }
    int32_t *order = out.query_order;
    if ( !order && n_tgt > 0 )
    {
        order_buf.resize( n_tgt, s );
        order = order_buf.get();
    }
    bool const share = out.sorted_src &&
                       static_cast<void const *>( out.src4 ) == src_v &&
                       sizeof( V ) == sizeof( double4 );
    DeviceBuffer<V> spts_buf;
    V *spts = reinterpret_cast<V *>( out.sorted_src );
    if ( !share )
    {
        spts_buf.resize( n_src, s );
        spts = spts_buf.get();
    }
    DeviceBuffer<T> box( 6, s );
    DeviceBuffer<uint64_t> scodes( n_src, s );
    if ( n_src <= kSmallSort && n_tgt <= kSmallSort )
    {
        SmallSortArgs<T, V> g;
        g.src = src;
        g.tgt = tgt;
        g.n_src = static_cast<int>( n_src );
        g.n_tgt = static_cast<int>( n_tgt );
        g.box = box.get();
        g.codes = scodes.get();
        g.src_ids = ids_sorted;
        g.src_pos = src_pos;
        g.tgt_ids = order;
        g.tgt_pos = out.query_pos;
        g.src_sorted = spts;
        if ( out.sorted_src && !share )
        {
            g.src4 = out.src4;
            g.src4_sorted = out.sorted_src;
        }
        small_sort( g, s );
    }
    else
    {
        // Sort state, one buffer: the digit counts of every pass, the tile
        // tickets and the look-back words of the first pass (all cleared by the
        // scene-box launch), then those of the second pass (cleared by the
        // first pass).
        int const src_tiles = rsort::tiles_for( n_src );
        int const tgt_tiles = rsort::tiles_for( n_tgt );
        std::size_t const head = ( kHistWords + 4 * rsort::kMaxPasses ) * 4;
        std::size_t const look_src = (std::size_t)src_tiles * rsort::kDigits * 8;
        std::size_t const look_tgt = (std::size_t)tgt_tiles * rsort::kDigits * 8;
        std::size_t const zero_bytes = head + look_src + look_tgt;
        static_assert( ( kHistWords + 4 * rsort::kMaxPasses ) * 4 % 16 == 0,
                       "uint4 clearing" );
        DeviceBuffer<uint4> state( ( zero_bytes + look_src + look_tgt ) / 16, s );
        char *const st = reinterpret_cast<char *>( state.get() );
        uint32_t *const hist = reinterpret_cast<uint32_t *>( st );
        uint32_t *const tickets = hist + kHistWords;
        uint64_t *const look0 = reinterpret_cast<uint64_t *>( st + head );
        uint64_t *const look1 = reinterpret_cast<uint64_t *>( st + zero_bytes );

        // scene box of the sources
        int nparts = static_cast<int>( std::min<int64_t>(
            1024, std::max<int64_t>( 1, ceil_div( n_src, kBlock ) ) ) );
        DeviceBuffer<T> partial( 6 * nparts, s );
        bbox_partial<T, V><<<nparts, kBlock, 0, s>>>(
            src, n_src, partial.get(), state.get(),
            static_cast<int64_t>( zero_bytes / 16 ) );
        bbox_final<T><<<1, kBlock, 0, s>>>( partial.get(), nparts, box.get() );
        DTKX_HIP( hipGetLastError() );

        // Hilbert codes of both point sets (the targets' order only has to be
        // local, so their top 48 bits do) with every pass's digit counts
        DeviceBuffer<uint64_t> scodes1( n_src, s );
        DeviceBuffer<uint64_t> tcodes( n_tgt, s ), tcodes1( n_tgt, s );
        curve_hist_kernel<T, V><<<src_tiles + tgt_tiles, rsort::kThreads, 0, s>>>(
            src, n_src, tgt, n_tgt, box.get(), nullptr, nullptr, src_tiles,
            scodes.get(), tcodes.get(), hist );
        DTKX_HIP( hipGetLastError() );

        DeviceBuffer<int32_t> svals( 2 * n_src, s ), tvals( 2 * n_tgt, s );

        rsort::PassArgs pa;
        pa.tickets = tickets;
        rsort::Array &a = pa.a[0];
        a.keys[0] = scodes.get();
        a.keys[1] = scodes1.get();
        a.vals[0] = svals.get();
        a.vals[1] = svals.get() + n_src;
        a.vals_out = ids_sorted;
        a.pos_out = src_pos;
        a.gather_in[0] = src;
        a.gather_out[0] = spts;
        a.gather_bytes[0] = sizeof( V );
        if ( out.sorted_src && !share )
        {
            a.gather_in[1] = out.src4;
            a.gather_out[1] = out.sorted_src;
            a.gather_bytes[1] = sizeof( double4 );
        }
        a.hist = hist;
        a.look[0] = look0;
        a.look[1] = look1;
        a.n = n_src;
        a.tiles = src_tiles;
        a.passes = kSrcPasses;
        a.key_bits = kSrcKeyBits;
        a.key_bytes = 8;
        a.keep_keys = true;
        rsort::Array &b = pa.a[1];
        if ( n_tgt > 0 )
        {
            b.keys[0] = tcodes.get();
            b.keys[1] = tcodes1.get();
            b.vals[0] = tvals.get();
            b.vals[1] = tvals.get() + n_tgt;
            b.vals_out = order;
            b.pos_out = out.query_pos;
            b.hist = hist + kSrcPasses * rsort::kDigits;
            b.look[0] = look0 + (std::size_t)src_tiles * rsort::kDigits;
            b.look[1] = look1 + (std::size_t)src_tiles * rsort::kDigits;
            b.n = n_tgt;
            b.tiles = tgt_tiles;
            b.passes = kTgtPasses;
            b.key_bits = kTgtKeyBits;
            b.key_bytes = 8;
        }
        rsort::sort( pa, s );
        // the sorted codes are back in scodes after an even number of passes
        static_assert( kSrcPasses % 2 == 0, "sorted codes in scodes" );
    }

    if ( n_tgt == 0 )
        return;
    int64_t const n_int = n_src - 1;
    DeviceBuffer<Node<T>> nodes( std::max<int64_t>( n_int, 1 ), s );
    DeviceBuffer<int32_t> sizes( std::max<int64_t>( n_int, 1 ), s );
    bool const grouped = n_src >= kGroupSources;
    DeviceBuffer<CurveBox<T>> box_buf;
    BoxLevels<T> boxes;
    if ( grouped )
        build_boxes<T, V>( spts, nullptr, nullptr, n_src, box_buf, boxes, s );
    auto build_tree = [&]( int32_t const *left_count ) {
        if ( n_int == 0 )
            return;
        karras_kernel<T, V><<<ceil_div( n_int, kBlock ), kBlock, 0, s>>>(
            scodes.get(), ids_sorted, src, spts, n_int, box.get(), boxes,
            nullptr, 1, nodes.get(), sizes.get(), left_count );
        DTKX_HIP( hipGetLastError() );
    };
    QueryArgs<T> qa;
    qa.nodes = nodes.get();
    qa.node_size = kSeed ? sizes.get() : nullptr;
    qa.src = src;
    qa.tgt = tgt;
    qa.order = order;
    qa.n_src = n_src;
    qa.kk = kk;
    qa.out_idx = out.indices;
    qa.out_dist = out.dist;
    qa.src_pos = out.morton_layout ? src_pos : nullptr;
    if ( info && info->query_begin )
        DTKX_HIP( hipEventRecord( info->query_begin, s ) );
    run_queries<T>( {{0, n_tgt, kk}}, qa, n_tgt, (double)n_src / (double)n_tgt,
                    grouped ? &boxes : nullptr, spts, ids_sorted, box.get(),
                    build_tree, info, s );
    if ( info && info->query_end )
        DTKX_HIP( hipEventRecord( info->query_end, s ) );
    // buffers are released at scope exit, ordered on the stream
}


// ------------------------------------------------------------- batched
template <typename T, typename V>
__global__ void __launch_bounds__( kBlock )
    bbox_segments( V const *pts, int32_t const *src_off, T *boxes )
{
    int const pb = blockIdx.x;
    int64_t const b = src_off[pb], e = src_off[pb + 1];
    T lo[3] = {INFINITY, INFINITY, INFINITY};
    T hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for ( int64_t i = b + threadIdx.x; i < e; i += kBlock )
    {
        V p = pts[i];
        lo[0] = fmin( lo[0], p.x );
        lo[1] = fmin( lo[1], p.y );
        lo[2] = fmin( lo[2], p.z );
        hi[0] = fmax( hi[0], p.x );
        hi[1] = fmax( hi[1], p.y );
        hi[2] = fmax( hi[2], p.z );
    }
    __shared__ T sh[6][kBlock];
    for ( int d = 0; d < 3; ++d )
    {
        sh[d][threadIdx.x] = lo[d];
        sh[3 + d][threadIdx.x] = hi[d];
    }
    __syncthreads();
    for ( int off = kBlock / 2; off > 0; off >>= 1 )
    {
        if ( threadIdx.x < off )
            for ( int d = 0; d < 3; ++d )
            {
                sh[d][threadIdx.x] =
                    fmin( sh[d][threadIdx.x], sh[d][threadIdx.x + off] );
                sh[3 + d][threadIdx.x] = fmax(
                    sh[3 + d][threadIdx.x], sh[3 + d][threadIdx.x + off] );
            }
        __syncthreads();
    }
    if ( threadIdx.x == 0 )
        for ( int d = 0; d < 6; ++d )
            boxes[pb * 6 + d] = sh[d][0];
}

// Clears [a, a + na) and [b, b + nb) (uint4 units).
__global__ void __launch_bounds__( kBlock )
    clear2_kernel( uint4 *a, int64_t na, uint4 *b, int64_t nb )
{
    for ( int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < na + nb;
          i += (int64_t)gridDim.x * kBlock )
        ( i < na ? a[i] : b[i - na] ) = make_uint4( 0u, 0u, 0u, 0u );
}

// Second-stage keys of a batch's sorts, read through the first stage's
// order: a source's problem, a target's row key (row_key[problem]), with
// the digit counts of their passes added into hist (sources' first, zero on
// entry); one sort tile of keys a block, blocks [0, src_blocks) take the
// sources.
__global__ void __launch_bounds__( rsort::kThreads )
    group_keys_kernel( int32_t const *src_ids, int32_t const *src_prob,
                       int64_t n_src, int src_passes, int32_t const *tgt_ids,
                       int32_t const *tgt_prob, int32_t const *row_key,
                       int64_t n_tgt, int tgt_passes, int src_blocks,
                       uint32_t *src_keys, uint32_t *tgt_keys, uint32_t *hist )
{
    __shared__ uint32_t h[4 * rsort::kDigits];
    bool const is_src = static_cast<int>( blockIdx.x ) < src_blocks;
    int const words = ( is_src ? src_passes : tgt_passes ) * rsort::kDigits;
    for ( int i = threadIdx.x; i < words; i += rsort::kThreads )
        h[i] = 0;
    __syncthreads();
    int64_t const c0 =
        (int64_t)( is_src ? blockIdx.x : blockIdx.x - src_blocks ) *
        rsort::kTile;
    int64_t const n = is_src ? n_src : n_tgt;
    int const passes = is_src ? src_passes : tgt_passes;
    for ( int s = 0; s < rsort::kItems; ++s )
    {
        int64_t const i = c0 + s * rsort::kThreads + threadIdx.x;
        if ( i >= n )
            break;
        uint32_t const key =
            is_src ? static_cast<uint32_t>( src_prob[src_ids[i]] )
                   : static_cast<uint32_t>( row_key[tgt_prob[tgt_ids[i]]] );
        ( is_src ? src_keys : tgt_keys )[i] = key;
        for ( int p = 0; p < passes; ++p )
            atomicAdd( &h[p * rsort::kDigits + ( ( key >> ( 8 * p ) ) & 255 )],
                       1u );
    }
    __syncthreads();
    uint32_t *g = hist + ( is_src ? 0 : src_passes * rsort::kDigits );
    for ( int i = threadIdx.x; i < words; i += rsort::kThreads )
    {
        uint32_t const v = h[i];
        if ( v )
            atomicAdd( g + i, v );
    }
}

__global__ void __launch_bounds__( kBlock )
    row_offsets_kernel( int32_t const *order, int32_t const *tgt_prob,
                        int64_t const *row_base, int32_t const *row_start,
                        int32_t const *kk_prob, int64_t n, int64_t nnz,
                        int64_t *row_off )
{
    int64_t r = blockIdx.x * (int64_t)kBlock + threadIdx.x;
    if ( r > n )
        return;
    if ( r == n )
    {
        row_off[n] = nnz;
        return;
    }
    int32_t const pb = tgt_prob[order[r]];
    row_off[r] = row_base[pb] + ( r - row_start[pb] ) * (int64_t)kk_prob[pb];
}

template <typename T>
void knn_batched_impl( void const *src_v, int64_t n_src, void const *tgt_v,
                       int64_t n_tgt, KnnBatch const &b,
                       KnnBatchOutput const &out, KnnInfo *info,
                       hipStream_t s )
{
    using V = typename Vec4<T>::type;
    V const *src = static_cast<V const *>( src_v );
    V const *tgt = static_cast<V const *>( tgt_v );
    int const P = b.n_problems;
    int prob_bits = 1;
    while ( ( int64_t( 1 ) << prob_bits ) < P )
        ++prob_bits;

    DeviceBuffer<T> boxes( 6 * (std::size_t)P, s );
    bbox_segments<T, V><<<P, kBlock, 0, s>>>( src, b.src_off, boxes.get() );
    DTKX_HIP( hipGetLastError() );

    // Two stable radix sorts of both point sets, in shared launches
    // (radix_sort.hpp): by Hilbert code in the problem's box (sources 63 bits,
    // targets 48, as one problem's search orders them), then by the
    // problem's key (sources: the problem; targets: its row key). The second
    // sorts positions of the first, and its last pass gathers the first's
    // indices (and the sources' codes) into the final order.
    int const src_tiles = rsort::tiles_for( n_src );
    int const tgt_tiles = rsort::tiles_for( n_tgt );
    int const src_passes2 = rsort::passes_for( prob_bits );
    int const tgt_passes2 = rsort::passes_for( b.key_bits );
    int const hist1 = kHistWords;
    int const hist2 = ( src_passes2 + tgt_passes2 ) * rsort::kDigits;
    std::size_t const sb1 = rsort::state_bytes( hist1, src_tiles + tgt_tiles );
    std::size_t const sb2 = rsort::state_bytes( hist2, src_tiles + tgt_tiles );
    DeviceBuffer<uint4> state( ( sb1 + sb2 ) / 16, s );
    rsort::State const st1 =
        rsort::carve_state( state.get(), hist1, src_tiles + tgt_tiles );
    rsort::State const st2 = rsort::carve_state(
        reinterpret_cast<char *>( state.get() ) + sb1, hist2,
        src_tiles + tgt_tiles );
    clear2_kernel<<<std::min<int64_t>( 1024, ceil_div( sb1 + sb2, 16 * kBlock ) ),
                    kBlock, 0, s>>>(
        static_cast<uint4 *>( st1.zero ), st1.zero_bytes / 16,
        static_cast<uint4 *>( st2.zero ), st2.zero_bytes / 16 );
    DTKX_HIP( hipGetLastError() );

    DeviceBuffer<uint64_t> scodes( n_src, s ), scodes1( n_src, s ),
        codes_sorted( n_src, s );
    DeviceBuffer<uint64_t> tcodes( n_tgt, s ), tcodes1( n_tgt, s );
    curve_hist_kernel<T, V><<<src_tiles + tgt_tiles, rsort::kThreads, 0, s>>>(
        src, n_src, tgt, n_tgt, boxes.get(), b.src_prob, b.tgt_prob,
        src_tiles, scodes.get(), tcodes.get(), st1.hist );
    DTKX_HIP( hipGetLastError() );
    DeviceBuffer<int32_t> svals( 2 * n_src, s ), tvals( 2 * n_tgt, s ),
        sids1( n_src, s ), tids1( n_tgt, s );
    auto first_stage = [&]( rsort::Array &a, rsort::Array &t ) {
        a.keys[0] = scodes.get();
        a.keys[1] = scodes1.get();
        a.vals[0] = svals.get();
        a.vals[1] = svals.get() + n_src;
        a.vals_out = sids1.get();
        a.hist = st1.hist;
        a.look[0] = st1.look0;
        a.look[1] = st1.look1;
        a.n = n_src;
        a.tiles = src_tiles;
        a.passes = kSrcPasses;
        a.key_bits = kSrcKeyBits;
        a.key_bytes = 8;
        a.keep_keys = true;
        if ( n_tgt == 0 )
            return;
        t.keys[0] = tcodes.get();
        t.keys[1] = tcodes1.get();
        t.vals[0] = tvals.get();
        t.vals[1] = tvals.get() + n_tgt;
        t.vals_out = tids1.get();
        t.hist = st1.hist + kSrcPasses * rsort::kDigits;
        t.look[0] = st1.look0 + (std::size_t)src_tiles * rsort::kDigits;
        t.look[1] = st1.look1 + (std::size_t)src_tiles * rsort::kDigits;
        t.n = n_tgt;
        t.tiles = tgt_tiles;
        t.passes = kTgtPasses;
        t.key_bits = kTgtKeyBits;
        t.key_bytes = 8;
    };
    rsort::PassArgs pa1;
    pa1.tickets = st1.tickets;
    first_stage( pa1.a[0], pa1.a[1] );
    rsort::sort( pa1, s );

    // second stage: keys through the first order; scodes holds the sorted
    // codes (an even number of passes), tcodes the targets' keys
    DeviceBuffer<uint32_t> skeys( n_src, s ), skeys1( n_src, s ),
        tkeys( n_tgt, s ), tkeys1( n_tgt, s );
    group_keys_kernel<<<src_tiles + tgt_tiles, rsort::kThreads, 0, s>>>(
        sids1.get(), b.src_prob, n_src, src_passes2, tids1.get(), b.tgt_prob,
        b.row_key, n_tgt, tgt_passes2, src_tiles, skeys.get(), tkeys.get(),
        st2.hist );
    DTKX_HIP( hipGetLastError() );
    DeviceBuffer<int32_t> spos1( n_src, s ), tpos1( n_tgt, s );
    rsort::PassArgs pa2;
    pa2.tickets = st2.tickets;
    {
        rsort::Array &a = pa2.a[0];
        a.keys[0] = skeys.get();
        a.keys[1] = skeys1.get();
        a.vals[0] = svals.get();
        a.vals[1] = svals.get() + n_src;
        a.vals_out = spos1.get();
        a.gather_in[0] = sids1.get();
        a.gather_out[0] = out.src_perm;
        a.gather_bytes[0] = 4;
        a.gather_in[1] = scodes.get();
        a.gather_out[1] = codes_sorted.get();
        a.gather_bytes[1] = 8;
        a.hist = st2.hist;
        a.look[0] = st2.look0;
        a.look[1] = st2.look1;
        a.n = n_src;
        a.tiles = src_tiles;
        a.passes = src_passes2;
        a.key_bits = prob_bits;
        a.key_bytes = 4;
        if ( n_tgt > 0 )
        {
            rsort::Array &t = pa2.a[1];
            t.keys[0] = tkeys.get();
            t.keys[1] = tkeys1.get();
            t.vals[0] = tvals.get();
            t.vals[1] = tvals.get() + n_tgt;
            t.vals_out = tpos1.get();
            t.gather_in[0] = tids1.get();
            t.gather_out[0] = out.order;
            t.gather_bytes[0] = 4;
            t.hist = st2.hist + src_passes2 * rsort::kDigits;
            t.look[0] = st2.look0 + (std::size_t)src_tiles * rsort::kDigits;
            t.look[1] = st2.look1 + (std::size_t)src_tiles * rsort::kDigits;
            t.n = n_tgt;
            t.tiles = tgt_tiles;
            t.passes = tgt_passes2;
            t.key_bits = b.key_bits;
            t.key_bytes = 4;
        }
    }
    rsort::sort( pa2, s );
    invert_permutation( out.src_perm, n_src, out.src_pos, s );

    if ( n_tgt == 0 )
        return;
    // one hierarchy per problem, all in one launch
    int64_t const n_int = n_src - P;
    DeviceBuffer<Node<T>> nodes( std::max<int64_t>( n_int, 1 ), s );
    DeviceBuffer<int32_t> sizes( std::max<int64_t>( n_int, 1 ), s );
    bool const grouped = n_src >= kGroupSources;
    DeviceBuffer<V> spts( grouped ? n_src : 0, s );
    DeviceBuffer<CurveBox<T>> box_buf;
    BoxLevels<T> levels;
    if ( grouped )
        build_boxes<T, V>( src, out.src_perm, spts.get(), n_src, box_buf, levels,
                           s );
    auto build_tree = [&]( int32_t const *left_count ) {
        if ( n_int == 0 )
            return;
        karras_kernel<T, V><<<ceil_div( n_int, kBlock ), kBlock, 0, s>>>(
            codes_sorted.get(), out.src_perm, src, nullptr, n_int,
            boxes.get(), levels, b.src_off, P, nodes.get(), sizes.get(), left_count );
        DTKX_HIP( hipGetLastError() );
    };

    // rows: ordered by (row key of the problem, Hilbert code)
    row_offsets_kernel<<<ceil_div( n_tgt + 1, kBlock ), kBlock, 0, s>>>(
        out.order, b.tgt_prob, b.row_base, b.row_start, b.kk_prob, n_tgt,
        b.nnz, out.row_off );
    DTKX_HIP( hipGetLastError() );

    if ( info && info->query_begin )
        DTKX_HIP( hipEventRecord( info->query_begin, s ) );
    QueryArgs<T> qa;
    qa.nodes = nodes.get();
    qa.node_size = kSeed ? sizes.get() : nullptr;
    qa.src = src;
    qa.tgt = tgt;
    qa.order = out.order;
    qa.src_off = b.src_off;
    qa.tgt_prob = b.tgt_prob;
    qa.kk_prob = b.kk_prob;
    qa.row_off = out.row_off;
    qa.out_idx = out.indices;
    qa.src_pos = out.src_pos;
    run_queries<T>( b.launches, qa, n_tgt, (double)n_src / (double)n_tgt,
                    grouped ? &levels : nullptr, spts.get(), out.src_perm,
                    boxes.get(), build_tree, info, s );
    if ( info && info->query_end )
        DTKX_HIP( hipEventRecord( info->query_end, s ) );
}

} // namespace

int knn_bucket( int k ) { return group_slots( k ); }

void knn_search_batched( int geometry, void const *src, int64_t n_src,
                         void const *tgt, int64_t n_tgt, KnnBatch const &b,
                         KnnBatchOutput const &out, KnnInfo *info,
                         hipStream_t s )
{
    DTKX_REQUIRE( b.n_problems >= 1, DTKX_ERR_INVALID_ARGUMENT );
    DTKX_REQUIRE( n_src >= b.n_problems, DTKX_ERR_EMPTY_SOURCE );
    DTKX_REQUIRE( n_src < INT32_MAX && n_tgt < INT32_MAX,
                  DTKX_ERR_UNSUPPORTED );
    if ( geometry == DTKX_GEOMETRY_FLOAT )
        knn_batched_impl<float>( src, n_src, tgt, n_tgt, b, out, info, s );
    else
        knn_batched_impl<double>( src, n_src, tgt, n_tgt, b, out, info, s );
}

void knn_search( int geometry, void const *src, int64_t n_src,
                 void const *tgt, int64_t n_tgt, int k, KnnOutput const &out,
                 KnnInfo *info, hipStream_t s )
{
    DTKX_REQUIRE( n_src > 0, DTKX_ERR_EMPTY_SOURCE );
    DTKX_REQUIRE( k >= 1 && k <= knn_max_k, DTKX_ERR_UNSUPPORTED );
    DTKX_REQUIRE( n_src < INT32_MAX && n_tgt < INT32_MAX,
                  DTKX_ERR_INVALID_ARGUMENT );
    if ( geometry == DTKX_GEOMETRY_FLOAT )
        knn_impl<float>( src, n_src, tgt, n_tgt, k, out, info, s );
    else
        knn_impl<double>( src, n_src, tgt, n_tgt, k, out, info, s );
}

} // namespace dtkx
