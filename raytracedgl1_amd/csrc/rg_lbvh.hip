// Linear BVH build for gfx950: FP64 bounds and Morton quantisation, stable
// LSD radix sort with wave-ballot ranking, the Karras (2012) hierarchy joined
// bottom-up with its boxes, and a deterministic collapse into 8-wide nodes.
//
// This replaces the driver-side acceleration-structure build of the reference
// (ASBuilder::BuildBottomLevel / BuildTopLevel, Source/ASBuilder.cpp:141-206);
// the reference has no BVH code of its own, so the build follows the
// published algorithms named above.
#include "rg_bvh.h"
#include "rg_device_math.h"
#include "rg_scan.h"

#include <cfloat>
#include <cmath>

namespace rg
{
namespace
{

constexpr int      THREADS     = 256;
constexpr int      RS_ITEMS    = 8;
constexpr int      RS_TILE     = THREADS * RS_ITEMS;
constexpr uint32_t MORTON_BITS = 21;
constexpr double   MORTON_CELLS = 2097152.0; // 2^21

// ------------------------------------------------------------- bounds

__device__ __forceinline__ void LoadTri( const float* tris, uint32_t i, v3& a, v3& b, v3& c )
{
    const float* t = tris + size_t( i ) * 9;
    a              = mk3( t[ 0 ], t[ 1 ], t[ 2 ] );
    b              = mk3( t[ 3 ], t[ 4 ], t[ 5 ] );
    c              = mk3( t[ 6 ], t[ 7 ], t[ 8 ] );
}

// Centroid in FP64: ((v0 + v1) + v2) / 3 per axis.
__device__ __forceinline__ void Centroid( const float* tris, uint32_t i, double c[ 3 ] )
{
    const float* t = tris + size_t( i ) * 9;
    for( int k = 0; k < 3; k++ )
    {
        c[ k ] = ( ( double( t[ k ] ) + double( t[ 3 + k ] ) ) + double( t[ 6 + k ] ) ) / 3.0;
    }
}

__global__ __launch_bounds__( THREADS ) void k_centroid_bounds( const float* tris, uint32_t n, double* partials )
{
    __shared__ double s[ 6 ][ THREADS ];
    double            lo[ 3 ] = { DBL_MAX, DBL_MAX, DBL_MAX };
    double            hi[ 3 ] = { -DBL_MAX, -DBL_MAX, -DBL_MAX };
    for( uint32_t i = blockIdx.x * THREADS + threadIdx.x; i < n; i += gridDim.x * THREADS )
    {
        double c[ 3 ];
        Centroid( tris, i, c );
        for( int k = 0; k < 3; k++ )
        {
            lo[ k ] = fmin( lo[ k ], c[ k ] );
            hi[ k ] = fmax( hi[ k ], c[ k ] );
        }
    }
    for( int k = 0; k < 3; k++ )
    {
        s[ k ][ threadIdx.x ]     = lo[ k ];
        s[ 3 + k ][ threadIdx.x ] = hi[ k ];
    }
    __syncthreads();
    for( int stride = THREADS / 2; stride > 0; stride >>= 1 )
    {
        if( int( threadIdx.x ) < stride )
        {
            for( int k = 0; k < 3; k++ )
            {
                s[ k ][ threadIdx.x ]     = fmin( s[ k ][ threadIdx.x ], s[ k ][ threadIdx.x + stride ] );
                s[ 3 + k ][ threadIdx.x ] = fmax( s[ 3 + k ][ threadIdx.x ], s[ 3 + k ][ threadIdx.x + stride ] );
            }
        }
        __syncthreads();
    }
    if( threadIdx.x < 6 )
    {
        partials[ blockIdx.x * 6 + threadIdx.x ] = s[ threadIdx.x ][ 0 ];
    }
}

// One block of THREADS: strided partial reductions, then an LDS tree.
__global__ __launch_bounds__( THREADS ) void k_bounds_final( const double* partials, uint32_t blocks, double* out )
{
    __shared__ double s[ 6 ][ THREADS ];
    double            v[ 6 ] = { DBL_MAX, DBL_MAX, DBL_MAX, -DBL_MAX, -DBL_MAX, -DBL_MAX };
    for( uint32_t b = threadIdx.x; b < blocks; b += THREADS )
    {
        for( int k = 0; k < 3; k++ )
        {
            v[ k ]     = fmin( v[ k ], partials[ b * 6 + k ] );
            v[ 3 + k ] = fmax( v[ 3 + k ], partials[ b * 6 + 3 + k ] );
        }
    }
    for( int k = 0; k < 6; k++ )
    {
        s[ k ][ threadIdx.x ] = v[ k ];
    }
    __syncthreads();
    for( int stride = THREADS / 2; stride > 0; stride >>= 1 )
    {
        if( int( threadIdx.x ) < stride )
        {
            for( int k = 0; k < 3; k++ )
            {
                s[ k ][ threadIdx.x ]     = fmin( s[ k ][ threadIdx.x ], s[ k ][ threadIdx.x + stride ] );
                s[ 3 + k ][ threadIdx.x ] = fmax( s[ 3 + k ][ threadIdx.x ], s[ 3 + k ][ threadIdx.x + stride ] );
            }
        }
        __syncthreads();
    }
    if( threadIdx.x < 6 )
    {
        out[ threadIdx.x ] = s[ threadIdx.x ][ 0 ];
    }
}

// ------------------------------------------------------------- morton

__device__ __forceinline__ uint64_t ExpandBits21( uint32_t v )
{
    uint64_t x = v & 0x1fffffu;
    x          = ( x | x << 32 ) & 0x1f00000000ffffull;
    x          = ( x | x << 16 ) & 0x1f0000ff0000ffull;
    x          = ( x | x << 8 ) & 0x100f00f00f00f00full;
    x          = ( x | x << 4 ) & 0x10c30c30c30c30c3ull;
    x          = ( x | x << 2 ) & 0x1249249249249249ull;
    return x;
}

__device__ __forceinline__ uint32_t Quantize21( double c, double lo, double hi )
{
    const double extent = hi - lo;
    if( !( extent > 0.0 ) )
    {
        return 0;
    }
    const double f = floor( ( ( c - lo ) / extent ) * MORTON_CELLS );
    return f >= MORTON_CELLS - 1.0 ? ( 1u << MORTON_BITS ) - 1u : ( f <= 0.0 ? 0u : uint32_t( f ) );
}

// Key of the traversal's tree: the axes share one cell size, a 2^21st of the
// longest extent.  Cells of the per-axis quantisation are as flat as the
// scene, and so were the boxes: rays over a 256 x 256 terrain with 10 units
// of height visited 13.5 (camera), 19.9 (bounce) and 20.8 (shadow) nodes,
// and 8.3, 11.5 and 16.7 with cubic cells.
__device__ __forceinline__ uint64_t CubicCode( const double c[ 3 ], const double* bounds )
{
    const double e = fmax( bounds[ 3 ] - bounds[ 0 ], fmax( bounds[ 4 ] - bounds[ 1 ], bounds[ 5 ] - bounds[ 2 ] ) );
    return ( ExpandBits21( Quantize21( c[ 0 ], bounds[ 0 ], bounds[ 0 ] + e ) ) << 2 ) |
           ( ExpandBits21( Quantize21( c[ 1 ], bounds[ 1 ], bounds[ 1 ] + e ) ) << 1 ) | ExpandBits21( Quantize21( c[ 2 ], bounds[ 2 ], bounds[ 2 ] + e ) );
}

__device__ __forceinline__ uint64_t AxisCode( const double c[ 3 ], const double* bounds )
{
    return ( ExpandBits21( Quantize21( c[ 0 ], bounds[ 0 ], bounds[ 3 ] ) ) << 2 ) | ( ExpandBits21( Quantize21( c[ 1 ], bounds[ 1 ], bounds[ 4 ] ) ) << 1 ) |
           ExpandBits21( Quantize21( c[ 2 ], bounds[ 2 ], bounds[ 5 ] ) );
}

// Where a build's keys go: the traversal's tree, and the published one (null
// codes: not asked for).
struct KeyOut
{
    uint64_t* codes;
    uint64_t* viewKeys;
    uint32_t* viewVals;
    uint64_t* keys;
    uint32_t* vals;
};

__global__ __launch_bounds__( THREADS ) void k_morton( const float* tris, uint32_t n, const double* bounds, KeyOut o )
{
    uint32_t i = blockIdx.x * THREADS + threadIdx.x;
    if( i >= n )
    {
        return;
    }
    double c[ 3 ];
    Centroid( tris, i, c );
    o.keys[ i ] = CubicCode( c, bounds );
    o.vals[ i ] = i;
    if( o.codes )
    {
        const uint64_t code = AxisCode( c, bounds );
        o.codes[ i ]        = code;
        o.viewKeys[ i ]     = code;
        o.viewVals[ i ]     = i;
    }
}

// ------------------------------------------------------ batched scenes
// S scenes concatenated: scene s owns triangles [offsets[s], offsets[s+1]).

__device__ __forceinline__ uint32_t SceneOf( const uint32_t* offsets, uint32_t S, uint32_t i )
{
    uint32_t lo = 0, hi = S; // last scene with offsets[s] <= i
    while( hi - lo > 1 )
    {
        const uint32_t mid = ( lo + hi ) / 2;
        if( offsets[ mid ] <= i )
        {
            lo = mid;
        }
        else
        {
            hi = mid;
        }
    }
    return lo;
}

// Block b of scene s (blockIdx.x = s * B + b) reduces part of that scene.
__global__ __launch_bounds__( THREADS ) void k_centroid_bounds_seg( const float* tris, const uint32_t* offsets, uint32_t B, double* partials )
{
    __shared__ double s[ 6 ][ THREADS ];
    const uint32_t    scene = blockIdx.x / B, b = blockIdx.x % B;
    const uint32_t    first = offsets[ scene ], last = offsets[ scene + 1 ];
    double            lo[ 3 ] = { DBL_MAX, DBL_MAX, DBL_MAX };
    double            hi[ 3 ] = { -DBL_MAX, -DBL_MAX, -DBL_MAX };
    for( uint32_t i = first + b * THREADS + threadIdx.x; i < last; i += B * THREADS )
    {
        double c[ 3 ];
        Centroid( tris, i, c );
        for( int k = 0; k < 3; k++ )
        {
            lo[ k ] = fmin( lo[ k ], c[ k ] );
            hi[ k ] = fmax( hi[ k ], c[ k ] );
        }
    }
    for( int k = 0; k < 3; k++ )
    {
        s[ k ][ threadIdx.x ]     = lo[ k ];
        s[ 3 + k ][ threadIdx.x ] = hi[ k ];
    }
    __syncthreads();
    for( int stride = THREADS / 2; stride > 0; stride >>= 1 )
    {
        if( int( threadIdx.x ) < stride )
        {
            for( int k = 0; k < 3; k++ )
            {
                s[ k ][ threadIdx.x ]     = fmin( s[ k ][ threadIdx.x ], s[ k ][ threadIdx.x + stride ] );
                s[ 3 + k ][ threadIdx.x ] = fmax( s[ 3 + k ][ threadIdx.x ], s[ 3 + k ][ threadIdx.x + stride ] );
            }
        }
        __syncthreads();
    }
    if( threadIdx.x < 6 )
    {
        partials[ size_t( blockIdx.x ) * 6 + threadIdx.x ] = s[ threadIdx.x ][ 0 ];
    }
}

// Block s combines scene s's B partials.
__global__ void k_bounds_final_seg( const double* partials, uint32_t B, double* out )
{
    if( threadIdx.x < 6 )
    {
        const bool isMin = threadIdx.x < 3;
        double     v     = isMin ? DBL_MAX : -DBL_MAX;
        for( uint32_t b = 0; b < B; b++ )
        {
            const double p = partials[ ( size_t( blockIdx.x ) * B + b ) * 6 + threadIdx.x ];
            v              = isMin ? fmin( v, p ) : fmax( v, p );
        }
        out[ size_t( blockIdx.x ) * 6 + threadIdx.x ] = v;
    }
}

// Morton code in the scene's own bounds; the sort key carries the scene in
// its top 7 bits above the code's top 57 bits (19 per axis), so one sort
// groups the scenes and orders each by its Morton curve, and the Karras
// hierarchy over the keys splits at scene boundaries first.
__global__ __launch_bounds__( THREADS ) void k_morton_seg( const float* tris, uint32_t n, const uint32_t* offsets, uint32_t S,
                                                           const double* bounds, KeyOut o )
{
    uint32_t i = blockIdx.x * THREADS + threadIdx.x;
    if( i >= n )
    {
        return;
    }
    const uint64_t scene = SceneOf( offsets, S, i );
    const double*  bb    = bounds + scene * 6;
    double         c[ 3 ];
    Centroid( tris, i, c );
    o.keys[ i ] = ( scene << 57 ) | ( CubicCode( c, bb ) >> 6 );
    o.vals[ i ] = i;
    if( o.codes )
    {
        const uint64_t code = AxisCode( c, bb );
        o.codes[ i ]        = code;
        o.viewKeys[ i ]     = ( scene << 57 ) | ( code >> 6 );
        o.viewVals[ i ]     = i;
    }
}

// The internal node whose range is exactly scene s (its keys differ from its
// neighbours' in the scene bits); none for a one-triangle scene.
__global__ __launch_bounds__( THREADS ) void k_scene_roots( uint32_t internal, const uint32_t* rf, const uint32_t* rl, const uint32_t* offsets,
                                                            uint32_t S, uint32_t* roots )
{
    const uint32_t i = blockIdx.x * THREADS + threadIdx.x;
    if( i >= internal )
    {
        return;
    }
    const uint32_t scene = SceneOf( offsets, S, rf[ i ] );
    if( rf[ i ] == offsets[ scene ] && rl[ i ] + 1u == offsets[ scene + 1 ] )
    {
        roots[ scene ] = i;
    }
}

// The words a build starts from: the collapse's level counts at 0, the node
// flags at 0 and the scene roots at none; one launch for what were up to
// four memsets of two kernels each.
__global__ __launch_bounds__( THREADS ) void k_build_init( uint32_t* levels, uint32_t levelWords, uint32_t* isNode, uint32_t nodeWords, uint32_t* roots0,
                                                           uint32_t* roots1, uint32_t rootWords )
{
    for( uint32_t i = blockIdx.x * THREADS + threadIdx.x; i < levelWords || i < nodeWords || i < rootWords; i += gridDim.x * THREADS )
    {
        if( i < levelWords )
        {
            levels[ i ] = 0u;
        }
        if( i < nodeWords )
        {
            isNode[ i ] = 0u;
        }
        if( i < rootWords && roots0 )
        {
            roots0[ i ] = RG_EXT_MISS;
        }
        if( i < rootWords && roots1 )
        {
            roots1[ i ] = RG_EXT_MISS;
        }
    }
}

// Seeds a collapse with every scene root.  A one-triangle scene (frame
// segments only) has no internal node: the published tree leaves it out, the
// traversal's tree gives it a node of one leaf, so that scene s's root is
// its node s.  With boxes: each root's box (lo xyz, hi xyz, 2 unused).
__global__ void k_seed_frontier_seg( const uint32_t* roots, uint32_t S, const uint32_t* offsets, uint32_t internal, bool leaves, uint32_t* queue,
                                     uint32_t* counts, const float* bounds, float* boxes )
{
    if( threadIdx.x == 0 )
    {
        uint32_t k = 0;
        for( uint32_t s = 0; s < S; s++ )
        {
            if( roots[ s ] != 0xFFFFFFFFu )
            {
                queue[ k++ ] = roots[ s ];
            }
            else if( leaves )
            {
                queue[ k++ ] = internal + offsets[ s ];
            }
        }
        counts[ 0 ] = k;
    }
    if( boxes && threadIdx.x < S )
    {
        const uint32_t s  = threadIdx.x;
        const uint32_t id = roots[ s ] != 0xFFFFFFFFu ? roots[ s ] : internal + offsets[ s ];
        for( int k = 0; k < 6; k++ )
        {
            boxes[ s * 8 + k ] = bounds[ size_t( id ) * 6 + k ];
        }
        boxes[ s * 8 + 6 ] = boxes[ s * 8 + 7 ] = 0.0f;
    }
}

// 8-wide root of each scene of the published tree.
__global__ void k_gather_roots8( const uint32_t* roots, uint32_t S, const uint32_t* node8Index, uint32_t* roots8 )
{
    for( uint32_t s = threadIdx.x; s < S; s += blockDim.x )
    {
        roots8[ s ] = roots[ s ] != 0xFFFFFFFFu ? node8Index[ roots[ s ] ] : 0xFFFFFFFFu;
    }
}

// --------------------------------------------------------- radix sort
// One pass = three launches: digit counts per tile, one block per digit that
// scans its counts over the tiles, and the scatter.  The two trees of a
// build go through every launch together (blockIdx.y): the launches are
// bound by their latency far more than by the keys they move.
struct SortSet
{
    uint64_t* keys[ 2 ];
    uint32_t* vals[ 2 ];
    uint32_t* hist;   // 256 x tiles
    uint32_t* totals; // 256
};
struct SortSets
{
    SortSet s[ 2 ];
};

__global__ __launch_bounds__( THREADS ) void k_radix_hist( SortSets sets, int from, uint32_t n, int shift, uint32_t numBlocks )
{
    const uint64_t* keys = sets.s[ blockIdx.y ].keys[ from ];
    uint32_t*       hist = sets.s[ blockIdx.y ].hist;
    __shared__ uint32_t cnt[ 256 ];
    cnt[ threadIdx.x ] = 0;
    __syncthreads();
    const uint32_t base = blockIdx.x * RS_TILE;
#pragma unroll
    for( int k = 0; k < RS_ITEMS; k++ )
    {
        const uint32_t i = base + k * THREADS + threadIdx.x;
        if( i < n )
        {
            atomicAdd( &cnt[ uint32_t( keys[ i ] >> shift ) & 255u ], 1u );
        }
    }
    __syncthreads();
    hist[ threadIdx.x * numBlocks + blockIdx.x ] = cnt[ threadIdx.x ];
}

// Inclusive sum over a wave.
__device__ __forceinline__ uint32_t WaveInclusive( uint32_t v, int lane )
{
#pragma unroll
    for( int off = 1; off < 64; off <<= 1 )
    {
        const uint32_t o = __shfl_up( v, off, 64 );
        v += lane >= off ? o : 0u;
    }
    return v;
}

// Exclusive sum over a block of THREADS; *total is the block's sum.
__device__ __forceinline__ uint32_t BlockExclusive( uint32_t v, uint32_t* s_wave, uint32_t* total )
{
    const int      lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t inc  = WaveInclusive( v, lane );
    if( lane == 63 )
    {
        s_wave[ wave ] = inc;
    }
    __syncthreads();
    uint32_t before = 0, sum = 0;
#pragma unroll
    for( int w = 0; w < THREADS / 64; w++ )
    {
        before += w < wave ? s_wave[ w ] : 0u;
        sum += s_wave[ w ];
    }
    __syncthreads();
    *total = sum;
    return before + inc - v;
}

// Block d: the exclusive sums of digit d's counts over the tiles, in place,
// and the digit's total.
__global__ __launch_bounds__( THREADS ) void k_radix_scan( SortSets sets, uint32_t numBlocks )
{
    __shared__ uint32_t s_wave[ THREADS / 64 ];
    uint32_t*           h   = sets.s[ blockIdx.y ].hist + size_t( blockIdx.x ) * numBlocks;
    uint32_t            run = 0;
    for( uint32_t base = 0; base < numBlocks; base += THREADS )
    {
        const uint32_t i = base + threadIdx.x;
        const uint32_t v = i < numBlocks ? h[ i ] : 0u;
        uint32_t       sum;
        const uint32_t ex = BlockExclusive( v, s_wave, &sum );
        if( i < numBlocks )
        {
            h[ i ] = run + ex;
        }
        run += sum;
    }
    if( threadIdx.x == 0 )
    {
        sets.s[ blockIdx.y ].totals[ blockIdx.x ] = run;
    }
}

// Stable scatter.  Each wave owns a run of the tile and ranks its keys item
// by item (64 consecutive keys at a time, equal digits by ballot matching
// over its own counters), so no barrier stands between items; the tile is
// then ordered in LDS and written out digit by digit, in runs.  1M pairs:
// 19 us with one barrier-separated round per 256 keys and scattered stores,
// 11 us like this (24 MB moved).
__global__ __launch_bounds__( THREADS ) void k_radix_scatter( SortSets sets, int from, uint32_t n, int shift, uint32_t numBlocks )
{
    const SortSet&      set     = sets.s[ blockIdx.y ];
    const uint64_t*     keysIn  = set.keys[ from ];
    const uint32_t*     valsIn  = set.vals[ from ];
    uint64_t*           keysOut = set.keys[ from ^ 1 ];
    uint32_t*           valsOut = set.vals[ from ^ 1 ];
    const uint32_t*     offsets = set.hist;
    const uint32_t*     totals  = set.totals;
    constexpr int       WAVES = THREADS / 64;
    __shared__ uint32_t s_cnt[ WAVES ][ 256 ]; // per wave: counts, then first positions in the tile
    __shared__ uint32_t s_out[ 256 ];          // global position of a digit's keys minus their position in the tile
    __shared__ uint32_t s_wave[ WAVES ];
    __shared__ uint64_t s_key[ RS_TILE ];
    __shared__ uint32_t s_val[ RS_TILE ];

    const int      tid    = threadIdx.x;
    const int      lane   = tid & 63;
    const int      wave   = tid >> 6;
    const uint64_t ltMask = ( lane == 0 ) ? 0ull : ( ~0ull >> ( 64 - lane ) );
    const uint32_t tile   = blockIdx.x * RS_TILE;
    const uint32_t here   = n - tile < uint32_t( RS_TILE ) ? n - tile : uint32_t( RS_TILE );

#pragma unroll
    for( int w = 0; w < WAVES; w++ )
    {
        s_cnt[ w ][ tid ] = 0;
    }
    __syncthreads();

    uint32_t* cnt = s_cnt[ wave ];
    uint64_t           key[ RS_ITEMS ];
    uint32_t           val[ RS_ITEMS ], rank[ RS_ITEMS ];
#pragma unroll
    for( int r = 0; r < RS_ITEMS; r++ )
    {
        const uint32_t i = uint32_t( wave * RS_ITEMS + r ) * 64u + lane;
        key[ r ]         = i < here ? keysIn[ tile + i ] : 0ull;
        val[ r ]         = i < here ? valsIn[ tile + i ] : 0u;
    }
#pragma unroll
    for( int r = 0; r < RS_ITEMS; r++ )
    {
        const bool     valid = uint32_t( wave * RS_ITEMS + r ) * 64u + lane < here;
        const uint32_t digit = uint32_t( key[ r ] >> shift ) & 255u;
        uint64_t       peers = __ballot( valid );
#pragma unroll
        for( int b = 0; b < 8; b++ )
        {
            const bool     bit = ( digit >> b ) & 1u;
            const uint64_t m   = __ballot( bit );
            peers &= bit ? m : ~m;
        }
        const uint32_t before = cnt[ digit ];
        const uint32_t lower  = __popcll( peers & ltMask );
        rank[ r ]             = before + lower;
        // every lane has read before the first of its peers counts them
        __builtin_amdgcn_fence( __ATOMIC_ACQ_REL, "wavefront" );
        __builtin_amdgcn_wave_barrier();
        if( valid && lower == 0 )
        {
            cnt[ digit ] = before + __popcll( peers );
        }
        __builtin_amdgcn_fence( __ATOMIC_ACQ_REL, "wavefront" );
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();

    // thread d: digit d's first position in the tile, per wave, and in the output
    uint32_t c[ WAVES ], sum = 0, all;
#pragma unroll
    for( int w = 0; w < WAVES; w++ )
    {
        c[ w ] = s_cnt[ w ][ tid ];
        sum += c[ w ];
    }
    uint32_t       first = BlockExclusive( sum, s_wave, &all );
    const uint32_t start = BlockExclusive( totals[ tid ], s_wave, &all );
    s_out[ tid ]         = start + offsets[ size_t( tid ) * numBlocks + blockIdx.x ] - first;
#pragma unroll
    for( int w = 0; w < WAVES; w++ )
    {
        s_cnt[ w ][ tid ] = first;
        first += c[ w ];
    }
    __syncthreads();
#pragma unroll
    for( int r = 0; r < RS_ITEMS; r++ )
    {
        if( uint32_t( wave * RS_ITEMS + r ) * 64u + lane < here )
        {
            const uint32_t pos = s_cnt[ wave ][ uint32_t( key[ r ] >> shift ) & 255u ] + rank[ r ];
            s_key[ pos ]       = key[ r ];
            s_val[ pos ]       = val[ r ];
        }
    }
    __syncthreads();
#pragma unroll
    for( int r = 0; r < RS_ITEMS; r++ )
    {
        const uint32_t i = r * THREADS + tid;
        if( i < here )
        {
            const uint64_t k   = s_key[ i ];
            const uint32_t out = s_out[ uint32_t( k >> shift ) & 255u ] + i;
            keysOut[ out ]     = k;
            valsOut[ out ]     = s_val[ i ];
        }
    }
}

// ----------------------------------------------------------- hierarchy
// The binary radix tree over the sorted keys (Karras 2012) with its boxes,
// built bottom-up (Apetrei 2014): a subtree over the sorted range [l, r]
// joins its left or its right neighbour, whichever shares the longer key
// prefix with it, and of two siblings the one that is done last makes their
// parent.  Node ids are Karras's: an internal node is the right end of its
// range as a left child, the left end as a right child, 0 as the root;
// leaf k is n - 1 + k.
//
// A block joins what lies within its own run of elements, with the meeting
// points in LDS; the subtrees whose sibling lies outside go to a list, and
// the next launch joins those of BUILD_LISTS lists.  Nothing is exchanged
// between blocks of a launch, so no fence or atomic leaves the CU.  A run is
// cut by at most two root paths, so its list holds at most two subtrees per
// level of the tree (63 key bits and 28 index bits).
// Bound by the latency of a run's climb and the 80 bytes written per node:
// 135 us for 1M triangles in 5 launches, where separate kernels for the
// topology, the depths by pointer jumping, a sort by depth and one union
// launch per level took 345 us in 56.
constexpr uint32_t BUILD_LIST_CAP = 192;
constexpr uint32_t BUILD_LISTS    = 8;

// Length of the prefix that sorted keys i and i + 1 share, equal keys by
// their positions; -1 at the ends.
__device__ __forceinline__ int PrefixAt( const uint64_t* keys, uint32_t n, int64_t i )
{
    if( i < 0 || i + 1 >= int64_t( n ) )
    {
        return -1;
    }
    const uint64_t x = keys[ i ] ^ keys[ i + 1 ];
    return x ? __clzll( x ) : 64 + __clz( uint32_t( i ) ^ uint32_t( i + 1 ) );
}

__device__ __forceinline__ float HalfArea( const float b[ 6 ] )
{
    const float dx = b[ 3 ] - b[ 0 ], dy = b[ 4 ] - b[ 1 ], dz = b[ 5 ] - b[ 2 ];
    return dx * dy + dy * dz + dz * dx;
}

constexpr uint32_t OPEN_BIT = 0x80000000u;

struct TreeArgs
{
    const float*    tris;
    const uint64_t* keys;      // sorted
    const uint32_t* order;     // triangle of each sorted position
    uint32_t        n;
    uint32_t        leafMax;
    uint2*          children;  // per internal node
    uint32_t*       rangeFirst;
    uint32_t*       rangeLast;
    float*          bounds;    // 6 per node, internal then leaves
    uint4*          info;      // per internal node: the collapse's record (below)
    const uint2*    listIn;    // ranges of the subtrees of the launch before
    const uint32_t* countIn;
    uint32_t        lists;
    uint2*          listOut;
    uint32_t*       countOut;
    bool            sizes;     // the low 4 bits of the half areas hold the child's triangle count (at most 15)
};

// LEAVES: the elements are PER * THREADS sorted triangles, else the subtrees
// of BUILD_LISTS lists.  The collapse's record of an internal node: its two
// children, each with OPEN_BIT set when it may be opened (internal, more
// than leafMax triangles), and their half areas (-1 for the others).
struct TreeSets
{
    TreeArgs s[ 2 ];
};
template< bool LEAVES, int PER >
__global__ __launch_bounds__( THREADS ) void k_tree( TreeSets sets )
{
    const TreeArgs&     a = sets.s[ blockIdx.y ];
    constexpr int       CAP = PER * THREADS;
    static_assert( LEAVES || CAP >= int( BUILD_LISTS * BUILD_LIST_CAP ), "element capacity" );
    __shared__ float    s_box[ 6 ][ CAP ];
    __shared__ uint32_t s_first[ LEAVES ? 1 : CAP ], s_last[ LEAVES ? 1 : CAP ];
    __shared__ uint32_t s_meet[ CAP ]; // between elements e and e + 1: 1 + the far end of the subtree that came first
    __shared__ int8_t   s_prefix[ CAP + 1 ];
    __shared__ uint32_t s_wave[ THREADS / 64 ];
    constexpr uint32_t  TAKEN = 0xFFFFFFFFu;

    const uint32_t tid = threadIdx.x, n = a.n, I = a.n - 1;
    uint32_t       count = 0, base = 0;
    if constexpr( LEAVES )
    {
        base  = blockIdx.x * CAP;
        count = n - base < uint32_t( CAP ) ? n - base : uint32_t( CAP );
    }
    else
    {
        for( uint32_t k = 0; k < BUILD_LISTS; k++ )
        {
            const uint32_t list = blockIdx.x * BUILD_LISTS + k;
            const uint32_t c    = list < a.lists ? a.countIn[ list ] : 0u;
            if( tid < c )
            {
                const uint2 rng        = a.listIn[ size_t( list ) * BUILD_LIST_CAP + tid ];
                s_first[ count + tid ] = rng.x;
                s_last[ count + tid ]  = rng.y;
            }
            count += c;
        }
        __syncthreads();
    }
    auto first = [ & ]( uint32_t e ) { return LEAVES ? base + e : s_first[ LEAVES ? 0 : e ]; };
    auto last  = [ & ]( uint32_t e ) { return LEAVES ? base + e : s_last[ LEAVES ? 0 : e ]; };
    for( uint32_t e = tid; e < count; e += THREADS )
    {
        s_prefix[ e ] = int8_t( PrefixAt( a.keys, n, int64_t( first( e ) ) - 1 ) );
        s_meet[ e ]   = 0u;
    }
    if( tid == 0 )
    {
        s_prefix[ count ] = int8_t( PrefixAt( a.keys, n, last( count - 1 ) ) );
    }
    __syncthreads();

    // the subtrees at the run's ends (one at either at most): [endA, count) and [0, startB]
    constexpr uint32_t NONE = 0xFFFFFFFFu;
    uint32_t           endA = NONE, startB = NONE;
    for( uint32_t e = tid; e < count; e += THREADS )
    {
        uint32_t A = e, B = e; // the subtree's elements
        float    box[ 6 ];
        if constexpr( LEAVES )
        {
            v3 p, q, r;
            LoadTri( a.tris, a.order[ base + e ], p, q, r );
            const v3 lo = vmin( vmin( p, q ), r ), hi = vmax( vmax( p, q ), r );
            box[ 0 ] = lo.x, box[ 1 ] = lo.y, box[ 2 ] = lo.z, box[ 3 ] = hi.x, box[ 4 ] = hi.y, box[ 5 ] = hi.z;
            float2* o = reinterpret_cast< float2* >( a.bounds + ( size_t( I ) + base + e ) * 6 );
            o[ 0 ]    = make_float2( box[ 0 ], box[ 1 ] );
            o[ 1 ]    = make_float2( box[ 2 ], box[ 3 ] );
            o[ 2 ]    = make_float2( box[ 4 ], box[ 5 ] );
        }
        else
        {
            const uint32_t l = first( e ), r = last( e );
            const uint32_t id = l == r ? I + l : ( s_prefix[ e + 1 ] > s_prefix[ e ] ? r : l );
            const float2*  o  = reinterpret_cast< const float2* >( a.bounds + size_t( id ) * 6 );
            const float2   x = o[ 0 ], y = o[ 1 ], z = o[ 2 ];
            box[ 0 ] = x.x, box[ 1 ] = x.y, box[ 2 ] = y.x, box[ 3 ] = y.y, box[ 4 ] = z.x, box[ 5 ] = z.y;
        }
        while( true )
        {
            const int before = s_prefix[ A ], after = s_prefix[ B + 1 ];
            if( before < 0 && after < 0 )
            {
                break; // the whole tree
            }
            const bool left = after > before;
            if( left ? B + 1 == count : A == 0 )
            {
                if( left )
                {
                    endA = A;
                }
                else
                {
                    startB = B;
                }
                break; // its sibling is not in this run
            }
            const uint32_t at = left ? B : A; // where this subtree's box is kept; the sibling's is next to it
#pragma unroll
            for( int k = 0; k < 6; k++ )
            {
                s_box[ k ][ at ] = box[ k ];
            }
            __builtin_amdgcn_fence( __ATOMIC_RELEASE, "workgroup" );
            const uint32_t meet = left ? B : A - 1;
            const uint32_t far  = __hip_atomic_exchange( &s_meet[ meet ], 1u + ( left ? A : B ), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP );
            if( far == 0u )
            {
                break; // the sibling goes on from here
            }
            __builtin_amdgcn_fence( __ATOMIC_ACQUIRE, "workgroup" );
            s_meet[ meet ]    = TAKEN;
            const uint32_t sA = left ? B + 1 : far - 1, sB = left ? far - 1 : A - 1;
            const uint32_t sat = left ? sA : sB;
            float          sib[ 6 ];
#pragma unroll
            for( int k = 0; k < 6; k++ )
            {
                sib[ k ] = s_box[ k ][ sat ];
            }
            // the children in order
            const uint32_t lA = left ? A : sA, lB = left ? B : sB, rA = left ? sA : A, rB = left ? sB : B;
            const uint32_t lf = first( lA ), ll = last( lB ), rf = first( rA ), rl = last( rB );
            const uint32_t lid = lf == ll ? I + lf : ll, rid = rf == rl ? I + rf : rf;
            const bool     lo = lf != ll && ll - lf + 1u > a.leafMax, ro = rf != rl && rl - rf + 1u > a.leafMax;
            const float    areaOwn = HalfArea( box ), areaSib = HalfArea( sib );
            float          la = lo ? ( left ? areaOwn : areaSib ) : -1.0f, ra = ro ? ( left ? areaSib : areaOwn ) : -1.0f;
            if( a.sizes )
            {
                // (an infinite area with these bits would be a NaN, which is never opened)
                la = lo ? __uint_as_float( ( __float_as_uint( fminf( la, FLT_MAX ) ) & ~15u ) | min( ll - lf + 1u, 15u ) ) : la;
                ra = ro ? __uint_as_float( ( __float_as_uint( fminf( ra, FLT_MAX ) ) & ~15u ) | min( rl - rf + 1u, 15u ) ) : ra;
            }
#pragma unroll
            for( int k = 0; k < 3; k++ )
            {
                const float x = left ? box[ k ] : sib[ k ], y = left ? sib[ k ] : box[ k ];
                const float z = left ? box[ 3 + k ] : sib[ 3 + k ], w = left ? sib[ 3 + k ] : box[ 3 + k ];
                box[ k ]      = fminf( x, y );
                box[ 3 + k ]  = fmaxf( z, w );
            }
            A = lA;
            B = rB;
            const int      pb = s_prefix[ A ], pa = s_prefix[ B + 1 ];
            const uint32_t id = pb < 0 && pa < 0 ? 0u : ( pa > pb ? rl : lf );
            a.children[ id ]   = make_uint2( lid, rid );
            a.rangeFirst[ id ] = lf;
            a.rangeLast[ id ]  = rl;
            float2* o          = reinterpret_cast< float2* >( a.bounds + size_t( id ) * 6 );
            o[ 0 ]             = make_float2( box[ 0 ], box[ 1 ] );
            o[ 1 ]             = make_float2( box[ 2 ], box[ 3 ] );
            o[ 2 ]             = make_float2( box[ 4 ], box[ 5 ] );
            a.info[ id ] = make_uint4( lid | ( lo ? OPEN_BIT : 0u ), rid | ( ro ? OPEN_BIT : 0u ), __float_as_uint( la ), __float_as_uint( ra ) );
        }
    }
    __syncthreads();
    if( gridDim.x == 1 )
    {
        return; // one run: the tree is whole
    }

    // The list of this run's subtrees, in order: s_meet becomes, per element,
    // 1 + the last element of the subtree that starts there (0: none).
    uint32_t seen[ PER ];
#pragma unroll
    for( int k = 0; k < PER; k++ )
    {
        const uint32_t e = k * THREADS + tid;
        seen[ k ]        = e < count ? s_meet[ e ] : 0u;
    }
    __syncthreads();
#pragma unroll
    for( int k = 0; k < PER; k++ )
    {
        s_meet[ k * THREADS + tid ] = 0u;
    }
    __syncthreads();
#pragma unroll
    for( int k = 0; k < PER; k++ )
    {
        const uint32_t e = k * THREADS + tid;
        if( seen[ k ] != 0u && seen[ k ] != TAKEN )
        {
            // nobody came to meet it: a left child [far, e] or a right child [e + 1, far]
            const uint32_t far                    = seen[ k ] - 1u;
            s_meet[ far <= e ? far : e + 1u ] = 1u + ( far <= e ? e : far );
        }
    }
    if( endA != NONE )
    {
        s_meet[ endA ] = count;
    }
    if( startB != NONE )
    {
        s_meet[ 0 ] = 1u + startB;
    }
    __syncthreads();
    uint32_t mine = 0;
#pragma unroll
    for( int k = 0; k < PER; k++ )
    {
        mine += s_meet[ tid * PER + k ] != 0u ? 1u : 0u;
    }
    uint32_t total;
    uint32_t pos = BlockExclusive( mine, s_wave, &total );
#pragma unroll
    for( int k = 0; k < PER; k++ )
    {
        const uint32_t e = tid * PER + k, end = s_meet[ e ];
        if( end != 0u )
        {
            if( pos < BUILD_LIST_CAP )
            {
                a.listOut[ size_t( blockIdx.x ) * BUILD_LIST_CAP + pos ] = make_uint2( first( e ), last( end - 1u ) );
            }
            pos++;
        }
    }
    if( tid == 0 )
    {
        a.countOut[ blockIdx.x ] = total < BUILD_LIST_CAP ? total : BUILD_LIST_CAP;
    }
}

// ------------------------------------------------------------ collapse

__device__ __forceinline__ uint32_t NodeCount( uint32_t id, uint32_t n, const uint32_t* rf, const uint32_t* rl )
{
    return id >= n - 1 ? 1u : rl[ id ] - rf[ id ] + 1u;
}

// Expands binary node b into up to 8 children by repeatedly opening the
// child with the largest surface area (first one on ties) among those that
// are internal and hold more than leafMax triangles.  Level by level: the
// nodes of this level are queue[levelBase[0] ..  + levelCount[0]), the next
// level's follow them, each wave taking room for its nodes with one atomic
// (one per child on a single address took 131 and 197 us for the two widest
// levels of a 1M-triangle build).
struct CollapseArgs
{
    uint32_t*       queue;
    uint32_t*       levelBase;
    uint32_t*       levelCount;
    uint32_t        n;
    uint32_t        leafMax;
    const uint4*    info;
    const uint32_t* rf;
    const uint32_t* rl;
    uint32_t*       expansion;
    uint32_t*       isNode8;   // published tree: marks, by binary node
    uint2*          nodeBase;  // traversal's tree: first child node and first triangle of each node
    uint32_t*       triCount;
};
struct CollapseSets
{
    CollapseArgs s[ 2 ];
};

__global__ __launch_bounds__( THREADS ) void k_collapse_level( CollapseSets sets, uint32_t level )
{
    const CollapseArgs& a          = sets.s[ blockIdx.y ];
    uint32_t* const     queue      = a.queue;
    uint32_t* const     levelBase  = a.levelBase + level;
    uint32_t* const     levelCount = a.levelCount + level;
    const uint32_t      n = a.n, leafMax = a.leafMax;
    const uint4* const  info = a.info;
    const uint32_t count = levelCount[ 0 ], first = levelBase[ 0 ];
    const int      lane  = threadIdx.x & 63;
    if( blockIdx.x == 0 && threadIdx.x == 0 )
    {
        levelBase[ 1 ] = first + count;
    }
    // whole waves stay in the loop, for the sums over their lanes
    for( uint32_t w = ( blockIdx.x * THREADS + threadIdx.x ) & ~63u; w < count; w += gridDim.x * THREADS )
    {
        const uint32_t t    = w + lane;
        const bool     have = t < count;
        const uint32_t b    = have ? queue[ first + t ] : 0u;
        // The node's children so far, each with whether it may be opened
        // (internal, more than leafMax triangles) and its half area.  Every
        // index into these arrays is a compile-time constant (the loops are
        // unrolled and the updates predicated), so they stay in registers.
        uint32_t ch[ 8 ];
        float    ar[ 8 ];
        bool     ex[ 8 ];
#pragma unroll
        for( int k = 0; k < 8; k++ )
        {
            ch[ k ] = 0xFFFFFFFFu;
            ar[ k ] = -1.0f;
            ex[ k ] = false;
        }
        int nch = 0;
        if( !have )
        {
        }
        else if( b >= n - 1 || NodeCount( b, n, a.rf, a.rl ) <= leafMax )
        {
            ch[ 0 ] = b; // a root that is small enough is a single leaf
            nch     = 1;
        }
        else
        {
            const uint4 q = info[ b ];
            ch[ 0 ]       = q.x & ~OPEN_BIT;
            ch[ 1 ]       = q.y & ~OPEN_BIT;
            ex[ 0 ]       = ( q.x & OPEN_BIT ) != 0u;
            ex[ 1 ]       = ( q.y & OPEN_BIT ) != 0u;
            ar[ 0 ]       = __uint_as_float( q.z );
            ar[ 1 ]       = __uint_as_float( q.w );
            nch           = 2;
            while( nch < 8 )
            {
                // the first child of largest area among those that open
                int   best     = -1;
                float bestArea = -1.0f;
                if( !a.nodeBase )
                {
#pragma unroll
                    for( int k = 0; k < 8; k++ )
                    {
                        if( k < nch && ex[ k ] && ar[ k ] > bestArea )
                        {
                            bestArea = ar[ k ];
                            best     = k;
                        }
                    }
                }
                else
                {
                    // The traversal's tree: a subtree of at most 8 triangles is
                    // opened last, and only where there is room for all of
                    // it: else it is a node of its own.  As many visits per
                    // ray as by area alone, in 198k nodes of 6.1 children
                    // where area alone leaves 364k of 3.7 (1M triangles).
                    int   small = -1;
                    float smallArea = -1.0f;
#pragma unroll
                    for( int k = 0; k < 8; k++ )
                    {
                        const int size = int( __float_as_uint( ar[ k ] ) & 15u );
                        const bool may = k < nch && ex[ k ];
                        if( may && size > 8 && ar[ k ] > bestArea )
                        {
                            bestArea = ar[ k ];
                            best     = k;
                        }
                        if( may && size - 1 <= 8 - nch && ar[ k ] > smallArea )
                        {
                            smallArea = ar[ k ];
                            small     = k;
                        }
                    }
                    best = best >= 0 ? best : small;
                }
                if( best < 0 )
                {
                    break;
                }
                uint32_t c = 0;
#pragma unroll
                for( int k = 0; k < 8; k++ )
                {
                    c = k == best ? ch[ k ] : c;
                }
                const uint4    q   = info[ c ];
                const uint32_t l   = q.x & ~OPEN_BIT, r = q.y & ~OPEN_BIT;
                const bool     el  = ( q.x & OPEN_BIT ) != 0u, er = ( q.y & OPEN_BIT ) != 0u;
                const float    al  = __uint_as_float( q.z ), arr = __uint_as_float( q.w );
                // ch[best + 2 ..] = old ch[best + 1 .. nch - 1]; then the two
                // children take slots best and best + 1
#pragma unroll
                for( int k = 7; k >= 1; k-- )
                {
                    if( k <= nch && k > best + 1 )
                    {
                        ch[ k ] = ch[ k - 1 ];
                        ar[ k ] = ar[ k - 1 ];
                        ex[ k ] = ex[ k - 1 ];
                    }
                }
#pragma unroll
                for( int k = 0; k < 8; k++ )
                {
                    if( k == best )
                    {
                        ch[ k ] = l;
                        ar[ k ] = al;
                        ex[ k ] = el;
                    }
                    else if( k == best + 1 )
                    {
                        ch[ k ] = r;
                        ar[ k ] = arr;
                        ex[ k ] = er;
                    }
                }
                nch++;
            }
        }
        if( have )
        {
            uint32_t out[ 8 ];
#pragma unroll
            for( int k = 0; k < 8; k++ )
            {
                out[ k ] = k < nch ? ( ch[ k ] | ( ex[ k ] ? OPEN_BIT : 0u ) ) : 0xFFFFFFFFu;
            }
            uint4* e = reinterpret_cast< uint4* >( a.expansion ) + size_t( first + t ) * 2;
            e[ 0 ]   = make_uint4( out[ 0 ], out[ 1 ], out[ 2 ], out[ 3 ] );
            e[ 1 ]   = make_uint4( out[ 4 ], out[ 5 ], out[ 6 ], out[ 7 ] );
            if( a.isNode8 )
            {
                a.isNode8[ b < n - 1 ? b : 0 ] = 1u;
            }
        }
        uint32_t kids = 0;
#pragma unroll
        for( int k = 0; k < 8; k++ )
        {
            kids += k < nch && ex[ k ] ? 1u : 0u;
        }
        // child nodes in the low half, leaf children in the high half
        const uint32_t own  = kids | ( uint32_t( nch ) - kids ) << 16;
        const uint32_t inc  = WaveInclusive( own, lane );
        uint32_t       base = 0, tri = 0;
        if( lane == 63 )
        {
            if( ( inc & 0xFFFFu ) != 0u )
            {
                base = atomicAdd( levelCount + 1, inc & 0xFFFFu );
            }
            if( a.nodeBase && ( inc >> 16 ) != 0u )
            {
                tri = atomicAdd( a.triCount, inc >> 16 );
            }
        }
        uint32_t pos = first + count + __shfl( base, 63, 64 ) + ( ( inc - own ) & 0xFFFFu );
        if( a.nodeBase )
        {
            tri = __shfl( tri, 63, 64 ) + ( ( inc - own ) >> 16 );
            if( have )
            {
                a.nodeBase[ first + t ] = make_uint2( pos, tri );
            }
        }
#pragma unroll
        for( int k = 0; k < 8; k++ )
        {
            if( k < nch && ex[ k ] )
            {
                queue[ pos++ ] = ch[ k ];
            }
        }
    }
}

__device__ __forceinline__ uint32_t LeafRef( uint32_t first, uint32_t count )
{
    return RG_EXT_BVH_CHILD_LEAF_BIT | ( first << 3 ) | ( count - 1u );
}

__global__ __launch_bounds__( THREADS ) void k_write_nodes( uint32_t        count,
                                                            uint32_t        n,
                                                            const uint32_t* queue,
                                                            const uint32_t* node8Index,
                                                            const uint32_t* expansion,
                                                            const uint32_t* rf,
                                                            const uint32_t* rl,
                                                            const float*    bounds,
                                                            BvhNode8*       nodes )
{
    // one thread per (node of the collapse's queue, child): the 8 threads of
    // a node write its SoA arrays as contiguous 32-byte runs
    const uint64_t t = uint64_t( blockIdx.x ) * THREADS + threadIdx.x;
    const uint32_t q = uint32_t( t >> 3 );
    const int      k = int( t & 7u );
    if( q >= count )
    {
        return;
    }
    const uint32_t b    = queue[ q ];
    BvhNode8&      node = nodes[ node8Index[ b < n - 1 ? b : 0 ] ];
    const uint32_t e    = expansion[ t ];
    if( e == 0xFFFFFFFFu )
    {
        node.lo_x[ k ] = node.lo_y[ k ] = node.lo_z[ k ] = INFINITY;
        node.hi_x[ k ] = node.hi_y[ k ] = node.hi_z[ k ] = -INFINITY;
        node.child[ k ] = RG_EXT_BVH_CHILD_EMPTY;
        node.pad[ k ]   = 0;
        return;
    }
    const uint32_t c  = e & ~OPEN_BIT;
    const float2*  bb = reinterpret_cast< const float2* >( bounds + size_t( c ) * 6 );
    const float2   x = bb[ 0 ], y = bb[ 1 ], z = bb[ 2 ];
    node.lo_x[ k ]  = x.x;
    node.lo_y[ k ]  = x.y;
    node.lo_z[ k ]  = y.x;
    node.hi_x[ k ]  = y.y;
    node.hi_y[ k ]  = z.x;
    node.hi_z[ k ]  = z.y;
    node.pad[ k ]   = 0;
    node.child[ k ] = e & OPEN_BIT ? node8Index[ c ] : ( c >= n - 1 ? LeafRef( c - ( n - 1 ), 1 ) : LeafRef( rf[ c ], rl[ c ] - rf[ c ] + 1u ) );
}

// Outward rounding to half: the half nearest to v - origin, stepped down
// (lo) or up (hi) until origin + float(h), in FP32, is on the outside of v.
__device__ __forceinline__ uint16_t HalfBitsOf( _Float16 h )
{
    return __builtin_bit_cast( uint16_t, h );
}
__device__ __forceinline__ _Float16 HalfOfBits( uint16_t b )
{
    return __builtin_bit_cast( _Float16, b );
}
__device__ _Float16 HalfStep( _Float16 h, bool up )
{
    const uint16_t b = HalfBitsOf( h );
    if( ( b & 0x7C00u ) == 0x7C00u )
    {
        return h; // inf (or NaN) stays
    }
    if( ( b & 0x7FFFu ) == 0u )
    {
        return HalfOfBits( up ? 0x0001u : 0x8001u ); // +-0 -> smallest subnormal
    }
    const bool neg = ( b & 0x8000u ) != 0u;
    return HalfOfBits( uint16_t( ( neg != up ) ? b + 1u : b - 1u ) );
}
__device__ uint16_t EncodeOffset( float v, float origin, bool up )
{
    _Float16 h = _Float16( v - origin );
    if( !up && HalfBitsOf( h ) == 0x7C00u )
    {
        h = HalfOfBits( 0x7BFFu ); // beyond the half range: the largest finite offset is still below v
    }
    for( int i = 0; i < 64; i++ )
    {
        const float d = origin + float( h );
        if( up ? !( d < v ) : !( d > v ) )
        {
            break;
        }
        h = HalfStep( h, up );
    }
    return HalfBitsOf( h );
}

__global__ __launch_bounds__( THREADS ) void k_half_nodes( const BvhNode8* in, uint32_t count, BvhNode8H* out )
{
    const uint32_t i = blockIdx.x * THREADS + threadIdx.x;
    if( i >= count )
    {
        return;
    }
    const BvhNode8& a = in[ i ];
    BvhNode8H       h;
    float           o[ 3 ] = { INFINITY, INFINITY, INFINITY };
    for( int k = 0; k < 8; k++ )
    {
        if( a.child[ k ] != RG_EXT_BVH_CHILD_EMPTY )
        {
            o[ 0 ] = fminf( o[ 0 ], a.lo_x[ k ] );
            o[ 1 ] = fminf( o[ 1 ], a.lo_y[ k ] );
            o[ 2 ] = fminf( o[ 2 ], a.lo_z[ k ] );
        }
    }
    for( int c = 0; c < 3; c++ )
    {
        h.origin[ c ] = o[ c ] < INFINITY ? o[ c ] : 0.0f;
    }
    h.pad = 0;
    for( int k = 0; k < 8; k++ )
    {
        h.child[ k ] = a.child[ k ];
        if( a.child[ k ] == RG_EXT_BVH_CHILD_EMPTY )
        {
            h.lo_x[ k ] = h.lo_y[ k ] = h.lo_z[ k ] = 0x7C00u; // +inf
            h.hi_x[ k ] = h.hi_y[ k ] = h.hi_z[ k ] = 0xFC00u; // -inf
            continue;
        }
        h.lo_x[ k ] = EncodeOffset( a.lo_x[ k ], h.origin[ 0 ], false );
        h.lo_y[ k ] = EncodeOffset( a.lo_y[ k ], h.origin[ 1 ], false );
        h.lo_z[ k ] = EncodeOffset( a.lo_z[ k ], h.origin[ 2 ], false );
        h.hi_x[ k ] = EncodeOffset( a.hi_x[ k ], h.origin[ 0 ], true );
        h.hi_y[ k ] = EncodeOffset( a.hi_y[ k ], h.origin[ 1 ], true );
        h.hi_z[ k ] = EncodeOffset( a.hi_z[ k ], h.origin[ 2 ], true );
    }
    out[ i ] = h;
}

__global__ __launch_bounds__( THREADS ) void k_sorted_tris( const float* tris, const uint32_t* sortedIdx, uint32_t n, float4* out )
{
    const uint32_t k = blockIdx.x * THREADS + threadIdx.x;
    if( k >= n )
    {
        return;
    }
    const uint32_t id = sortedIdx[ k ];
    v3             a, b, c;
    LoadTri( tris, id, a, b, c );
    out[ size_t( k ) * 3 + 0 ] = make_float4( a.x, a.y, a.z, __uint_as_float( id ) );
    out[ size_t( k ) * 3 + 1 ] = make_float4( b.x, b.y, b.z, 0.0f );
    out[ size_t( k ) * 3 + 2 ] = make_float4( c.x, c.y, c.z, 0.0f );
}

// ----------------------------------------------------- traversal nodes

// Box planes of an axis as whole numbers: scale 2^k and origin such that
// origin + q * 2^k, q in 0..GRID_MAX, covers [lo, hi] with room to spare; 2^k
// is no finer than four units in the last place of the coordinates, so that
// the origin, half a step below lo and rounded to float, stays below it.  An
// axis whose box is not finite gets an infinite scale and zeros: the
// traversal's distances are then NaN, which its min / max leave out.
constexpr double GRID_MAX  = 2047.0;
constexpr double GRID_SPAN = 2040.0;
struct AxisGrid
{
    float    origin;
    uint32_t exponent; // of the scale, biased as in a float
};
__device__ __forceinline__ AxisGrid MakeGrid( float lo, float hi )
{
    AxisGrid     g;
    const double ext = double( hi ) - double( lo ), big = fmax( fabs( double( lo ) ), fabs( double( hi ) ) );
    if( !( ext >= 0.0 && big < 1e36 ) )
    {
        g.origin   = 0.0f;
        g.exponent = 255u;
        return g;
    }
    int k = ext > 0.0 ? ilogb( ext / GRID_SPAN ) : -126;
    k     = ext > 0.0 && ldexp( GRID_SPAN, k ) < ext ? k + 1 : k;
    const int fine = big > 0.0 ? ilogb( big ) - 21 : -126;
    k              = k < fine ? fine : k;
    k              = k < -126 ? -126 : k;
    g.origin       = float( double( lo ) - ldexp( 0.5, k ) );
    g.exponent     = uint32_t( k + 127 );
    return g;
}
// The plane below lo or above hi.  The traversal evaluates
// fma(q, 2^k / d, (origin - o) / d) with up to 2^-10 steps of rounding error
// beyond a relative one of its second term, which it covers itself; 2^-9 steps
// of margin cover the steps.
__device__ __forceinline__ uint16_t GridBits( double q )
{
    return __builtin_bit_cast( uint16_t, _Float16( float( q ) ) ); // whole and at most 2047: exact
}
__device__ __forceinline__ uint16_t GridLo( const AxisGrid& g, float v )
{
    if( g.exponent == 255u )
    {
        return 0u;
    }
    const double q = floor( ldexp( double( v ) - double( g.origin ), 127 - int( g.exponent ) ) - 0x1p-9 );
    return GridBits( q > 0.0 ? fmin( q, GRID_MAX ) : 0.0 ); // NaN: 0
}
__device__ __forceinline__ uint16_t GridHi( const AxisGrid& g, float v )
{
    if( g.exponent == 255u )
    {
        return 0u;
    }
    const double q = ceil( ldexp( double( v ) - double( g.origin ), 127 - int( g.exponent ) ) + 0x1p-9 );
    return GridBits( q < GRID_MAX ? fmax( q, 0.0 ) : GRID_MAX ); // NaN: the largest
}

// One traversal node per node of the collapse's queue, eight lanes a node
// (one per child), and its leaves' triangles side by side.
__global__ __launch_bounds__( THREADS ) void k_pack_nodes( uint32_t count, uint32_t n, const uint32_t* expansion, const uint2* nodeBase,
                                                           const float* bounds, const uint32_t* order, const float* tris, BvhNodeQ* nodes,
                                                           float4* nodeTris )
{
    const uint64_t t    = uint64_t( blockIdx.x ) * THREADS + threadIdx.x;
    const uint32_t q    = uint32_t( t >> 3 );
    const bool     have = q < count;
    const uint32_t e    = have ? expansion[ t ] : 0xFFFFFFFFu;
    const bool     full = e != 0xFFFFFFFFu, inner = full && ( e & OPEN_BIT ) != 0u;
    const uint32_t c    = e & ~OPEN_BIT;
    const int      lane = threadIdx.x & 63, first = lane & ~7;

    float lo[ 3 ] = { INFINITY, INFINITY, INFINITY }, hi[ 3 ] = { -INFINITY, -INFINITY, -INFINITY };
    if( full )
    {
        const float2* bb = reinterpret_cast< const float2* >( bounds + size_t( c ) * 6 );
        const float2  x = bb[ 0 ], y = bb[ 1 ], z = bb[ 2 ];
        lo[ 0 ] = x.x, lo[ 1 ] = x.y, lo[ 2 ] = y.x, hi[ 0 ] = y.y, hi[ 1 ] = z.x, hi[ 2 ] = z.y;
    }
    const uint32_t inMask   = uint32_t( __ballot( inner ) >> first ) & 0xFFu;
    const uint32_t leafMask = uint32_t( __ballot( full && !inner ) >> first ) & 0xFFu;
    const uint32_t below    = ( 1u << ( lane & 7 ) ) - 1u;
    const uint32_t inner8 = __popc( inMask ), leaf8 = __popc( leafMask );
    // child nodes take the first slots, leaves the next ones
    const uint32_t slot = inner ? __popc( inMask & below ) : ( full ? inner8 + __popc( leafMask & below ) : inner8 + leaf8 + __popc( ~( inMask | leafMask ) & below ) );
    AxisGrid       g[ 3 ];
#pragma unroll
    for( int ax = 0; ax < 3; ax++ )
    {
        float l = lo[ ax ], h = hi[ ax ];
#pragma unroll
        for( int m = 1; m < 8; m <<= 1 )
        {
            l = fminf( l, __shfl_xor( l, m, 64 ) );
            h = fmaxf( h, __shfl_xor( h, m, 64 ) );
        }
        g[ ax ] = MakeGrid( l, h );
    }
    if( !have )
    {
        return;
    }
    BvhNodeQ&   node = nodes[ q ];
    const uint2 base = nodeBase[ q ];
#pragma unroll
    for( int ax = 0; ax < 3; ax++ )
    {
        node.planes[ ax ][ 0 ][ slot ] = full ? GridLo( g[ ax ], lo[ ax ] ) : GridBits( GRID_MAX );
        node.planes[ ax ][ 1 ][ slot ] = full ? GridHi( g[ ax ], hi[ ax ] ) : GridBits( 0.0 );
    }
    if( ( lane & 7 ) == 0 )
    {
        node.origin[ 0 ] = g[ 0 ].origin;
        node.origin[ 1 ] = g[ 1 ].origin;
        node.origin[ 2 ] = g[ 2 ].origin;
        node.meta        = g[ 0 ].exponent | g[ 1 ].exponent << 8 | g[ 2 ].exponent << 16 | inner8 << 24 | leaf8 << 28;
        node.childBase   = base.x;
        node.triBase     = base.y - inner8; // leaf slot s holds triangle triBase + s
        node.pad[ 0 ] = node.pad[ 1 ] = 0u;
    }
    if( full && !inner )
    {
        const uint32_t id = order[ c - ( n - 1 ) ];
        v3             v0, v1, v2;
        LoadTri( tris, id, v0, v1, v2 );
        float4* o = nodeTris + size_t( base.y + slot - inner8 ) * 3;
        o[ 0 ]    = make_float4( v0.x, v0.y, v0.z, __uint_as_float( id ) );
        o[ 1 ]    = make_float4( v1.x, v1.y, v1.z, 0.0f );
        o[ 2 ]    = make_float4( v2.x, v2.y, v2.z, 0.0f );
    }
}

__global__ void k_seed_frontier( CollapseSets sets, uint32_t count )
{
    if( threadIdx.x < count )
    {
        sets.s[ threadIdx.x ].queue[ 0 ]      = 0;
        sets.s[ threadIdx.x ].levelCount[ 0 ] = 1;
    }
}

} // namespace

namespace
{
// Stable sort of n (key, value) pairs of `count` sets by key bits [0, 64):
// an even number of passes, so the result is where the input was.
void RadixSort( const SortSets& sets, uint32_t count, uint32_t n, hipStream_t stream )
{
    const uint32_t blocks = DivUp( n, RS_TILE );
    for( int pass = 0; pass < 8; pass++ )
    {
        const int from = pass & 1, shift = pass * 8;
        k_radix_hist<<< dim3( blocks, count ), THREADS, 0, stream >>>( sets, from, n, shift, blocks );
        CheckLaunch( "k_radix_hist" );
        k_radix_scan<<< dim3( 256, count ), THREADS, 0, stream >>>( sets, blocks );
        CheckLaunch( "k_radix_scan" );
        k_radix_scatter<<< dim3( blocks, count ), THREADS, 0, stream >>>( sets, from, n, shift, blocks );
        CheckLaunch( "k_radix_scatter" );
    }
}

// Runs of the hierarchy's first launch: 256 triangles while that fills the
// chip with blocks, 1024 (and a quarter of the subtrees left over) beyond.
constexpr uint32_t TREE_RUN_SMALL = THREADS, TREE_RUN = 4 * THREADS;
constexpr uint32_t TREE_SMALL     = 128 * TREE_RUN_SMALL;

uint32_t TreeRuns( uint32_t n )
{
    return n <= TREE_SMALL ? DivUp( n, TREE_RUN_SMALL ) : DivUp( n, TREE_RUN );
}

// Two sets of lists (the first launch's and the second's) and their counts.
size_t TreeListBytes( uint32_t n )
{
    const size_t runs = TreeRuns( n ), next = DivUp( runs, BUILD_LISTS );
    return ( runs + next ) * ( BUILD_LIST_CAP * sizeof( uint2 ) + sizeof( uint32_t ) );
}

void BuildTree( TreeSets a, uint2* const lists[ 2 ], uint32_t count, hipStream_t stream )
{
    const uint32_t n    = a.s[ 0 ].n;
    uint32_t       runs = TreeRuns( n );
    const uint32_t first = runs, next = DivUp( runs, BUILD_LISTS );
    auto           point = [ & ]( bool flip, bool in ) {
        for( uint32_t k = 0; k < count; k++ )
        {
            uint2*    listA = lists[ k ];
            uint2*    listB = listA + size_t( first ) * BUILD_LIST_CAP;
            uint32_t* cntA  = reinterpret_cast< uint32_t* >( listB + size_t( next ) * BUILD_LIST_CAP );
            uint32_t* cntB  = cntA + first;
            if( in )
            {
                a.s[ k ].listIn  = flip ? listB : listA;
                a.s[ k ].countIn = flip ? cntB : cntA;
            }
            else
            {
                a.s[ k ].listOut  = flip ? listB : listA;
                a.s[ k ].countOut = flip ? cntB : cntA;
            }
        }
    };
    bool flip = false;
    point( flip, false );
    if( n <= TREE_SMALL )
    {
        k_tree< true, 1 ><<< dim3( runs, count ), THREADS, 0, stream >>>( a );
    }
    else
    {
        k_tree< true, 4 ><<< dim3( runs, count ), THREADS, 0, stream >>>( a );
    }
    CheckLaunch( "k_tree" );
    while( runs > 1 )
    {
        point( flip, true );
        flip = !flip;
        point( flip, false );
        for( uint32_t k = 0; k < count; k++ )
        {
            a.s[ k ].lists = runs;
        }
        runs = DivUp( runs, BUILD_LISTS );
        k_tree< false, int( BUILD_LISTS * BUILD_LIST_CAP / THREADS ) ><<< dim3( runs, count ), THREADS, 0, stream >>>( a );
        CheckLaunch( "k_tree" );
    }
}

// Carves aligned arrays out of one allocation.
struct Carver
{
    char*  base = nullptr;
    size_t used = 0;
    template< typename T >
    T* Take( size_t count )
    {
        T* p = base ? reinterpret_cast< T* >( base + used ) : nullptr;
        used += ( count * sizeof( T ) + 255 ) & ~size_t( 255 );
        return p;
    }
};

// Scratch of the traversal's tree.  What the nodes' launch (k_pack_nodes) no
// longer reads lies in its output buffer, nodeTris, and with a published tree
// the boxes lie in sortedTris, which is written last: 63 bytes a triangle are
// left of 155, and a published BVH of 1M triangles with 3 a leaf takes 390 in
// all, not 482.
struct TreeScratch
{
    uint64_t *keys0, *keys1;
    uint32_t *vals0, *vals1, *hist;
    uint2*    children;
    uint32_t *rf, *rl;
    float*    bounds;
    uint4*    info;
    uint2*    lists;
    uint32_t *expansion, *queue;
    uint2*    nodeBase;
    uint32_t* roots;
    float*    boxes;
    uint32_t* levels; // per set: nodes of each level, then its first node; one more word for the triangle count
    size_t    bytes;      // of base
    size_t    earlyBytes; // of nodeTris, which its own contents may exceed

    TreeScratch( char* base, char* nodeTris, float* sortedTris, bool view, uint32_t n, uint32_t sceneCount )
    {
        const size_t slots = n > 1 ? n - 1 : 1;
        Carver       e{ nodeTris };
        keys0      = e.Take< uint64_t >( n );
        keys1      = e.Take< uint64_t >( n );
        vals1      = e.Take< uint32_t >( n );
        rf         = e.Take< uint32_t >( slots );
        rl         = e.Take< uint32_t >( slots );
        info       = e.Take< uint4 >( slots );
        earlyBytes = e.used;
        Carver c{ base };
        vals0      = c.Take< uint32_t >( n );
        hist       = c.Take< uint32_t >( size_t( 256 ) * ( DivUp( n, RS_TILE ) + 1 ) );
        children   = c.Take< uint2 >( slots );
        bounds     = view ? sortedTris : c.Take< float >( ( 2 * size_t( n ) - 1 ) * 6 ); // 48 n - 24 bytes
        lists      = c.Take< uint2 >( TreeListBytes( n ) / sizeof( uint2 ) + 1 );
        expansion  = c.Take< uint32_t >( ( slots + sceneCount ) * 8 ); // one-triangle scenes have nodes of their own
        queue      = c.Take< uint32_t >( slots + sceneCount );
        nodeBase   = c.Take< uint2 >( slots + sceneCount );
        roots      = c.Take< uint32_t >( sceneCount + 1 );
        boxes      = c.Take< float >( size_t( sceneCount + 1 ) * 8 );
        levels     = c.Take< uint32_t >( LEVEL_WORDS * 2 + 1 );
        bytes      = c.used;
    }
    static constexpr uint32_t LEVEL_WORDS = ( BVH_MAX_LEVELS + 1 ) * 2;
};

// Builds the traversal's tree (nodesQ, nodeTris) over the cubic keys and,
// with `view`, the published LBVH (codes, order, binary tree, nodes) over
// the per-axis ones, the two side by side through the same launches.
// batchOffsets (host, S + 1 of them) switches to per-scene bounds and keys
// and seeds the collapse with every scene's root.
void BuildBvhImpl( BvhObject& bvh, const float* d_tris, uint32_t n, const RgExtBvhBuildParams& params, const uint32_t* batchOffsets,
                   uint32_t sceneCount, hipStream_t stream, bool view )
{
    RG_REQUIRE( n > 0, RG_RESULT_WRONG_FUNCTION_ARGUMENT, "triangle count must be > 0" );
    RG_REQUIRE( n < ( 1u << 28 ), RG_RESULT_WRONG_FUNCTION_ARGUMENT, "triangle count must be < 2^28" );
    RG_REQUIRE( params.maxLeafSize >= 1 && params.maxLeafSize <= 8, RG_RESULT_WRONG_FUNCTION_ARGUMENT, "maxLeafSize must be in [1, 8]" );
    RG_REQUIRE( params.nodeFormat == RG_EXT_BVH_NODE_FP32 || params.nodeFormat == RG_EXT_BVH_NODE_FP16, RG_RESULT_WRONG_FUNCTION_ARGUMENT,
                "unknown node format" );

    const bool batched = batchOffsets != nullptr;
    bvh.n              = n;
    bvh.leafMax        = params.maxLeafSize;
    bvh.nodeFormat     = params.nodeFormat;
    bvh.nodeCount      = 0; // until the build is done
    bvh.nodeCountQ     = 0;
    bvh.sceneCount     = batched ? sceneCount : 0u;

    const uint32_t internal  = n - 1;
    const uint32_t slots     = internal > 0 ? internal : 1;
    const uint32_t rsBlocks  = DivUp( n, RS_TILE );
    const uint32_t bndBlocks = DivUp( n, THREADS ) < 1024 ? DivUp( n, THREADS ) : 1024;
    const uint32_t sets      = view ? 2 : 1; // set 0: the traversal's tree, set 1: the published one
    const uint32_t S         = batched ? sceneCount : 0u;

    const TreeScratch size( nullptr, nullptr, nullptr, view, n, S );
    bvh.scratch.Reserve( size.bytes );
    bvh.nodeTris.Reserve( std::max( size_t( n ) * 48, size.earlyBytes ) );
    if( view )
    {
        bvh.sortedTris.Reserve( size_t( n ) * 48 );
    }
    const TreeScratch ts( bvh.scratch.as< char >(), bvh.nodeTris.as< char >(), bvh.sortedTris.as< float >(), view, n, S );
    bvh.boundsPartials.Reserve( size_t( bndBlocks + 1 ) * 6 * 8 );
    if( !bvh.hostLevels )
    {
        RG_HIP_CHECK( hipHostMalloc( reinterpret_cast< void** >( &bvh.hostLevels ), TreeScratch::LEVEL_WORDS * 2 * 4, hipHostMallocDefault ) );
    }
    if( view )
    {
        bvh.codes.Reserve( size_t( n ) * 8 );
        bvh.keysA.Reserve( size_t( n ) * 8 );
        bvh.keysB.Reserve( size_t( n ) * 8 );
        bvh.valsA.Reserve( size_t( n ) * 4 );
        bvh.valsB.Reserve( size_t( n ) * 4 );
        bvh.hist.Reserve( size_t( 256 ) * ( rsBlocks + 1 ) * 4 );
        bvh.scanScratch.Reserve( ScanScratchBytes( slots ) );
        bvh.children.Reserve( size_t( slots ) * 8 );
        bvh.rangeFirst.Reserve( size_t( slots ) * 4 );
        bvh.rangeLast.Reserve( size_t( slots ) * 4 );
        bvh.nodeBounds.Reserve( ( 2 * size_t( n ) - 1 ) * 24 );
        bvh.expandInfo.Reserve( size_t( slots ) * sizeof( uint4 ) );
        bvh.treeLists.Reserve( TreeListBytes( n ) );
        bvh.expansion.Reserve( size_t( slots ) * 32 );
        bvh.isNode8.Reserve( size_t( slots ) * 4 );
        bvh.node8Index.Reserve( size_t( slots ) * 4 );
        bvh.queue.Reserve( size_t( slots ) * 4 );
    }

    // 1. FP64 centroid bounds and 2. Morton keys (input order) with the
    // identity permutation, per scene in a batch.
    double*  partials    = bvh.boundsPartials.as< double >();
    double*  sceneBounds = partials + size_t( bndBlocks ) * 6;
    uint32_t* offs       = nullptr;
    KeyOut   ko{ nullptr, nullptr, nullptr, ts.keys0, ts.vals0 };
    if( view )
    {
        ko.codes    = bvh.codes.as< uint64_t >();
        ko.viewKeys = bvh.keysA.as< uint64_t >();
        ko.viewVals = bvh.valsA.as< uint32_t >();
    }
    if( !batched || view )
    {
        // (a batch keeps these for the view's fields alone)
        k_centroid_bounds<<< bndBlocks, THREADS, 0, stream >>>( d_tris, n, partials );
        CheckLaunch( "k_centroid_bounds" );
        k_bounds_final<<< 1, THREADS, 0, stream >>>( partials, bndBlocks, sceneBounds );
        CheckLaunch( "k_bounds_final" );
    }
    if( !batched )
    {
        k_morton<<< DivUp( n, THREADS ), THREADS, 0, stream >>>( d_tris, n, sceneBounds, ko );
        CheckLaunch( "k_morton" );
    }
    else
    {
        const uint32_t B = 16;
        bvh.sceneOffsets.Reserve( size_t( sceneCount + 1 ) * 4 );
        bvh.sceneRoots.Reserve( size_t( sceneCount ) * 4 );
        bvh.sceneRoots8.Reserve( size_t( sceneCount ) * 4 );
        bvh.sceneBounds.Reserve( size_t( sceneCount ) * 6 * 8 );
        bvh.scenePartials.Reserve( size_t( sceneCount ) * B * 6 * 8 );
        bvh.hostSceneOffsets.assign( batchOffsets, batchOffsets + sceneCount + 1 );
        RG_HIP_CHECK( hipMemcpyAsync( bvh.sceneOffsets.ptr, bvh.hostSceneOffsets.data(), size_t( sceneCount + 1 ) * 4, hipMemcpyHostToDevice, stream ) );
        offs = bvh.sceneOffsets.as< uint32_t >();
        k_centroid_bounds_seg<<< sceneCount * B, THREADS, 0, stream >>>( d_tris, offs, B, bvh.scenePartials.as< double >() );
        CheckLaunch( "k_centroid_bounds_seg" );
        k_bounds_final_seg<<< sceneCount, 64, 0, stream >>>( bvh.scenePartials.as< double >(), B, bvh.sceneBounds.as< double >() );
        CheckLaunch( "k_bounds_final_seg" );
        k_morton_seg<<< DivUp( n, THREADS ), THREADS, 0, stream >>>( d_tris, n, offs, sceneCount, bvh.sceneBounds.as< double >(), ko );
        CheckLaunch( "k_morton_seg" );
    }

    // 3. Stable LSD radix sort, 8 passes of 8 bits.
    SortSets ss{};
    ss.s[ 0 ] = SortSet{ { ts.keys0, ts.keys1 }, { ts.vals0, ts.vals1 }, ts.hist, ts.hist + size_t( 256 ) * rsBlocks };
    if( view )
    {
        ss.s[ 1 ] = SortSet{ { bvh.keysA.as< uint64_t >(), bvh.keysB.as< uint64_t >() },
                             { bvh.valsA.as< uint32_t >(), bvh.valsB.as< uint32_t >() },
                             bvh.hist.as< uint32_t >(),
                             bvh.hist.as< uint32_t >() + size_t( 256 ) * rsBlocks };
    }
    RadixSort( ss, sets, n, stream );
    bvh.sortedIdx = view ? bvh.valsA.as< uint32_t >() : nullptr;

    // 4. The binary hierarchies with their boxes.
    uint32_t* rf     = view ? bvh.rangeFirst.as< uint32_t >() : nullptr;
    uint32_t* rl     = view ? bvh.rangeLast.as< uint32_t >() : nullptr;
    float*    bounds = view ? bvh.nodeBounds.as< float >() : nullptr;
    TreeSets  ta{};
    ta.s[ 0 ]       = TreeArgs{ d_tris, ts.keys0, ts.vals0, n, 1, ts.children, ts.rf, ts.rl, ts.bounds, ts.info };
    ta.s[ 0 ].sizes = true;
    if( view )
    {
        ta.s[ 1 ] = TreeArgs{ d_tris, bvh.keysA.as< uint64_t >(), bvh.valsA.as< uint32_t >(), n, bvh.leafMax, bvh.children.as< uint2 >(), rf, rl, bounds,
                              bvh.expandInfo.as< uint4 >() };
    }
    uint2* const lists[ 2 ] = { ts.lists, view ? bvh.treeLists.as< uint2 >() : nullptr };
    BuildTree( ta, lists, sets, stream );

    // 5. Collapse to 8-wide nodes, level by level; the traversal's tree with
    // one triangle per leaf.
    constexpr uint32_t LW     = TreeScratch::LEVEL_WORDS;
    uint32_t* const    levels = ts.levels;
    CollapseSets       cs{};
    cs.s[ 0 ] = CollapseArgs{ ts.queue, levels + BVH_MAX_LEVELS + 1, levels, n, 1, ts.info, ts.rf, ts.rl, ts.expansion, nullptr, ts.nodeBase,
                              levels + LW * 2 };
    if( view )
    {
        cs.s[ 1 ] = CollapseArgs{ bvh.queue.as< uint32_t >(), levels + LW + BVH_MAX_LEVELS + 1, levels + LW, n, bvh.leafMax, bvh.expandInfo.as< uint4 >(),
                                  rf, rl, bvh.expansion.as< uint32_t >(), bvh.isNode8.as< uint32_t >(), nullptr, nullptr };
    }
    uint32_t* const roots[ 2 ] = { batched ? ts.roots : nullptr, batched && view ? bvh.sceneRoots.as< uint32_t >() : nullptr };
    const uint32_t  nodeWords  = view ? slots : 0u;
    const uint32_t  initWords  = std::max( std::max( nodeWords, LW * 2 + 1 ), batched ? sceneCount : 0u );
    k_build_init<<< std::min( DivUp( initWords, THREADS ), 1024u ), THREADS, 0, stream >>>( levels, LW * 2 + 1, view ? bvh.isNode8.as< uint32_t >() : nullptr,
                                                                                          nodeWords, roots[ 0 ], roots[ 1 ], batched ? sceneCount : 0u );
    CheckLaunch( "k_build_init" );
    if( !batched )
    {
        k_seed_frontier<<< 1, 64, 0, stream >>>( cs, sets );
        CheckLaunch( "k_seed_frontier" );
    }
    else
    {
        for( uint32_t k = 0; k < sets; k++ )
        {
            if( internal > 0 )
            {
                k_scene_roots<<< DivUp( internal, THREADS ), THREADS, 0, stream >>>( internal, ta.s[ k ].rangeFirst, ta.s[ k ].rangeLast, offs, sceneCount,
                                                                                   roots[ k ] );
                CheckLaunch( "k_scene_roots" );
            }
            k_seed_frontier_seg<<< 1, 256, 0, stream >>>( roots[ k ], sceneCount, offs, internal, k == 0, cs.s[ k ].queue, cs.s[ k ].levelCount,
                                                          ta.s[ k ].bounds, k == 0 ? ts.boxes : nullptr );
            CheckLaunch( "k_seed_frontier_seg" );
        }
        bvh.hostSegBoxes.resize( size_t( sceneCount ) * 8 );
        RG_HIP_CHECK( hipMemcpyAsync( bvh.hostSegBoxes.data(), ts.boxes, size_t( sceneCount ) * 8 * sizeof( float ), hipMemcpyDeviceToHost, stream ) );
    }

    const uint32_t maxFrontier  = n / 2 + 1 + S;
    const uint32_t collapseGrid = DivUp( maxFrontier, THREADS ) < 4096 ? DivUp( maxFrontier, THREADS ) : 4096;
    // levels before the first look at how many nodes are left: an 8-wide
    // node stands for about 1.75 binary levels
    uint32_t bits = 1;
    while( bits < 28 && ( n >> bits ) != 0 )
    {
        bits++;
    }
    uint32_t        level = 0, batch = bits * 4 / 7 + 2;
    uint32_t* const host  = bvh.hostLevels;
    do
    {
        for( uint32_t k = 0; k < batch; k++, level++ )
        {
            RG_REQUIRE( level + 1 < BVH_MAX_LEVELS, RG_RESULT_INTERNAL_ERROR, "BVH deeper than the level limit" );
            k_collapse_level<<< dim3( collapseGrid, sets ), THREADS, 0, stream >>>( cs, level );
            CheckLaunch( "k_collapse_level" );
        }
        RG_HIP_CHECK( hipMemcpyAsync( host, levels, LW * 2 * 4, hipMemcpyDeviceToHost, stream ) );
        RG_HIP_CHECK( hipStreamSynchronize( stream ) );
        batch = 4;
    } while( host[ level ] != 0 || host[ LW + level ] != 0 );
    const uint32_t countQ    = host[ BVH_MAX_LEVELS + 1 + level ];
    const uint32_t countView = host[ LW + BVH_MAX_LEVELS + 1 + level ];
    RG_REQUIRE( countQ >= 1 && ( !view || countView >= 1 ), RG_RESULT_INTERNAL_ERROR, "BVH collapse produced no nodes" );

    // 6. The nodes.
    bvh.nodesQ.Reserve( size_t( countQ ) * sizeof( BvhNodeQ ) );
    k_pack_nodes<<< DivUp( uint64_t( countQ ) * 8u, THREADS ), THREADS, 0, stream >>>( countQ, n, ts.expansion, ts.nodeBase, ts.bounds, ts.vals0, d_tris,
                                                                                     bvh.nodesQ.as< BvhNodeQ >(), bvh.nodeTris.as< float4 >() );
    CheckLaunch( "k_pack_nodes" );
    if( view )
    {
        ExclusiveScan( bvh.isNode8.as< uint32_t >(), slots, bvh.node8Index.as< uint32_t >(), nullptr, bvh.scanScratch.as< uint32_t >(), stream );
        const bool    half    = params.nodeFormat == RG_EXT_BVH_NODE_FP16;
        DeviceBuffer& fp32Out = half ? bvh.nodes32 : bvh.nodes;
        fp32Out.Reserve( size_t( countView ) * sizeof( BvhNode8 ) );
        k_write_nodes<<< DivUp( uint64_t( countView ) * 8u, THREADS ), THREADS, 0, stream >>>(
            countView, n, bvh.queue.as< uint32_t >(), bvh.node8Index.as< uint32_t >(), bvh.expansion.as< uint32_t >(), rf, rl, bounds, fp32Out.as< BvhNode8 >() );
        CheckLaunch( "k_write_nodes" );
        k_sorted_tris<<< DivUp( n, THREADS ), THREADS, 0, stream >>>( d_tris, bvh.sortedIdx, n, bvh.sortedTris.as< float4 >() );
        CheckLaunch( "k_sorted_tris" );
        if( batched )
        {
            k_gather_roots8<<< 1, 256, 0, stream >>>( bvh.sceneRoots.as< uint32_t >(), sceneCount, bvh.node8Index.as< uint32_t >(),
                                                      bvh.sceneRoots8.as< uint32_t >() );
            CheckLaunch( "k_gather_roots8" );
            bvh.hostSceneRoots.resize( sceneCount );
            RG_HIP_CHECK( hipMemcpyAsync( bvh.hostSceneRoots.data(), bvh.sceneRoots8.ptr, size_t( sceneCount ) * 4, hipMemcpyDeviceToHost, stream ) );
        }
        if( half )
        {
            bvh.nodes.Reserve( size_t( countView ) * sizeof( BvhNode8H ) );
            k_half_nodes<<< DivUp( countView, THREADS ), THREADS, 0, stream >>>( bvh.nodes32.as< BvhNode8 >(), countView, bvh.nodes.as< BvhNode8H >() );
            CheckLaunch( "k_half_nodes" );
        }
        RG_HIP_CHECK( hipMemcpyAsync( bvh.sceneMin, sceneBounds, 3 * sizeof( double ), hipMemcpyDeviceToHost, stream ) );
        RG_HIP_CHECK( hipMemcpyAsync( bvh.sceneMax, sceneBounds + 3, 3 * sizeof( double ), hipMemcpyDeviceToHost, stream ) );
    }
    RG_HIP_CHECK( hipStreamSynchronize( stream ) );
    bvh.nodeCountQ = countQ;
    bvh.nodeCount  = view ? countView : countQ;
}
} // namespace

void BuildBvh( BvhObject& bvh, const float* d_tris, uint32_t n, const RgExtBvhBuildParams& params, hipStream_t stream )
{
    BuildBvhImpl( bvh, d_tris, n, params, nullptr, 0, stream, true );
    bvh.frameSegs.clear();
}

void BuildBvhBatch( BvhObject& bvh, const float* d_tris, const uint32_t* offsets, uint32_t sceneCount, const RgExtBvhBuildParams& params,
                    hipStream_t stream, bool view )
{
    RG_REQUIRE( offsets && sceneCount >= 1 && sceneCount <= 128, RG_RESULT_WRONG_FUNCTION_ARGUMENT, "1..128 scenes" );
    RG_REQUIRE( offsets[ 0 ] == 0, RG_RESULT_WRONG_FUNCTION_ARGUMENT, "scene offsets must start at 0" );
    for( uint32_t s = 0; s < sceneCount; s++ )
    {
        RG_REQUIRE( offsets[ s + 1 ] >= offsets[ s ] + 2, RG_RESULT_WRONG_FUNCTION_ARGUMENT, "every scene needs at least 2 triangles" );
    }
    BuildBvhImpl( bvh, d_tris, offsets[ sceneCount ], params, offsets, sceneCount, stream, view );
    bvh.frameSegs.clear();
    for( uint32_t s = 0; view && s < sceneCount; s++ )
    {
        RG_REQUIRE( bvh.hostSceneRoots[ s ] < bvh.nodeCount, RG_RESULT_INTERNAL_ERROR, "a scene has no root node" );
    }
}

void BuildFrameBvh( BvhObject& bvh, const float* d_tris, const uint32_t* classTris, uint32_t classCount, const RgExtBvhBuildParams& params,
                    hipStream_t stream )
{
    std::vector< uint32_t > offsets( 1, 0u ), cls;
    for( uint32_t c = 0; c < classCount; c++ )
    {
        if( classTris[ c ] > 0 )
        {
            offsets.push_back( offsets.back() + classTris[ c ] );
            cls.push_back( c );
        }
    }
    const uint32_t S = uint32_t( cls.size() ), n = offsets.back();
    RG_REQUIRE( S > 0 && S <= 8, RG_RESULT_INTERNAL_ERROR, "a frame BVH has 1..8 segments" );
    bvh.frameSegs.assign( S, BvhObject::FrameSegment{} );
    if( S == 1 )
    {
        // one class: the single-scene build (21 Morton bits per axis); rays
        // whose mask admits it start at its root
        BuildBvhImpl( bvh, d_tris, n, params, nullptr, 0, stream, false );
        bvh.frameSegs[ 0 ].cls  = cls[ 0 ];
        bvh.frameSegs[ 0 ].root = 0;
        for( int k = 0; k < 3; k++ )
        {
            bvh.frameSegs[ 0 ].box[ k ]     = -INFINITY;
            bvh.frameSegs[ 0 ].box[ 3 + k ] = INFINITY;
        }
        return;
    }
    // several classes: one batched build, each class a segment with its own
    // root (node s of segment s) and root box
    BuildBvhImpl( bvh, d_tris, n, params, offsets.data(), S, stream, false );
    for( uint32_t s = 0; s < S; s++ )
    {
        bvh.frameSegs[ s ].cls  = cls[ s ];
        bvh.frameSegs[ s ].root = s;
        std::memcpy( bvh.frameSegs[ s ].box, &bvh.hostSegBoxes[ size_t( s ) * 8 ], 6 * sizeof( float ) );
    }
    bvh.sceneCount = 0; // traced as a frame (TraceRaysFrame), not as a batch of scenes
}

} // namespace rg
