// tiles_dev.h -- device helpers shared by the tiled list build (tiles.hip)
// and the tiled force kernels (lj.hip).  See tiles.hip for the layout.
#pragma once

#include "internal.h"

namespace cmd
{
// A tile is W x W interior columns of the binning grid (W = 1, 2 or 3) over E
// cells [e0, e1).  Its atoms are the local atoms of those cells: one
// contiguous run per atom column (the cell-sorted order runs along a
// column), taken in atom-column order c = ca * W + cb.  Every neighbour
// candidate of those atoms lies in the (W + 2) x (W + 2) staged columns
// around them, cells [e0 - 1, e1]: per staged column one contiguous run of
// locals and one of cell-sorted ghosts (segments 2q and 2q + 1 of staged
// column q = da * (W + 2) + db).  Staged columns past the padded grid (the
// right edge of a tile whose second atom column does not exist) are empty.
constexpr int TILE_WMAX = 3;
constexpr int TILE_QMAX = ( TILE_WMAX + 2 ) * ( TILE_WMAX + 2 ); // staged columns
constexpr int TILE_CMAX = TILE_WMAX * TILE_WMAX;                 // atom columns
static constexpr int TILE_SEGS = 2 * TILE_QMAX; // segments: locals and ghosts of each column
enum
{
    TI_LB = 0,                         // [Q] first local index of each staged column run
    TI_LLEN = TILE_QMAX,               // [Q] local run lengths
    TI_GB = 2 * TILE_QMAX,             // [Q] first sorted-ghost slot of each run
    TI_GLEN = 3 * TILE_QMAX,           // [Q] ghost run lengths
    TI_AL = 4 * TILE_QMAX,             // [C] first local atom of each atom column
    TI_AN = 4 * TILE_QMAX + TILE_CMAX, // [C] atoms of each atom column
    TI_NAT = 4 * TILE_QMAX + 2 * TILE_CMAX, // atoms in the tile
    TI_TOTAL,                               // staged positions
    TI_EA,                                  // first staged cell (e0 - 1, clamped)
    TI_NST,                                 // staged cells per column
    TI_SEG,                                 // [SEGS + 1] segment offsets in slots (segment
                                            // 2q = locals of staged column q, 2q + 1 = its
                                            // ghosts; TOTAL past the tile's segments)
    TI_AOFF = TI_SEG + TILE_SEGS + 1,       // [C + 1] tile-atom offsets of the atom columns
    TI_WORDS = TI_AOFF + TILE_CMAX + 1
};

constexpr int TILE_STRIP = 4;

__host__ __device__ constexpr int tile_q( int W ) { return ( W + 2 ) * ( W + 2 ); }

__device__ __forceinline__ void tile_coords( const TileGrid &T, int t, int &a0,
                                             int &b0, int &e0, int &e1 )
{
    // tile columns in strips of TILE_STRIP rows of a, b outer and a inner
    // within a strip: the columns around a tile are staged by its neighbours
    // close together in time, so a staged column is mostly re-read from L2
    t -= T.tile0;
    const int col = t / T.tpc, z = t % T.tpc;
    const int strip = col / ( TILE_STRIP * T.nt1 ), r = col % ( TILE_STRIP * T.nt1 );
    const int h = min( TILE_STRIP, T.nt0 - strip * TILE_STRIP );
    a0 = 1 + T.W * ( strip * TILE_STRIP + r % h );
    b0 = 1 + T.W * ( r / h );
    e0 = 1 + z * T.E;
    e1 = min( e0 + T.E, T.g.n[2] - 1 );
}

__device__ __forceinline__ int col_base( const TileGrid &T, int a, int b )
{
    return T.cell0 + ( a * T.g.n[1] + b ) * T.g.n[2];
}

// Round-robin dispatch puts block b on XCD b % 8; give XCD k the k-th
// contiguous slice of tiles.
__device__ __forceinline__ int xcd_tile( int b, int nb )
{
    const int q = nb >> 3, r = nb & 7;
    const int xcd = b & 7, k = b >> 3;
    return ( xcd < r ) ? xcd * ( q + 1 ) + k : r * ( q + 1 ) + ( xcd - r ) * q + k;
}

// Shared tile header: the info words (the segment offsets and atom-column
// offsets are among them, laid out by k_tile_info).
struct TileHead
{
    int info[TI_WORDS];
    int nseg; // 2 (W + 2)^2
    __device__ const int *segoff() const { return info + TI_SEG; }
    __device__ const int *aoff() const { return info + TI_AOFF; }
};

__device__ inline void load_head( const int *__restrict__ info, int t, int W, TileHead &H )
{
    const int *I = info + (size_t)t * TI_WORDS;
    for ( int k = threadIdx.x; k < TI_WORDS; k += blockDim.x )
        H.info[k] = I[k];
    if ( threadIdx.x == 0 )
        H.nseg = 2 * tile_q( W );
    __syncthreads();
}

// System index of tile atom ta (ta < the tile's atom count).
__device__ __forceinline__ int tile_atom( const TileHead &H, int W, int ta )
{
    int c = 0;
    while ( c + 1 < W * W && ta >= H.aoff()[c + 1] )
        ++c;
    return H.info[TI_AL + c] + ( ta - H.aoff()[c] );
}

// Staged column of atom column c.
__device__ __forceinline__ int atom_col_q( int W, int c )
{
    return ( c / W + 1 ) * ( W + 2 ) + ( c % W + 1 );
}

// Position of a tile's sentinel slot (slot TOTAL, just past the staged
// atoms): list rows are padded with it, and its distance to any atom is far
// beyond every cutoff, so a padded pair contributes exact zeros.
static constexpr double TILE_FAR = 1.0e30;

// Record sizes (TILE_REC, TILE_REC32) are defined with the neighbour list
// (internal.h): tiled list entries are byte offsets of records.

// Lanes per atom of slab wave w of a tile with nat atoms, for tiled lists
// built with G lanes per atom (64 / G atoms per full wave): G, doubled up to
// 8 while the wave's atoms still fill the 64 lanes.  A tile's last wave is
// usually part full; spreading its rows over more lanes shortens its walk.
__device__ __forceinline__ int wave_lanes( int G, int nat, int w )
{
    const int na = min( 64 / G, nat - w * ( 64 / G ) );
    int g = G;
    while ( g < 8 && na * g * 2 <= 64 )
        g *= 2;
    return g;
}

// The segment s (0 <= s < nseg) with off[s] <= k < off[s + 1], for
// off[0] <= k < off[nseg]: a binary search, so that the searches of a
// thread's several slots are independent chains of a few LDS reads (a walk
// from segment to segment would chain one read per segment passed).
__device__ __forceinline__ int find_seg( const int *off, int nseg, int k )
{
    int lo = 0, hi = nseg;
    while ( hi - lo > 1 )
    {
        const int mid = ( lo + hi ) >> 1;
        if ( off[mid] <= k )
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

// Largest value of the wave's lanes (values >= 0), in row shifts and row
// broadcasts of the adder's operand rather than LDS permutes.
__device__ __forceinline__ int wave_max_i32( int v )
{
#define CMD_MAX_DPP( CTRL )                                                                \
    v = max( v, __builtin_amdgcn_update_dpp( 0, v, CTRL, 0xf, 0xf, true ) )
    CMD_MAX_DPP( 0x111 ); // row_shr 1, 2, 4, 8: lane 15 of each row holds its maximum
    CMD_MAX_DPP( 0x112 );
    CMD_MAX_DPP( 0x114 );
    CMD_MAX_DPP( 0x118 );
    CMD_MAX_DPP( 0x142 ); // row_bcast 15, then 31: lane 63 holds the wave's
    CMD_MAX_DPP( 0x143 );
#undef CMD_MAX_DPP
    return __builtin_amdgcn_readlane( v, 63 );
}

// v plus the value of the lane O away (lane ^ O), O = 8, 16 or 32.
template <int O>
__device__ __forceinline__ double add_lane_xor( double v )
{
    const unsigned long long b = (unsigned long long)__double_as_longlong( v );
    const unsigned lo = (unsigned)b, hi = (unsigned)( b >> 32 );
    auto join = []( unsigned l, unsigned h )
    { return __longlong_as_double( (long long)( ( (unsigned long long)h << 32 ) | l ) ); };
    if constexpr ( O == 8 )
    {
        // row_ror:8 turns each row of 16 lanes by half
        const unsigned l = (unsigned)__builtin_amdgcn_update_dpp( 0, (int)lo, 0x128, 0xf, 0xf, true );
        const unsigned h = (unsigned)__builtin_amdgcn_update_dpp( 0, (int)hi, 0x128, 0xf, 0xf, true );
        return v + join( l, h );
    }
    else
    {
        // the swap leaves one half's (or row pair's) values in all lanes of
        // one result and the other's in the other
        const auto l = O == 32 ? __builtin_amdgcn_permlane32_swap( lo, lo, false, false )
                               : __builtin_amdgcn_permlane16_swap( lo, lo, false, false );
        const auto h = O == 32 ? __builtin_amdgcn_permlane32_swap( hi, hi, false, false )
                               : __builtin_amdgcn_permlane16_swap( hi, hi, false, false );
        return join( l[0], h[0] ) + join( l[1], h[1] );
    }
}

// Sum over the lanes of one atom: lane pairs apw, 2 apw, ... apart (apw = 8,
// 16 or 32 atoms per wave; wave-uniform).
__device__ __forceinline__ void sum_atom_lanes( int apw, double &a, double &b, double &c )
{
    if ( apw <= 8 )
    {
        a = add_lane_xor<8>( a );
        b = add_lane_xor<8>( b );
        c = add_lane_xor<8>( c );
    }
    if ( apw <= 16 )
    {
        a = add_lane_xor<16>( a );
        b = add_lane_xor<16>( b );
        c = add_lane_xor<16>( c );
    }
    a = add_lane_xor<32>( a );
    b = add_lane_xor<32>( b );
    c = add_lane_xor<32>( c );
}

// Walk of a tile's staged positions for the full-list force kernel, straight
// from the tile's info words: the segments (lane s of a wave holds segment
// s: 50 at most) are cut into chunks of 64 and wave w of nw takes chunks w,
// w + nw, ...; put(slot, p) gets each lane's position with its slot.  A
// chunk's segment is the number of segments that end at or before it (one
// compare and a scalar count), so no lane searches for its segment, the
// loads of a wave are consecutive, and up to B chunks are in flight.  A block
// that first copied the info words to LDS, chained the segment offsets in one
// thread and searched them per slot spent about a tenth of its time there:
// with this walk and the cross-lane sums above the force kernel went from 222
// to 194 us (2,048,000 atoms, mixed), 152 to 133 us (864,000, FP64) and 17.2
// to 13.1 us (48,000, two types, mixed).
template <class Put>
__device__ __forceinline__ void stage_chunks( const int *__restrict__ I, int nseg, int wid,
                                              int nw, const double4 *__restrict__ x,
                                              const double4 *__restrict__ xg, Put put )
{
    const int lane = threadIdx.x & 63;
    int src = 0, len = 0, dst = 0;
    if ( lane < nseg )
    {
        const int q = lane >> 1, g = lane & 1;
        src = I[( g ? TI_GB : TI_LB ) + q];
        len = I[( g ? TI_GLEN : TI_LLEN ) + q];
        dst = I[TI_SEG + lane];
    }
    // chunks of the segments up to and including the lane's
    int inc = ( len + 63 ) >> 6;
#define CMD_SCAN_DPP( CTRL, ROWS )                                                         \
    inc += __builtin_amdgcn_update_dpp( 0, inc, CTRL, ROWS, 0xf, true )
    CMD_SCAN_DPP( 0x111, 0xf );
    CMD_SCAN_DPP( 0x112, 0xf );
    CMD_SCAN_DPP( 0x114, 0xf );
    CMD_SCAN_DPP( 0x118, 0xf );
    CMD_SCAN_DPP( 0x142, 0xa ); // rows 1 and 3 take the row before's total
    CMD_SCAN_DPP( 0x143, 0xc ); // rows 2 and 3 take the first half's
#undef CMD_SCAN_DPP
    const int nch = __builtin_amdgcn_readlane( inc, 63 );
    constexpr int B = 8; // chunks of a wave in flight together
    for ( int c0 = wid; c0 < nch; c0 += B * nw )
    {
        double4 p[B];
        int slot[B];
#pragma unroll
        for ( int u = 0; u < B; ++u )
        {
            const int c = c0 + u * nw;
            slot[u] = -1;
            if ( c < nch ) // wave-uniform
            {
                const int s =
                    (int)__popcll( __builtin_amdgcn_ballot_w64( inc <= c ) );
                const int sl = __builtin_amdgcn_readlane( len, s );
                const int first = __builtin_amdgcn_readlane( inc, s ) - ( ( sl + 63 ) >> 6 );
                const int o = ( ( c - first ) << 6 ) + lane;
                const double4 *__restrict__ base = ( s & 1 ) ? xg : x;
                // lanes past the segment's end reload its last position
                p[u] = base[__builtin_amdgcn_readlane( src, s ) + min( o, sl - 1 )];
                if ( o < sl )
                    slot[u] = __builtin_amdgcn_readlane( dst, s ) + o;
            }
        }
#pragma unroll
        for ( int u = 0; u < B; ++u )
            if ( slot[u] >= 0 )
                put( slot[u], p[u] );
    }
}

// Centre of tile t's staged region, the origin of its FP32 records.
__device__ __forceinline__ void tile_centre( const TileGrid &T, int t, double &ox, double &oy,
                                             double &oz )
{
    int a0, b0, e0, e1;
    tile_coords( T, t, a0, b0, e0, e1 );
    // columns a0 - 1 .. a0 + W, cells e0 - 1 .. e1
    ox = T.g.min[0] + ( a0 - 1 + 0.5 * ( T.W + 2 ) ) / T.g.rd[0];
    oy = T.g.min[1] + ( b0 - 1 + 0.5 * ( T.W + 2 ) ) / T.g.rd[1];
    oz = T.g.min[2] + 0.5 * ( e0 + e1 ) / T.g.rd[2];
}

} // namespace cmd
