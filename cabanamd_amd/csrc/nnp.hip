// nnp.hip -- Behler-Parrinello neural-network potential: ForceNNP
// (force_types/force_nnp_cabana_neigh_impl.h:41-130) on one GPU.
//
// The reference runs n2p2's ModeCabana in three phases per force call
// (impl.h:93-98): symmetry functions, atomic networks, forces.  Here:
//   k_nnp_sf     one wave per atom: the atom's neighbours inside rc are
//                compacted into LDS (FP32 relative vectors from FP64
//                positions), radial functions with lanes over neighbours and
//                angular functions with lanes over neighbour pairs; per-lane
//                partial sums are combined with a reduce-scatter butterfly.
//   k_nnp_mlp    all elements in one launch, 16 atoms of one element per
//                wave: the two hidden layers and the backward pass on the
//                matrix cores over the scaled symmetry functions (split BF16
//                products, or FP32 ones); output layer, tanh and scaling on
//                the VALU.
//   k_nnp_force  one wave per atom: dE/dG chained into dG/dr on the same
//                pairs; reactions on neighbours gather in LDS and reach
//                f by FP64 atomics (ghost rows included, folded by
//                update_force as in the reference, cabanamd_impl.h:346-353).
// Definitions (n2p2's, for the input.nn keywords used by input/nnp):
// cosine cutoff fc(r) = (cos(pi r/rc) + 1)/2; radial G = sum_j
// exp(-eta (r-rs)^2) fc; angular G = 2^(1-zeta) sum_{j<k} (1 + lambda cos)^zeta
// exp(-eta sum (r-rs)^2) fc fc fc; min-max scaling; tanh/linear layers.
//
// The symmetry-function set of an element must be a grid: radial functions
// = {(eta, rs)} x {neighbour element or any}, angular = {(eta, rs)} x
// {(lambda, zeta)} over any neighbour pair.  Each pair then needs one exp
// per (eta, rs) and one power per (lambda, zeta), and every term is a
// product of the two.  Both the reference fixture and the benchmark model
// have this form; other sets are rejected at setup.
#include "internal.h"
#include "roofline.h"

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <fstream>
#include <map>
#include <sstream>
#include <string>
#include <vector>

// The NNP kernels compute in FP32 against a tolerance, not bit for bit:
// multiply-adds may fuse here (the library builds with contraction off for
// the FP64 paths, whose sums must match the oracle exactly).
#pragma clang fp contract( fast )

namespace cmd
{
static constexpr int NNP_MAXEL = 4;
static constexpr int RG_MAX = 16; // radial (eta, rs) values
static constexpr int RE_MAX = 2;  // radial neighbour-element filters
static constexpr int AG_MAX = 8;  // angular (eta, rs) values
static constexpr int AP_MAX = 8;  // angular (lambda, zeta) values
static constexpr int NR_MAX = RG_MAX * RE_MAX; // 32
static constexpr int NA_MAX = AG_MAX * AP_MAX; // 64
static constexpr int NSF_LD = 96;              // row stride of G / dE/dG
static constexpr int KPAD = 96;                // MFMA K of layer 1 (6 x 16)
static constexpr int HPAD = 32;                // hidden width (2 x 16)
static constexpr int NN_MAX = 128;             // neighbours inside rc
static constexpr int TCAP = 512;               // compacted neighbour pairs per wave
static constexpr int NNP_TPB = 256;
// The (lambda, zeta) grid of zeta = 1, 2, 4, 16 and both signs of lambda:
// its powers are a few squarings, so it has kernels of its own.  Entry p:
// lambda = -1 for p < 4, else +1; zeta = POW_ZETA[p % 4].
static constexpr double POW_ZETA[4] = { 1.0, 2.0, 4.0, 16.0 };
static constexpr int POW_NAP = 8;

struct NnpElemPlan
{
    int nsf;
    int nrg, nre, nag, nap;
    float r_eta[RG_MAX], r_rs[RG_MAX];
    int r_el[RE_MAX];              // neighbour element, -1 = any
    int r_out[RG_MAX][RE_MAX];     // model index of radial (g, e)
    float a_eta[AG_MAX], a_rs[AG_MAX];
    float a_lam[AP_MAX], a_zeta[AP_MAX], a_lpref[AP_MAX]; // lpref = 1 - zeta
    int a_out[AG_MAX][AP_MAX];     // model index of angular (g, p)
    int pow2;                      // (lambda, zeta) are the POW_* grid, in its order
    alignas( 16 ) float g_mul[NSF_LD]; // Gs = g_mul * G + g_add
    alignas( 16 ) float g_add[NSF_LD];
    int h1, h2;
    int act1, act2, act3; // 1 = tanh, 0 = linear
    // layer weights, zero padded: [out][in] as the forward products' B
    // operands read them, [in][out] for the backward ones
    alignas( 16 ) float W1[HPAD][KPAD];
    alignas( 16 ) float W1T[KPAD][HPAD];
    float b1[HPAD];
    alignas( 16 ) float W2[HPAD][HPAD];
    alignas( 16 ) float W2T[HPAD][HPAD];
    float b2[HPAD];
    float w3[HPAD];
    float b3;
    // The layer weights as three BF16 parts (w = hi + mid + lo to FP32
    // precision), laid out as the MFMA B operands read them: [out][in] for
    // the forward products, [in][out] for the backward ones.
    alignas( 16 ) unsigned short W1s[3][HPAD][KPAD];
    alignas( 16 ) unsigned short W1Ts[3][KPAD][HPAD];
    alignas( 16 ) unsigned short W2s[3][HPAD][HPAD];
    alignas( 16 ) unsigned short W2Ts[3][HPAD][HPAD];
};

struct NnpPlan
{
    int nelem;
    float rc, rc2, pi_rc; // pi_rc = pi / rc
    NnpElemPlan el[NNP_MAXEL];
};
} // namespace cmd

// Host-side model: what input.nn, scaling.data and weights.NNN.data hold.
struct cmd_nnp_model
{
    struct SF
    {
        int type, e1, e2;
        double eta, rs, lambda, zeta, rc;
    };
    struct Elem
    {
        std::string name;
        int z = 0;
        std::vector<SF> sf;
        std::vector<double> gmin, gmax;
        std::vector<std::vector<double>> W, b; // per layer [out][in], [out]
        double atom_energy = 0.0;
    };
    int nelem = 0;
    int nlayers = 3;
    std::vector<int> hidden;
    std::string act = "ttl";
    bool scale = true;
    double smin = 0.0, smax = 1.0;
    std::vector<Elem> el;
};

struct cmd_nnp
{
    cmd_nnp_model model;
    cmd::NnpPlan plan{};
    cmd::DevBuf<cmd::NnpPlan> dplan;
    bool plan_ok = false;
    int prec = CMD_PREC_MIXED; // MIXED: BF16 MFMA layers; FP64: FP32 layers
    cmd::DevBuf<float> G, dEdG, Ei;
    cmd::DevBuf<int> flag;
    cmd::DevBuf<double> part;
    cmd::DevBuf<int4> terms; // per atom: neighbours, triplets, element (last compute)
    int cap = 0;
    int n_last = 0;
    // a time loop's stream and (pinned) the step that stopped it; its steps so
    // far and the marks among them, two events in turn
    hipStream_t run_stream = nullptr;
    cmd::HostWords stop;
    hipEvent_t mark[2] = {};
    long steps = 0, marks = 0;
    ~cmd_nnp()
    {
        for ( hipEvent_t e : mark )
            if ( e )
                (void)hipEventDestroy( e );
    }
};

namespace cmd
{
// ---------------------------------------------------------------- plan
static int find_or_add( std::vector<std::pair<double, double>> &v, double a,
                        double b )
{
    for ( size_t k = 0; k < v.size(); ++k )
        if ( v[k].first == a && v[k].second == b )
            return (int)k;
    v.push_back( { a, b } );
    return (int)v.size() - 1;
}

// BF16 bits of a float, rounded to nearest even (the format's NaN and
// infinity are not produced from the finite weights and activations here).
__host__ __device__ inline unsigned short bf16_bits( float f )
{
    unsigned u;
    std::memcpy( &u, &f, sizeof( u ) );
    u += 0x7fffu + ( ( u >> 16 ) & 1u );
    return (unsigned short)( u >> 16 );
}

__host__ __device__ inline float bf16_value( unsigned short b )
{
    const unsigned u = (unsigned)b << 16;
    float f;
    std::memcpy( &f, &u, sizeof( f ) );
    return f;
}

// x = hi + mid + lo: each part the BF16 rounding of what the parts before it
// leave, so the three hold the 24 significant bits of an FP32 value.
__host__ __device__ inline void bf16_split3( float x, unsigned short part[3] )
{
    part[0] = bf16_bits( x );
    const float r1 = x - bf16_value( part[0] );
    part[1] = bf16_bits( r1 );
    const float r2 = r1 - bf16_value( part[1] );
    part[2] = bf16_bits( r2 );
}

static cmd_status build_plan( const cmd_nnp_model &m, NnpPlan &P )
{
    std::memset( &P, 0, sizeof( P ) );
    CMD_REQUIRE( m.nelem >= 1 && m.nelem <= NNP_MAXEL, CMD_ERR_ARG,
                 "NNP models with 1..%d elements are supported", NNP_MAXEL );
    CMD_REQUIRE( m.hidden.size() == 2, CMD_ERR_ARG,
                 "NNP networks with two hidden layers are supported" );
    CMD_REQUIRE( m.hidden[0] >= 1 && m.hidden[0] <= HPAD && m.hidden[1] >= 1 &&
                     m.hidden[1] <= HPAD,
                 CMD_ERR_ARG, "hidden layers wider than %d nodes", HPAD );
    CMD_REQUIRE( m.act.size() == 3 && m.act[2] == 'l', CMD_ERR_ARG,
                 "activations must be t/l for the hidden layers and l for "
                 "the output" );
    P.nelem = m.nelem;
    double rc = -1.0;
    for ( int e = 0; e < m.nelem; ++e )
    {
        const auto &E = m.el[e];
        NnpElemPlan &Q = P.el[e];
        const int ns = (int)E.sf.size();
        CMD_REQUIRE( ns >= 1 && ns <= NSF_LD && ns <= KPAD, CMD_ERR_ARG,
                     "element %d has %d symmetry functions (1..%d supported)",
                     e, ns, KPAD );
        Q.nsf = ns;
        std::vector<std::pair<double, double>> rg, ag, ap;
        std::vector<int> re;
        for ( const auto &s : E.sf )
        {
            if ( rc < 0 )
                rc = s.rc;
            CMD_REQUIRE( s.rc == rc, CMD_ERR_ARG,
                         "all symmetry functions must share one cutoff" );
            if ( s.type == 2 )
            {
                find_or_add( rg, s.eta, s.rs );
                const int ne = m.nelem == 1 ? -1 : s.e1;
                if ( std::find( re.begin(), re.end(), ne ) == re.end() )
                    re.push_back( ne );
            }
            else if ( s.type == 3 )
            {
                CMD_REQUIRE( m.nelem == 1 || s.e1 < 0, CMD_ERR_ARG,
                             "angular functions must accept any neighbour "
                             "pair" );
                find_or_add( ag, s.eta, s.rs );
                find_or_add( ap, s.lambda, s.zeta );
            }
            else
            {
                set_error( "symmetry function type %d is not supported", s.type );
                return CMD_ERR_ARG;
            }
        }
        // the power-of-two grid in its own order, whatever the model's
        Q.pow2 = (int)ap.size() == POW_NAP;
        std::vector<std::pair<double, double>> pg;
        for ( int p = 0; p < POW_NAP; ++p )
        {
            pg.push_back( { p < 4 ? -1.0 : 1.0, POW_ZETA[p % 4] } );
            if ( std::find( ap.begin(), ap.end(), pg.back() ) == ap.end() )
                Q.pow2 = 0;
        }
        if ( Q.pow2 )
            ap = pg;
        CMD_REQUIRE( (int)rg.size() <= RG_MAX && (int)re.size() <= RE_MAX &&
                         (int)ag.size() <= AG_MAX && (int)ap.size() <= AP_MAX,
                     CMD_ERR_ARG, "symmetry-function grid too large" );
        Q.nrg = (int)rg.size();
        Q.nre = (int)re.size();
        Q.nag = (int)ag.size();
        Q.nap = (int)ap.size();
        for ( int g = 0; g < RG_MAX; ++g )
            for ( int k = 0; k < RE_MAX; ++k )
                Q.r_out[g][k] = -1;
        for ( int g = 0; g < AG_MAX; ++g )
            for ( int k = 0; k < AP_MAX; ++k )
                Q.a_out[g][k] = -1;
        for ( int g = 0; g < Q.nrg; ++g )
        {
            Q.r_eta[g] = (float)rg[g].first;
            Q.r_rs[g] = (float)rg[g].second;
        }
        for ( int k = 0; k < Q.nre; ++k )
            Q.r_el[k] = re[k];
        for ( int g = 0; g < Q.nag; ++g )
        {
            Q.a_eta[g] = (float)ag[g].first;
            Q.a_rs[g] = (float)ag[g].second;
        }
        for ( int p = 0; p < Q.nap; ++p )
        {
            Q.a_lam[p] = (float)ap[p].first;
            Q.a_zeta[p] = (float)ap[p].second;
            Q.a_lpref[p] = (float)( 1.0 - ap[p].second );
        }
        for ( int s = 0; s < ns; ++s )
        {
            const auto &f = E.sf[s];
            if ( f.type == 2 )
            {
                const int g = find_or_add( rg, f.eta, f.rs );
                const int ne = m.nelem == 1 ? -1 : f.e1;
                const int k = (int)( std::find( re.begin(), re.end(), ne ) - re.begin() );
                CMD_REQUIRE( Q.r_out[g][k] < 0, CMD_ERR_ARG,
                             "duplicate radial symmetry function" );
                Q.r_out[g][k] = s;
            }
            else
            {
                const int g = find_or_add( ag, f.eta, f.rs );
                const int p = find_or_add( ap, f.lambda, f.zeta );
                CMD_REQUIRE( Q.a_out[g][p] < 0, CMD_ERR_ARG,
                             "duplicate angular symmetry function" );
                Q.a_out[g][p] = s;
            }
        }
        for ( int g = 0; g < Q.nrg; ++g )
            for ( int k = 0; k < Q.nre; ++k )
                CMD_REQUIRE( Q.r_out[g][k] >= 0, CMD_ERR_ARG,
                             "radial functions do not form a grid" );
        for ( int g = 0; g < Q.nag; ++g )
            for ( int p = 0; p < Q.nap; ++p )
                CMD_REQUIRE( Q.a_out[g][p] >= 0, CMD_ERR_ARG,
                             "angular functions do not form a grid" );
        for ( int s = 0; s < NSF_LD; ++s )
        {
            Q.g_mul[s] = 0.0f;
            Q.g_add[s] = 0.0f;
        }
        for ( int s = 0; s < ns; ++s )
        {
            if ( m.scale )
            {
                const double w = E.gmax[s] - E.gmin[s];
                const double mul = w > 0.0 ? ( m.smax - m.smin ) / w : 0.0;
                Q.g_mul[s] = (float)mul;
                Q.g_add[s] = (float)( m.smin - mul * E.gmin[s] );
            }
            else
                Q.g_mul[s] = 1.0f;
        }
        Q.h1 = m.hidden[0];
        Q.h2 = m.hidden[1];
        Q.act1 = m.act[0] == 't';
        Q.act2 = m.act[1] == 't';
        Q.act3 = 0;
        CMD_REQUIRE( E.W.size() == 3 && E.W[0].size() == (size_t)Q.h1 * ns &&
                         E.W[1].size() == (size_t)Q.h2 * Q.h1 &&
                         E.W[2].size() == (size_t)Q.h2,
                     CMD_ERR_ARG, "network weights of element %d are missing", e );
        for ( int o = 0; o < Q.h1; ++o )
        {
            for ( int k = 0; k < ns; ++k )
                Q.W1[o][k] = (float)E.W[0][(size_t)o * ns + k];
            Q.b1[o] = (float)E.b[0][o];
        }
        for ( int o = 0; o < Q.h2; ++o )
        {
            for ( int k = 0; k < Q.h1; ++k )
                Q.W2[o][k] = (float)E.W[1][(size_t)o * Q.h1 + k];
            Q.b2[o] = (float)E.b[1][o];
        }
        for ( int k = 0; k < Q.h2; ++k )
            Q.w3[k] = (float)E.W[2][k];
        Q.b3 = (float)E.b[2][0];
        for ( int o = 0; o < HPAD; ++o )
        {
            for ( int k = 0; k < KPAD; ++k )
            {
                unsigned short part[3];
                Q.W1T[k][o] = Q.W1[o][k];
                bf16_split3( Q.W1[o][k], part );
                for ( int q = 0; q < 3; ++q )
                {
                    Q.W1s[q][o][k] = part[q];
                    Q.W1Ts[q][k][o] = part[q];
                }
            }
            for ( int k = 0; k < HPAD; ++k )
            {
                unsigned short part[3];
                Q.W2T[k][o] = Q.W2[o][k];
                bf16_split3( Q.W2[o][k], part );
                for ( int q = 0; q < 3; ++q )
                {
                    Q.W2s[q][o][k] = part[q];
                    Q.W2Ts[q][k][o] = part[q];
                }
            }
        }
    }
    P.rc = (float)rc;
    P.rc2 = (float)( rc * rc );
    P.pi_rc = (float)( 3.14159265358979323846 / rc );
    return CMD_OK;
}

// ---------------------------------------------------------------- device
// Cosine cutoff 0.5 (cos(pi r / rc) + 1) and its derivative; k = pi / rc.
__device__ __forceinline__ float fcut( float r, float rc, float k )
{
    return r < rc ? 0.5f * ( __cosf( k * r ) + 1.0f ) : 0.0f;
}
__device__ __forceinline__ float dfcut( float r, float rc, float k )
{
    return r < rc ? -0.5f * k * __sinf( k * r ) : 0.0f;
}

// The angular constants of one element, held in scalar registers through
// the triplet loops (read once per wave from LDS, so the compiler cannot
// reload them from memory inside the loop).
struct AngK
{
    int nag, nap;
    unsigned lampos; // bit pp: lambda_pp > 0
    float eta[AG_MAX], rs[AG_MAX];
    float zeta[AP_MAX], lpref[AP_MAX], zm1[AP_MAX], zl[AP_MAX];
};

__device__ __forceinline__ AngK load_angk( const NnpElemPlan &Q, float *stage )
{
    const int lane = threadIdx.x & 63;
    // stage: eta[8] rs[8] zeta[8] lpref[8] lam[8]
    if ( lane < 40 )
    {
        const int k = lane & 7, w = lane >> 3;
        float v = 0.f;
        if ( w == 0 )
            v = Q.a_eta[k];
        else if ( w == 1 )
            v = Q.a_rs[k];
        else if ( w == 2 )
            v = Q.a_zeta[k];
        else if ( w == 3 )
            v = Q.a_lpref[k];
        else
            v = Q.a_lam[k];
        stage[lane] = v;
    }
    __builtin_amdgcn_fence( __ATOMIC_SEQ_CST, "wavefront" );
    AngK K;
    K.nag = __builtin_amdgcn_readfirstlane( Q.nag );
    K.nap = __builtin_amdgcn_readfirstlane( Q.nap );
    K.lampos = 0u;
#pragma unroll
    for ( int k = 0; k < AG_MAX; ++k )
    {
        K.eta[k] = __builtin_bit_cast( float, __builtin_amdgcn_readfirstlane(
                                                   __builtin_bit_cast( int, stage[k] ) ) );
        K.rs[k] = __builtin_bit_cast( float, __builtin_amdgcn_readfirstlane(
                                                  __builtin_bit_cast( int, stage[8 + k] ) ) );
    }
#pragma unroll
    for ( int k = 0; k < AP_MAX; ++k )
    {
        const float z = __builtin_bit_cast( float, __builtin_amdgcn_readfirstlane(
                                                       __builtin_bit_cast( int, stage[16 + k] ) ) );
        const float lp = __builtin_bit_cast( float, __builtin_amdgcn_readfirstlane(
                                                        __builtin_bit_cast( int, stage[24 + k] ) ) );
        const float lam = __builtin_bit_cast( float, __builtin_amdgcn_readfirstlane(
                                                         __builtin_bit_cast( int, stage[32 + k] ) ) );
        K.zeta[k] = z;
        K.lpref[k] = lp;
        K.zm1[k] = z - 1.f;
        K.zl[k] = z * lam;
        if ( lam > 0.f )
            K.lampos |= 1u << k;
    }
    __builtin_amdgcn_fence( __ATOMIC_SEQ_CST, "wavefront" );
    return K;
}

// Angular factors of the element's (lambda, zeta) grid for cos theta = cs:
// Pw = 2^(1-zeta) (1 + lambda cs)^zeta through the hardware log2/exp2
// (exp2(-inf) = 0), and Dw = zeta lambda 2^(1-zeta) (1 + lambda cs)^(zeta-1),
// the derivative of Pw with respect to cs, as zeta lambda Pw / base.  For
// zeta = 1, Dw = lambda, also at base = 0 (collinear neighbours); for
// zeta > 1 at base = 0 both are 0 (the reciprocal is taken as 0 there).
template <bool WANT_D>
__device__ __forceinline__ void ang_powers( const AngK &K, float cs, float *Pw, float *Dw )
{
    const float bp = fmaxf( 1.0f + cs, 0.0f ), bm = fmaxf( 1.0f - cs, 0.0f );
    const float lbp = __builtin_amdgcn_logf( bp );
    const float lbm = __builtin_amdgcn_logf( bm );
    float ibp = 0.0f, ibm = 0.0f;
    if ( WANT_D )
    {
        ibp = bp > 0.0f ? __builtin_amdgcn_rcpf( bp ) : 0.0f;
        ibm = bm > 0.0f ? __builtin_amdgcn_rcpf( bm ) : 0.0f;
    }
#pragma unroll
    for ( int pp = 0; pp < AP_MAX; ++pp )
    {
        Pw[pp] = 0.0f;
        if ( WANT_D )
            Dw[pp] = 0.0f;
        if ( pp < K.nap )
        {
            const bool pos = ( K.lampos >> pp ) & 1u;
            const float lb = pos ? lbp : lbm;
            Pw[pp] = __builtin_amdgcn_exp2f( K.zeta[pp] * lb + K.lpref[pp] );
            if ( WANT_D )
                Dw[pp] = K.zm1[pp] != 0.f ? K.zl[pp] * Pw[pp] * ( pos ? ibp : ibm ) : K.zl[pp];
        }
    }
}

// Reduce-scatter across the 64 lanes: in: v[S] per lane; out: v[0] of
// lane l = the sum over lanes of value l (S = 64) or l & 31 (S = 32).
// Each halving step keeps the half selected by one lane bit and sends the
// other half to the partner lane, so S values cost S - 1 exchanges in all.
// The 32- and 16-lane exchanges are one swap of the two halves' registers
// (after it, one register holds the kept value of every lane and the other
// the received one); the shorter ones go through the row rotations and quad
// permutes of the adder's operand, so no step waits on LDS.
template <int CTRL>
__device__ __forceinline__ float dpp_f( float v )
{
    return __builtin_bit_cast( float, __builtin_amdgcn_update_dpp(
                                          0, __builtin_bit_cast( int, v ), CTRL, 0xf, 0xf, true ) );
}

template <int O>
__device__ __forceinline__ float lane_xor( float v )
{
    if constexpr ( O == 8 )
        return dpp_f<0x128>( v ); // row_ror:8
    else if constexpr ( O == 2 )
        return dpp_f<0x4e>( v ); // quad_perm [2,3,0,1]
    else if constexpr ( O == 1 )
        return dpp_f<0xb1>( v ); // quad_perm [1,0,3,2]
    else
        return __shfl_xor( v, O, 64 );
}

template <int M>
__device__ __forceinline__ void rs_step( float *v, int lane )
{
    if constexpr ( M > 1 )
    {
        constexpr int O = M / 2;
        if constexpr ( O >= 16 )
        {
#pragma unroll
            for ( int k = 0; k < O; ++k )
            {
                const unsigned a = __builtin_bit_cast( unsigned, v[k] ),
                               b = __builtin_bit_cast( unsigned, v[O + k] );
                const auto r = O == 32 ? __builtin_amdgcn_permlane32_swap( a, b, false, false )
                                       : __builtin_amdgcn_permlane16_swap( a, b, false, false );
                v[k] = __builtin_bit_cast( float, (unsigned)r[0] ) +
                       __builtin_bit_cast( float, (unsigned)r[1] );
            }
        }
        else
        {
            const bool hi = lane & O;
#pragma unroll
            for ( int k = 0; k < O; ++k )
            {
                const float keep = hi ? v[O + k] : v[k];
                const float send = hi ? v[k] : v[O + k];
                v[k] = keep + lane_xor<O>( send );
            }
        }
        rs_step<O>( v, lane );
    }
}

template <int S>
__device__ __forceinline__ void wave_reduce_scatter( float *v )
{
    const int lane = threadIdx.x & 63;
    rs_step<S>( v, lane );
    if constexpr ( S == 32 )
        v[0] += __shfl_xor( v[0], 32, 64 );
}

// Neighbours of one atom inside rc: d = (x_j - x_i, r) and
// e = (1 / r, fc(r), dfc(r), element as float bits), two 16-byte reads each.
struct NbLds
{
    float4 d[NN_MAX];
    float4 e[NN_MAX];
    int j[NN_MAX];
};

// Compact the neighbours of atom i inside rc into LDS; returns the count
// (wave-uniform).  Sets *flag on overflow.
__device__ int gather_neighbours( int i, const double4 *__restrict__ x,
                                  const int64_t *__restrict__ off,
                                  const int *__restrict__ idx, float rc,
                                  float rc2, float kpi, NbLds &L,
                                  int *__restrict__ flag )
{
    const int lane = threadIdx.x & 63;
    const double4 xi = x[i];
    const int64_t o0 = off[i];
    const int n = (int)( off[i + 1] - o0 );
    int cnt = 0;
    for ( int base = 0; base < n; base += 64 )
    {
        const int k = base + lane;
        bool in = false;
        float dx = 0.f, dy = 0.f, dz = 0.f, r2 = 0.f;
        int j = 0;
        if ( k < n )
        {
            j = idx[o0 + k];
            const double4 xj = x[j];
            dx = (float)( xj.x - xi.x );
            dy = (float)( xj.y - xi.y );
            dz = (float)( xj.z - xi.z );
            r2 = dx * dx + dy * dy + dz * dz;
            in = r2 < rc2;
        }
        const unsigned long long m = __ballot( in );
        const int pos = cnt + (int)__builtin_amdgcn_mbcnt_hi(
                                  (unsigned)( m >> 32 ),
                                  __builtin_amdgcn_mbcnt_lo( (unsigned)m, 0u ) );
        if ( in && pos < NN_MAX )
        {
            const float r = __builtin_amdgcn_sqrtf( r2 );
            L.d[pos] = make_float4( dx, dy, dz, r );
            L.e[pos] = make_float4( __builtin_amdgcn_rcpf( r ), fcut( r, rc, kpi ),
                                    dfcut( r, rc, kpi ),
                                    __builtin_bit_cast( float, (int)x[j].w ) );
            L.j[pos] = j;
        }
        cnt += (int)__popcll( m );
    }
    if ( cnt > NN_MAX )
    {
        if ( lane == 0 )
            atomicOr( flag, 1 );
        cnt = NN_MAX;
    }
    __builtin_amdgcn_fence( __ATOMIC_SEQ_CST, "wavefront" );
    return cnt;
}

// Pair index p of n items -> (a, q), a < q, row-major over a.
__device__ __forceinline__ void pair_of( int p, int n, int &a, int &q )
{
    const float tn = 2.0f * n - 1.0f;
    int aa = (int)( ( tn - sqrtf( tn * tn - 8.0f * (float)p ) ) * 0.5f );
    aa = max( 0, min( aa, n - 2 ) );
    // start of row aa: aa*(2n - aa - 1)/2
    while ( aa > 0 && aa * ( 2 * n - aa - 1 ) / 2 > p )
        --aa;
    while ( ( aa + 1 ) * ( 2 * n - aa - 2 ) / 2 <= p )
        ++aa;
    a = aa;
    q = p - aa * ( 2 * n - aa - 1 ) / 2 + aa + 1;
}

// The neighbour pairs (a < q) of the gathered list whose third side is
// inside the cutoff, |x_q - x_a| < rc: tested 64 at a time and compacted
// into buf (CAP entries per wave, a | q << 8; NN_MAX <= 256), then handed to body(a, q)
// with every lane busy (lane l takes entries l*per .. l*per + per - 1).
// Used where the body keeps many accumulators in registers.
// A wave that shares the atom with others takes every its-th test from it0.
// With ALL the body runs in every lane of the wave, as body(a, q, ok): lanes
// past the list repeat its last pair with ok false.
// With PAIRS the body takes two pairs at once, (a0, q0) and (a1, q1), the
// second valid when ok1 (else a repeat of the first): the two gradient
// chains are independent, so their latencies overlap.
template <bool PAIRS = false, int CAP = TCAP, bool ALL = false, class Body>
__device__ __forceinline__ void for_triplets( const NbLds &L, int n, float rc2,
                                             unsigned short *buf, Body body,
                                             int *count = nullptr, int it0 = 0, int its = 1 )
{
    const int lane = threadIdx.x & 63;
    // candidate pairs, 64 per test: with n <= 64 rows a and n - 2 - a side
    // by side (n - 1 - a and a + 1 entries: n in all), else the flat pair
    // index through pair_of
    const bool rows = n <= 64;
    const int np = n * ( n - 1 ) / 2;
    const int nit = rows ? n / 2 : ( np + 63 ) / 64; // rows: pairs of rows
    for ( int it = it0; it < nit; )
    {
        int cnt = 0;
        while ( cnt <= CAP - 64 && it < nit )
        {
            bool ok = false;
            unsigned short code = 0;
            int a = 0, q = 0;
            bool have;
            if ( rows )
            {
                // rows a1 < a2 hold n - 1 - a1 and n - 1 - a2 = a1 + 1
                // entries; the middle row of an even n comes alone
                const int a1 = it, a2 = n - 2 - it;
                const int len1 = n - 1 - a1, len2 = a2 > a1 ? n - 1 - a2 : 0;
                have = lane < len1 + len2;
                if ( lane < len1 )
                {
                    a = a1;
                    q = a1 + 1 + lane;
                }
                else
                {
                    a = a2;
                    q = a2 + 1 + ( lane - len1 );
                }
            }
            else
            {
                const int p = it * 64 + lane;
                have = p < np;
                if ( have )
                    pair_of( p, n, a, q );
            }
            if ( have )
            {
                const float4 A = L.d[a], B = L.d[q];
                const float cx = B.x - A.x, cy = B.y - A.y, cz = B.z - A.z;
                ok = cx * cx + cy * cy + cz * cz < rc2;
                code = (unsigned short)( a | ( q << 8 ) );
            }
            const unsigned long long m = __ballot( ok );
            if ( ok )
                buf[cnt + (int)__builtin_amdgcn_mbcnt_hi(
                              (unsigned)( m >> 32 ),
                              __builtin_amdgcn_mbcnt_lo( (unsigned)m, 0u ) )] = code;
            cnt += (int)__popcll( m );
            it += its;
        }
        __builtin_amdgcn_fence( __ATOMIC_SEQ_CST, "wavefront" );
        if ( count )
            *count += cnt;
        const int per = ( cnt + 63 ) >> 6;
        if constexpr ( PAIRS )
        {
            for ( int j = 0; j < per; j += 2 )
            {
                const int e = lane * per + j;
                if ( e < cnt )
                {
                    const unsigned c0 = buf[e];
                    const bool ok1 = j + 1 < per && e + 1 < cnt;
                    const unsigned c1 = ok1 ? buf[e + 1] : c0;
                    body( (int)( c0 & 0xffu ), (int)( c0 >> 8 ), (int)( c1 & 0xffu ),
                          (int)( c1 >> 8 ), ok1 );
                }
            }
        }
        else if constexpr ( ALL )
        {
            for ( int j = 0; j < per; ++j )
            {
                const int e = lane * per + j;
                const unsigned c = buf[min( e, cnt - 1 )];
                body( (int)( c & 0xffu ), (int)( c >> 8 ), e < cnt );
            }
        }
        else
        {
            for ( int j = 0; j < per; ++j )
            {
                const int e = lane * per + j;
                if ( e < cnt )
                {
                    const unsigned c = buf[e];
                    body( (int)( c & 0xffu ), (int)( c >> 8 ) );
                }
            }
        }
        __builtin_amdgcn_fence( __ATOMIC_SEQ_CST, "wavefront" );
    }
}

// Walk of the neighbour pairs of an atom with n <= 64 neighbours whose third
// side is inside the cutoff, with every lane busy and no atomics.  Row d
// (1 <= d <= n / 2) pairs neighbour l with neighbour (l + d) mod n in lane l,
// so a row's test reads the partners from consecutive LDS records and its
// valid pairs are one 64-bit mask.  The valid pairs of consecutive rows are
// compacted into a ring of PAIR_RING codes; step(slot, l, p, ok) runs on 64 of
// them at a time: in every lane of the wave with ROWS (lanes past the last pair
// repeat it with ok false), else in the lanes that have one.  Once all pairs of a row are done, row(d, mask, start) may
// collect what step left at ring slots start, start + 1, ... (one per mask
// bit in lane order) -- each neighbour meets each of its pairs there in its
// own lane, which replaces reactions added with LDS atomics: at 192,000 atoms
// those took half of the force kernel's 3794 us, which the ring, the matrix
// products of the coefficients (k_nnp_force_pow) and six blocks per CU brought
// to 1795 us, 87 % of them VALU issue (1742 us with the steps' loads outside
// the branch of the lanes that have a pair); the symmetry functions, which use
// the steps alone, went from 996 to 893 us.
constexpr int PAIR_RING = 256;

// set bits of m below the lane's
__device__ __forceinline__ int lanes_below( unsigned long long m )
{
    return (int)__builtin_amdgcn_mbcnt_hi( (unsigned)( m >> 32 ),
                                           __builtin_amdgcn_mbcnt_lo( (unsigned)m, 0u ) );
}

// the partner (l + d) mod n, for l < n and d < n
__device__ __forceinline__ int pair_partner( int l, int d, int n )
{
    const int p = l + d;
    return p >= n ? p - n : p;
}

// Without ROWS only the steps run (row is not called).  With WPA waves on an
// atom, wave `part` takes the rows part + 1, part + 1 + WPA, ...
template <bool ROWS, int WPA, class Step, class Row>
__device__ __forceinline__ int pair_ring( const NbLds &L, int n, float rc2, int part,
                                          unsigned short *code, Step step, Row row )
{
    const int lane = threadIdx.x & 63;
    const int nrow = ( n / 2 + WPA - 1 - part ) / WPA; // this wave's rows
    const float4 own = L.d[lane]; // lanes past n are masked out
    // prod pairs compacted, comp of them stepped; rows below made are
    // compacted, rows below done are collected and first is where row done
    // starts: a ring slot is reused only after its row is collected
    int prod = 0, comp = 0, made = 1, done = 1, first = 0;
    int mlo = 0, mhi = 0, mst = 0; // the k-th row's mask and start in lane k - 1
    auto row_d = [&]( int k ) { return part + 1 + WPA * ( k - 1 ); };
    while ( ROWS ? done <= nrow : ( made <= nrow || comp < prod ) )
    {
        if ( !ROWS )
            first = comp;
        while ( made <= nrow && prod - first <= PAIR_RING - 64 )
        {
            const int d = row_d( made );
            const int p = pair_partner( lane, d, n );
            // the middle row of an even n holds each pair once in its first
            // half
            const int lim = 2 * d == n ? d : n;
            bool ok = false;
            if ( lane < lim )
            {
                const float4 B = L.d[p];
                const float cx = B.x - own.x, cy = B.y - own.y, cz = B.z - own.z;
                ok = cx * cx + cy * cy + cz * cz < rc2;
            }
            const unsigned long long m = __ballot( ok );
            if ( ok )
                code[( prod + lanes_below( m ) ) & ( PAIR_RING - 1 )] =
                    (unsigned short)( lane | ( p << 8 ) );
            if ( ROWS )
            {
                const bool mine = lane == made - 1;
                mlo = mine ? (int)m : mlo;
                mhi = mine ? (int)( m >> 32 ) : mhi;
                mst = mine ? prod : mst;
            }
            prod += (int)__popcll( m );
            ++made;
        }
        __builtin_amdgcn_fence( __ATOMIC_SEQ_CST, "wavefront" );
        while ( prod - comp >= 64 || ( made > nrow && comp < prod ) )
        {
            const int e = comp + lane;
            if ( ROWS || e < prod )
            {
                const int slot = min( e, prod - 1 ) & ( PAIR_RING - 1 );
                const unsigned c = code[slot];
                step( slot, (int)( c & 0xffu ), (int)( c >> 8 ), e < prod );
            }
            comp = min( comp + 64, prod );
        }
        __builtin_amdgcn_fence( __ATOMIC_SEQ_CST, "wavefront" );
        while ( ROWS && done < made )
        {
            const unsigned lo = __builtin_amdgcn_readlane( mlo, done - 1 ),
                           hi = __builtin_amdgcn_readlane( mhi, done - 1 );
            const unsigned long long mu = lo | ( (unsigned long long)hi << 32 );
            first = __builtin_amdgcn_readlane( mst, done - 1 );
            const int end = first + (int)__popcll( mu );
            if ( end > comp )
                break;
            row( row_d( done ), mu, first );
            first = end;
            ++done;
        }
    }
    return prod;
}

// Radial symmetry functions of one atom, lanes over its neighbours.
__device__ __forceinline__ void radial_sf( const NnpElemPlan &Q, const NbLds &L, int n,
                                           float *__restrict__ Gi )
{
    const int lane = threadIdx.x & 63;
    float acc[NR_MAX];
#pragma unroll
    for ( int s = 0; s < NR_MAX; ++s )
        acc[s] = 0.0f;
    for ( int a = lane; a < n; a += 64 )
    {
        const float4 Ea = L.e[a];
        const float r = L.d[a].w, fc = Ea.y;
        const int ej = __builtin_bit_cast( int, Ea.w );
#pragma unroll
        for ( int g = 0; g < RG_MAX; ++g )
        {
            if ( g < Q.nrg )
            {
                const float t = r - Q.r_rs[g];
                const float v = __expf( -Q.r_eta[g] * t * t ) * fc;
#pragma unroll
                for ( int k = 0; k < RE_MAX; ++k )
                    if ( k < Q.nre && ( Q.r_el[k] < 0 || Q.r_el[k] == ej ) )
                        acc[g * RE_MAX + k] += v;
            }
        }
    }
    wave_reduce_scatter<NR_MAX>( acc );
    if ( lane < NR_MAX )
    {
        const int g = lane / RE_MAX, k = lane % RE_MAX;
        if ( g < Q.nrg && k < Q.nre )
            Gi[Q.r_out[g][k]] = acc[0];
    }
}

// f = 0 over the nt local and ghost rows and the G columns past the atom's
// functions, by the first kernel of a force call (no launches of their own).
__device__ __forceinline__ void zero_forces( double *__restrict__ f, int fcap, int nt )
{
    for ( int k = blockIdx.x * blockDim.x + threadIdx.x; k < nt; k += gridDim.x * blockDim.x )
    {
        f[k] = 0.0;
        f[fcap + k] = 0.0;
        f[2 * fcap + k] = 0.0;
    }
}

__device__ __forceinline__ void zero_tail( const NnpElemPlan &Q, float *__restrict__ Gi )
{
    for ( int k = Q.nsf + ( threadIdx.x & 63 ); k < NSF_LD; k += 64 )
        Gi[k] = 0.f;
}

// NAG, NAP > 0: the angular (eta, rs) and (lambda, zeta) grid sizes of
// every element, fixed at compile time (loops unrolled straight); 0: read
// from the plan.  RS0: every element's angular rs are 0, so the Gaussian
// argument r_ij^2 + r_ik^2 + r_jk^2 is shared by all eta (a kernel of its
// own: with both paths in one kernel the registers of the longer one would
// cost occupancy).
template <int NAG, int NAP, bool RS0>
__global__ __launch_bounds__( NNP_TPB ) void k_nnp_sf(
    int n_local, const double4 *__restrict__ x, const int64_t *__restrict__ off,
    const int *__restrict__ idx, const NnpPlan *__restrict__ P,
    float *__restrict__ G, int *__restrict__ flag, int4 *__restrict__ terms,
    double *__restrict__ f, int fcap, int nt )
{
    __shared__ NbLds lds[NNP_TPB / 64];
    __shared__ unsigned short tbuf[NNP_TPB / 64][TCAP];
    __shared__ float kst[NNP_TPB / 64][64];
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    zero_forces( f, fcap, nt );
    const int i = blockIdx.x * ( NNP_TPB / 64 ) + wv;
    if ( i >= n_local )
        return;
    NbLds &L = lds[wv];
    const float rc = P->rc, rc2 = P->rc2, kpi = P->pi_rc;
    const int n = gather_neighbours( i, x, off, idx, rc, rc2, kpi, L, flag );
    const int e = __builtin_amdgcn_readfirstlane( (int)x[i].w );
    const NnpElemPlan &Q = P->el[e];
    AngK K = load_angk( Q, kst[wv] );
    if constexpr ( NAG > 0 )
        K.nag = NAG;
    if constexpr ( NAP > 0 )
        K.nap = NAP;
    float *Gi = G + (size_t)i * NSF_LD;
    zero_tail( Q, Gi );
    radial_sf( Q, L, n, Gi );
    // angular: lanes over the compacted neighbour pairs
    {
        float acc[NA_MAX];
#pragma unroll
        for ( int s = 0; s < NA_MAX; ++s )
            acc[s] = 0.0f;
        int ntrip = 0;
        for_triplets(
            L, n, rc2, tbuf[wv], [&]( int a, int q ) {
            const float4 A = L.d[a], B = L.d[q], Ea = L.e[a], Eb = L.e[q];
            const float cx = B.x - A.x, cy = B.y - A.y, cz = B.z - A.z;
            const float r3 = __builtin_amdgcn_sqrtf( cx * cx + cy * cy + cz * cz );
            const float F = Ea.y * Eb.y * fcut( r3, rc, kpi );
            const float cs = ( A.x * B.x + A.y * B.y + A.z * B.z ) * ( Ea.x * Eb.x );
            float Pw[AP_MAX];
            ang_powers<false>( K, cs, Pw, nullptr );
            if constexpr ( RS0 )
            {
                // one Gaussian argument, and the cutoff product joins the
                // Gaussian (nag multiplies, not nap)
                const float s2 = A.w * A.w + B.w * B.w + r3 * r3;
#pragma unroll
                for ( int g = 0; g < AG_MAX; ++g )
                {
                    if ( g < K.nag )
                    {
                        const float EgF = __expf( -K.eta[g] * s2 ) * F;
#pragma unroll
                        for ( int pp = 0; pp < AP_MAX; ++pp )
                            acc[g * AP_MAX + pp] += EgF * Pw[pp];
                    }
                }
            }
            else
            {
#pragma unroll
                for ( int pp = 0; pp < AP_MAX; ++pp )
                    Pw[pp] *= F;
#pragma unroll
                for ( int g = 0; g < AG_MAX; ++g )
                {
                    if ( g < K.nag )
                    {
                        const float rs = K.rs[g];
                        const float t1 = A.w - rs, t2 = B.w - rs, t3 = r3 - rs;
                        const float Eg = __expf( -K.eta[g] * ( t1 * t1 + t2 * t2 + t3 * t3 ) );
#pragma unroll
                        for ( int pp = 0; pp < AP_MAX; ++pp )
                            acc[g * AP_MAX + pp] += Eg * Pw[pp];
                    }
                }
            }
            },
            &ntrip );
        // the work model's term counts (roofline.h) of this atom: its
        // neighbours and triplets, and its element for the per-element
        // grids (one store per atom, summed when asked for)
        if ( terms && lane == 0 )
            terms[i] = make_int4( n, ntrip, e, 0 );
        wave_reduce_scatter<NA_MAX>( acc );
        const int g = lane / AP_MAX, pp = lane % AP_MAX;
        if ( g < Q.nag && pp < Q.nap )
            Gi[Q.a_out[g][pp]] = acc[0];
    }
}

// ---- the power-of-two (lambda, zeta) grid, angular rs = 0
//
// Both kernels below run on the models whose every element has the POW_*
// grid, NAG (the number of angular etas, the same for all elements) and
// angular rs of 0 -- the usual n2p2 form -- in place of the general ones.
// They are bound by FP32 VALU issue, so they are written for few operations
// per triplet: (1 + lambda cos)^zeta by squarings (no log2 and exp2, and
// exact to a few roundings for zeta = 16), 2^(1 - zeta) applied to the
// finished sum or the coefficients, one reciprocal square root for r_jk and
// 1 / r_jk, and constants in scalar registers.

// A constant of the lane-held table t as a wave-uniform value.
__device__ __forceinline__ float lane_value( float t, int k )
{
    return __builtin_bit_cast(
        float, __builtin_amdgcn_readlane( __builtin_bit_cast( int, t ), k ) );
}

// b^1, b^2, b^4, b^16
__device__ __forceinline__ void pow_grid( float b, float *p )
{
    p[0] = b;
    p[1] = b * b;
    p[2] = p[1] * p[1];
    const float b8 = p[2] * p[2];
    p[3] = b8 * b8;
}

template <int NAG, int WPA>
__global__ __launch_bounds__( NNP_TPB ) void k_nnp_sf_pow(
    int n_local, const double4 *__restrict__ x, const int64_t *__restrict__ off,
    const int *__restrict__ idx, const NnpPlan *__restrict__ P,
    float *__restrict__ G, int *__restrict__ flag, int4 *__restrict__ terms,
    double *__restrict__ f, int fcap, int nt )
{
    __shared__ NbLds lds[NNP_TPB / 64];
    __shared__ unsigned short tbuf[NNP_TPB / 64][TCAP];
    const int wv = __builtin_amdgcn_readfirstlane( threadIdx.x >> 6 ), lane = threadIdx.x & 63;
    zero_forces( f, fcap, nt );
    // with WPA = 4 the block's waves share an atom (one exit for all)
    const int part = WPA > 1 ? wv : 0;
    const int i = WPA > 1 ? (int)blockIdx.x : blockIdx.x * ( NNP_TPB / 64 ) + wv;
    if ( i >= n_local )
        return;
    NbLds &L = lds[wv];
    const float rc = P->rc, rc2 = P->rc2, kpi = P->pi_rc;
    const int n = gather_neighbours( i, x, off, idx, rc, rc2, kpi, L, flag );
    const int e = __builtin_amdgcn_readfirstlane( (int)x[i].w );
    const NnpElemPlan &Q = P->el[e];
    float *Gi = G + (size_t)i * NSF_LD;
    if ( part == 0 )
    {
        zero_tail( Q, Gi );
        radial_sf( Q, L, n, Gi );
    }
    // exp(-eta s) = exp2(k s)
    const float kl = -1.44269504f * Q.a_eta[lane & ( AG_MAX - 1 )];
    float ke[NAG];
#pragma unroll
    for ( int g = 0; g < NAG; ++g )
        ke[g] = lane_value( kl, g );
    const float kcos = 0.5f / rc; // cos(pi r / rc) in revolutions
    float acc[NA_MAX];
#pragma unroll
    for ( int s = 0; s < NA_MAX; ++s )
        acc[s] = 0.0f;
    auto triplet = [&]( int a, int q )
    {
        const float4 A = L.d[a], B = L.d[q], Ea = L.e[a], Eb = L.e[q];
        const float cx = B.x - A.x, cy = B.y - A.y, cz = B.z - A.z;
        const float c2 = cx * cx + cy * cy + cz * cz;
        const float f3 =
            0.5f + 0.5f * __builtin_amdgcn_cosf( __builtin_amdgcn_sqrtf( c2 ) * kcos );
        const float F = Ea.y * Eb.y * f3;
        const float cs = ( A.x * B.x + A.y * B.y + A.z * B.z ) * ( Ea.x * Eb.x );
        const float s2 = A.w * A.w + ( B.w * B.w + c2 );
        float Pw[POW_NAP];
        pow_grid( fmaxf( 1.0f - cs, 0.0f ), Pw );
        pow_grid( fmaxf( 1.0f + cs, 0.0f ), Pw + 4 );
#pragma unroll
        for ( int g = 0; g < NAG; ++g )
        {
            const float EgF = __builtin_amdgcn_exp2f( ke[g] * s2 ) * F;
#pragma unroll
            for ( int pp = 0; pp < POW_NAP; ++pp )
                acc[g * AP_MAX + pp] += EgF * Pw[pp];
        }
    };
    int ntrip = 0;
    if ( n <= 64 )
        ntrip = pair_ring<false, WPA>(
            L, n, rc2, part, tbuf[wv], [&]( int, int a, int q, bool ) { triplet( a, q ); },
            []( int, unsigned long long, int ) {} );
    else
        for_triplets( L, n, rc2, tbuf[wv], triplet, &ntrip, part, WPA );
    wave_reduce_scatter<NA_MAX>( acc );
    if constexpr ( WPA > 1 )
    {
        // the waves' sums and counts, through the neighbour tables
        lds[wv].e[lane].x = acc[0];
        if ( lane == 0 )
            lds[wv].j[0] = ntrip;
        __syncthreads();
        if ( part != 0 )
            return;
        for ( int w = 1; w < WPA; ++w )
        {
            acc[0] += lds[w].e[lane].x;
            ntrip += lds[w].j[0];
        }
    }
    // the work model's term counts, as in k_nnp_sf
    if ( terms && lane == 0 )
        terms[i] = make_int4( n, ntrip, e, 0 );
    const int g = lane / AP_MAX, pp = lane % AP_MAX;
    if ( g < NAG )
        Gi[Q.a_out[g][pp]] = acc[0] * __builtin_amdgcn_exp2f( Q.a_lpref[pp] );
}

// ---- network: split-BF16 MFMA, 16 atoms of one element per wave
//
// Every layer product runs on gfx950's 16x16x32 BF16 MFMA with FP32
// accumulation.  Each FP32 operand is split into three BF16 parts (a = ah +
// am + al, exact for FP32 values), and a product sums the six part products
// of order up to 2^-16 relative (ah bh, ah bm, am bh, am bm, ah bl, al bh),
// smallest first: the result matches an FP32 product to about 2^-24, while a
// single BF16 product carries 2^-8.  The weights come pre-split from the
// plan; activations are split as they are loaded.
typedef __bf16 bf16x8 __attribute__( ( ext_vector_type( 8 ) ) );
typedef short s16x8 __attribute__( ( ext_vector_type( 8 ) ) );
typedef float f32x4 __attribute__( ( ext_vector_type( 4 ) ) );

__device__ __forceinline__ float act_f( float z, int tanh_ )
{
    return tanh_ ? tanhf( z ) : z;
}

// The three BF16 parts of 8 consecutive FP32 values.
__device__ __forceinline__ void split8( const float *v, bf16x8 &h, bf16x8 &m, bf16x8 &l )
{
    s16x8 sh, sm, sl;
#pragma unroll
    for ( int u = 0; u < 8; ++u )
    {
        unsigned short part[3];
        bf16_split3( v[u], part );
        sh[u] = (short)part[0];
        sm[u] = (short)part[1];
        sl[u] = (short)part[2];
    }
    h = __builtin_bit_cast( bf16x8, sh );
    m = __builtin_bit_cast( bf16x8, sm );
    l = __builtin_bit_cast( bf16x8, sl );
}

__device__ __forceinline__ bf16x8 load8( const unsigned short *p )
{
    return __builtin_bit_cast( bf16x8, *reinterpret_cast<const s16x8 *>( p ) );
}

// c += A B over one 32-deep K block, A from the three parts of the lane's
// 8 activations, B from the three weight parts at w[0], w[stride], w[2 stride].
__device__ __forceinline__ f32x4 mfma_split( const float *a8, const unsigned short *w,
                                             size_t stride, f32x4 c )
{
    bf16x8 ah, am, al;
    split8( a8, ah, am, al );
    const bf16x8 bh = load8( w ), bm = load8( w + stride ), bl = load8( w + 2 * stride );
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16( al, bh, c, 0, 0, 0 );
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16( ah, bl, c, 0, 0, 0 );
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16( am, bm, c, 0, 0, 0 );
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16( am, bh, c, 0, 0, 0 );
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16( ah, bm, c, 0, 0, 0 );
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16( ah, bh, c, 0, 0, 0 );
    return c;
}

// The same K block in FP32 on the 16x16x4 FP32 MFMA.  Any order of k serves
// the sum, so MFMA (j, u) takes k = 16 j + 4 (l / 16) + u in lane l and both
// operands are read 16 bytes at a time.
__device__ __forceinline__ f32x4 mfma_f32( const float *a, const float *w, f32x4 c )
{
#pragma unroll
    for ( int j = 0; j < 2; ++j )
    {
        const f32x4 av = *reinterpret_cast<const f32x4 *>( a + 16 * j );
        const f32x4 wv = *reinterpret_cast<const f32x4 *>( w + 16 * j );
#pragma unroll
        for ( int u = 0; u < 4; ++u )
            c = __builtin_amdgcn_mfma_f32_16x16x4f32( av[u], wv[u], c, 0, 0, 0 );
    }
    return c;
}

// The network of every element in one launch: energies and dE/dG, forward
// and backward, 16 atoms of one element per wave.  A block takes 64
// consecutive atoms and groups them by element in LDS (sum_e ceil(c_e / 16)
// <= 3 + nelem tiles, one per wave), so no grouping pass over the system and
// no per-element launch is needed.  F32 runs the products on the FP32 MFMA
// (FP32 operands and sums, as the per-atom dot products it replaces), else
// on split BF16 parts.  A tile is a serial chain of five products and two
// activations: latency bounds it, so the tiles of a block sit in separate
// waves and K ends at the element's function count.  Against one launch per
// element after a grouping pass, and one atom per lane in FP32, a whole step
// took: 19,652 atoms, 27-24-24-1, FP32 layers 437 -> 237 us; 3,000 atoms,
// two 70-25-25-1 networks, BF16 parts 288 -> 243 us (192,000 atoms: 5.63 ->
// 5.53 ms).
//
// MFMA 16x16x32 operand layout (per lane l): A[row = l % 16][k = 8 (l / 16)
// + 0..7], B[k = 8 (l / 16) + 0..7][col = l % 16], D[row = 4 (l / 16) + 0..3]
// [col = l % 16]; 16x16x4: A[row = l % 16][k = l / 16], B[k = l / 16]
// [col = l % 16], D as above.
constexpr int MLP_ATOMS = 64; // atoms per block
constexpr int MLP_WAVES = MLP_ATOMS / 16 + NNP_MAXEL - 1;

template <bool F32>
__global__ __launch_bounds__( 64 * MLP_WAVES ) void k_nnp_mlp(
    int n_local, int nelem, const double4 *__restrict__ x, const float *__restrict__ G,
    const NnpPlan *__restrict__ P, float *__restrict__ dEdG, float *__restrict__ Ei )
{
    extern __shared__ __align__( 16 ) float s_mlp[]; // per wave: row-major 16 x (KPAD + 4)
    __shared__ int s_atom[MLP_ATOMS];
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    // every wave groups the block's atoms the same way: rank of each atom in
    // element order, and the element and atoms of this wave's tile
    const int at = blockIdx.x * MLP_ATOMS + lane;
    const int el = at < n_local ? (int)x[at].w : -1;
    int elem = -1, first = 0, cnt = 0; // this wave's tile: s_atom[first ..)
    {
        int base = 0, tile = 0;
        for ( int e = 0; e < nelem; ++e )
        {
            const unsigned long long m = __ballot( el == e );
            const int c = (int)__popcll( m );
            if ( wv == 0 && el == e )
                s_atom[base + (int)__builtin_amdgcn_mbcnt_hi(
                                  (unsigned)( m >> 32 ),
                                  __builtin_amdgcn_mbcnt_lo( (unsigned)m, 0u ) )] = at;
            const int nt = ( c + 15 ) >> 4;
            if ( wv >= tile && wv < tile + nt )
            {
                elem = e;
                first = base + 16 * ( wv - tile );
                cnt = min( 16, c - 16 * ( wv - tile ) );
            }
            tile += nt;
            base += c;
        }
    }
    __syncthreads();
    elem = __builtin_amdgcn_readfirstlane( elem );
    if ( elem < 0 )
        return;
    const NnpElemPlan &Q = P->el[elem];
    constexpr int LDA = KPAD + 4;
    float *A = s_mlp + wv * 16 * LDA;
    const int row = lane & 15, kq = ( lane >> 4 ) * 4, k8 = ( lane >> 4 ) * 8;
    const int ka = F32 ? kq : k8; // first k of the lane in a 32-deep block
    const int nsf = Q.nsf, nkb = ( nsf + 31 ) >> 5;
    // scaled inputs, row-major in LDS, zero past nsf and past the tile's
    // atoms: lane group l / 16 takes every fourth quad of row l % 16
    {
        const bool have = row < cnt;
        const float *Gi = G + (size_t)s_atom[first + ( have ? row : 0 )] * NSF_LD;
        for ( int c = kq; c < 32 * nkb; c += 16 )
        {
            const f32x4 g = *reinterpret_cast<const f32x4 *>( Gi + c );
            const f32x4 mu = *reinterpret_cast<const f32x4 *>( Q.g_mul + c );
            const f32x4 ad = *reinterpret_cast<const f32x4 *>( Q.g_add + c );
            f32x4 v;
#pragma unroll
            for ( int u = 0; u < 4; ++u )
                v[u] = have && c + u < nsf ? mu[u] * g[u] + ad[u] : 0.f;
            *reinterpret_cast<f32x4 *>( A + row * LDA + c ) = v;
        }
    }
    __builtin_amdgcn_fence( __ATOMIC_SEQ_CST, "wavefront" );
    // one 32-deep K block: A row at k0, W in [col][k] order (split parts Ws)
    auto block = [&]( int k0, const float *W, const unsigned short *Ws, size_t stride, int ld,
                      int col, f32x4 c ) -> f32x4
    {
        if constexpr ( F32 )
            return mfma_f32( A + row * LDA + k0 + ka, W + (size_t)col * ld + k0 + ka, c );
        else
            return mfma_split( A + row * LDA + k0 + ka, Ws + (size_t)col * ld + k0 + ka, stride,
                               c );
    };
    const f32x4 zero = { 0.f, 0.f, 0.f, 0.f };
    // layer 1: h1[16 x 32] = Gs[16 x K] W1^T, B[k][col] = W1[col][k]
    f32x4 h1[2] = { zero, zero };
    for ( int kb = 0; kb < nkb; ++kb )
#pragma unroll
        for ( int nt = 0; nt < 2; ++nt )
            h1[nt] = block( kb * 32, &Q.W1[0][0], &Q.W1s[0][0][0], (size_t)HPAD * KPAD, KPAD,
                            nt * 16 + row, h1[nt] );
    __builtin_amdgcn_fence( __ATOMIC_SEQ_CST, "wavefront" );
    // bias + activation; h1 to LDS (row-major 16 x 32)
#pragma unroll
    for ( int nt = 0; nt < 2; ++nt )
#pragma unroll
        for ( int u = 0; u < 4; ++u )
        {
            const int r = kq + u, col = nt * 16 + row;
            const float z = h1[nt][u] + ( col < Q.h1 ? Q.b1[col] : 0.f );
            const float h = col < Q.h1 ? act_f( z, Q.act1 ) : 0.f;
            h1[nt][u] = h;
            A[r * LDA + col] = h;
        }
    __builtin_amdgcn_fence( __ATOMIC_SEQ_CST, "wavefront" );
    // layer 2: h2[16 x 32] = h1 W2^T, B[k][col] = W2[col][k]
    f32x4 h2[2];
#pragma unroll
    for ( int nt = 0; nt < 2; ++nt )
        h2[nt] = block( 0, &Q.W2[0][0], &Q.W2s[0][0][0], (size_t)HPAD * HPAD, HPAD,
                        nt * 16 + row, zero );
    __builtin_amdgcn_fence( __ATOMIC_SEQ_CST, "wavefront" );
    // output layer and the first backward step (VALU, FP32):
    // E = w3 . h2 + b3; delta2 = w3 * act'(z2)
    float epart[4] = { 0.f, 0.f, 0.f, 0.f };
#pragma unroll
    for ( int nt = 0; nt < 2; ++nt )
#pragma unroll
        for ( int u = 0; u < 4; ++u )
        {
            const int r = kq + u, col = nt * 16 + row;
            const float z = h2[nt][u] + ( col < Q.h2 ? Q.b2[col] : 0.f );
            const float h = col < Q.h2 ? act_f( z, Q.act2 ) : 0.f;
            const float w = col < Q.h2 ? Q.w3[col] : 0.f;
            epart[u] += h * w;
            A[r * LDA + col] = Q.act2 ? w * ( 1.f - h * h ) : w; // delta2, row-major
        }
    // sum the 16 columns held by the 16 lanes of each row group
#pragma unroll
    for ( int u = 0; u < 4; ++u )
    {
        float s = epart[u];
#pragma unroll
        for ( int o = 1; o < 16; o <<= 1 )
            s += __shfl_xor( s, o, 64 );
        epart[u] = s;
    }
    if ( row == 0 )
#pragma unroll
        for ( int u = 0; u < 4; ++u )
            if ( kq + u < cnt )
                Ei[s_atom[first + kq + u]] = epart[u] + Q.b3;
    __builtin_amdgcn_fence( __ATOMIC_SEQ_CST, "wavefront" );
    // delta1[16 x 32] = (delta2 W2) * act'(z1): B[k][col] = W2[k][col]
    f32x4 d1[2];
#pragma unroll
    for ( int nt = 0; nt < 2; ++nt )
        d1[nt] = block( 0, &Q.W2T[0][0], &Q.W2Ts[0][0][0], (size_t)HPAD * HPAD, HPAD,
                        nt * 16 + row, zero );
    __builtin_amdgcn_fence( __ATOMIC_SEQ_CST, "wavefront" );
#pragma unroll
    for ( int nt = 0; nt < 2; ++nt )
#pragma unroll
        for ( int u = 0; u < 4; ++u )
        {
            const int r = kq + u, col = nt * 16 + row;
            const float h = h1[nt][u];
            A[r * LDA + col] =
                col < Q.h1 ? ( Q.act1 ? d1[nt][u] * ( 1.f - h * h ) : d1[nt][u] ) : 0.f;
        }
    __builtin_amdgcn_fence( __ATOMIC_SEQ_CST, "wavefront" );
    // dE/dGs[16 x nsf] = delta1 W1: B[k][col] = W1[k][col]
    for ( int nt = 0; 16 * nt < nsf; ++nt )
    {
        const f32x4 c = block( 0, &Q.W1T[0][0], &Q.W1Ts[0][0][0], (size_t)KPAD * HPAD, HPAD,
                               nt * 16 + row, zero );
        const int col = nt * 16 + row;
#pragma unroll
        for ( int u = 0; u < 4; ++u )
            if ( kq + u < cnt && col < nsf )
                dEdG[(size_t)s_atom[first + kq + u] * NSF_LD + col] = c[u] * Q.g_mul[col];
    }
}

// ---- forces
// sum_s c_s dG_s/dr / r of the radial functions for neighbour a.
__device__ __forceinline__ float radial_force( const NnpElemPlan &Q, const NbLds &L, int a,
                                               const float *c )
{
    const float4 Ea = L.e[a];
    const float r = L.d[a].w, fc = Ea.y, dfc = Ea.z;
    const int ej = __builtin_bit_cast( int, Ea.w );
    float gsum = 0.f;
#pragma unroll
    for ( int g = 0; g < RG_MAX; ++g )
    {
        if ( g < Q.nrg )
        {
            const float t = r - Q.r_rs[g];
            const float ex = __expf( -Q.r_eta[g] * t * t );
            const float d = ex * ( -2.f * Q.r_eta[g] * t * fc + dfc );
            float cw = 0.f;
#pragma unroll
            for ( int k = 0; k < RE_MAX; ++k )
                if ( k < Q.nre && ( Q.r_el[k] < 0 || Q.r_el[k] == ej ) )
                    cw += c[Q.r_out[g][k]];
            gsum = fmaf( cw, d, gsum );
        }
    }
    return gsum * Ea.x;
}

template <int NAG, int NAP, bool RS0>
__global__ __launch_bounds__( NNP_TPB ) void k_nnp_force(
    int n_local, int fcap, const double4 *__restrict__ x,
    const int64_t *__restrict__ off, const int *__restrict__ idx,
    const NnpPlan *__restrict__ P, const float *__restrict__ dEdG,
    double *__restrict__ f, int *__restrict__ flag )
{
    __shared__ NbLds lds[NNP_TPB / 64];
    __shared__ float sF[NNP_TPB / 64][NN_MAX][3];
    __shared__ float sC[NNP_TPB / 64][NSF_LD];
    __shared__ float4 sCg[NNP_TPB / 64][NA_MAX / 4]; // c of angular (g, p) in grid order
    __shared__ unsigned short tbuf[NNP_TPB / 64][TCAP];
    __shared__ float kst[NNP_TPB / 64][64];
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int i = blockIdx.x * ( NNP_TPB / 64 ) + wv;
    if ( i >= n_local )
        return;
    NbLds &L = lds[wv];
    const float rc = P->rc, rc2 = P->rc2, kpi = P->pi_rc;
    const int n = gather_neighbours( i, x, off, idx, rc, rc2, kpi, L, flag );
    const int e = __builtin_amdgcn_readfirstlane( (int)x[i].w );
    const NnpElemPlan &Q = P->el[e];
    AngK K = load_angk( Q, kst[wv] );
    if constexpr ( NAG > 0 )
        K.nag = NAG;
    if constexpr ( NAP > 0 )
        K.nap = NAP;
    for ( int k = lane; k < NSF_LD; k += 64 )
        sC[wv][k] = k < Q.nsf ? dEdG[(size_t)i * NSF_LD + k] : 0.f;
    for ( int a = lane; a < n; a += 64 )
    {
        sF[wv][a][0] = 0.f;
        sF[wv][a][1] = 0.f;
        sF[wv][a][2] = 0.f;
    }
    __builtin_amdgcn_fence( __ATOMIC_SEQ_CST, "wavefront" );
    const float *c = sC[wv];
    float fix = 0.f, fiy = 0.f, fiz = 0.f;
    // radial
    for ( int a = lane; a < n; a += 64 )
    {
        const float4 A = L.d[a];
        const float s = radial_force( Q, L, a, c );
        const float vx = s * A.x, vy = s * A.y, vz = s * A.z;
        // dG/dx_j = g' u; F_j -= c g' u, F_i += c g' u
        sF[wv][a][0] -= vx;
        sF[wv][a][1] -= vy;
        sF[wv][a][2] -= vz;
        fix += vx;
        fiy += vy;
        fiz += vz;
    }
    __builtin_amdgcn_fence( __ATOMIC_SEQ_CST, "wavefront" );
    // angular: coefficients in grid order in LDS (the generic grid reads
    // them per pair, which keeps 64 registers free for occupancy)
    {
        float *cg = reinterpret_cast<float *>( sCg[wv] );
        for ( int k = lane; k < NA_MAX; k += 64 )
        {
            const int g = k / AP_MAX, pp = k % AP_MAX;
            cg[k] = ( g < Q.nag && pp < Q.nap ) ? c[Q.a_out[g][pp]] : 0.f;
        }
    }
    __builtin_amdgcn_fence( __ATOMIC_SEQ_CST, "wavefront" );
    const float4 *cg4 = sCg[wv];
    // with the grid fixed at compile time the coefficients are read once per
    // atom as wave-uniform values (scalar registers, the excess spilled to
    // lanes of vector registers) instead of from LDS per triplet: 4 % off
    // the kernel at 192,000 atoms
    float cgr[( NAG > 0 ? NAG : 1 ) * ( NAP > 0 ? NAP : 1 )];
    if constexpr ( NAG > 0 && NAP > 0 )
    {
        const float *cgf = reinterpret_cast<const float *>( sCg[wv] );
#pragma unroll
        for ( int g = 0; g < NAG; ++g )
#pragma unroll
            for ( int pp = 0; pp < NAP; ++pp )
                cgr[g * NAP + pp] = __builtin_bit_cast(
                    float, __builtin_amdgcn_readfirstlane(
                               __builtin_bit_cast( int, cgf[g * AP_MAX + pp] ) ) );
    }
    // angular: each lane takes a contiguous block of the compacted (a-major)
    // pair list, so the reaction on a stays in registers until a changes;
    // the one on q goes to LDS.
    int cur = -1;
    float ax = 0.f, ay = 0.f, az = 0.f; // reaction on row atom cur
    // gradients of sum_s c_s T_s of the triplet (i, a, q) with respect to
    // A = x_a - x_i (ga) and B = x_q - x_i (gb): no side effects, so two of
    // them run interleaved
    auto grad = [&]( int a, int q, float ( &ga )[3], float ( &gb )[3] ) {
        const float4 A = L.d[a], Ea = L.e[a];
        const float4 B = L.d[q], Eb = L.e[q];
        const float cx = B.x - A.x, cy = B.y - A.y, cz = B.z - A.z;
        const float r1 = A.w, r2 = B.w;
        const float r3 = __builtin_amdgcn_sqrtf( cx * cx + cy * cy + cz * cz );
        const float ia = Ea.x, ib = Eb.x, ic = __builtin_amdgcn_rcpf( r3 );
        const float f1 = Ea.y, f2 = Eb.y, f3 = fcut( r3, rc, kpi );
        const float d1 = Ea.z, d2 = Eb.z, d3 = dfcut( r3, rc, kpi );
        const float F = f1 * f2 * f3;
        const float inv12 = ia * ib;
        const float cs = ( A.x * B.x + A.y * B.y + A.z * B.z ) * inv12;
        float Pw[AP_MAX], Dw[AP_MAX];
        ang_powers<true>( K, cs, Pw, Dw );
        float Gs = 0.f, As = 0.f, B1 = 0.f, B2 = 0.f, B3 = 0.f;
        // sum_p c_gp P_p and sum_p c_gp D_p of one (eta, rs)
        auto cdots = [&]( int g, float &sp, float &sd )
        {
            sp = 0.f;
            sd = 0.f;
            if constexpr ( NAG > 0 && NAP > 0 )
            {
#pragma unroll
                for ( int pp = 0; pp < NAP; ++pp )
                {
                    sp = fmaf( cgr[g * NAP + pp], Pw[pp], sp );
                    sd = fmaf( cgr[g * NAP + pp], Dw[pp], sd );
                }
            }
            else
            {
#pragma unroll
                for ( int q4 = 0; q4 < AP_MAX / 4; ++q4 )
                {
                    const float4 cc = cg4[g * ( AP_MAX / 4 ) + q4];
                    const float cv[4] = { cc.x, cc.y, cc.z, cc.w };
#pragma unroll
                    for ( int u = 0; u < 4; ++u )
                    {
                        sp = fmaf( cv[u], Pw[q4 * 4 + u], sp );
                        sd = fmaf( cv[u], Dw[q4 * 4 + u], sd );
                    }
                }
            }
        };
        if constexpr ( RS0 )
        {
            // one Gaussian argument, and the distance gradients share one
            // factor, sum_g -2 eta_g w_g
            const float s2 = r1 * r1 + r2 * r2 + r3 * r3;
            float M2 = 0.f;
#pragma unroll
            for ( int g = 0; g < AG_MAX; ++g )
            {
                if ( g < K.nag )
                {
                    const float Eg = __expf( -K.eta[g] * s2 );
                    float sp, sd;
                    cdots( g, sp, sd );
                    const float w = sp * Eg; // sum_p c P E
                    Gs += w;
                    As = fmaf( sd, Eg, As );
                    M2 = fmaf( -2.f * K.eta[g], w, M2 );
                }
            }
            B1 = M2 * r1;
            B2 = M2 * r2;
            B3 = M2 * r3;
        }
        else
        {
#pragma unroll
            for ( int g = 0; g < AG_MAX; ++g )
            {
                if ( g < K.nag )
                {
                    const float rs = K.rs[g];
                    const float t1 = r1 - rs, t2 = r2 - rs, t3 = r3 - rs;
                    const float Eg = __expf( -K.eta[g] * ( t1 * t1 + t2 * t2 + t3 * t3 ) );
                    float sp, sd;
                    cdots( g, sp, sd );
                    const float w = sp * Eg; // sum_p c P E
                    Gs += w;
                    As = fmaf( sd, Eg, As );
                    const float m2 = -2.f * K.eta[g] * w;
                    B1 = fmaf( m2, t1, B1 );
                    B2 = fmaf( m2, t2, B2 );
                    B3 = fmaf( m2, t3, B3 );
                }
            }
        }
        // (T = pref P E F, r3 = |B - A|)
        const float dFa1 = d1 * f2 * f3, dF3 = f1 * f2 * d3, dFb2 = f1 * d2 * f3;
        const float Av[3] = { A.x, A.y, A.z }, Bv[3] = { B.x, B.y, B.z },
                    Cv[3] = { cx, cy, cz };
#pragma unroll
        for ( int k = 0; k < 3; ++k )
        {
            const float u1 = Av[k] * ia, u2 = Bv[k] * ib, u3 = Cv[k] * ic;
            const float dca = Bv[k] * inv12 - cs * Av[k] * ia * ia;
            const float dcb = Av[k] * inv12 - cs * Bv[k] * ib * ib;
            ga[k] = F * ( As * dca + B1 * u1 - B3 * u3 ) + Gs * ( dFa1 * u1 - dF3 * u3 );
            gb[k] = F * ( As * dcb + B2 * u2 + B3 * u3 ) + Gs * ( dFb2 * u2 + dF3 * u3 );
        }
    };
    // the reactions of one triplet: on a in registers while the row atom
    // stays the same (the stream is a-major), on q through LDS
    auto apply = [&]( int a, int q, const float ( &ga )[3], const float ( &gb )[3] ) {
        if ( a != cur )
        {
            if ( cur >= 0 )
            {
                atomicAdd( &sF[wv][cur][0], ax );
                atomicAdd( &sF[wv][cur][1], ay );
                atomicAdd( &sF[wv][cur][2], az );
            }
            cur = a;
            ax = ay = az = 0.f;
        }
        ax -= ga[0];
        ay -= ga[1];
        az -= ga[2];
        atomicAdd( &sF[wv][q][0], -gb[0] );
        atomicAdd( &sF[wv][q][1], -gb[1] );
        atomicAdd( &sF[wv][q][2], -gb[2] );
        fix += ga[0] + gb[0];
        fiy += ga[1] + gb[1];
        fiz += ga[2] + gb[2];
    };
    if constexpr ( NAG > 0 && NAP > 0 )
        for_triplets<true>( L, n, rc2, tbuf[wv],
                            [&]( int a0, int q0, int a1, int q1, bool ok1 ) {
                                float ga0[3], gb0[3], ga1[3], gb1[3];
                                grad( a0, q0, ga0, gb0 );
                                grad( a1, q1, ga1, gb1 );
                                apply( a0, q0, ga0, gb0 );
                                if ( ok1 )
                                    apply( a1, q1, ga1, gb1 );
                            } );
    else
        // the generic grid's registers leave no room for a second chain
        for_triplets( L, n, rc2, tbuf[wv], [&]( int a, int q ) {
            float ga[3], gb[3];
            grad( a, q, ga, gb );
            apply( a, q, ga, gb );
        } );
    if ( cur >= 0 )
    {
        atomicAdd( &sF[wv][cur][0], ax );
        atomicAdd( &sF[wv][cur][1], ay );
        atomicAdd( &sF[wv][cur][2], az );
    }
    __builtin_amdgcn_fence( __ATOMIC_SEQ_CST, "wavefront" );
#pragma unroll
    for ( int o = 32; o > 0; o >>= 1 )
    {
        fix += __shfl_xor( fix, o, 64 );
        fiy += __shfl_xor( fiy, o, 64 );
        fiz += __shfl_xor( fiz, o, 64 );
    }
    if ( lane == 0 )
    {
        unsafeAtomicAdd( &f[i], (double)fix );
        unsafeAtomicAdd( &f[fcap + i], (double)fiy );
        unsafeAtomicAdd( &f[2 * fcap + i], (double)fiz );
    }
    for ( int a = lane; a < n; a += 64 )
    {
        const int j = L.j[a];
        unsafeAtomicAdd( &f[j], (double)sF[wv][a][0] );
        unsafeAtomicAdd( &f[fcap + j], (double)sF[wv][a][1] );
        unsafeAtomicAdd( &f[2 * fcap + j], (double)sF[wv][a][2] );
    }
}

// LDS of a wave's pair walk beyond its neighbours'.  Up to 64 neighbours
// leave the upper halves of L.d and L.e free: the ring's records (pa, pm,
// pb) lie there and here, which keeps six blocks on a CU.
union ForceBuf
{
    float coef[NSF_LD];
    struct
    {
        float pb[PAIR_RING];
        unsigned short code[PAIR_RING];
    } ring;
    struct
    {
        float f[NN_MAX][3];
        unsigned short code[PAIR_RING];
    } flat;
};
static_assert( PAIR_RING * sizeof( float ) == ( NN_MAX - 64 ) * sizeof( float4 ),
               "a ring of floats fits the upper half of L.d" );

// Forces of the power-of-two grid (see k_nnp_sf_pow).  With T = sum_s c_s
// T_s of a triplet (i, a, q), A = x_a - x_i and B = x_q - x_i, the gradients
// are combinations of A and B alone,
//   dT/dA = pa A + pm B,  dT/dB = pb B + pm A,
//   pm = F T' / (r1 r2) - s3,
//   pa = F M + s3 - F T' cos / r1^2 + S f2 f3 fc'(r1) / r1  (pb likewise),
//   s3 = F M + S f1 f2 fc'(r3) / r3,
// where S, T' and M are the coefficient sums of P E, (dP/dcos) E and
// -2 eta P E: two scalars per neighbour and triplet in place of gradients by
// component.  The atom's own force is minus the sum of its neighbours'
// reactions.
template <int NAG, int WPA>
__global__ __launch_bounds__( NNP_TPB, 5 ) void k_nnp_force_pow(
    int n_local, int fcap, const double4 *__restrict__ x,
    const int64_t *__restrict__ off, const int *__restrict__ idx,
    const NnpPlan *__restrict__ P, const float *__restrict__ dEdG,
    double *__restrict__ f, int *__restrict__ flag )
{
    __shared__ NbLds lds[NNP_TPB / 64];
    __shared__ ForceBuf buf[NNP_TPB / 64];
    const int wv = __builtin_amdgcn_readfirstlane( threadIdx.x >> 6 ), lane = threadIdx.x & 63;
    // with WPA = 4 the block's waves share an atom (one exit for all)
    const int part = WPA > 1 ? wv : 0;
    const int i = WPA > 1 ? (int)blockIdx.x : blockIdx.x * ( NNP_TPB / 64 ) + wv;
    if ( i >= n_local )
        return;
    NbLds &L = lds[wv];
    const float rc = P->rc, rc2 = P->rc2, kpi = P->pi_rc;
    const int n = gather_neighbours( i, x, off, idx, rc, rc2, kpi, L, flag );
    const int e = __builtin_amdgcn_readfirstlane( (int)x[i].w );
    const NnpElemPlan &Q = P->el[e];
    // dE/dG of the atom, in LDS until the coefficients below are read
    float *c = buf[wv].coef;
    for ( int k = lane; k < NSF_LD; k += 64 )
        c[k] = k < Q.nsf ? dEdG[(size_t)i * NSF_LD + k] : 0.f;
    __builtin_amdgcn_fence( __ATOMIC_SEQ_CST, "wavefront" );
    // the radial factors, kept for the end; e.z becomes fc' / r, d.w r^2
    float srad[NN_MAX / 64];
#pragma unroll
    for ( int u = 0; u < NN_MAX / 64; ++u )
    {
        const int a = lane + 64 * u;
        srad[u] = 0.f;
        if ( a < n )
        {
            if ( part == 0 )
                srad[u] = radial_force( Q, L, a, c );
            L.e[a].z *= L.e[a].x;
            L.d[a].w *= L.d[a].w;
        }
    }
    // the coefficients as rows of 4x4x1 MFMAs: lane l holds row l % 4, that
    // is c_gp 2^(1 - zeta_p) for p = l % 4 (half 0) and 4 + l % 4 (half 1);
    // exp(-eta s) = exp2(k s)
    const float kl = -1.44269504f * Q.a_eta[lane & ( AG_MAX - 1 )];
    const float ml = -2.0f * Q.a_eta[lane & ( AG_MAX - 1 )];
    float ct[NAG][2], ke[NAG], me[NAG];
#pragma unroll
    for ( int g = 0; g < NAG; ++g )
    {
        ke[g] = lane_value( kl, g );
        me[g] = lane_value( ml, g );
#pragma unroll
        for ( int h = 0; h < 2; ++h )
        {
            const int pp = 4 * h + ( lane & 3 );
            ct[g][h] = c[Q.a_out[g][pp]] * __builtin_amdgcn_exp2f( Q.a_lpref[pp] );
        }
    }
    __builtin_amdgcn_fence( __ATOMIC_SEQ_CST, "wavefront" );
    const float krev = 0.5f / rc; // pi r / rc in revolutions
    const float kd = -0.5f * kpi;
    // pa, pb and pm of the triplet (i, a, q); run by all lanes of the wave
    auto grad = [&]( const float4 &A, const float4 &B, const float4 &Ea, const float4 &Eb,
                     float &pa, float &pb, float &pm )
    {
        const float cx = B.x - A.x, cy = B.y - A.y, cz = B.z - A.z;
        const float c2 = cx * cx + cy * cy + cz * cz;
        const float ic = __builtin_amdgcn_rsqf( c2 );
        const float rev = c2 * ic * krev;
        const float f3 = 0.5f + 0.5f * __builtin_amdgcn_cosf( rev );
        const float d3 = kd * __builtin_amdgcn_sinf( rev ) * ic; // fc'(r3) / r3
        const float f12 = Ea.y * Eb.y, F = f12 * f3;
        const float inv12 = Ea.x * Eb.x;
        const float cs = ( A.x * B.x + A.y * B.y + A.z * B.z ) * inv12;
        const float s2 = A.w + B.w + c2;
        float Pw[POW_NAP];
        const float bm = fmaxf( 1.0f - cs, 0.0f ), bp = fmaxf( 1.0f + cs, 0.0f );
        pow_grid( bm, Pw );
        pow_grid( bp, Pw + 4 );
        // T_p = sum_g c_gp E_g and U_p = sum_g -2 eta_g c_gp E_g on the FP32
        // matrix cores: in 16 blocks of 4 x 4 with the coefficients as rows
        // and the Gaussians as columns, lane l is column l % 4 of block
        // l / 4 and receives its own triplet's four sums, so no operand
        // changes lanes.  The coefficient rows of a block come from all four
        // of its lanes, also where only some of them have a pair, and an MFMA
        // reads a lane's registers whether it is in the exec mask or not: so
        // every lane of the wave runs this (the compiler keeps the values of
        // masked-out lanes only by chance)
        f32x4 T[2] = { { 0.f, 0.f, 0.f, 0.f }, { 0.f, 0.f, 0.f, 0.f } }, U[2] = { T[0], T[0] };
#pragma unroll
        for ( int g = 0; g < NAG; ++g )
        {
            const float Eg = __builtin_amdgcn_exp2f( ke[g] * s2 ), Mg = me[g] * Eg;
#pragma unroll
            for ( int h = 0; h < 2; ++h )
            {
                T[h] = __builtin_amdgcn_mfma_f32_4x4x1f32( ct[g][h], Eg, T[h], 0, 0, 0 );
                U[h] = __builtin_amdgcn_mfma_f32_4x4x1f32( ct[g][h], Mg, U[h], 0, 0, 0 );
            }
        }
        // S = sum_p T_p P_p, M = sum_p U_p P_p and T' = sum_p T_p zeta lambda
        // b^(zeta - 1), b^3 and b^15 from the grid
        float S = 0.f, Mg = 0.f;
#pragma unroll
        for ( int u = 0; u < 4; ++u )
        {
            S = fmaf( T[1][u], Pw[4 + u], fmaf( T[0][u], Pw[u], S ) );
            Mg = fmaf( U[1][u], Pw[4 + u], fmaf( U[0][u], Pw[u], Mg ) );
        }
        const float m3 = Pw[1] * bm, p3 = Pw[5] * bp;
        const float m15 = Pw[2] * Pw[2] * Pw[2] * m3, p15 = Pw[6] * Pw[6] * Pw[6] * p3;
        float Td = T[1][0] - T[0][0];
        Td = fmaf( 2.f, T[1][1] * bp - T[0][1] * bm, Td );
        Td = fmaf( 4.f, T[1][2] * p3 - T[0][2] * m3, Td );
        Td = fmaf( 16.f, T[1][3] * p15 - T[0][3] * m15, Td );
        const float X = F * Td, FM = F * Mg;
        const float s3 = fmaf( S * f12, d3, FM );
        const float Xc = X * cs, Sf3 = S * f3, base = FM + s3;
        pm = fmaf( X, inv12, -s3 );
        pa = fmaf( Sf3 * Eb.y, Ea.z, fmaf( -Xc * Ea.x, Ea.x, base ) );
        pb = fmaf( Sf3 * Ea.y, Eb.z, fmaf( -Xc * Eb.x, Eb.x, base ) );
    };
    float fix = 0.f, fiy = 0.f, fiz = 0.f;
    auto finish = [&]( int a, float rx, float ry, float rz )
    {
        const int j = L.j[a];
        fix -= rx;
        fiy -= ry;
        fiz -= rz;
        unsafeAtomicAdd( &f[j], (double)rx );
        unsafeAtomicAdd( &f[fcap + j], (double)ry );
        unsafeAtomicAdd( &f[2 * fcap + j], (double)rz );
    };
    if ( n <= 64 )
    {
        float *rpa = reinterpret_cast<float *>( L.d + 64 ),
              *rpm = reinterpret_cast<float *>( L.e + 64 ), *rpb = buf[wv].ring.pb;
        // of the lane's neighbour: sum of its pa (or pb), sum of pm X_partner
        float sp = srad[0], sx = 0.f, sy = 0.f, sz = 0.f;
        pair_ring<true, WPA>(
            L, n, rc2, part, buf[wv].ring.code,
            [&]( int slot, int a, int q, bool ok ) {
                float pa, pb, pm;
                grad( L.d[a], L.d[q], L.e[a], L.e[q], pa, pb, pm );
                if ( ok )
                {
                    rpa[slot] = pa;
                    rpm[slot] = pm;
                    rpb[slot] = pb;
                }
            },
            [&]( int d, unsigned long long m, int s0 ) {
                // as the pair's first neighbour, the partner d further on
                if ( __builtin_amdgcn_inverse_ballot_w64( m ) )
                {
                    const int k = ( s0 + lanes_below( m ) ) & ( PAIR_RING - 1 );
                    const float4 X = L.d[pair_partner( lane, d, n )];
                    const float w = rpm[k];
                    sp += rpa[k];
                    sx = fmaf( w, X.x, sx );
                    sy = fmaf( w, X.y, sy );
                    sz = fmaf( w, X.z, sz );
                }
                // as its second, the first neighbour p d before: lanes from
                // d on have p = lane - d, those below p = lane - d + n, so
                // the row's mask turns by d within n bits
                const unsigned long long up = m << d, wrap = m >> ( n - d );
                const unsigned long long turned =
                    ( up & ( ~0ull >> ( 64 - n ) ) ) | wrap;
                if ( __builtin_amdgcn_inverse_ballot_w64( turned ) )
                {
                    const int nw = (int)__popcll( wrap );
                    const int before = s0 + ( lane >= d ? -nw : (int)__popcll( m ) - nw );
                    const int k = ( before + lanes_below( turned ) ) & ( PAIR_RING - 1 );
                    const float4 X = L.d[pair_partner( lane, n - d, n )];
                    const float w = rpm[k];
                    sp += rpb[k];
                    sx = fmaf( w, X.x, sx );
                    sy = fmaf( w, X.y, sy );
                    sz = fmaf( w, X.z, sz );
                }
            } );
        if constexpr ( WPA > 1 )
        {
            // the waves' sums meet in the first wave
            L.e[lane] = make_float4( sp, sx, sy, sz );
            __syncthreads();
            if ( part != 0 )
                return;
            for ( int w = 1; w < WPA; ++w )
            {
                const float4 o = lds[w].e[lane];
                sp += o.x;
                sx += o.y;
                sy += o.z;
                sz += o.w;
            }
        }
        if ( lane < n )
        {
            const float4 A = L.d[lane];
            finish( lane, -fmaf( sp, A.x, sx ), -fmaf( sp, A.y, sy ), -fmaf( sp, A.z, sz ) );
        }
    }
    else
    {
        // more neighbours than lanes: each lane takes a contiguous block of
        // the compacted (a-major) pair list, the sums of pa and pm B of the
        // row atom stay in registers until a changes and the reaction on q
        // goes to LDS
        float( *sF )[3] = buf[wv].flat.f;
        for ( int a = lane; a < n; a += 64 )
            sF[a][0] = sF[a][1] = sF[a][2] = 0.f;
        __builtin_amdgcn_fence( __ATOMIC_SEQ_CST, "wavefront" );
        int cur = -1;
        float spa = 0.f, bx = 0.f, by = 0.f, bz = 0.f;
        auto flush = [&]()
        {
            const float4 A = L.d[cur];
            atomicAdd( &sF[cur][0], -( spa * A.x + bx ) );
            atomicAdd( &sF[cur][1], -( spa * A.y + by ) );
            atomicAdd( &sF[cur][2], -( spa * A.z + bz ) );
        };
        for_triplets<false, PAIR_RING, true>( L, n, rc2, buf[wv].flat.code,
                                              [&]( int a, int q, bool ok ) {
            const float4 A = L.d[a], B = L.d[q];
            float pa, pb, pm;
            grad( A, B, L.e[a], L.e[q], pa, pb, pm );
            if ( !ok )
                return;
            if ( a != cur )
            {
                if ( cur >= 0 )
                    flush();
                cur = a;
                spa = bx = by = bz = 0.f;
            }
            spa += pa;
            bx = fmaf( pm, B.x, bx );
            by = fmaf( pm, B.y, by );
            bz = fmaf( pm, B.z, bz );
            atomicAdd( &sF[q][0], -fmaf( pb, B.x, pm * A.x ) );
            atomicAdd( &sF[q][1], -fmaf( pb, B.y, pm * A.y ) );
            atomicAdd( &sF[q][2], -fmaf( pb, B.z, pm * A.z ) );
        }, nullptr, part, WPA );
        if ( cur >= 0 )
            flush();
        __builtin_amdgcn_fence( __ATOMIC_SEQ_CST, "wavefront" );
        if constexpr ( WPA > 1 )
        {
            __syncthreads();
            if ( part != 0 )
                return;
            for ( int a = lane; a < n; a += 64 )
                for ( int w = 1; w < WPA; ++w )
                    for ( int k = 0; k < 3; ++k )
                        sF[a][k] += buf[w].flat.f[a][k];
        }
#pragma unroll
        for ( int u = 0; u < NN_MAX / 64; ++u )
        {
            const int a = lane + 64 * u;
            if ( a < n )
            {
                const float4 A = L.d[a];
                finish( a, fmaf( -srad[u], A.x, sF[a][0] ), fmaf( -srad[u], A.y, sF[a][1] ),
                        fmaf( -srad[u], A.z, sF[a][2] ) );
            }
        }
    }
#pragma unroll
    for ( int o = 32; o > 0; o >>= 1 )
    {
        fix += __shfl_xor( fix, o, 64 );
        fiy += __shfl_xor( fiy, o, 64 );
        fiz += __shfl_xor( fiz, o, 64 );
    }
    if ( lane == 0 )
    {
        unsafeAtomicAdd( &f[i], (double)fix );
        unsafeAtomicAdd( &f[fcap + i], (double)fiy );
        unsafeAtomicAdd( &f[2 * fcap + i], (double)fiz );
    }
}

__global__ void k_nnp_esum( int n, const float *__restrict__ Ei,
                            double *__restrict__ part )
{
    __shared__ double s[256];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    s[threadIdx.x] = i < n ? (double)Ei[i] : 0.0;
    __syncthreads();
    for ( int o = 128; o > 0; o >>= 1 )
    {
        if ( (int)threadIdx.x < o )
            s[threadIdx.x] += s[threadIdx.x + o];
        __syncthreads();
    }
    if ( threadIdx.x == 0 )
        part[blockIdx.x] = s[0];
}

// ---------------------------------------------------------------- host
static cmd_status nnp_prepare( cmd_nnp *M, int n_local, hipStream_t st )
{
    if ( !M->plan_ok )
    {
        CMD_TRY( build_plan( M->model, M->plan ) );
        CMD_TRY( M->dplan.reserve( 1 ) );
        CMD_HIP( hipMemcpyAsync( M->dplan.p, &M->plan, sizeof( NnpPlan ),
                                 hipMemcpyHostToDevice, st ) );
        M->plan_ok = true;
    }
    const int n = std::max( n_local, 1 );
    if ( n > M->cap )
    {
        M->cap = n;
        CMD_TRY( M->G.reserve( (size_t)n * NSF_LD ) );
        CMD_TRY( M->dEdG.reserve( (size_t)n * NSF_LD ) );
        CMD_TRY( M->Ei.reserve( n ) );
    }
    CMD_TRY( M->flag.reserve( 1 ) );
    return CMD_OK;
}

// The neighbour-count check of a force call: begin clears the flag that the
// kernels raise, end waits for the stream and reads it.
static cmd_status too_many_neighbours()
{
    set_error( "an atom has more than %d neighbours inside the NNP cutoff", NN_MAX );
    return CMD_ERR_CAPACITY;
}

static cmd_status nnp_check_begin( cmd_nnp *M, hipStream_t st )
{
    CMD_TRY( M->flag.reserve( 1 ) );
    return fill_i32( M->flag.p, 0, 1, st );
}

static cmd_status nnp_check_end( cmd_nnp *M, hipStream_t st )
{
    int fl = 0;
    CMD_HIP( hipMemcpyAsync( &fl, M->flag.p, sizeof( int ),
                             hipMemcpyDeviceToHost, st ) );
    CMD_HIP( hipStreamSynchronize( st ) );
    return fl == 0 ? CMD_OK : too_many_neighbours();
}

// The same for the steps of a time loop (internal.h).  The flag stays up once
// raised, so every later integrator of the loop leaves the state alone too.
cmd_status nnp_run_begin( cmd_nnp *M, hipStream_t st )
{
    CMD_TRY( M->stop.init( 1 ) );
    // (no step of an earlier loop is unfinished: loops end with nnp_run_stop)
    M->stop.p[0] = 0;
    // (no fence at the marks, which would write the caches back between steps:
    // they only pace the host)
    for ( hipEvent_t &e : M->mark )
        if ( !e )
            CMD_HIP( hipEventCreateWithFlags( &e, hipEventDisableTiming |
                                                      hipEventDisableSystemFence ) );
    M->steps = M->marks = 0;
    M->run_stream = st;
    return nnp_check_begin( M, st );
}

void nnp_run_gate( cmd_nnp *M, StepCtl &ctl, int step )
{
    ctl.stop = M->flag.p;
    ctl.stop_step = M->stop.d;
    ctl.step = step;
}

cmd_status nnp_run_check( cmd_nnp *M, bool wait )
{
    if ( wait )
        CMD_HIP( hipStreamSynchronize( M->run_stream ) );
    return *(volatile int *)M->stop.p == 0 ? CMD_OK : too_many_neighbours();
}

// The host waits for the mark before the last, so that two steps are queued at
// most: the device always has work, and other streams' waits that take in the
// whole device (freeing a buffer that grows) stand behind two steps.  With a
// rebuild interval queued, the first LJ jobs that joined beside NNP systems of
// 0.4 million atoms (6.4 ms a step) took 0.22 s instead of 0.13.  A mark
// takes the device about 2.5 us, 2 % of a step of 3,000 atoms, so below 32,768
// atoms (up to 0.55 ms a step) eight steps share one and 16 are queued at most.
static constexpr int MARK_EACH = 32768, MARK_SMALL = 8;

cmd_status nnp_run_mark( cmd_nnp *M, int n_local )
{
    if ( ++M->steps % ( n_local < MARK_EACH ? MARK_SMALL : 1 ) != 0 )
        return CMD_OK;
    CMD_HIP( hipEventRecord( M->mark[M->marks & 1], M->run_stream ) );
    if ( ++M->marks >= 2 )
        CMD_HIP( hipEventSynchronize( M->mark[M->marks & 1] ) );
    return nnp_run_check( M, false );
}

int nnp_run_stop( cmd_nnp *M )
{
    (void)hipStreamSynchronize( M->run_stream );
    return *(volatile int *)M->stop.p;
}

// Where the power-of-two kernels put four waves on an atom.  One wave each
// leaves SIMDs with too few waves to cover their latencies, but the gather and
// set-up are repeated in each of the four.  A block is then an atom, and up to
// 1,536 of them (six to a CU) run in one round; with few pairs to share the
// repeats win there too.  Beyond that only atoms past the ring's 64 neighbours
// gain, whose walk with LDS atomics one wave does slowly.  In systems with
// thermal displacements (0.25 on a spacing of 2.5) they are some from about 66
// listed on average (near a perfect lattice from 72), and the gain is down to
// 5 % at 3,072 atoms.  Step with four waves / with one (us), by atoms and
// listed neighbours:
//              24          36          53          61          69          76
//   729      52 / 53
//   1,331    59 / 57     62 / 63     69 / 73     71 / 78     86 / 115   118 / 154
//   1,728    67 / 57     71 / 63     76 / 72     79 / 79     92 / 118   139 / 157
//   2,744    73 / 59     77 / 66     84 / 78     89 / 84    112 / 121   173 / 184
//   4,096    87 / 62     94 / 71    103 / 84    109 / 93    133 / 140   223 / 217
//   4,913    98 / 65    103 / 75    114 / 90    121 / 100   147 / 146   254 / 247
static bool nnp_split( int n, int64_t listed )
{
    return ( n <= 1536 && listed >= 32 * (int64_t)n ) ||
           ( n <= 3072 && listed >= 66 * (int64_t)n );
}

cmd_status nnp_compute( cmd_nnp *M, cmd_system *S, cmd_neigh *N, bool check )
{
    const hipStream_t st = S->stream;
    const int n = S->n_local;
    CMD_TRY( nnp_prepare( M, n, st ) );
    CMD_REQUIRE( S->ntypes <= M->plan.nelem, CMD_ERR_ARG,
                 "the system has %d atom types but the model %d elements",
                 S->ntypes, M->plan.nelem );
    CMD_REQUIRE( !N->half, CMD_ERR_ARG,
                 "the NNP force needs a full neighbour list (the reference "
                 "supports only full lists, force_nnp_cabana_neigh_impl.h)" );
    // A list shorter than the symmetry-function cutoff truncates the
    // functions to the listed neighbours, as in the reference (in.nnp lists
    // 3.9 + skin against rc 7.37 in input/nnp/input.nn).
    CMD_TRY( neigh_csr( N ) );
    const int nt = S->n_local + S->n_ghost;
    if ( check )
        CMD_TRY( nnp_check_begin( M, st ) );
    if ( n == 0 )
    {
        // no kernel below clears the rows of uploaded ghosts
        for ( int c = 0; c < 3; ++c )
            CMD_TRY( fill_f64( S->f.p + (size_t)c * S->cap, 0.0, nt, st ) );
        return CMD_OK;
    }
    CMD_TRY( M->terms.reserve( std::max( n, 1 ) ) );
    M->n_last = n;
    const int nbw = ( n + NNP_TPB / 64 - 1 ) / ( NNP_TPB / 64 );
    // the angular grid of every element: its number of etas where they
    // agree (0: they do not), whether all its rs are 0 and whether its
    // (lambda, zeta) are the power-of-two grid
    int nag = M->plan.nelem > 0 ? M->plan.el[0].nag : 0;
    bool nap8 = true, rs0 = true, pow2 = true;
    for ( int e = 0; e < M->plan.nelem; ++e )
    {
        const NnpElemPlan &Q = M->plan.el[e];
        if ( Q.nag != nag )
            nag = 0;
        nap8 = nap8 && Q.nap == 8;
        pow2 = pow2 && Q.pow2;
        for ( int g = 0; g < Q.nag; ++g )
            rs0 = rs0 && Q.a_rs[g] == 0.f;
    }
    // squarings in place of log2 and exp2 and fixed grid sizes: the fewest
    // operations wherever the grid allows them
    const bool pow = nag >= 1 && rs0 && pow2;
    const bool g58 = nag == 5 && nap8;
    const bool split = nnp_split( n, N->nnz );
#define CMD_POW( LAUNCH )                                                                 \
    switch ( nag )                                                                        \
    {                                                                                     \
    case 1: LAUNCH( 1 ); break;                                                           \
    case 2: LAUNCH( 2 ); break;                                                           \
    case 3: LAUNCH( 3 ); break;                                                           \
    case 4: LAUNCH( 4 ); break;                                                           \
    case 5: LAUNCH( 5 ); break;                                                           \
    case 6: LAUNCH( 6 ); break;                                                           \
    case 7: LAUNCH( 7 ); break;                                                           \
    default: LAUNCH( 8 ); break;                                                          \
    }
#define CMD_SF_POW( A )                                                                   \
    if ( split )                                                                          \
        k_nnp_sf_pow<A, 4><<<n, NNP_TPB, 0, st>>>( n, S->x.p, N->offsets.p, N->idx.p,      \
                                                   M->dplan.p, M->G.p, M->flag.p,         \
                                                   M->terms.p, S->f.p, S->cap, nt );      \
    else                                                                                  \
        k_nnp_sf_pow<A, 1><<<nbw, NNP_TPB, 0, st>>>( n, S->x.p, N->offsets.p, N->idx.p,    \
                                                     M->dplan.p, M->G.p, M->flag.p,       \
                                                     M->terms.p, S->f.p, S->cap, nt )
#define CMD_FORCE_POW( A )                                                                \
    if ( split )                                                                          \
        k_nnp_force_pow<A, 4><<<n, NNP_TPB, 0, st>>>( n, S->cap, S->x.p, N->offsets.p,     \
                                                      N->idx.p, M->dplan.p, M->dEdG.p,    \
                                                      S->f.p, M->flag.p );                \
    else                                                                                  \
        k_nnp_force_pow<A, 1><<<nbw, NNP_TPB, 0, st>>>( n, S->cap, S->x.p, N->offsets.p,   \
                                                        N->idx.p, M->dplan.p, M->dEdG.p,  \
                                                        S->f.p, M->flag.p )
#define CMD_SF( A, P, R )                                                                 \
    k_nnp_sf<A, P, R><<<nbw, NNP_TPB, 0, st>>>( n, S->x.p, N->offsets.p, N->idx.p, M->dplan.p, \
                                                M->G.p, M->flag.p, M->terms.p, S->f.p,    \
                                                S->cap, nt )
    if ( pow )
        CMD_POW( CMD_SF_POW )
    else if ( g58 )
    {
        if ( rs0 )
            CMD_SF( 5, 8, true );
        else
            CMD_SF( 5, 8, false );
    }
    else if ( rs0 )
        CMD_SF( 0, 0, true );
    else
        CMD_SF( 0, 0, false );
#undef CMD_SF
    CMD_LAUNCH_CHECK();
    {
        const int nb = ( n + MLP_ATOMS - 1 ) / MLP_ATOMS;
        const int waves = MLP_ATOMS / 16 + M->plan.nelem - 1;
        const size_t lds = (size_t)waves * 16 * ( KPAD + 4 ) * sizeof( float );
        if ( M->prec == CMD_PREC_MIXED )
            k_nnp_mlp<false><<<nb, 64 * waves, lds, st>>>( n, M->plan.nelem, S->x.p, M->G.p,
                                                           M->dplan.p, M->dEdG.p, M->Ei.p );
        else
            k_nnp_mlp<true><<<nb, 64 * waves, lds, st>>>( n, M->plan.nelem, S->x.p, M->G.p,
                                                          M->dplan.p, M->dEdG.p, M->Ei.p );
        CMD_LAUNCH_CHECK();
    }
#define CMD_FORCE( A, P, R )                                                               \
    k_nnp_force<A, P, R><<<nbw, NNP_TPB, 0, st>>>( n, S->cap, S->x.p, N->offsets.p, N->idx.p, \
                                                   M->dplan.p, M->dEdG.p, S->f.p, M->flag.p )
    if ( pow )
        CMD_POW( CMD_FORCE_POW )
    else if ( g58 )
    {
        if ( rs0 )
            CMD_FORCE( 5, 8, true );
        else
            CMD_FORCE( 5, 8, false );
    }
    else if ( rs0 )
        CMD_FORCE( 0, 0, true );
    else
        CMD_FORCE( 0, 0, false );
#undef CMD_FORCE
#undef CMD_POW
#undef CMD_SF_POW
#undef CMD_FORCE_POW
    CMD_LAUNCH_CHECK();
    return check ? nnp_check_end( M, st ) : CMD_OK;
}

// Sum of the atomic network outputs (FP64 reduction).
cmd_status nnp_energy_sum( cmd_nnp *M, cmd_system *S, double *sum )
{
    const int n = S->n_local;
    const int nb = ( n + 255 ) / 256;
    CMD_TRY( M->part.reserve( std::max( nb, 1 ) ) );
    if ( n > 0 )
    {
        k_nnp_esum<<<nb, 256, 0, S->stream>>>( n, M->Ei.p, M->part.p );
        CMD_LAUNCH_CHECK();
    }
    std::vector<double> h( std::max( nb, 1 ), 0.0 );
    if ( n > 0 )
        CMD_HIP( hipMemcpyAsync( h.data(), M->part.p, sizeof( double ) * nb,
                                 hipMemcpyDeviceToHost, S->stream ) );
    CMD_HIP( hipStreamSynchronize( S->stream ) );
    double s = 0.0;
    for ( int k = 0; k < nb; ++k )
        s += h[k];
    *sum = s;
    return CMD_OK;
}

// ---------------------------------------------------------------- n2p2 files
static std::vector<std::string> words_of( const std::string &line )
{
    std::vector<std::string> w;
    std::istringstream is( line.substr( 0, line.find( '#' ) ) );
    std::string t;
    while ( is >> t )
        w.push_back( t );
    return w;
}

// n2p2 orders an element's functions by type, then cutoff, then the
// parameters (eta, rs, zeta, lambda) and neighbour elements; scaling.data
// rows and the network inputs follow that order.
static bool sf_less( const cmd_nnp_model::SF &a, const cmd_nnp_model::SF &b )
{
    if ( a.type != b.type )
        return a.type < b.type;
    if ( a.rc != b.rc )
        return a.rc < b.rc;
    if ( a.eta != b.eta )
        return a.eta < b.eta;
    if ( a.rs != b.rs )
        return a.rs < b.rs;
    if ( a.zeta != b.zeta )
        return a.zeta < b.zeta;
    if ( a.lambda != b.lambda )
        return a.lambda < b.lambda;
    if ( a.e1 != b.e1 )
        return a.e1 < b.e1;
    return a.e2 < b.e2;
}

static cmd_status load_n2p2( const char *dir, int nelem, const char *const *names,
                             const int *znum, cmd_nnp_model &m )
{
    m = cmd_nnp_model{};
    m.nelem = nelem;
    m.el.resize( nelem );
    m.scale = false;
    for ( int e = 0; e < nelem; ++e )
    {
        m.el[e].name = names[e];
        m.el[e].z = znum[e];
    }
    auto elem_of = [&]( const std::string &s ) -> int
    {
        for ( int e = 0; e < nelem; ++e )
            if ( m.el[e].name == s )
                return e;
        return -1;
    };
    const std::string d( dir );
    {
        std::ifstream in( d + "/input.nn" );
        CMD_REQUIRE( in.good(), CMD_ERR_IO, "cannot read %s/input.nn", dir );
        std::string line;
        std::string act;
        while ( std::getline( in, line ) )
        {
            const auto w = words_of( line );
            if ( w.empty() )
                continue;
            try
            {
                if ( w[0] == "global_nodes_short" )
                {
                    m.hidden.clear();
                    for ( size_t k = 1; k < w.size(); ++k )
                        m.hidden.push_back( std::stoi( w[k] ) );
                }
                else if ( w[0] == "global_activation_short" )
                {
                    act.clear();
                    for ( size_t k = 1; k < w.size(); ++k )
                        act += w[k];
                }
                else if ( w[0] == "scale_symmetry_functions" )
                    m.scale = true;
                else if ( w[0] == "scale_min_short" )
                    m.smin = std::stod( w.at( 1 ) );
                else if ( w[0] == "scale_max_short" )
                    m.smax = std::stod( w.at( 1 ) );
                else if ( w[0] == "cutoff_type" )
                    CMD_REQUIRE( std::stoi( w.at( 1 ) ) == 1, CMD_ERR_IO,
                                 "only cutoff_type 1 (cosine) is supported" );
                else if ( w[0] == "atom_energy" )
                {
                    const int e = elem_of( w.at( 1 ) );
                    if ( e >= 0 )
                        m.el[e].atom_energy = std::stod( w.at( 2 ) );
                }
                else if ( w[0] == "symfunction_short" )
                {
                    const int e = elem_of( w.at( 1 ) );
                    CMD_REQUIRE( e >= 0, CMD_ERR_IO, "unknown element %s",
                                 w.at( 1 ).c_str() );
                    cmd_nnp_model::SF s{};
                    s.type = std::stoi( w.at( 2 ) );
                    if ( s.type == 2 )
                    {
                        s.e1 = elem_of( w.at( 3 ) );
                        s.e2 = -1;
                        s.eta = std::stod( w.at( 4 ) );
                        s.rs = std::stod( w.at( 5 ) );
                        s.rc = std::stod( w.at( 6 ) );
                    }
                    else if ( s.type == 3 )
                    {
                        s.e1 = elem_of( w.at( 3 ) );
                        s.e2 = elem_of( w.at( 4 ) );
                        s.eta = std::stod( w.at( 5 ) );
                        s.lambda = std::stod( w.at( 6 ) );
                        s.zeta = std::stod( w.at( 7 ) );
                        s.rc = std::stod( w.at( 8 ) );
                        s.rs = w.size() > 9 ? std::stod( w[9] ) : 0.0;
                    }
                    else
                    {
                        set_error( "symfunction_short type %d is not supported",
                                   s.type );
                        return CMD_ERR_IO;
                    }
                    m.el[e].sf.push_back( s );
                }
            }
            catch ( const std::exception & )
            {
                set_error( "malformed line in input.nn: %s", line.c_str() );
                return CMD_ERR_IO;
            }
        }
        m.act = act;
        m.nlayers = (int)m.hidden.size() + 1;
    }
    for ( auto &E : m.el )
    {
        std::stable_sort( E.sf.begin(), E.sf.end(), sf_less );
        E.gmin.assign( E.sf.size(), 0.0 );
        E.gmax.assign( E.sf.size(), 1.0 );
    }
    if ( m.scale )
    {
        std::ifstream in( d + "/scaling.data" );
        CMD_REQUIRE( in.good(), CMD_ERR_IO, "cannot read %s/scaling.data", dir );
        std::string line;
        while ( std::getline( in, line ) )
        {
            const auto w = words_of( line );
            if ( w.size() < 4 )
                continue;
            const int e = std::stoi( w[0] ) - 1, k = std::stoi( w[1] ) - 1;
            CMD_REQUIRE( e >= 0 && e < nelem && k >= 0 &&
                             k < (int)m.el[e].sf.size(),
                         CMD_ERR_IO, "scaling.data row %d %d out of range", e + 1,
                         k + 1 );
            m.el[e].gmin[k] = std::stod( w[2] );
            m.el[e].gmax[k] = std::stod( w[3] );
        }
    }
    for ( int e = 0; e < nelem; ++e )
    {
        auto &E = m.el[e];
        std::vector<int> sizes;
        sizes.push_back( (int)E.sf.size() );
        for ( int h : m.hidden )
            sizes.push_back( h );
        sizes.push_back( 1 );
        const int L = (int)sizes.size() - 1;
        E.W.assign( L, {} );
        E.b.assign( L, {} );
        for ( int l = 0; l < L; ++l )
        {
            E.W[l].assign( (size_t)sizes[l + 1] * sizes[l], 0.0 );
            E.b[l].assign( sizes[l + 1], 0.0 );
        }
        char fn[64];
        std::snprintf( fn, sizeof( fn ), "/weights.%03d.data", E.z );
        std::ifstream in( d + fn );
        CMD_REQUIRE( in.good(), CMD_ERR_IO, "cannot read %s%s", dir, fn );
        std::string line;
        while ( std::getline( in, line ) )
        {
            const auto w = words_of( line );
            if ( w.size() < 5 )
                continue;
            try
            {
                const double v = std::stod( w[0] );
                if ( w[1] == "a" && w.size() >= 7 )
                {
                    const int lf = std::stoi( w[3] ), nf = std::stoi( w[4] ),
                              nt = std::stoi( w[6] );
                    CMD_REQUIRE( lf >= 0 && lf < L && nf >= 1 && nf <= sizes[lf] &&
                                     nt >= 1 && nt <= sizes[lf + 1],
                                 CMD_ERR_IO, "weight index out of range" );
                    E.W[lf][(size_t)( nt - 1 ) * sizes[lf] + ( nf - 1 )] = v;
                }
                else if ( w[1] == "b" )
                {
                    const int l = std::stoi( w[3] ), nd = std::stoi( w[4] );
                    CMD_REQUIRE( l >= 1 && l <= L && nd >= 1 && nd <= sizes[l],
                                 CMD_ERR_IO, "bias index out of range" );
                    E.b[l - 1][nd - 1] = v;
                }
            }
            catch ( const std::exception & )
            {
                set_error( "malformed line in %s: %s", fn + 1, line.c_str() );
                return CMD_ERR_IO;
            }
        }
    }
    return CMD_OK;
}

// ---------------------------------------------------------------- synthetic
// splitmix64 stream for seeded weights (normal deviates by Box-Muller).
struct Mix
{
    uint64_t s;
    uint64_t next()
    {
        uint64_t z = ( s += 0x9e3779b97f4a7c15ull );
        z = ( z ^ ( z >> 30 ) ) * 0xbf58476d1ce4e5b9ull;
        z = ( z ^ ( z >> 27 ) ) * 0x94d049bb133111ebull;
        return z ^ ( z >> 31 );
    }
    double uniform() { return ( next() >> 11 ) * ( 1.0 / 9007199254740992.0 ); }
    double normal()
    {
        const double u1 = std::max( uniform(), 1e-300 ), u2 = uniform();
        return std::sqrt( -2.0 * std::log( u1 ) ) * std::cos( 6.283185307179586 * u2 );
    }
};

} // namespace cmd

using namespace cmd;

extern "C" {

cmd_status cmd_nnp_model_create( int nelem, int n_hidden, const int *hidden,
                                 const char *activations, cmd_nnp_model **out )
{
    CMD_REQUIRE( out && nelem >= 1 && nelem <= NNP_MAXEL && n_hidden >= 0 &&
                     activations && (int)std::strlen( activations ) == n_hidden + 1,
                 CMD_ERR_ARG, "bad NNP model description" );
    cmd_nnp_model *m = new cmd_nnp_model;
    m->nelem = nelem;
    m->el.resize( nelem );
    m->hidden.assign( hidden, hidden + n_hidden );
    m->nlayers = n_hidden + 1;
    m->act = activations;
    *out = m;
    return CMD_OK;
}

cmd_status cmd_nnp_model_destroy( cmd_nnp_model *m )
{
    delete m;
    return CMD_OK;
}

cmd_status cmd_nnp_model_set_scaling( cmd_nnp_model *m, int scale, double smin,
                                      double smax )
{
    CMD_REQUIRE( m, CMD_ERR_ARG, "model is NULL" );
    m->scale = scale != 0;
    m->smin = smin;
    m->smax = smax;
    return CMD_OK;
}

cmd_status cmd_nnp_model_add_sf( cmd_nnp_model *m, int elem, int type, int e1,
                                 int e2, double eta, double rs, double lambda,
                                 double zeta, double rc, double gmin, double gmax )
{
    CMD_REQUIRE( m && elem >= 0 && elem < m->nelem, CMD_ERR_ARG, "bad element" );
    CMD_REQUIRE( type == 2 || type == 3, CMD_ERR_ARG,
                 "symmetry function type %d is not supported", type );
    m->el[elem].sf.push_back( cmd_nnp_model::SF{ type, e1, e2, eta, rs, lambda, zeta, rc } );
    m->el[elem].gmin.push_back( gmin );
    m->el[elem].gmax.push_back( gmax );
    return CMD_OK;
}

cmd_status cmd_nnp_model_set_layer( cmd_nnp_model *m, int elem, int layer,
                                    int n_out, int n_in, const double *W,
                                    const double *b )
{
    CMD_REQUIRE( m && elem >= 0 && elem < m->nelem && layer >= 0 &&
                     layer < m->nlayers && W && b,
                 CMD_ERR_ARG, "bad layer" );
    auto &E = m->el[elem];
    if ( (int)E.W.size() < m->nlayers )
    {
        E.W.resize( m->nlayers );
        E.b.resize( m->nlayers );
    }
    E.W[layer].assign( W, W + (size_t)n_out * n_in );
    E.b[layer].assign( b, b + n_out );
    return CMD_OK;
}

cmd_status cmd_nnp_model_set_atom_energy( cmd_nnp_model *m, int elem, double e )
{
    CMD_REQUIRE( m && elem >= 0 && elem < m->nelem, CMD_ERR_ARG, "bad element" );
    m->el[elem].atom_energy = e;
    return CMD_OK;
}

cmd_status cmd_nnp_model_load_n2p2( const char *dir, int nelem,
                                    const char *const *names,
                                    const int *atomic_numbers,
                                    cmd_nnp_model **out )
{
    CMD_REQUIRE( dir && names && atomic_numbers && out && nelem >= 1 &&
                     nelem <= NNP_MAXEL,
                 CMD_ERR_ARG, "bad argument" );
    cmd_nnp_model *m = new cmd_nnp_model;
    const cmd_status st = load_n2p2( dir, nelem, names, atomic_numbers, *m );
    if ( st != CMD_OK )
    {
        delete m;
        return st;
    }
    *out = m;
    return CMD_OK;
}

// The benchmark model: 2 elements; per element 15 radial functions (eta
// log-spaced in [0.01, 2], rs = 0) for each neighbour element and 40
// angular ones (5 eta log-spaced in [0.001, 0.05] x lambda +-1 x zeta
// {1, 2, 4, 16}, any pair); cosine cutoff rc; network 70 -> 25 -> 25 -> 1
// (tanh, tanh, linear) with N(0, 1)/sqrt(fan_in) weights and zero biases
// from `seed`; scaling ranges [0, 1] until fitted to a frame.
cmd_status cmd_nnp_model_synthetic( uint64_t seed, double rc, cmd_nnp_model **out )
{
    CMD_REQUIRE( out && rc > 0, CMD_ERR_ARG, "bad argument" );
    cmd_nnp_model *m = new cmd_nnp_model;
    m->nelem = 2;
    m->el.resize( 2 );
    m->hidden = { 25, 25 };
    m->nlayers = 3;
    m->act = "ttl";
    m->scale = true;
    Mix rng{ seed };
    for ( int e = 0; e < 2; ++e )
    {
        auto &E = m->el[e];
        for ( int k = 0; k < 15; ++k )
        {
            const double eta = 0.01 * std::pow( 200.0, k / 14.0 );
            for ( int ne = 0; ne < 2; ++ne )
                E.sf.push_back( { 2, ne, -1, eta, 0.0, 0.0, 0.0, rc } );
        }
        const double zetas[4] = { 1.0, 2.0, 4.0, 16.0 };
        for ( int k = 0; k < 5; ++k )
        {
            const double eta = 0.001 * std::pow( 50.0, k / 4.0 );
            for ( double z : zetas )
                for ( double lam : { -1.0, 1.0 } )
                    E.sf.push_back( { 3, -1, -1, eta, 0.0, lam, z, rc } );
        }
        E.gmin.assign( E.sf.size(), 0.0 );
        E.gmax.assign( E.sf.size(), 1.0 );
        const int sizes[4] = { (int)E.sf.size(), 25, 25, 1 };
        E.W.resize( 3 );
        E.b.resize( 3 );
        for ( int l = 0; l < 3; ++l )
        {
            E.W[l].resize( (size_t)sizes[l + 1] * sizes[l] );
            for ( auto &w : E.W[l] )
                w = rng.normal() / std::sqrt( (double)sizes[l] );
            E.b[l].assign( sizes[l + 1], 0.0 );
        }
    }
    *out = m;
    return CMD_OK;
}

cmd_status cmd_nnp_model_info( const cmd_nnp_model *m, int elem, int *nsf,
                               int *n_hidden, int *hidden, double *atom_energy )
{
    CMD_REQUIRE( m && elem >= 0 && elem < m->nelem, CMD_ERR_ARG, "bad element" );
    if ( nsf )
        *nsf = (int)m->el[elem].sf.size();
    if ( n_hidden )
        *n_hidden = (int)m->hidden.size();
    if ( hidden )
        for ( size_t k = 0; k < m->hidden.size(); ++k )
            hidden[k] = m->hidden[k];
    if ( atom_energy )
        *atom_energy = m->el[elem].atom_energy;
    return CMD_OK;
}

// params: type, e1, e2, eta, rs, lambda, zeta, rc, gmin, gmax
cmd_status cmd_nnp_model_get_sf( const cmd_nnp_model *m, int elem, int k,
                                 double params[10] )
{
    CMD_REQUIRE( m && elem >= 0 && elem < m->nelem && k >= 0 &&
                     k < (int)m->el[elem].sf.size() && params,
                 CMD_ERR_ARG, "bad argument" );
    const auto &s = m->el[elem].sf[k];
    const double v[10] = { (double)s.type, (double)s.e1, (double)s.e2, s.eta, s.rs,
                           s.lambda, s.zeta, s.rc, m->el[elem].gmin[k],
                           m->el[elem].gmax[k] };
    std::memcpy( params, v, sizeof( v ) );
    return CMD_OK;
}

cmd_status cmd_nnp_model_get_layer( const cmd_nnp_model *m, int elem, int layer,
                                    double *W, double *b )
{
    CMD_REQUIRE( m && elem >= 0 && elem < m->nelem && layer >= 0 &&
                     layer < (int)m->el[elem].W.size(),
                 CMD_ERR_ARG, "bad argument" );
    if ( W )
        std::memcpy( W, m->el[elem].W[layer].data(),
                     sizeof( double ) * m->el[elem].W[layer].size() );
    if ( b )
        std::memcpy( b, m->el[elem].b[layer].data(),
                     sizeof( double ) * m->el[elem].b[layer].size() );
    return CMD_OK;
}

cmd_status cmd_force_nnp_create( const cmd_nnp_model *m, cmd_force **out )
{
    CMD_REQUIRE( m && out, CMD_ERR_ARG, "NULL argument" );
    cmd_force *f = new cmd_force;
    f->kind = 2;
    f->ntypes = m->nelem;
    f->nnp = new cmd_nnp;
    f->nnp->model = *m;
    std::vector<NnpPlan> probe( 1 ); // a plan holds the split weights: keep it off the stack
    const cmd_status st = build_plan( f->nnp->model, probe[0] );
    if ( st != CMD_OK )
    {
        delete f->nnp;
        delete f;
        return st;
    }
    f->prec = CMD_PREC_MIXED;
    *out = f;
    return CMD_OK;
}

// Scaling ranges fitted to the symmetry functions of the current frame
// (the benchmark model's "min-max scaling from the initial frame").
cmd_status cmd_force_nnp_fit_scaling( cmd_force *f, cmd_system *s, cmd_neigh *n )
{
    CMD_REQUIRE( f && f->kind == 2 && s && n, CMD_ERR_ARG, "bad argument" );
    cmd_nnp *M = f->nnp;
    const int nl = s->n_local;
    // raw symmetry functions with unit scaling
    cmd_nnp_model saved = M->model;
    for ( auto &E : M->model.el )
    {
        E.gmin.assign( E.sf.size(), 0.0 );
        E.gmax.assign( E.sf.size(), 1.0 );
    }
    M->model.smin = 0.0;
    M->model.smax = 1.0;
    M->plan_ok = false;
    cmd_status st = nnp_compute( M, s, n );
    std::vector<float> G( (size_t)std::max( nl, 1 ) * NSF_LD );
    std::vector<double4> x( std::max( nl, 1 ) );
    if ( st == CMD_OK && nl > 0 )
    {
        if ( hipMemcpy( G.data(), M->G.p, sizeof( float ) * G.size(),
                        hipMemcpyDeviceToHost ) != hipSuccess ||
             hipMemcpy( x.data(), s->x.p, sizeof( double4 ) * nl,
                        hipMemcpyDeviceToHost ) != hipSuccess )
        {
            set_error( "copy of symmetry functions failed" );
            st = CMD_ERR_HIP;
        }
    }
    M->model = saved;
    if ( st != CMD_OK )
        return st;
    for ( int e = 0; e < M->model.nelem; ++e )
    {
        auto &E = M->model.el[e];
        const int ns = (int)E.sf.size();
        std::vector<double> lo( ns, 1e300 ), hi( ns, -1e300 );
        for ( int i = 0; i < nl; ++i )
            if ( (int)x[i].w == e )
                for ( int k = 0; k < ns; ++k )
                {
                    lo[k] = std::min( lo[k], (double)G[(size_t)i * NSF_LD + k] );
                    hi[k] = std::max( hi[k], (double)G[(size_t)i * NSF_LD + k] );
                }
        for ( int k = 0; k < ns; ++k )
            if ( lo[k] <= hi[k] )
            {
                E.gmin[k] = lo[k];
                E.gmax[k] = hi[k];
            }
    }
    M->model.scale = true;
    M->plan_ok = false;
    return CMD_OK;
}

cmd_status cmd_nnp_lattice_create( int nx, int ny, int nz, double s,
                                   double jitter, double frac1, uint64_t seed,
                                   int *n, double *x, int *type, int *id )
{
    CMD_REQUIRE( nx > 0 && ny > 0 && nz > 0 && s > 0 && n && jitter >= 0 &&
                     jitter < 0.5 && frac1 >= 0 && frac1 <= 1,
                 CMD_ERR_ARG, "bad lattice description" );
    const int N = nx * ny * nz;
    *n = N;
    if ( !x )
        return CMD_OK;
    Mix rng{ seed };
    int k = 0;
    for ( int iz = 0; iz < nz; ++iz )
        for ( int iy = 0; iy < ny; ++iy )
            for ( int ix = 0; ix < nx; ++ix, ++k )
            {
                const int c[3] = { ix, iy, iz };
                for ( int d = 0; d < 3; ++d )
                    x[3 * k + d] =
                        ( c[d] + 0.5 + jitter * ( 2.0 * rng.uniform() - 1.0 ) ) * s;
                if ( id )
                    id[k] = k + 1;
            }
    if ( type )
    {
        const int n1 = (int)std::lround( N * frac1 );
        std::vector<int> t( N, 0 );
        for ( int i = 0; i < n1; ++i )
            t[i] = 1;
        for ( int i = N - 1; i > 0; --i )
        {
            const int j = (int)( rng.next() % (uint64_t)( i + 1 ) );
            std::swap( t[i], t[j] );
        }
        for ( int i = 0; i < N; ++i )
            type[i] = t[i];
    }
    return CMD_OK;
}

cmd_status cmd_force_nnp_model( const cmd_force *f, const cmd_nnp_model **m )
{
    CMD_REQUIRE( f && f->kind == 2 && m, CMD_ERR_ARG, "bad argument" );
    *m = &f->nnp->model;
    return CMD_OK;
}

// Work of the last compute under the flop model of roofline.h: out[0]
// neighbours inside rc, [1] triplets, [2] FP32 flops of the symmetry
// functions, [3] of the force chain, [4] of the network layers, [5] atoms.
cmd_status cmd_force_nnp_work( cmd_force *f, double out[6] )
{
    namespace F = cmd::nnp_flops;
    CMD_REQUIRE( f && f->kind == 2 && out, CMD_ERR_ARG, "bad argument" );
    cmd_nnp *M = f->nnp;
    double nb = 0.0, rad = 0.0, tri = 0.0, ang = 0.0, sf = 0.0, fc = 0.0;
    if ( M->n_last > 0 && M->terms.p )
    {
        std::vector<int4> t( M->n_last );
        CMD_HIP( hipMemcpy( t.data(), M->terms.p, sizeof( int4 ) * t.size(),
                            hipMemcpyDeviceToHost ) );
        // the kernels' path: the shorter one when every element's angular
        // rs are 0 (the launch in nnp_compute)
        bool rs0 = true;
        for ( int e = 0; e < M->plan.nelem; ++e )
            for ( int g = 0; g < M->plan.el[e].nag; ++g )
                rs0 = rs0 && M->plan.el[e].a_rs[g] == 0.f;
        for ( const int4 &a : t )
        {
            const int e = std::min( std::max( a.z, 0 ), M->plan.nelem - 1 );
            const cmd::NnpElemPlan &Q = M->plan.el[e];
            const double tr = a.y, angp = tr * Q.nap, angg = tr * Q.nag;
            nb += a.x;
            rad += (double)a.x * Q.nrg;
            tri += tr;
            ang += tr * Q.nag * Q.nap;
            sf += rs0 ? tr * F::SF_TRIP_RS0 + angp * F::SF_ANGP_RS0 + angg * F::SF_ANGG_RS0
                      : tr * F::SF_TRIP + angp * F::SF_ANGP + angg * F::SF_ANGG;
            fc += rs0 ? tr * F::F_TRIP_RS0 + angp * F::F_ANGP + angg * F::F_ANGG_RS0
                      : tr * F::F_TRIP + angp * F::F_ANGP + angg * F::F_ANGG;
        }
    }
    out[0] = nb;
    out[1] = tri;
    out[2] = nb * F::SF_NB + rad * F::SF_RAD + sf + ang * F::SF_ANG;
    out[3] = nb * F::F_NB + rad * F::F_RAD + fc + ang * F::F_ANG;
    // layers: the element with the largest network stands for all (the
    // models here give every element the same shape)
    double fwd = 0.0;
    for ( int e = 0; e < M->plan.nelem; ++e )
    {
        const cmd::NnpElemPlan &Q = M->plan.el[e];
        // nsf -> h1 -> h2 -> 1
        const double per = 2.0 * ( (double)Q.nsf * Q.h1 + (double)Q.h1 * Q.h2 + Q.h2 );
        fwd = std::max( fwd, per );
    }
    out[4] = F::MLP_PASSES * fwd * M->n_last;
    out[5] = M->n_last;
    return CMD_OK;
}

// Per-atom symmetry functions, dE/dG (both ld = stride floats per atom) and
// atomic energies of the last compute (any pointer may be NULL).
cmd_status cmd_force_nnp_atomic( cmd_force *f, cmd_system *s, int ld, float *G,
                                 float *dEdG, float *Ei )
{
    CMD_REQUIRE( f && f->kind == 2 && s && ld >= 1, CMD_ERR_ARG, "bad argument" );
    cmd_nnp *M = f->nnp;
    const int n = s->n_local;
    CMD_REQUIRE( M->cap >= n, CMD_ERR_STATE, "no NNP force computed yet" );
    std::vector<float> h( (size_t)std::max( n, 1 ) * NSF_LD );
    auto rows = [&]( const float *d, float *o ) -> cmd_status
    {
        CMD_HIP( hipMemcpy( h.data(), d, sizeof( float ) * (size_t)n * NSF_LD,
                            hipMemcpyDeviceToHost ) );
        for ( int i = 0; i < n; ++i )
            for ( int k = 0; k < std::min( ld, NSF_LD ); ++k )
                o[(size_t)i * ld + k] = h[(size_t)i * NSF_LD + k];
        return CMD_OK;
    };
    if ( G && n > 0 )
        CMD_TRY( rows( M->G.p, G ) );
    if ( dEdG && n > 0 )
        CMD_TRY( rows( M->dEdG.p, dEdG ) );
    if ( Ei && n > 0 )
        CMD_HIP( hipMemcpy( Ei, M->Ei.p, sizeof( float ) * n, hipMemcpyDeviceToHost ) );
    return CMD_OK;
}

} // extern "C"

namespace cmd
{
cmd_status nnp_model_copy( const cmd_nnp_model *m, cmd_nnp_model **out )
{
    *out = new cmd_nnp_model( *m );
    return CMD_OK;
}

// Atomic numbers of the element symbols n2p2 files name (weights.%03d.data).
static int atomic_number( const std::string &sym )
{
    static const char *const table[] = {
        "H",  "He", "Li", "Be", "B",  "C",  "N",  "O",  "F",  "Ne", "Na", "Mg",
        "Al", "Si", "P",  "S",  "Cl", "Ar", "K",  "Ca", "Sc", "Ti", "V",  "Cr",
        "Mn", "Fe", "Co", "Ni", "Cu", "Zn", "Ga", "Ge", "As", "Se", "Br", "Kr",
        "Rb", "Sr", "Y",  "Zr", "Nb", "Mo", "Tc", "Ru", "Rh", "Pd", "Ag", "Cd",
        "In", "Sn", "Sb", "Te", "I",  "Xe", "Cs", "Ba", "La", "Ce", "Pr", "Nd",
        "Pm", "Sm", "Eu", "Gd", "Tb", "Dy", "Ho", "Er", "Tm", "Yb", "Lu", "Hf",
        "Ta", "W",  "Re", "Os", "Ir", "Pt", "Au", "Hg", "Tl", "Pb", "Bi", "Po",
        "At", "Rn" };
    for ( int z = 0; z < (int)( sizeof( table ) / sizeof( table[0] ) ); ++z )
        if ( sym == table[z] )
            return z + 1;
    return 0;
}

cmd_status nnp_load_deck_model( const char *dir, cmd_nnp_model **out )
{
    CMD_REQUIRE( dir && dir[0], CMD_ERR_ARG,
                 "pair_style nnp needs a model directory (dir <path>)" );
    std::ifstream in( std::string( dir ) + "/input.nn" );
    CMD_REQUIRE( in.good(), CMD_ERR_IO, "cannot read %s/input.nn", dir );
    std::vector<std::string> names;
    std::string line;
    while ( std::getline( in, line ) )
    {
        const auto w = words_of( line );
        if ( w.size() >= 2 && w[0] == "elements" )
            names.assign( w.begin() + 1, w.end() );
    }
    CMD_REQUIRE( !names.empty() && (int)names.size() <= NNP_MAXEL, CMD_ERR_IO,
                 "input.nn must list 1..%d elements", NNP_MAXEL );
    std::vector<const char *> np;
    std::vector<int> z;
    for ( const auto &nm : names )
    {
        np.push_back( nm.c_str() );
        z.push_back( atomic_number( nm ) );
        CMD_REQUIRE( z.back() > 0, CMD_ERR_IO, "unknown element symbol %s",
                     nm.c_str() );
    }
    return cmd_nnp_model_load_n2p2( dir, (int)names.size(), np.data(), z.data(),
                                    out );
}

cmd_status nnp_destroy( cmd_nnp *M )
{
    delete M;
    return CMD_OK;
}
cmd_status nnp_set_precision( cmd_nnp *M, int prec )
{
    M->prec = prec;
    return CMD_OK;
}
// ForceNNP::compute_energy (impl.h:101-130): sum of atomic energies plus
// N_local times element 0's offset, over convEnergy (1: no normalisation),
// plus N times meanEnergy (0), times the hard-coded 27.211384021355236.
__global__ void k_nnp_ei_f64( int n, const float *__restrict__ Ei, double *__restrict__ out )
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if ( i < n )
        out[i] = (double)Ei[i];
}

cmd_status nnp_atom_energy( cmd_nnp *M, int n, double *out, hipStream_t st )
{
    if ( n <= 0 )
        return CMD_OK;
    CMD_REQUIRE( M->cap >= n, CMD_ERR_STATE, "no atomic energies for %d atoms", n );
    k_nnp_ei_f64<<<( n + 255 ) / 256, 256, 0, st>>>( n, M->Ei.p, out );
    CMD_LAUNCH_CHECK();
    return CMD_OK;
}

double nnp_energy_offset( const cmd_nnp *M ) { return M->model.el[0].atom_energy; }

cmd_status nnp_reference_energy( cmd_nnp *M, cmd_system *S, double *pe )
{
    double sum = 0.0;
    CMD_TRY( nnp_energy_sum( M, S, &sum ) );
    *pe = ( sum + S->n_local * M->model.el[0].atom_energy ) * 27.211384021355236;
    return CMD_OK;
}
} // namespace cmd
