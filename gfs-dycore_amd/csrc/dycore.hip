// Device-resident GFS hybrid sigma-pressure dynamical core step.
//
// State lives in HBM in a coefficient-major layout spec[k][field] (complex),
// field = member * nfs + {vrt[nlev], div[nlev], tv[nlev], trac[ntrac*nlev], lnps},
// so one launch covers every level, variable and ensemble member:
//   getdyntend (dyn_run.f90:33-305): one batched synthesis of all grid fields,
//     one column kernel (pressure_data.f90:58 calc_pressdata, dyn_run.f90:307
//     getomega, :375 getpresgrad, :453 getvadv, :190-272 tendency assembly), one
//     batched analysis scattered straight into tendency fields.
//   advance (run.f90:194-565): IMEX RK3 stages with the semi-implicit solve per
//     spectral coefficient (one wavefront per coefficient, lane = level), implicit
//     damping, then the time-split physics -- Held-Suarez (phy_run_hs.f90:22) or
//     the simple moist physics (phy_run_simple.f90:28, simple_physics_v5_1.f90) --
//     and the dry-mass fixer (dyn_run.f90:605) with FP64 global sums.
// Grid fields synthesised per member (nsyn): u, v, vrt, div, tv, dtv/dx, dtv/dy
// (nlev each), tracers q, dq/dx, dq/dy (ntrac*nlev each), ln ps', dlnps/dx, dlnps/dy.
// ln(ps) is synthesised without its global-mean coefficient c0 = q_00 / sqrt(4 pi):
// ps = exp(c0 + ln ps') is formed in FP64 and the mass fixer analyses
// ln ps' + ln(pcorr) (= log(ps pcorr) - c0), adding c0 back to q_00. This is the
// reference's arithmetic (ln(ps) and log(ps pcorr) transformed to spectral space),
// rearranged so that the FP32 path does not round a ~11.5 grid field to ~1e-6.
#include <cfloat>
#include <cmath>
#include <cstring>

#include "engine.h"
#include "mlp.h"

namespace gfsdc {

#define SGLF(x) ((double)(float)(x))

// IMEX tableau, semimp_data.f90:74-88 (default-real literals)
static const double TAB_A[3][3] = {{SGLF(1. / 3.), 0, 0}, {SGLF(1. / 6.), SGLF(1. / 2.), 0},
                                   {SGLF(1. / 2.), SGLF(-1. / 2.), 1.0}};
static const double TAB_AA[3][3] = {{SGLF(1. / 6.), 0, 0}, {SGLF(1. / 3.), 0.0, 0},
                                    {SGLF(3. / 8.), 0.0, SGLF(3. / 8.)}};
static const double TAB_IMP[3] = {SGLF(1. / 6.), SGLF(1. / 3.), SGLF(1. / 4.)};

constexpr int MAXLEV = 64;  // levels map onto the 64 lanes of a wavefront in the solve

// counter-based RNG: splitmix64 finaliser over a mixed (seed, stream, index) key
__host__ __device__ inline uint64_t rng_mix(uint64_t seed, uint64_t stream, uint64_t index) {
    uint64_t z = seed * 0x9E3779B97F4A7C15ULL ^ (stream + 0x632BE59BD9B4E019ULL) * 0xBF58476D1CE4E5B9ULL;
    z += index * 0x94D049BB133111EBULL + 0x9E3779B97F4A7C15ULL;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}

struct Coeffs3 {
    double a[3];
};

struct DycoreBuffers {
    int nl = 0, ntr = 0, nm = 0;
    int nfs = 0;    // state fields per member
    int nsyn = 0;   // synthesised grid fields per member
    int nan = 0;    // analysed grid fields per member
    int nhs = 0;    // Held-Suarez forcing fields per member (3 nlev + 1)
    int nsp = 0;    // simple-physics grid fields per member: dT, du, dv, dq (nlev each), mass fixer
    long ng = 0;
    void *spec = nullptr, *spec0 = nullptr, *ten[3] = {nullptr, nullptr, nullptr};
    // what the second and the third stage need of the earlier ones' tendencies and linear
    // terms (k_si_mfma's E1, E2; none in the explicit scheme): div[nl], tv[nl], lnps per member
    void *mix[2] = {nullptr, nullptr};
    void *tphys = nullptr;                       // physics tendencies
    void *gsyn = nullptr, *gan = nullptr;        // grid fields (T)
    void *gmean = nullptr;                       // global means added back by the Fourier synthesis (nm * nsyn)
    void *etadot = nullptr, *dlnpdt = nullptr;   // per member (nl+1)*ng, nl*ng
    void *psg = nullptr, *dlnpsdt = nullptr;     // per member ng
    void *dphisdx = nullptr, *dphisdy = nullptr; // per member ng
    void *topo = nullptr;                        // spectral orography per member (complex)
    void *Work = nullptr;                        // Work<T>*
    // operators (T)
    void *at = nullptr, *bt = nullptr, *dt3 = nullptr;  // transposed amhyb, bmhyb, d_hyb_m
    void *sv = nullptr, *tor = nullptr;
    void *disspec = nullptr, *diffp = nullptr, *dmpp = nullptr;
    void *ak = nullptr, *bk = nullptr, *ck = nullptr, *dbk = nullptr, *dak = nullptr;  // T
    void *sinlat = nullptr, *coslat = nullptr, *areaw = nullptr;      // T, nlat; areaw FP64 nlat
    int2 *si_tiles = nullptr;                    // (degree, first item) tiles of the matrix-core solve
    int n_si_tiles = 0;
    int *degree = nullptr;                       // degree of coefficient k
    double *pdryini = nullptr, *pmean = nullptr; // FP64 per member
    double *pspart = nullptr;                    // FP64 partial sums and ranges (4 x PS_BLOCKS per member)
    unsigned *psdone = nullptr;                  // workgroups and members that have arrived (k_area), zero between calls
    double *pwsum = nullptr;                     // FP64 area sum of pwat per member
    void *colq = nullptr;                        // T per member ng: column tracer mass sum(dpk q)
    void *pwat = nullptr, *precip = nullptr;     // T per member ng (simple physics)
    double *latd = nullptr;                      // FP64 latitude (radians), nlat
    // AR(1) temperature pattern (patterngenerator.f90), per member
    void *tpat = nullptr;                        // cplx<T> nm * nlm
    double *tpat_var = nullptr;                  // FP64 nlm, normalised variance spectrum
    void *tpat_vf = nullptr;                     // T nlev, vertical taper (bottom -> top)
    unsigned long long *tpat_ctr = nullptr;      // advances so far (random stream index)
    double tpat_phi = 0.0;
    // learned column physics (replaces the simple-physics column call when on)
    MlpNet *mlp = nullptr;
    float *ds_x = nullptr, *ds_y = nullptr;      // dataset: raw features / targets [cap][nin|nout]
    long ds_cap = 0, ds_n = 0;
    float *nrm = nullptr;                        // [mean_x | std_x | mean_y | std_y]
    bool nrm_ready = false, mlp_on = false;
    float *xin = nullptr, *yout = nullptr;       // inference rows [nm*ng][nin], [nm*ng][nout]
    float *tbx = nullptr, *tby = nullptr;        // training batch (normalised)
    int judge_stride = 50;
    double judge_thr = 0.5;
    void *ganj = nullptr, *pwatj = nullptr, *precipj = nullptr;  // plain physics on the judged columns
    double *jpart = nullptr, *jstat = nullptr;   // judge partial sums; [last error, fallbacks, judged steps]
    int *jflag = nullptr;                        // 1: this step falls back to the plain physics
    unsigned long long *jctr = nullptr;          // judge / sampling step counter
    unsigned long long bctr = 0;                 // training batch counter
    double *diag = nullptr;                      // FP64 4 per member
    // stochastic physics (stoch_data.f90): kinds 0 svc, 1 sppt, 2 shum (one
    // pattern per member each, st_pat2 [kind][member][nlm]) and 3 addnoise (one
    // per level and member, [member][level][nlm])
    gfsdc_stoch_cfg sc{};
    int st_on[4] = {0, 0, 0, 0}, st_nf[4] = {1, 1, 1, 1};
    double st_phi[4] = {0, 0, 0, 0}, st_sd[4] = {0, 0, 0, 0};
    unsigned long long st_seed[4] = {0, 0, 0, 0};
    void *st_pat2 = nullptr, *st_pat[4] = {nullptr, nullptr, nullptr, nullptr};
    double *st_var = nullptr;                    // FP64 [4][nlm]
    void *st_vf = nullptr;                       // T [4][nl]
    unsigned long long *st_ctr = nullptr;        // advances per kind [4]
    void *st_grd = nullptr;                      // T [kind 0..2][member][ng]
    SynthDesc *sd_pat = nullptr;                 // [kind 0..2][member]
    unsigned char *rf0 = nullptr;                // zero 1/cos flags
    bool vc_on = false;
    void *vcg = nullptr;                         // T [member][2 nl][ng] vorticity gradient
    SynthDesc *sd_vc = nullptr;                  // [member][2 nl]
    unsigned char *rf1 = nullptr;                // one 1/cos flags
    void *an_w = nullptr;                        // cplx<T> [group 3][member][nl][nlm]
    void *an_g = nullptr;                        // T [group 3][member][nl][ng]
    void *an_sm = nullptr;                       // T nlm smoothing factors
    SynthDesc *sd_an = nullptr;                  // [ud, vd, psi | group 1 copy | group 0 copy]
    AnalDesc *ad_an = nullptr;                   // [member][nl]
    unsigned char *rf_an = nullptr;              // [group][member][nl]: 1, 1, 0
    double *clock = nullptr;                     // model time (s) at the start of the next step
    // incremental analysis update (iau_module.f90): nfiles increments of the
    // whole state in the state layout, their times (h) and the forcing of a step
    int iau_n = 0;
    double *iau_hrs = nullptr, iau_dt = 0.0;
    void *iau_inc = nullptr, *iau_F = nullptr;
    // the dynamics synthesis: the gather and Legendre GEMM take nleg fields per
    // member (every grid field but the x-gradients dtv/dx, dq/dx, dlnps/dx,
    // which the Fourier synthesis forms from its scalar's Legendre output through
    // fmap_dyn); the Fourier synthesis writes all nsyn grid fields
    SynthDesc *sdesc = nullptr;                  // nm*nleg
    int nleg = 0;
    FieldMap fmap_dyn;
    // the physics pass synthesises every field but the temperature and tracer
    // gradients (nph per member): descriptors, 1/cos flags and grid slots
    int nph = 0;
    SynthDesc *sdesc_ph = nullptr;
    unsigned char *rflag_ph = nullptr;
    int *slot_ph = nullptr;
    // the lean Held-Suarez physics pass of the steps before an advance's last
    // synthesises only the grids the forcing reads (phy_run_hs.f90:66-76); the
    // winds, their gradients and getomega serve only the post-step grids and
    // diagnostics. Its fields: temperature and ln ps (nhla = nm (nl + 1),
    // member-major), then vorticity and divergence level-major from the lowest
    // level (nhlb = 2 nm nl: level k, member, vrt / div), of which it
    // transforms only the levels where the drag can act
    int nhla = 0, nhlb = 0;
    SynthDesc *sdesc_hl = nullptr;
    unsigned char *rflag_hl = nullptr;
    int *slot_hl = nullptr;
    // device counts of the lean pass, written by k_area: [0] fields of
    // the vorticity / divergence synthesis that follows the drag's count (0
    // where the first synthesis already held every level with drag), [1]
    // Held-Suarez forcing fields to analyse, [2] nact, the levels counted from
    // the lowest whose drag is evaluated, [3] fields of the next lean pass's
    // first synthesis, [4] the levels it takes (the last nact plus one)
    int *hsdyn = nullptr;
    // the grids after the last step are those of a lean pass (profile_step):
    // get_grid and step_diag refuse them
    bool grids_partial = false;
    // adesc_hsu: the Held-Suarez forcing's analysis applied to the state in
    // place (state += dt tendency, the mass fixer's ln ps update) for advance
    AnalDesc *adesc_dyn = nullptr, *adesc_hs = nullptr, *adesc_hsu = nullptr, *adesc_sp = nullptr;
    unsigned char *rflag_syn = nullptr, *rflag_an = nullptr, *rflag_hs = nullptr, *rflag_sp = nullptr;
    // host copies of the FP64 operators
    std::vector<double> amhyb, bmhyb, svhyb, tor_hyb, d_hyb_m, disspec_h, diff_h, dmp_h, sl;
    std::vector<double> ym;                       // tor (x) sv + amhyb bmhyb (semimp_data.f90:225-234)
    hipGraph_t graph = nullptr, graph_lean = nullptr;
    hipGraphExec_t gexec = nullptr, gexec_lean = nullptr;
    // profiling
    bool profiling = false;
    std::vector<hipEvent_t> ev;
    std::vector<std::string> evname;
};

// drop the captured steps: the next graph advance captures them again
static void drop_graph(DycoreBuffers *B) {
    if (B->gexec) (void)hipGraphExecDestroy(B->gexec);
    if (B->graph) (void)hipGraphDestroy(B->graph);
    if (B->gexec_lean) (void)hipGraphExecDestroy(B->gexec_lean);
    if (B->graph_lean) (void)hipGraphDestroy(B->graph_lean);
    B->gexec = B->gexec_lean = nullptr;
    B->graph = B->graph_lean = nullptr;
}

// ---------------------------------------------------------------------------
// kernels

// ps = exp(q_00 / sqrt(4 pi) + ln ps'), rounded alike in every kernel that forms it
template <typename T> __device__ __forceinline__ T full_ps(T q00, T lnps) {
    return (T)exp(fma((double)q00, 0.28209479177387814, (double)lnps));
}

// Layer coefficients of calc_pressdata / getpresgrad for K >= 2 (pressure_data.f90:
// 76-82, dyn_run.f90:393-410): rlnp = ln(p2/p1), alfa = 1 - p1/dp rlnp,
// cofa = -(bk_K p1/p2 - bk_{K-1} + rlnp (bk_{K-1} - p1 dbk/dp)) / dp and the cofb
// increment bk_K / p2 - bk_{K-1} / p1. With thin layers (dp/p of a few per cent)
// these expressions cancel to a few per cent of their terms; FP64 evaluates
// them as written, FP32 uses identities exact in real arithmetic that do not
// cancel (y = rlnp):
//   rlnp = ln(1 + x) = 2 atanh(u), x = dp / p1, u = x / (2 + x) <= 1/3 for x <= 1,
//          = 2 (u + u^3/3 + ... + u^15/15) (truncation 5e-9 at u = 1/3),
//   alfa = 1 - y / (e^y - 1) = y/2 - y^2/12 + y^4/720 - y^6/30240 + y^8/1209600
//          - y^10/47900160 (Bernoulli series, truncation 5e-10 at y = 1),
//   bk_K p1/p2 - bk_{K-1} = -ck / p2 and bk_{K-1} - p1 dbk / dp = ck / dp, so
//   cofa = (ck / dp) (e^-y - 1 + alfa) / p1 = (ck / dp) (alfa - dp / p2) / p1,
//   bk_K / p2 - bk_{K-1} / p1 = -ck / (p1 p2),
// with ck = ak_K bk_{K-1} - ak_{K-1} bk_K formed in FP64 on the host. The layer
// thickness is dp = dak + dbk ps from the FP64 differences of ak and bk (the
// difference of the rounded interface pressures would carry their rounding,
// amplified by p/dp).
// 1 / x: the hardware reciprocal (1 ulp) in FP32, where it feeds products and
// never a cancellation; a division in FP64
__device__ __forceinline__ float recip(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ double recip(double x) { return 1.0 / x; }
// x at p + v + s bytes (v in a vector, s in a scalar register), below 4 GiB past p
typedef unsigned bufu2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void *p) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, 0xFFFFFFFFu, 0x00020000);  // raw, 32-bit data
}
__device__ __forceinline__ float buf_load(const float *p, unsigned v, unsigned s) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(buf_rsrc(p), v, s, 0));
}
__device__ __forceinline__ double buf_load(const double *p, unsigned v, unsigned s) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(buf_rsrc(p), v, s, 0));
}
__device__ __forceinline__ void buf_store(float *p, unsigned v, unsigned s, float x) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, x), buf_rsrc(p), v, s, 0);
}
__device__ __forceinline__ void buf_store(double *p, unsigned v, unsigned s, double x) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(bufu2, x), buf_rsrc(p), v, s, 0);
}
template <typename T>
__device__ __forceinline__ void layer_log(T p1, T p2, T dpk, T rp1, T rdp, T &rlnp, T &alfa) {
    if constexpr (sizeof(T) == 4) {
        const T x = dpk * rp1;
        T y;
        if (x <= T(1)) {
            const T u = x * recip(T(2) + x), u2 = u * u;
            y = T(2) * u *
                (T(1) + u2 * (T(1.0 / 3.0) +
                              u2 * (T(0.2) + u2 * (T(1.0 / 7.0) + u2 * (T(1.0 / 9.0) +
                                                                       u2 * (T(1.0 / 11.0) +
                                                                             u2 * (T(1.0 / 13.0) + u2 * T(1.0 / 15.0))))))));
        } else {
            y = log1p(x);
        }
        rlnp = y;
        if (y <= T(1)) {
            const T y2 = y * y;
            alfa = y * T(0.5) -
                   y2 * (T(1.0 / 12.0) -
                         y2 * (T(1.0 / 720.0) -
                               y2 * (T(1.0 / 30240.0) - y2 * (T(1.0 / 1209600.0) - y2 * T(1.0 / 47900160.0)))));
        } else {
            alfa = T(1) - (p1 * rdp) * y;
        }
    } else {
        rlnp = log(p2 * rp1);
        alfa = T(1) - (p1 * rdp) * rlnp;
    }
}
// dbp = bk_K / p2 - bk_{K-1} / p1
template <typename T>
__device__ __forceinline__ void layer_rest(T p1, T dpk, T bk1, T bk2, T ck, T dbk, T rp1, T rp2, T rdp, T rlnp, T alfa,
                                           T &cofa, T &dbp) {
    if constexpr (sizeof(T) == 4) {
        cofa = ck * rdp * (alfa - dpk * rp2) * rp1;
        dbp = -ck * rp1 * rp2;
    } else {
        cofa = -rdp * (bk2 * p1 * rp2 - bk1 + rlnp * (bk1 - p1 * dbk * rdp));
        dbp = bk2 * rp2 - bk1 * rp1;
    }
}

// Column kernel: calc_pressdata + getomega (+ getpresgrad, getvadv, getvadv_tracers
// and the tendency assembly unless COL_INV). A workgroup holds NC grid columns of
// one member with the levels split over CH threads of each column, up to LPC
// consecutive layers a thread, so that a layer's inputs are read once, all loads
// of a thread are in flight together and the layers' terms stay in registers
// between the two halves: first every thread forms its layers' terms and their
// sums, then it takes the sums over the layers above (getomega's) and below
// (getpresgrad's) it from the other threads' sums in LDS.
// Measured in kernel traces, which start every kernel with cold caches (us a
// launch, against one thread per column, whose bottom-up pass read u, v and the
// divergence again): T254L64 FP32 192 from 228, 838 MB at 4.4 TB/s where a large
// copy reaches 4.6-5.3; 16 members T126L64 664 from 827; T126L64 54 from 106, with
// a tracer 87 from 223; T42L20 FP64 9 from 28. Whole steps: T42L20 FP64 1.17 times
// as fast, T126L64 with a tracer 1.07, T254L64 1.05. 8 chunks of 8 layers in 128
// registers keep two workgroups on a CU: 16 chunks of 4 took 270 at T254L64, 8
// without the bound (141 registers, one workgroup) 258.
// Index conventions: K counts interfaces/layers top -> bottom (1-based, as pk,
// dpk, alfa, rlnp, etadot), L = nl + 1 - K model levels bottom -> top (as u, v, tv).
// getomega's two running sums, of div dp and of (V . grad ln ps) dbk over the
// layers above, appear only as s = db + ps cb: omega / p = (workc - alfa t - rlnp s) / dp
// with the layer's own t = div dp + ps (V . grad ln ps) dbk, etadot = -s - ps bk dlnpsdt,
// dlnpsdt = -s(surface) / ps. s is summed in FP64.
// COL_VC adds the vorticity-confinement flux (dyn_run.f90:230-248) from the
// vorticity gradient vcg [member][2 nl][ng] (x then y), with speed vcamp
// times 1 + vfsvc[level] svcg (the svc pattern grid [member][ng]) when svcg is set.
enum ColMode { COL_DYN = 0, COL_VC = 1, COL_INV = 2 };
template <typename T> struct ColCfg { static constexpr int NC = 64, CH = 8; };
template <> struct ColCfg<double> { static constexpr int NC = 32, CH = 16; };  // twice the registers a value
template <typename T, int MODE, int LPC, bool TR>
__global__ __launch_bounds__(ColCfg<T>::NC * ColCfg<T>::CH, sizeof(T) * LPC <= 16 || sizeof(T) == 4 ? 4 : 2) void k_columns(
    const T *__restrict__ gsyn, T *__restrict__ gan, T *__restrict__ etadot, T *__restrict__ dlnpdt,
    T *__restrict__ psg_out, T *__restrict__ dlnpsdt_out, const T *__restrict__ dphisdx,
    const T *__restrict__ dphisdy, const T *__restrict__ ak_, const T *__restrict__ bk_,
    const T *__restrict__ ck_, const T *__restrict__ dbk_, const T *__restrict__ dak_, const T *__restrict__ sinlat,
    int nl, int ntr_, int nsyn, int nan, long ng, int nlon, T rd, T kappa, T cvcp, T twoom,
    const cplx<T> *__restrict__ spec, int nfs, T *__restrict__ colq, const T *__restrict__ vcg,
    const T *__restrict__ svcg, const T *__restrict__ vfsvc, T vcamp, int store) {
    constexpr int NC = ColCfg<T>::NC, CH = ColCfg<T>::CH;
    constexpr bool DYN = MODE != COL_INV, VC = MODE == COL_VC;
    const int ntr = TR ? ntr_ : 0;  // TR: there are tracers
    __shared__ T ak[MAXLEV + 1], bk[MAXLEV + 1], ck[MAXLEV], dbk[MAXLEV], dak[MAXLEV];
    __shared__ double ssum[CH][NC];
    // per chunk and column: the column tracer mass, getpresgrad's three sums, u, v
    // and tv of the chunk's first and last layer
    enum { S_CQ, S_COF, S_PX, S_PY, S_U0, S_V0, S_T0, S_U1, S_V1, S_T1, S_N };
    __shared__ T sh[DYN ? S_N : S_COF][CH][NC];
    const int tid = threadIdx.x, ln = tid % NC;
    const int w = NC == 64 ? __builtin_amdgcn_readfirstlane(tid / NC) : tid / NC;  // chunk
    for (int i = tid; i <= nl; i += NC * CH) {
        ak[i] = ak_[i];
        bk[i] = bk_[i];
        if (i < nl) {
            ck[i] = ck_[i];
            dbk[i] = dbk_[i];
            dak[i] = dak_[i];
        }
    }
    const int mem = blockIdx.y, lpc = (nl + CH - 1) / CH;
    const int K0 = w * lpc, cnt = min(max(nl - K0, 0), lpc);  // layers K0 + 1 .. K0 + cnt
    const long c_ = (long)xcd_tile(blockIdx.x, gridDim.x) * NC + ln;  // neighbours on one XCD: ensemble 708 -> 664 us
    const bool valid = c_ < ng;
    const unsigned col = (unsigned)(valid ? c_ : ng - 1), cb = col * (unsigned)sizeof(T);
    const T *G = gsyn + (long)mem * nsyn * ng;
    const T *U = G, *V = G + (long)nl * ng, *VRT = G + 2L * nl * ng, *DIV = G + 3L * nl * ng;
    const T *TV = G + 4L * nl * ng, *TX = G + 5L * nl * ng, *TY = G + 6L * nl * ng, *Q = G + 7L * nl * ng;
    const T *LNPS = G + (7L + 3L * ntr) * nl * ng;
    // This column's value at layer K = K0 + 1 + i (clamped to the column) of a field of
    // nl levels, level nl - K: the descriptor starts at the wavefront's lowest level, so
    // that a field may be of any size, the layer's offset is in a scalar register and the
    // column's in a vector register, where FP64 also has the distance between the
    // wavefront's two chunks (a layer's offset that differed between them would make
    // every access a loop over the two).
    constexpr bool TWO = NC < 64;
    const unsigned lb = (unsigned)(ng * sizeof(T));
    const int w0 = __builtin_amdgcn_readfirstlane(tid / NC);  // the wavefront's first chunk
    const int Kw = TWO ? (w0 + 1) * lpc : K0;                 // layers above its last one
    auto level = [&](int K, int i) { return min(max(nl - 1 - K - i, 0), nl - 1); };
    const int low = level(Kw, lpc + 1);  // tracers reach two layers past the chunk
    auto voff = [&](int i) { return TWO ? cb + (unsigned)(level(K0, i) - level(Kw, i)) * lb : cb; };
    auto soff = [&](int i) { return (unsigned)(level(Kw, i) - low) * lb; };
    auto ld = [&](const T *P, int i) { return buf_load(P + (long)low * ng, voff(i), soff(i)); };
    auto st = [&](T *P, int i, T x) { buf_store(P + (long)low * ng, voff(i), soff(i), x); };
    // etadot at interface K0 + i, counted from the top
    const int top = w0 * lpc;
    const unsigned ve = TWO ? cb + (unsigned)(K0 - top) * lb : cb;
    T *ET = etadot + (long)mem * (nl + 1) * ng;
    auto ste = [&](int i, T x) { buf_store(ET + (long)top * ng, ve, (unsigned)i * lb, x); };
    T u[LPC], v[LPC], dv[LPC], tv[LPC], tx[LPC], ty[LPC], vr[LPC], q1[LPC];
#pragma unroll
    for (int i = 0; i < LPC; i++)
        if (i < lpc) {
            u[i] = ld(U, i);  // past the lowest layer nothing is used
            v[i] = ld(V, i);
            dv[i] = ld(DIV, i);
            if constexpr (DYN) {
                tv[i] = ld(TV, i);
                tx[i] = ld(TX, i);
                ty[i] = ld(TY, i);
                vr[i] = ld(VRT, i);
                if constexpr (TR) q1[i] = ld(Q, i);
            }
        }
    const T dpx = LNPS[ng + col], dpy = LNPS[2 * ng + col];
    const T c00 = spec[(long)mem * nfs + 3L * nl + (long)ntr * nl].x;
    const T ps = full_ps(c00, LNPS[col]);
    const T gpx = ps * dpx, gpy = ps * dpy;
    const T alfa1 = T(SGLF(0.69314718055994530942)), rlnp1 = T(SGLF(99999.99));
    __syncthreads();  // the level tables
    auto pk = [&](int K) -> T { return ak[K - 1] + bk[K - 1] * ps; };
    auto dp = [&](int K) -> T { return fma(dbk[K - 1], ps, dak[K - 1]); };  // pk(K + 1) - pk(K), one rounding
    // the layers' terms, bottom -> top; fx0, fy0 are the fluxes with the pressure
    // gradient of the sums over the chunk's own layers below
    T f = T(0), dphx = T(0), dphy = T(0);
    if constexpr (DYN) {
        f = twoom * sinlat[col / (unsigned)nlon];
        dphx = dphisdx[(long)mem * ng + col];
        dphy = dphisdy[(long)mem * ng + col];
    }
    T q[LPC], w1[LPC], w2[LPC], adv[LPC], fx0[LPC], fy0[LPC];
    T cof = T(0), px = T(0), py = T(0);
    T p2 = pk(min(K0 + cnt, nl) + 1), rp2 = recip(p2);
#pragma unroll
    for (int i = LPC - 1; i >= 0; i--)
        if (i < cnt) {
            const int K = K0 + 1 + i;
            const T dpk = dp(K), p1 = pk(K), rp1 = recip(p1), cg = gpx * u[i] + gpy * v[i];
            const T t = fma(cg, dbk[K - 1], dv[i] * dpk);
            q[i] = t;
            const T rdp = recip(dpk);
            T rlnp = rlnp1, alfa = alfa1, cofa, dbp, cofb0, workc, workb = t;
            if (K == 1) {
                cofa = -rdp * (bk[1] * p1 * rp2 - bk[0] + rlnp * (bk[0] - p1 * dbk[0] * rdp));
                dbp = T(0);  // no layer above takes it
                cofb0 = -rdp * (alfa * dbk[0]);
                workc = cg * dbk[0];
                workb = dv[i] * dpk + workc * dbk[0];
                w1[i] = T(0);
            } else {
                layer_log(p1, p2, dpk, rp1, rdp, rlnp, alfa);
                layer_rest(p1, dpk, bk[K - 1], bk[K], ck[K - 1], dbk[K - 1], rp1, rp2, rdp, rlnp, alfa, cofa, dbp);
                cofb0 = -rdp * (bk[K - 1] * rlnp + alfa * dbk[K - 1]);
                w1[i] = rlnp * rdp;
                workc = cg * (dbk[K - 1] + ck[K - 1] * w1[i]);
            }
            w2[i] = (workc - alfa * workb) * rdp;
            if constexpr (DYN) {
                // prsgx = c ps dpx + px - rd alfa tx - dphx, c and px with the sums below
                const T rt = rd * tv[i], c = (cofb0 - cofa) * rt + cof, z = vr[i] + f;
                fx0[i] = u[i] * z - (c * gpy + (py - rd * alfa * ty[i]));
                fy0[i] = v[i] * z + (c * gpx + (px - rd * alfa * tx[i]));
                adv[i] = -u[i] * tx[i] - v[i] * ty[i];
                cof -= dbp * rt;
                px -= rd * rlnp * tx[i];
                py -= rd * rlnp * ty[i];
            }
            p2 = p1;
            rp2 = rp1;
        }
    // s within the chunk, over the layers down to and including i
    double sum = 0.0;
#pragma unroll
    for (int i = 0; i < LPC; i++)
        if (i < cnt) {
            sum += (double)q[i];
            q[i] = (T)sum;
        }
    ssum[w][ln] = sum;
    if constexpr (DYN) {
        sh[S_COF][w][ln] = cof;
        sh[S_PX][w][ln] = px;
        sh[S_PY][w][ln] = py;
        sh[S_U0][w][ln] = u[0];
        sh[S_V0][w][ln] = v[0];
        sh[S_T0][w][ln] = tv[0];
#pragma unroll
        for (int i = 0; i < LPC; i++)
            if (i == cnt - 1) {
                sh[S_U1][w][ln] = u[i];
                sh[S_V1][w][ln] = v[i];
                sh[S_T1][w][ln] = tv[i];
            }
    }
    if (TR && colq) {
        // column tracer mass of the dry-mass diagnostic (dyn_run.f90:138-145)
        T s = T(0);
        for (int i = 0; i < cnt; i++) {
            T qs = T(0);
            for (int nt = 0; nt < ntr; nt++) qs += ld(Q + (long)nt * nl * ng, i);
            s += dp(K0 + 1 + i) * qs;
        }
        sh[S_CQ][w][ln] = s;
    }
    __syncthreads();
    // s over the chunks above this one, over those and this one, over the column
    double sa = 0.0, sb = 0.0, tot = 0.0;
#pragma unroll
    for (int c = 0; c < CH; c++) {
        if (c == w) sa = tot;
        tot += ssum[c][ln];
        if (c == w) sb = tot;
    }
    const T dlnpsdt = -(T)tot / ps, ah = (T)sa, al = (T)(sa - (double)ah), bh = (T)sb;
    if (w == 0 && valid) {
        psg_out[(long)mem * ng + col] = ps;
        dlnpsdt_out[(long)mem * ng + col] = dlnpsdt;
        if (TR && colq) {
            T s = T(0);
            for (int c = 0; c < CH; c++) s += sh[S_CQ][c][ln];
            colq[(long)mem * ng + col] = s;
        }
    }
    if (!valid) return;
    // s over the layers above layer i of the chunk (i = cnt: above the next chunk)
    auto above = [&](int i) { return i == 0 ? ah : i == cnt ? bh : ah + (al + q[i > 0 ? i - 1 : 0]); };
    // etadot at the top interface of layer i of the chunk, K = K0 + i (0 and nl: zero)
    auto eta = [&](int i, T s) {
        const int K = K0 + i;
        return (K > 0 && K < nl) ? -s - (ps * bk[K]) * dlnpsdt : T(0);
    };
    T *WD = dlnpdt + (long)mem * nl * ng;
    if constexpr (!DYN) {
#pragma unroll
        for (int i = 0; i < LPC; i++)
            if (i < cnt) {
                const int K = K0 + 1 + i;
                const T s = above(i);
                st(WD, i, w2[i] - w1[i] * s);
                ste(i, eta(i, s));
                if (K == nl) ste(i + 1, T(0));
            }
    } else {
        cof = px = py = T(0);
#pragma unroll
        for (int c = CH - 1; c > 0; c--)
            if (c > w) {  // getpresgrad's sums over the chunks below
                cof += sh[S_COF][c][ln];
                px += sh[S_PX][c][ln];
                py += sh[S_PY][c][ln];
            }
        const T bx = cof * gpx + (px - dphx), by = cof * gpy + (py - dphy);
        T *A = gan + (long)mem * nan * ng;
        T *TT = A, *FX = A + (long)nl * ng, *FY = A + 2L * nl * ng, *KE = A + 3L * nl * ng;
        if (w == 0) A[4L * nl * ng + col] = dlnpsdt;
        T um = T(0), vm = T(0), tm = T(0);  // the level below the chunk
        if (K0 + cnt < nl) {
            um = sh[S_U0][w + 1][ln];
            vm = sh[S_V0][w + 1][ln];
            tm = sh[S_T0][w + 1][ln];
        }
        T ua = T(0), va = T(0), ta = T(0);  // the level above it
        if (w > 0) {
            ua = sh[S_U1][w - 1][ln];
            va = sh[S_V1][w - 1][ln];
            ta = sh[S_T1][w - 1][ln];
        }
        T eb = eta(cnt, bh);  // etadot at the bottom of layer i; zero at the surface, and at the top
#pragma unroll
        for (int i = LPC - 1; i >= 0; i--)
            if (i < cnt) {
                const int K = K0 + 1 + i;
                const T up = i > 0 ? u[i > 0 ? i - 1 : 0] : ua, vp = i > 0 ? v[i > 0 ? i - 1 : 0] : va;
                const T tp = i > 0 ? tv[i > 0 ? i - 1 : 0] : ta;
                const T s = above(i), ea = eta(i, s), om = w2[i] - w1[i] * s;
                if (store) {
                    st(WD, i, om);
                    ste(i, ea);
                    if (K == nl) ste(i + 1, T(0));
                }
                // getvadv for u, v, tv
                const T h = T(0.5) * recip(dp(K)), hb = h * eb, ha = h * ea;
                const T vu = hb * (um - u[i]) + ha * (u[i] - up);
                const T vv = hb * (vm - v[i]) + ha * (v[i] - vp);
                const T vt = hb * (tm - tv[i]) + ha * (tv[i] - tp);
                T vq = kappa * om * tv[i];
                if constexpr (TR) vq = vq / (T(1) + cvcp * q1[i]);
                st(TT, i, adv[i] - vt + vq);
                T fx = fx0[i] + vv - by, fy = fy0[i] - vu + bx;
                if constexpr (VC) {
                    // up-gradient vorticity flux vc |vrt| grad(vrt) / |grad(vrt)|
                    const T *VCX = vcg + (long)mem * 2 * nl * ng, *VCY = VCX + (long)nl * ng;
                    const T gx = ld(VCX, i), gy = ld(VCY, i), ag = sqrt(gx * gx + gy * gy);
                    T vcl = vcamp;
                    if (svcg) vcl = (T(1) + vfsvc[nl - K] * svcg[(long)mem * ng + col]) * vcl;
                    if (ag > T(FLT_MIN)) {
                        const T av = fabs(ld(VRT, i));
                        fx += vcl * (gx / ag) * av;
                        fy += vcl * (gy / ag) * av;
                    }
                }
                st(FX, i, fx);
                st(FY, i, fy);
                st(KE, i, T(0.5) * (u[i] * u[i] + v[i] * v[i]));
                um = u[i];
                vm = v[i];
                tm = tv[i];
                eb = ea;
            }
        // tracers (dyn_run.f90:279-291): horizontal advection with the synthesised
        // gradient and the Thuburn (1993) flux-limited vertical advection of
        // getvadv_tracers (dyn_run.f90:478-603) with layer values D_K = q at L = nl + 1 - K.
        // Half-level values need D from two layers above to two below; a chunk
        // recomputes that of its top interface.
        const T *QX = Q + (long)ntr * nl * ng, *QY = QX + (long)ntr * nl * ng;
        const T tiny = std::numeric_limits<T>::min();
        auto guard = [&](T d) { return fabs(d) < tiny ? copysign(tiny, d) : d; };
        for (int nt = 0; nt < ntr && cnt > 0; nt++) {
            const T *Qn = Q + (long)nt * nl * ng, *QXn = QX + (long)nt * nl * ng, *QYn = QY + (long)nt * nl * ng;
            T *DQ = A + (4L * nl + 1 + (long)nt * nl) * ng;
            T D[LPC + 4], gx[LPC], gy[LPC];  // D[i] = D_{K0 - 1 + i}, clamped to the column
#pragma unroll
            for (int i = 0; i < LPC + 4; i++)
                if (i < lpc + 4) D[i] = ld(Qn, i - 2);
#pragma unroll
            for (int i = 0; i < LPC; i++)
                if (i < lpc) {
                    gx[i] = ld(QXn, i);
                    gy[i] = ld(QYn, i);
                }
            // dd_K, K = K0 - 1 + i: D_{K+1} - D_K, guarded; at the top and the surface from two layers
            auto dd = [&](int i) {
                const int K = K0 - 1 + i;
                if (K <= 0) {
                    const T a = D[i + 1], mx = T(2) * a - D[i + 2];
                    return a >= T(0) ? a - fmax(T(0), mx) : a - fmin(T(0), mx);
                }
                if (K >= nl) {
                    const T a = D[i], mb = T(2) * a - D[i > 0 ? i - 1 : 0];
                    return a >= T(0) ? fmax(T(0), mb) - a : fmin(T(0), mb) - a;
                }
                return guard(D[i + 1] - D[i]);
            };
            // the value at interface K0 + i, where etadot is e
            auto half = [&](int i, T e) {
                const int K = K0 + i;
                if (K <= 0) return D[i + 2];
                if (K >= nl) return D[i + 1];
                const T a = D[i + 1], b = D[i + 2], h = T(0.5) * (b + a), dk = dd(i + 1);
                const T phi = (e > T(0) ? dd(i) : dd(i + 2)) / dk;
                const T lim = (phi + fabs(phi)) / (T(1) + fabs(phi));
                return e > T(0) ? a + lim * (h - a) : b + lim * (h - b);
            };
            T et = eta(0, ah), hp = half(0, et);
#pragma unroll
            for (int i = 0; i < LPC; i++)
                if (i < cnt) {
                    const int K = K0 + 1 + i;
                    const T eb2 = eta(i + 1, above(i + 1));
                    const T hk = half(i + 1, eb2), Dk = D[i + 2];
                    const T vadv = recip(dp(K)) * ((hk * eb2 - hp * et) + (Dk * (et - eb2)));
                    st(DQ, i, -u[i] * gx[i] - v[i] * gy[i] - vadv);
                    hp = hk;
                    et = eb2;
                }
        }
    }
}

// getomega's layer terms, evaluated identically wherever they are needed: with
// contraction off, each is one rounded product of the same operands, so the
// column total of pass 1 and the suffix sums of pass 3 add the same numbers.
template <typename T> struct OmegaTerms {
    T cg, tdb, tcb;  // V . grad ln ps, div dp_K, cg dbk_K
};
template <typename T>
__device__ __forceinline__ OmegaTerms<T> omega_terms(T u, T v, T dv, T dpx, T dpy, T dpk, T dbk) {
#pragma clang fp contract(off)
    OmegaTerms<T> o;
    o.cg = u * dpx + v * dpy;
    o.tdb = dv * dpk;
    o.tcb = o.cg * dbk;
    return o;
}
// A sum carried as an unevaluated pair hi + lo (Neumaier's compensated
// summation with the two-sum of Knuth): its error stays at eps^2 of the summed
// magnitudes, so a prefix sum of the top layers can be formed as the column
// total minus the sum of the layers below without cancelling its digits.
template <typename T> struct PairSum {
    T hi = 0, lo = 0;
    __device__ __forceinline__ void add(T t) {
#pragma clang fp contract(off)
        const T s = hi + t, bp = s - hi;
        lo += (hi - (s - bp)) + (t - bp);
        hi = s;
    }
    // this - o, rounded once
    __device__ __forceinline__ T minus(const PairSum &o) const {
#pragma clang fp contract(off)
        const T s = hi - o.hi, bp = s - hi;
        const T e = (hi - (s - bp)) + (-o.hi - bp);
        return s + (e + (lo - o.lo));
    }
};

// Whether a dynamics pass takes k_columns_serial. FP32: a getdyntend call of a member with
// 100 000 columns, which so keeps its order of sums (see there). FP64: any pass without
// tracers that has columns enough for a thread each. k_columns and this kernel in
// us a launch, FP64: 64 levels T84 (33 000 columns) 58 and 90, T126 (73 000) 128 and 142,
// two members at T95 (83 000) 148 and 142, T170 218 and 189, T254 444 and 446; 28 levels,
// where k_columns takes half the registers, two members at T84 (66 000) 44 and 50, T126 49
// and 62, eight at T62 (144 000) 86 and 98, but T170 (131 000) 91 and 73, T254 185 and 186.
// With 33 to 43 levels its 16 threads a column have three layers each and up to a third of
// them few or none: 36 levels two members at T84 77 and 67, 44 levels 85 and 84, T126 95 and
// 102. With a tracer a T126 moist step takes 1.30 and 1.41 ms: here it is advected in a pass
// of its own.
template <typename T> static bool columns_serial(long ng, int nm, int ntr, int nl, bool grids) {
    if (sizeof(T) == 4) return grids && ng >= 100000;
    return ntr == 0 && nm * ng >= (nl <= 32 ? 100000 : nl < 44 ? 50000 : 80000);
}
// The dynamics columns with one thread per column, every sum in the order of the
// reference's recursions. In FP64 (three wavefronts a SIMD) the faster kernel where the
// columns are enough, for its fewer operations: bound by them, where k_columns forms prefix
// sums over its threads besides.
// In FP32 it is the slower one (232 us at T254L64, k_columns 193) and no closer to 64
// bits. The vorticity tendency shows the rounding most, as the curl of the pressure gradient
// nearly vanishes; its error in the 2-norm here and in k_columns, rough states of 64
// levels: T84 6.69e-6 and 6.68e-6, T126 9.12e-6 and 9.01e-6, T170 1.207e-5 and 1.213e-5,
// T254 1.780e-5 and 1.778e-5; states of a Held-Suarez run T126 1.10e-6 and 1.09e-6, T254
// 9.9e-7 and 9.9e-7; the other tendencies' alike, ln ps' up to 8 % smaller in k_columns. What the FP32 rule keeps is the order
// of sums itself, by which a large getdyntend call's single coefficients differ by up to
// 3e-5 of the largest, and k_columns' passes inside advance by a few parts in 1e6 of the state.
template <typename T, bool VC>
__global__ __launch_bounds__(256, sizeof(T) == 8 ? 3 : 4) void k_columns_serial(
    const T *__restrict__ gsyn, T *__restrict__ gan, T *__restrict__ etadot, T *__restrict__ dlnpdt,
    T *__restrict__ psg_out, T *__restrict__ dlnpsdt_out, const T *__restrict__ dphisdx,
    const T *__restrict__ dphisdy, const T *__restrict__ ak_, const T *__restrict__ bk_,
    const T *__restrict__ ck_, const T *__restrict__ dbk_, const T *__restrict__ dak_, const T *__restrict__ sinlat,
    int nl, int ntr_, int nsyn, int nan, long ng, int nlon, T rd, T kappa, T cvcp, T twoom,
    const cplx<T> *__restrict__ spec, int nfs, T *__restrict__ colq, const T *__restrict__ vcg,
    const T *__restrict__ svcg, const T *__restrict__ vfsvc, T vcamp, int store) {
    const int ntr = sizeof(T) == 8 ? 0 : ntr_;  // in FP64 no pass with tracers comes here
    __shared__ T ak[MAXLEV + 1], bk[MAXLEV + 1], ck[MAXLEV], dbk[MAXLEV], dak[MAXLEV];
    for (int i = threadIdx.x; i <= nl; i += blockDim.x) {
        ak[i] = ak_[i];
        bk[i] = bk_[i];
        if (i < nl) {
            ck[i] = ck_[i];
            dbk[i] = dbk_[i];
            dak[i] = dak_[i];
        }
    }
    __syncthreads();
    const long col = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int mem = blockIdx.y;
    if (col >= ng) return;
    const T *G = gsyn + (long)mem * nsyn * ng + col;
    const T *U = G, *V = G + (long)nl * ng, *VRT = G + 2L * nl * ng, *DIV = G + 3L * nl * ng;
    const T *TV = G + 4L * nl * ng, *TX = G + 5L * nl * ng, *TY = G + 6L * nl * ng, *Q = G + 7L * nl * ng;
    const T *QX = Q + (long)ntr * nl * ng, *QY = QX + (long)ntr * nl * ng;
    const T *LNPS = G + (7L + 3L * ntr) * nl * ng;
    const T dpx = LNPS[ng], dpy = LNPS[2 * ng];
    const T c00 = spec[(long)mem * nfs + 3L * nl + (long)ntr * nl].x;
    const T ps = full_ps(c00, LNPS[0]);
    T *ET = etadot + (long)mem * (nl + 1) * ng + col;
    T *WD = dlnpdt + (long)mem * nl * ng + col;
    const T alfa1 = T(SGLF(0.69314718055994530942)), rlnp1 = T(SGLF(99999.99));
#define LV(P, L) (P)[(long)((L) - 1) * ng]
    auto pk = [&](int K) -> T { return ak[K - 1] + bk[K - 1] * ps; };
    auto dp = [&](int K) -> T { return fma(dbk[K - 1], ps, dak[K - 1]); };  // pk(K + 1) - pk(K), one rounding
    // omega / p of layer K (getomega's workb, workc) from the sums db, cb over
    // the layers above it
    auto omega_p = [&](int K, T dba, T cba, const OmegaTerms<T> &o, T dv, T dpk, T rdp, T rlnp, T alfa) {
        T workb, workc;
        if (K == 1) {
            workb = alfa * (dv * dpk + ps * (o.cg * dbk[0]) * dbk[0]);
            workc = ps * o.cg * dbk[0];
        } else {
            workb = rlnp * (dba + ps * cba) + alfa * (dv * dpk + ps * o.cg * dbk[K - 1]);
            workc = ps * o.cg * (dbk[K - 1] + ck[K - 1] * rlnp * rdp);
        }
        return (workc - workb) * rdp;
    };
    // pass 1 (top -> bottom): getomega's sums db, cb and their column totals
    T db = 0, cb = 0;
    PairSum<T> sdb, scb;
    // FP32 always stores the grids (its calls hand them out), without a branch: one there
    // changes how the interface pressures are fused, which the vorticity tendency shows
    const bool st_om = sizeof(T) == 4 || store, st_et = st_om || ntr > 0;  // the tracers read etadot back
    if (st_et) ET[(long)nl * ng] = T(0);
    constexpr int P1G = 4;  // levels whose loads are issued together
    for (int K0 = 1; K0 <= nl; K0 += P1G) {
        T gu[P1G], gv[P1G], gd[P1G];
#pragma unroll
        for (int i = 0; i < P1G; i++) {
            const int Lc = max(nl + 1 - (K0 + i), 1);  // clamped: past the bottom level nothing is used
            gu[i] = LV(U, Lc);
            gv[i] = LV(V, Lc);
            gd[i] = LV(DIV, Lc);
        }
#pragma unroll
        for (int i = 0; i < P1G; i++) {
            const int K = K0 + i;
            if (K > nl) break;
            const OmegaTerms<T> o = omega_terms(gu[i], gv[i], gd[i], dpx, dpy, dp(K), dbk[K - 1]);
            db += o.tdb;
            cb += o.tcb;
            sdb.add(o.tdb);
            scb.add(o.tcb);
        }
    }
    const T dlnpsdt = -db / ps - cb;
    psg_out[(long)mem * ng + col] = ps;
    dlnpsdt_out[(long)mem * ng + col] = dlnpsdt;
    if (ntr > 0 && colq) {
        // column tracer mass of the dry-mass diagnostic (dyn_run.f90:138-145)
        T s = 0;
        for (int K = 1; K <= nl; K++) {
            T dpk = dp(K), qs = 0;
            for (int nt = 0; nt < ntr; nt++) qs += Q[((long)nt * nl + (nl - K)) * ng];
            s += dpk * qs;
        }
        colq[(long)mem * ng + col] = s;
    }
    T *A = gan + (long)mem * nan * ng + col;
    T *TT = A, *FX = A + (long)nl * ng, *FY = A + 2L * nl * ng, *KE = A + 3L * nl * ng;
    A[4L * nl * ng] = dlnpsdt;
    const T f = twoom * sinlat[col / nlon];
    const T dphx = dphisdx[(long)mem * ng + col], dphy = dphisdy[(long)mem * ng + col];
    // pass 3: bottom -> top (K = nl..1): getpresgrad accumulations, getvadv, assembly.
    // u, v, tv of the levels below / at / above L slide through registers. The
    // getomega sums over the layers above K are the column totals less the sums
    // over K..nl (rdb, rcb), from which omega / p of the layer and etadot at its
    // top interface follow; etadot at its bottom interface is the previous top.
    T cofb_acc = 0, px3u = 0, px3v = 0;
    T um = 0, vm = 0, tm = 0;                          // level L - 1
    T u = LV(U, 1), v = LV(V, 1), tv = LV(TV, 1);      // level L
    T eb = T(0);                                       // etadot at the layer's bottom interface
    T rpb = recip(pk(nl + 1));                         // and the reciprocal of the pressure there
    PairSum<T> rdb, rcb;
    constexpr int P3G = 2;  // levels whose loads are issued together
    for (int K0 = nl; K0 >= 1; K0 -= P3G) {
        T gup[P3G], gvp[P3G], gtp[P3G], gtx[P3G], gty[P3G], gdv[P3G], gvr[P3G];
#pragma unroll
        for (int i = 0; i < P3G; i++) {
            const int Lc = min(nl + 1 - (K0 - i), nl), Lp = min(Lc + 1, nl);  // clamped to the top level
            gup[i] = LV(U, Lp);
            gvp[i] = LV(V, Lp);
            gtp[i] = LV(TV, Lp);
            gtx[i] = LV(TX, Lc);
            gty[i] = LV(TY, Lc);
            gdv[i] = LV(DIV, Lc);
            gvr[i] = LV(VRT, Lc);
        }
#pragma unroll
        for (int i = 0; i < P3G; i++) {
            const int K = K0 - i;
            if (K < 1) break;
            int L = nl + 1 - K;
            T up = 0, vp = 0, tp = 0;                      // level L + 1
            if (L < nl) {
                up = gup[i];
                vp = gvp[i];
                tp = gtp[i];
            }
            T p1 = pk(K), p2 = pk(K + 1), dpk = dp(K), rdp = recip(dpk);
            const T dv = gdv[i];
            const OmegaTerms<T> o = omega_terms(u, v, dv, dpx, dpy, dpk, dbk[K - 1]);
            rdb.add(o.tdb);
            rcb.add(o.tcb);
            const T dba = sdb.minus(rdb), cba = scb.minus(rcb);  // sums over the layers above K
            T ea = T(0);                                   // etadot at the top interface K - 1
            if (K > 1) ea = (-(ps * cba) - dba) - (ps * bk[K - 1]) * dlnpsdt;
            if (st_et) ET[(long)(K - 1) * ng] = ea;
            T rlnp = rlnp1, alfa = alfa1, cofa, dbp;
            // FP64, bound by its operations, takes the reciprocal from the layer below
            const T rp1 = recip(p1), rp2 = sizeof(T) == 4 ? recip(p2) : rpb;
            rpb = rp1;
            if (K == 1) {
                cofa = -rdp * (bk[K] * p1 * rp2 - bk[K - 1] + rlnp * (bk[K - 1] - p1 * dbk[K - 1] * rdp));
                dbp = bk[K] * rp2 - bk[K - 1] * rp1;
            } else {
                layer_log(p1, p2, dpk, rp1, rdp, rlnp, alfa);
                layer_rest(p1, dpk, bk[K - 1], bk[K], ck[K - 1], dbk[K - 1], rp1, rp2, rdp, rlnp, alfa, cofa, dbp);
            }
            T cofb0 = (K == 1) ? -rdp * (alfa * dbk[0]) : -rdp * (bk[K - 1] * rlnp + alfa * dbk[K - 1]);
            T tx = gtx[i], ty = gty[i];
            T prsgx = cofb0 * rd * tv * ps * dpx - dphx + cofb_acc * ps * dpx + px3u - rd * alfa * tx -
                      cofa * rd * tv * ps * dpx;
            T prsgy = cofb0 * rd * tv * ps * dpy - dphy + cofb_acc * ps * dpy + px3v - rd * alfa * ty -
                      cofa * rd * tv * ps * dpy;
            // getvadv for u, v, tv at level L
            T vu, vv, vt;
            T h = T(0.5) * rdp;
            if (L == nl) {  // top layer: etadot at interface 1 (its bottom)
                vu = h * eb * (um - u);
                vv = h * eb * (vm - v);
                vt = h * eb * (tm - tv);
            } else if (L == 1) {  // bottom layer: etadot at interface nl - 1 (its top)
                vu = h * ea * (u - up);
                vv = h * ea * (v - vp);
                vt = h * ea * (tv - tp);
            } else {
                vu = h * (eb * (um - u) + ea * (u - up));
                vv = h * (eb * (vm - v) + ea * (v - vp));
                vt = h * (eb * (tm - tv) + ea * (tv - tp));
            }
            const T om = omega_p(K, dba, cba, o, dv, dpk, rdp, rlnp, alfa);
            if (st_om) LV(WD, L) = om;
            T vq = kappa * om * tv;
            if (ntr > 0) vq = vq / (T(1) + cvcp * LV(Q, L));
            vv -= prsgy;
            vu -= prsgx;
            T z = gvr[i] + f;
            LV(TT, L) = -u * tx - v * ty - vt + vq;
            T fx = u * z + vv, fy = v * z - vu;
            if constexpr (VC) {
                // up-gradient vorticity flux vc |vrt| grad(vrt) / |grad(vrt)|
                const T *VCX = vcg + (long)mem * 2 * nl * ng + col, *VCY = VCX + (long)nl * ng;
                const T gx = LV(VCX, L), gy = LV(VCY, L), ag = sqrt(gx * gx + gy * gy);
                T vcl = vcamp;
                if (svcg) vcl = (T(1) + vfsvc[L - 1] * svcg[(long)mem * ng + col]) * vcl;
                if (ag > T(FLT_MIN)) {
                    fx += vcl * (gx / ag) * fabs(gvr[i]);
                    fy += vcl * (gy / ag) * fabs(gvr[i]);
                }
            }
            LV(FX, L) = fx;
            LV(FY, L) = fy;
            LV(KE, L) = T(0.5) * (u * u + v * v);
            // accumulations for the layer above (getpresgrad cofb and px3 recursions)
            cofb_acc -= rd * dbp * tv;
            px3u -= rd * rlnp * tx;
            px3v -= rd * rlnp * ty;
            um = u;
            vm = v;
            tm = tv;
            u = up;
            v = vp;
            tv = tp;
            eb = ea;
        }
    }

    // pass 4: tracers (dyn_run.f90:279-291): horizontal advection with the
    // synthesised gradient and the Thuburn (1993) flux-limited vertical
    // advection of getvadv_tracers (dyn_run.f90:478-603), top -> bottom with a
    // sliding window of layer values D_K, K = 1..nl (D_K = q at L = nl+1-K).
    const T tiny = std::numeric_limits<T>::min();
    auto guard = [&](T d) { return fabs(d) < tiny ? copysign(tiny, d) : d; };
    for (int nt = 0; nt < ntr; nt++) {
        const T *Qn = Q + (long)nt * nl * ng, *QXn = QX + (long)nt * nl * ng, *QYn = QY + (long)nt * nl * ng;
        T *DQ = A + (4L * nl + 1 + (long)nt * nl) * ng;
        T Dk = LV(Qn, nl), Dk1 = LV(Qn, nl - 1);
        T mx = T(2) * Dk - Dk1;
        T ddprev = (Dk >= T(0)) ? Dk - fmax(T(0), mx) : Dk - fmin(T(0), mx);  // dd_0 (unguarded)
        T ddk = guard(Dk1 - Dk);                                                    // dd_1
        T hprev = Dk;                                                                // half_0
        for (int K = 1; K <= nl; K++) {
            const T etop = ET[(long)(K - 1) * ng], ebot = ET[(long)K * ng];
            const T dpk = dp(K);
            T hk, Dk2 = T(0), ddn = T(0);
            if (K <= nl - 1) {
                if (K + 1 <= nl - 1) {
                    Dk2 = LV(Qn, nl - 1 - K);  // D_{K+2}
                    ddn = guard(Dk2 - Dk1);
                } else {  // dd_nl from the two lowest layers (unguarded)
                    T mb = T(2) * Dk1 - Dk;
                    ddn = (Dk1 >= T(0)) ? fmax(T(0), mb) - Dk1 : fmin(T(0), mb) - Dk1;
                }
                T h = T(0.5) * (Dk1 + Dk);
                if (ebot > T(0)) {
                    T phi = ddprev / ddk;
                    hk = Dk + (phi + fabs(phi)) / (T(1) + fabs(phi)) * (h - Dk);
                } else {
                    T phi = ddn / ddk;
                    hk = Dk1 + (phi + fabs(phi)) / (T(1) + fabs(phi)) * (h - Dk1);
                }
            } else {
                hk = Dk;  // half_nl = lowest layer value
            }
            T vadv = recip(dpk) * ((hk * ebot - hprev * etop) + (Dk * (etop - ebot)));
            const int L = nl + 1 - K;
            LV(DQ, L) = -LV(U, L) * LV(QXn, L) - LV(V, L) * LV(QYn, L) - vadv;
            hprev = hk;
            ddprev = ddk;
            ddk = ddn;
            Dk = Dk1;
            Dk1 = Dk2;
        }
    }
#undef LV
}

// Phillips layer pressure ((p2^(k+1) - p1^(k+1)) / ((k+1)(p2 - p1)))^(1/k) of
// pressure_data.f90:87-88. In FP32 the difference of powers cancels (a layer is
// a few per cent thick), losing 3e-5 relative; float therefore evaluates the
// same quantity as sqrt(p1 p2) exp(S(y)), y = ln(p2 / p1), from the series
// ln((e^z - 1) / z) = z/2 + sum_j B_2j z^2j / (2j (2j)!) taken at z = (k+1) y and
// z = y (B_2j Bernoulli numbers; five terms, truncation 3e-9 at y = 1), which
// keeps it to a few ulp. The top layer (p1 = 0) has no cancellation.
// coefficients d1..d5 of the series S(y) above; they depend on kappa only
template <typename T> struct PrsSeries {
    T d1, d2, d3, d4, d5;
};
template <typename T> __device__ inline PrsSeries<T> prs_series(T kappa) {
    const T a = kappa + T(1), a2 = a * a, a4 = a2 * a2, a6 = a4 * a2, a8 = a4 * a4, a10 = a8 * a2;
    return PrsSeries<T>{(a2 - T(1)) / (T(24) * kappa), -(a4 - T(1)) / (T(2880) * kappa),
                        (a6 - T(1)) / (T(181440) * kappa), -(a8 - T(1)) / (T(9676800) * kappa),
                        (a10 - T(1)) / (T(479001600) * kappa)};
}
// FP32 natural logarithm and exponential on the hardware base-2 instructions
// (v_log_f32 / v_exp_f32, about 1 ulp for the normal positive arguments here)
__device__ __forceinline__ float ln_hw(float x) { return __builtin_amdgcn_logf(x) * 0.693147180559945309f; }
__device__ __forceinline__ float exp_hw(float x) { return __builtin_amdgcn_exp2f(x * 1.44269504088896341f); }

template <typename T> __device__ inline T phillips_prs(T p1, T p2, T kappa, const PrsSeries<T> &c) {
    if constexpr (sizeof(T) == 4) {
        if (p1 > T(0)) {
            // y only enters through S = O(y^2 / 12): the rounding of 1 + x in the
            // hardware logarithm leaves S, and the pressure, exact to far below an ulp
            const T y = ln_hw(T(1) + (p2 - p1) * recip(p1));
            if (y <= T(1)) {
                const T y2 = y * y;
                const T S = y2 * (c.d1 + y2 * (c.d2 + y2 * (c.d3 + y2 * (c.d4 + y2 * c.d5))));
                return sqrt(p1 * p2) * exp_hw(S);
            }
        }
    }
    return pow((pow(p2, kappa) * p2 - pow(p1, kappa) * p1) / ((kappa + T(1)) * (p2 - p1)), T(1) / kappa);
}
template <typename T> __device__ inline T phillips_prs(T p1, T p2, T kappa) {
    return phillips_prs(p1, p2, kappa, prs_series(kappa));
}

// Held-Suarez forcing fields in the analysis grid buffer: every member's
// temperature forcing of levels 0..nl-1 (level 0 the lowest) with its
// mass-fixer field as level nl, then the vorticity and divergence forcing
// level-major from the lowest level (level k, member, vrt / div), so that the
// levels where the drag acts form a prefix of the buffer.
enum { HS_T = 0, HS_VRT = 1, HS_DIV = 2 };
__host__ __device__ inline int hs_field(int nl, int nm, int mem, int kind, int k) {
    return kind == HS_T ? mem * (nl + 1) + k : nm * (nl + 1) + 2 * (k * nm + mem) + (kind - HS_VRT);
}

// The levels on which the Held-Suarez drag can act, for the lean pass.
// phy_run_hs.f90:52-58 sets the drag profile max(0, (p_k / ps - sigbot) /
// (1 - sigbot)): where p_k / ps stays below sigbot in every column, a level's
// vorticity and divergence forcing -0 * vrtg is zero on the whole grid, and so
// is its transform. The layer pressure p_k lies below the layer's lower
// interface ak + bk ps, and (ak + bk ps) / ps = ak / ps + bk is monotone in ps,
// so over all columns it is largest at the least or the greatest ps (1 / ps =
// rmin, rmax). A level where it stays below 0.999 sigbot at both (a margin far
// above the rounding of p_k) has no drag. The lean pass takes the levels up
// to the highest other one (nact, which k_area turns into the counts the
// pass's kernels read).
template <typename T>
__device__ inline bool hs_level_drags(int k, double rmin, double rmax, const T *__restrict__ ak,
                                      const T *__restrict__ bk, int nl) {
    const double thr = 0.999 * SGLF(0.7);
    const double a = (double)ak[nl - k], b = (double)bk[nl - k];  // grid level k: interfaces nl - k - 1, nl - k
    return a * rmin + b > thr || a * rmax + b > thr;
}

// Held-Suarez forcing on the post-dynamics grid fields (phy_run_hs.f90:42-77)
// and the dry-mass-fixer field log(ps * pcorr) (dyn_run.f90:626-631), into the
// forcing fields of hs_field. With cnt (the lean pass) the vorticity and
// divergence forcing is formed on the levels below cnt[2] only: hs_level_drags
// found the drag zero on every level above them, and their vorticity and
// divergence were not synthesised.
constexpr int HS_LCH = 8;  // level chunks of the Held-Suarez kernel (levels are independent)

template <typename T>
__global__ __launch_bounds__(256) void k_hs_columns(const T *__restrict__ gsyn, const T *__restrict__ psg,
                                                    T *__restrict__ gan, const T *__restrict__ ak_,
                                                    const T *__restrict__ bk_, const T *__restrict__ sinlat,
                                                    const double *__restrict__ pdryini,
                                                    const double *__restrict__ pmean, int nl, int ntr, int nsyn,
                                                    int nm, long ng, int nlon, T kappa, int massfix,
                                                    const int *__restrict__ cnt) {
    __shared__ T ak[MAXLEV + 1], bk[MAXLEV + 1];
    for (int i = threadIdx.x; i <= nl; i += blockDim.x) {
        ak[i] = ak_[i];
        bk[i] = bk_[i];
    }
    __syncthreads();
    // the levels are independent: blockIdx.y = member * HS_LCH + level chunk
    const long col = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int mem = blockIdx.y / HS_LCH, ch = blockIdx.y - mem * HS_LCH;
    const int CS = (nl + HS_LCH - 1) / HS_LCH, L0 = ch * CS + 1, L1 = min(nl, (ch + 1) * CS);
    if (col >= ng) return;
    const int nact = cnt ? cnt[2] : nl;
    const T *G = gsyn + (long)mem * nsyn * ng + col;
    const T *VRT = G + 2L * nl * ng, *DIV = G + 3L * nl * ng, *TV = G + 4L * nl * ng;
    T *AT = gan + (long)hs_field(nl, nm, mem, HS_T, 0) * ng + col;
    const T ps = psg[(long)mem * ng + col];
    const T sl = sinlat[col / nlon];
    const T cl2 = T(1) - sl * sl;
    const T sigbot = T(SGLF(0.7)), delthz = T(10), tempstrat = T(200);
    const T kdrag = T(SGLF(1.f / 86400.f)), krada = T(SGLF(1.f / (40.f * 86400.f)));
    const T kradb = T(SGLF(1.f / (4.f * 86400.f))), p0 = T(1.e5), deltmp = T(60);
    const T expo = T(SGLF(2.f / 7.f));
    // per column: the layer-pressure series, 1 / ps, 1 / (1 - sigbot)
    const PrsSeries<T> prc = prs_series(kappa);
    const T rps = recip(ps), rsb = T(1) / (T(1) - sigbot);
    // the chunk's grid values first, all loads in flight together (levels
    // clamped into the chunk; the vorticity and divergence where the chunk has
    // a level with drag)
    constexpr int CSM = (MAXLEV + HS_LCH - 1) / HS_LCH;
    const bool drag = L0 - 1 < nact;
    T tv[CSM], vr[CSM], dv[CSM];
#pragma unroll
    for (int i = 0; i < CSM; i++) {
        const long o = (long)(min(L0 + i, L1) - 1) * ng;
        tv[i] = TV[o];
        vr[i] = dv[i] = T(0);
        if (drag) {
            vr[i] = VRT[o];
            dv[i] = DIV[o];
        }
    }
#pragma unroll
    for (int i = 0; i < CSM; i++) {
        const int L = L0 + i;
        if (L > L1) break;
        int K = nl + 1 - L;
        T p1 = ak[K - 1] + bk[K - 1] * ps, p2 = ak[K] + bk[K] * ps;
        T prs = phillips_prs(p1, p2, kappa, prc);
        T blprof = prs * rps;
        // (prs / p0)^(2/7) as exp(2/7 ln(prs / p0)), sharing the logarithm of the
        // temperature profile (in FP32 the base-2 hardware instructions)
        T lr, pw;
        if constexpr (sizeof(T) == 4) {
            const float l2 = __builtin_amdgcn_logf(prs / p0);  // log2, on the hardware
            lr = l2 * 0.693147180559945309f;
            pw = __builtin_amdgcn_exp2f(expo * l2);
        } else {
            lr = log(prs / p0);
            pw = exp(expo * lr);
        }
        T teq = pw * (T(315) - deltmp * sl * sl - delthz * lr * cl2);
        blprof = (blprof - sigbot) * rsb;
        if (blprof < T(0)) blprof = T(0);
        if (teq < tempstrat) teq = tempstrat;
        long o = (long)(L - 1) * ng;
        AT[o] = (krada + (kradb - krada) * blprof * cl2 * cl2) * (teq - tv[i]);
        if (L - 1 < nact) {
            T *AV = gan + (long)hs_field(nl, nm, mem, HS_VRT, L - 1) * ng + col;  // divergence follows it
            AV[0] = -(blprof * kdrag) * vr[i];
            AV[ng] = -(blprof * kdrag) * dv[i];
        }
    }
    if (massfix && ch == 0) {
        // log(ps * pcorr) - c0 = ln ps' + log(pcorr)
        const T *LNPS = G + (7L + 3L * ntr) * nl * ng;
        AT[(long)nl * ng] = LNPS[0] + (T)log(pdryini[mem] / pmean[mem]);
    }
}

// Area-weighted global sums per member in FP64 (areawts sum to 1, so these are
// global means): S_a of field a (ps) and, when b is given, S_b of field b (the
// column tracer mass, or pwat); pdryini = S_a - S_b where it is still 0
// (dyn_run.f90:135-149). PS_BLOCKS workgroups per member write partial sums, and
// the last of them to arrive adds these up in the order of the workgroups, so the
// result does not depend on which one it is. part holds four values per (member,
// workgroup): S_a, S_b and the least and the greatest a of its columns; done
// counts the workgroups that have arrived, per member, and after those the
// members, and is left at zero.
// With PSG (the lean pass) a is formed here from ln ps, as the column kernel
// forms it: ps = exp(mean + ln ps'), the mean from the spectral state in FP64; and
// the last member's last workgroup takes the range of ps over all members, finds
// the levels with drag from it (hs_level_drags) and writes the lean pass's counts
// (cnt[0..4], as DycoreBuffers::hsdyn describes them).
// Bound by latency: the lean pass's ps, sums, range and counts take 8.8 us at T42
// FP64 and 12.8 us at T254 FP32 as one launch (13.5 and 17 us as three, without
// the gaps between them); the dynamics' call, once the dry mass is set, ends at once.
constexpr int PS_BLOCKS = 128;
static_assert(MAXLEV <= PS_BLOCKS, "k_area tests one level per thread");

template <typename T, bool PSG>
__global__ __launch_bounds__(256) void k_area(T *__restrict__ a, const T *__restrict__ b,
                                              const double *__restrict__ areaw, double *__restrict__ part,
                                              unsigned *__restrict__ done, long ng, int nlon,
                                              double *__restrict__ out_a, double *__restrict__ out_b,
                                              double *__restrict__ pdryini, const T *__restrict__ ak,
                                              const T *__restrict__ bk, int nl, int *__restrict__ cnt,
                                              const T *__restrict__ gsyn, const cplx<T> *__restrict__ spec, int ntr,
                                              int nsyn, int nfs) {
    const int mem = blockIdx.y, nm = gridDim.y, tid = threadIdx.x;
    // nothing to find out about a member whose dry mass is set
    if (!PSG && !out_a && !out_b && (!pdryini || pdryini[mem] != 0.0)) return;
    T *pa = a + (long)mem * ng;
    const T *pb = b ? b + (long)mem * ng : nullptr;
    const T *in = PSG ? gsyn + (long)mem * nsyn * ng + (7L + 3L * ntr) * nl * ng : pa;
    const T c00 = PSG ? spec[(long)mem * nfs + 3L * nl + (long)ntr * nl].x : T(0);
    double sa = 0.0, sb = 0.0, lo = INFINITY, hi = -INFINITY;
    constexpr int AB = 4;  // columns whose loads are in flight together
    const long step = (long)PS_BLOCKS * 256;
    for (long i0 = (long)blockIdx.x * 256 + tid; i0 < ng; i0 += AB * step) {
        T x[AB], y[AB];
        double w[AB];
#pragma unroll
        for (int u = 0; u < AB; u++) {
            const long i = min(i0 + u * step, ng - 1);
            x[u] = in[i];
            y[u] = pb ? pb[i] : T(0);
            w[u] = areaw[(unsigned)i / (unsigned)nlon];  // a member has less than 2^31 columns
        }
#pragma unroll
        for (int u = 0; u < AB; u++) {
            const long i = i0 + u * step;
            if (i >= ng) break;
            if constexpr (PSG) pa[i] = x[u] = full_ps(c00, x[u]);
            const double v = (double)x[u];
            sa += w[u] * v;
            lo = fmin(lo, v);
            hi = fmax(hi, v);
            if (pb) sb += w[u] * (double)y[u];
        }
    }
    __shared__ double ra[256], rb[256], rl[256], rh[256];
    __shared__ int last;
    auto reduce = [&](int n) {
        for (int w = n / 2; w > 0; w >>= 1) {
            __syncthreads();
            if (tid < w) {
                ra[tid] += ra[tid + w];
                rb[tid] += rb[tid + w];
                rl[tid] = fmin(rl[tid], rl[tid + w]);
                rh[tid] = fmax(rh[tid], rh[tid + w]);
            }
        }
        __syncthreads();
    };
    // counts this workgroup in (thread 0) and says whether it was the n-th. Thread 0 has
    // stored the workgroup's part with device-scope stores and waits for them here, and
    // they are read with device-scope loads. That orders them by what gfx950 does (other
    // chips are refused when a context is made) and not by the memory model, for which the
    // count would have to release and acquire: here such a store is written through to
    // where every XCD's device-scope loads read, and vmcnt counts it until it is there. A
    // release would write back the L2 of the XCD for each workgroup (16 members at T126:
    // 60 us)
    auto arrive = [&](unsigned *at, int n) {
        if (tid == 0) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            last = __hip_atomic_fetch_add(at, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)n - 1u;
            asm volatile("" ::: "memory");
            if (last) __hip_atomic_store(at, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        return last != 0;
    };
    auto get = [&](long i) { return __hip_atomic_load(part + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
    ra[tid] = sa;
    rb[tid] = sb;
    rl[tid] = lo;
    rh[tid] = hi;
    reduce(256);
    if (tid == 0) {
        double *q = part + 4 * (mem * PS_BLOCKS + blockIdx.x);
        const double r[4] = {ra[0], rb[0], rl[0], rh[0]};
#pragma unroll
        for (int u = 0; u < 4; u++) __hip_atomic_store(q + u, r[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (!arrive(done + mem, PS_BLOCKS)) return;
    if (tid < PS_BLOCKS) {
        ra[tid] = get(4 * (mem * PS_BLOCKS + tid));
        rb[tid] = get(4 * (mem * PS_BLOCKS + tid) + 1);
    }
    reduce(PS_BLOCKS);
    if (tid == 0) {
        if (out_a) out_a[mem] = ra[0];
        if (out_b) out_b[mem] = rb[0];
        if (pdryini && pdryini[mem] == 0.0) pdryini[mem] = ra[0] - rb[0];
    }
    if constexpr (PSG) {
        __syncthreads();  // last, ra and rb are read
        if (!arrive(done + nm, nm)) return;
        lo = INFINITY;
        hi = -INFINITY;
        for (int i = tid; i < nm * PS_BLOCKS; i += 256) {
            lo = fmin(lo, get(4 * i + 2));
            hi = fmax(hi, get(4 * i + 3));
        }
        rl[tid] = lo;
        rh[tid] = hi;
        reduce(256);
        // one level per thread; every level for a state without a finite positive ps
        const double pmin = rl[0], pmax = rh[0];
        const bool ok = pmin > 0.0 && pmax < INFINITY;
        __shared__ int top;
        if (tid == 0) top = 0;
        __syncthreads();
        if (tid < nl && (!ok || hs_level_drags(tid, 1.0 / pmin, 1.0 / pmax, ak, bk, nl))) atomicMax(&top, tid + 1);
        __syncthreads();
        if (tid == 0) {
            const int nact = top, took = cnt[4], next = min(nl, nact + 1);
            cnt[0] = nact > took ? 2 * nm * nact : 0;
            cnt[1] = nm * (nl + 1) + 2 * nm * nact;
            cnt[2] = nact;
            cnt[3] = nm * (nl + 1) + 2 * nm * next;
            cnt[4] = next;
        }
    }
}

// Simple moist physics on the post-dynamics grid (phy_run_simple.f90:50-107
// around simple_physics_v5_1.f90), column arithmetic in FP64 as the reference's
// r8 routine. The column runs top -> bottom (c = 1 model top .. nl lowest level;
// grid level L = nl + 1 - c): large-scale condensation (265-292) and the surface
// fluxes (344-366) level by level, then the upward (bottom -> top) elimination
// and the downward back-substitution (375-447) of the implicit boundary layer.
// Output per member (nsp fields): dT(Tv), du, dv, dq (nlev each; changes over the
// step, the 1/dt is applied in the analysis) and the mass-fixer slot.
struct SimpleCfg {
    double dt, fv, qmin, grav;
    int sst_mode, turbflux;
};

// column selection of the column kernels: every column, or (judge and data
// sampling) columns i * stride + off with off drawn from the counter RNG by a
// device step counter; gate: when set and 0, the launch does nothing (the
// plain-physics fallback of the learned physics)
struct ColSel {
    int stride;
    const unsigned long long *ctr;
    const int *gate;
};

__device__ inline long sel_col(const ColSel &cs, long i, long ng) {
    if (cs.stride <= 0) return i < ng ? i : -1;
    const long nsel = ng / cs.stride;
    if (i >= nsel) return -1;
    const long off = (long)(rng_mix(0x4A554447ULL, cs.ctr ? cs.ctr[0] : 0ULL, 0) % (uint64_t)cs.stride);
    return i * cs.stride + off;
}

__device__ __forceinline__ double simple_sst(int mode, double lat) {
    if (mode == 1) {
        // simple_physics_v5_1.f90:231-239 (moist baroclinic wave)
        const double pi = 3.14159265358979323846;
        const double rair = 287.0, a = 6371220.0, om = 7.29212e-5, zvir = (461.5 / 287.0) - 1.0;
        const double T00 = 288.0, u0 = 35.0, latw = 2.0 * pi / 9.0, eta0 = 0.252;
        const double etav = (1.0 - eta0) * 0.5 * pi, q0 = (double)0.021f;
        const double s = sin(lat), c = cos(lat);
        const double num = T00 + pi * u0 / rair * 1.5 * sin(etav) * pow(cos(etav), 0.5) *
                                     ((-2.0 * pow(s, 6.0) * (c * c + 1.0 / 3.0) + 10.0 / 63.0) * u0 * pow(cos(etav), 1.5) +
                                      (8.0 / 5.0 * c * c * c * (s * s + 2.0 / 3.0) - pi / 4.0) * a * om * 0.5);
        return num / (1.0 + zvir * q0 * exp(-pow(lat / latw, 4.0)));
    }
    if (mode == 2) {
        const double s = sin(lat);
        return 302.15 - 30.0 * s * s;  // build-defined latitude falloff
    }
    return 302.15;
}

// Simple physics, SP_C columns a workgroup: everything that belongs to a level
// (layer pressure, condensation, Exner factors, diffusivities, the changes at the
// end) over SP_C x 16 threads, up to four levels each, and the two tridiagonal
// sweeps of the boundary layer over one wavefront, a lane for each of u, v, T and
// q of a column. The profiles stay in LDS in FP64 (49 KB: three workgroups a CU);
// one thread per column, with the sweeps' coefficients through memory, ran
// 1100 long FP64 wavefronts at T126. Bound by FP64 arithmetic (the powers and
// exponentials) and the sweeps' chain of divisions: FP32, T126 64 levels, 150 us
// a step (one thread per column 370; with 57 KB, two workgroups a CU, 194).
constexpr int SP_C = 16, SP_L = MAXLEV / 16;
template <typename T>
__global__ __launch_bounds__(256) void k_simple_columns(
    const T *__restrict__ gsyn, const T *__restrict__ psg, T *__restrict__ gan, T *__restrict__ pwat_out,
    T *__restrict__ precip_out, const T *__restrict__ ak_, const T *__restrict__ bk_, const double *__restrict__ latd,
    int nl, int ntr, int nsyn, int nsp, long ng, int nlon, T kappa, SimpleCfg sc, ColSel cs) {
    if (cs.gate && cs.gate[0] == 0) return;
    __shared__ T ak[MAXLEV + 1], bk[MAXLEV + 1];
    // profiles [position c - 1, top -> bottom][column]: T (then T / Exner), q, u, v; Y, then
    // the momentum sweep's CE; layer pressure, then 1 / dp, then the heat sweep's CE
    __shared__ double st[MAXLEV][SP_C], sq[MAXLEV][SP_C], su[MAXLEV][SP_C], sv[MAXLEV][SP_C];
    __shared__ double sy[MAXLEV][SP_C], srp[MAXLEV][SP_C], skm[SP_C], ske[SP_C];
    const int tid = threadIdx.x, cl = tid % SP_C, lg = tid / SP_C;
    for (int i = tid; i <= nl; i += 256) {
        ak[i] = ak_[i];
        bk[i] = bk_[i];
    }
    __syncthreads();
    const long col_ = sel_col(cs, (long)xcd_tile(blockIdx.x, gridDim.x) * SP_C + cl, ng);
    const bool valid = col_ >= 0;
    const long col = valid ? col_ : 0;  // a column past the last repeats the first and stores nothing
    const int mem = blockIdx.y;
    // simple_physics_v5_1.f90:175-222
    const double gravit = 9.80616, rair = 287.0, cpair = 1.0045e3, latvap = 2.5e6, rh2o = 461.5;
    const double epsilo = rair / rh2o, zvir = (rh2o / rair) - 1.0, Csfc = 0.0011, T0 = 273.16;
    const double e0 = 610.78, rhow = 1000.0, Cd0 = 0.0007, Cd1 = 0.000065, Cm = 0.002, v20 = 20.0;
    const double p0 = 100000.0, pbltop = 85000.0, pblconst = 10000.0, rk = rair / cpair;
    const double dt = sc.dt;
    const T *G = gsyn + (long)mem * nsyn * ng + col;
    const T *U = G, *V = G + (long)nl * ng, *TV = G + 4L * nl * ng, *Q = G + 7L * nl * ng;
    T *A = gan + (long)mem * nsp * ng + col;
    T *DT = A, *DU = A + (long)nl * ng, *DV = A + 2L * nl * ng, *DQ = A + 3L * nl * ng;
    const T ps = psg[(long)mem * ng + col];
    const T fvT = (T)sc.fv, qminT = (T)sc.qmin;
    // column positions c = 1..nl top -> bottom; this thread's are lg + 1 + 16 i
    auto lvl = [&](int c) { return (long)(nl - c) * ng; };
    auto pint = [&](int c) { return (double)(ak[c - 1] + bk[c - 1] * ps); };
    T tv0[SP_L], q0[SP_L], u0[SP_L], v0[SP_L];
#pragma unroll
    for (int i = 0; i < SP_L; i++) {
        const long o = lvl(min(lg + 1 + 16 * i, nl));
        tv0[i] = TV[o];
        q0[i] = Q[o];
        u0[i] = U[o];
        v0[i] = V[o];
    }
    double precl = 0.0, pw = 0.0, ex[SP_L];
#pragma unroll
    for (int i = 0; i < SP_L; i++) {
        const int c = lg + 1 + 16 * i;
        if (c > nl) break;
        // Phillips layer pressure of pressure_data.f90:87-88 in the grid precision
        const double pm = (double)phillips_prs(ak[c - 1] + bk[c - 1] * ps, ak[c] + bk[c] * ps, kappa);
        // T = Tv / (1 + fv max(qmin, q)) (phy_run_simple.f90:56)
        const double tin = (double)(tv0[i] / (T(1) + fvT * fmax(qminT, q0[i])));
        double t = tin, q = (double)q0[i], u = (double)u0[i], v = (double)v0[i];
        // large-scale condensation
        const double qsat = epsilo * e0 / pm * exp(-latvap / rh2o * ((1.0 / t) - 1.0 / T0));
        if (q > qsat) {
            const double tmp = 1.0 / dt * (q - qsat) / (1.0 + (latvap / cpair) * (epsilo * latvap * qsat / (rair * (t * t))));
            t = t + (latvap / cpair * tmp) * dt;
            q = q + (-tmp) * dt;
            precl = precl + tmp * (pint(c + 1) - pint(c)) / (gravit * rhow);
        }
        if (sc.turbflux && c == nl) {
            // za from the lowest level before any update (225-229); drag and eddy
            // diffusivities (300-335); surface fluxes (344-366)
            const double zab = rair / gravit * tin * (1.0 + zvir * (double)q0[i]) * 0.5 * (log((double)ps) - log(pint(nl)));
            const double wind = sqrt(u * u + v * v), lat = latd[col / nlon];
            const double cd = wind < v20 ? Cd0 + Cd1 * wind : Cm;
            skm[cl] = cd * wind * zab;
            ske[cl] = Csfc * wind * zab;
            const double tsurf = simple_sst(sc.sst_mode, lat);
            const double qsats = epsilo * e0 / (double)ps * exp(-latvap / rh2o * ((1.0 / tsurf) - 1.0 / T0));
            u = u / (1.0 + cd * wind * dt / zab);
            v = v / (1.0 + cd * wind * dt / zab);
            t = (t + Csfc * wind * tsurf * dt / zab) / (1.0 + Csfc * wind * dt / zab);
            q = (q + Csfc * wind * qsats * dt / zab) / (1.0 + Csfc * wind * dt / zab);
        }
        st[c - 1][cl] = t;
        sq[c - 1][cl] = q;
        su[c - 1][cl] = u;
        sv[c - 1][cl] = v;
        srp[c - 1][cl] = pm;
        ex[i] = 1.0;
    }
    if (sc.turbflux) {
        __syncthreads();
        // interface c (between c - 1 and c): the sweeps' coefficients are 1 / dp of the
        // layer above or below times the diffusivity times Y (407-431)
        double th[SP_L], rp[SP_L];
#pragma unroll
        for (int i = 0; i < SP_L; i++) {
            const int c = lg + 1 + 16 * i;
            if (c > nl) break;
            const double pi_ = pint(c), pm = srp[c - 1][cl], t = st[c - 1][cl];
            double y = 0.0;
            if (c >= 2) {
                const double rho = pi_ / (rair * (t + st[c - 2][cl]) / 2.0);
                double prof = 1.0;  // taper above pbltop
                if (pi_ < pbltop) prof = exp(-((pbltop - pi_) * (pbltop - pi_)) / (pblconst * pblconst));
                y = dt * gravit * gravit * rho * rho / (pm - srp[c - 2][cl]) * prof;
            }
            sy[c - 1][cl] = y;
            rp[i] = 1.0 / (pint(c + 1) - pi_);
            const double pf = pow(p0 / pm, rk);
            th[i] = pf * t;
            ex[i] = 1.0 / pf;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < SP_L; i++)
            if (lg + 1 + 16 * i <= nl) {
                st[lg + 16 * i][cl] = th[i];
                srp[lg + 16 * i][cl] = rp[i];
            }
        __syncthreads();
        if (tid < 4 * SP_C) {
            // lanes of one wavefront in step: u, v (momentum), T, q (heat) of each column
            const int f = tid / SP_C;
            double(*x)[SP_C] = f == 0 ? su : f == 1 ? sv : f == 2 ? st : sq;
            double(*e)[SP_C] = f < 2 ? sy : srp;  // where this sweep's CE goes
            const double k = f < 2 ? skm[cl] : ske[cl];
            // lanes that share a row write the same CE, one step after all have read it;
            // a step's values are loaded a step ahead, above what it stores
            double ce1 = 0.0, cf1 = 0.0, ca = 0.0;  // CE, CF at c + 1; CA(c), zero at c = nl
            double rp = srp[nl - 1][cl], y = sy[nl - 1][cl], rhs = x[nl - 1][cl];
            for (int c = nl; c >= 1; c--) {  // upward elimination
                const int up = max(c - 2, 0);
                const double rpn = srp[up][cl], yn = sy[up][cl], rhsn = x[up][cl];
                const double cc = rp * (k * y);
                const double r = 1.0 / (1.0 + ca + cc - ca * ce1);
                ce1 = cc * r;
                cf1 = (rhs + ca * cf1) * r;
                ca = rpn * (k * y);  // unused above the top
                e[c - 1][cl] = ce1;
                x[c - 1][cl] = cf1;
                rp = rpn;
                y = yn;
                rhs = rhsn;
            }
            double xp = 0.0;
            int c = 0;
            for (; c + 8 <= nl; c += 8) {  // downward back-substitution (432-447)
                double ev[8], xv[8];
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    ev[j] = e[c + j][cl];
                    xv[j] = x[c + j][cl];
                }
#pragma unroll
                for (int j = 0; j < 8; j++) x[c + j][cl] = xp = ev[j] * xp + xv[j];
            }
            for (; c < nl; c++) x[c][cl] = xp = e[c][cl] * xp + x[c][cl];
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < SP_L; i++) {
        const int c = lg + 1 + 16 * i;
        if (c > nl) break;
        // Tv, changes and column water (phy_run_simple.f90:92-107)
        const double t = st[c - 1][cl] * ex[i], q = sq[c - 1][cl];
        const long o = lvl(c);
        const T dq = (T)(q - (double)q0[i]);
        pw += (pint(c + 1) - pint(c)) * (double)(dq + q0[i]);
        if (valid) {
            const double tv = t * (1.0 + sc.fv * fmax(sc.qmin, q));
            DT[o] = (T)(tv - (double)tv0[i]);
            DQ[o] = dq;
            DU[o] = (T)(su[c - 1][cl] - (double)u0[i]);
            DV[o] = (T)(sv[c - 1][cl] - (double)v0[i]);
        }
    }
    __syncthreads();
    srp[lg][cl] = pw;
    sy[lg][cl] = precl;
    __syncthreads();
    if (lg == 0 && valid) {
        for (int g = 1; g < 16; g++) {
            pw += srp[g][cl];
            precl += sy[g][cl];
        }
        pwat_out[(long)mem * ng + col] = (T)(pw / sc.grav);
        precip_out[(long)mem * ng + col] = (T)(precl * 1000.0);
    }
}

// ---- learned column physics: features, targets, application, judge --------
// Column features (top -> bottom, the plain physics' inputs): T (= Tv / (1 + fv
// max(qmin, q))), q, u, v (nlev each), ps, sea-surface temperature, sin(lat);
// targets: the plain physics' changes of Tv, q, u, v over the step. Optional
// normalisation nrm = [mean_x | std_x | mean_y | std_y].
// Feature rows of the column MLP, one row per selected column: T (= Tv / (1 + fv
// max(qmin, q)), as the plain physics sees it), q, u, v top -> bottom, then ps,
// SST and sin(lat), normalised when nrm is given. A workgroup gathers MLP_CB
// columns with lanes along columns (coalesced level rows), transposes them in
// LDS, and writes their rows, which are contiguous in x, as one coalesced block.
constexpr int MLP_CB = 32;

template <typename T>
__global__ __launch_bounds__(256) void k_mlp_features(const T *__restrict__ gsyn, const T *__restrict__ psg,
                                                      const double *__restrict__ latd, int nl, int nsyn, long ng,
                                                      int nlon, SimpleCfg sc, ColSel cs, long nsel,
                                                      const float *__restrict__ nrm, float *__restrict__ x,
                                                      long row0) {
    extern __shared__ float tile[];  // MLP_CB rows x pitch
    const int nin = 4 * nl + 3, pitch = nin | 1;
    const long i0 = (long)blockIdx.x * MLP_CB;
    const int mem = blockIdx.y;
    const int r = threadIdx.x % MLP_CB, grp = threadIdx.x / MLP_CB, ngrp = blockDim.x / MLP_CB;
    const long col = sel_col(cs, i0 + r, ng);
    const long cc = col < 0 ? 0 : col;  // rows past the selection gather column 0 and are not written
    const T *G = gsyn + (long)mem * nsyn * ng + cc;
    const T *U = G, *V = G + (long)nl * ng, *TV = G + 4L * nl * ng, *Q = G + 7L * nl * ng;
    const T fvT = (T)sc.fv, qminT = (T)sc.qmin;
    float *tr = tile + r * pitch;
    for (int c = 1 + grp; c <= nl; c += ngrp) {
        const long o = (long)(nl - c) * ng;
        const T q = Q[o];
        tr[c - 1] = (float)(TV[o] / (T(1) + fvT * fmax(qminT, q)));
        tr[nl + c - 1] = (float)q;
        tr[2 * nl + c - 1] = (float)U[o];
        tr[3 * nl + c - 1] = (float)V[o];
    }
    if (grp == 0) {
        const double lat = latd[cc / nlon];
        tr[4 * nl] = (float)psg[(long)mem * ng + cc];
        tr[4 * nl + 1] = (float)simple_sst(sc.sst_mode, lat);
        tr[4 * nl + 2] = (float)sin(lat);
    }
    __syncthreads();
    const int nrow = (int)min((long)MLP_CB, nsel - i0);
    float *xb = x + (row0 + (long)mem * nsel + i0) * nin;
    for (int e = threadIdx.x; e < nrow * nin; e += blockDim.x) {
        const int rr = e / nin, f = e - rr * nin;
        float v = tile[rr * pitch + f];
        if (nrm) v = (v - nrm[f]) / nrm[nin + f];
        xb[e] = v;
    }
}

template <typename T>
__global__ __launch_bounds__(256) void k_mlp_targets(const T *__restrict__ gan, int nl, int nsp, long ng, ColSel cs,
                                                     long nsel, float *__restrict__ y, long row0) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long col = sel_col(cs, i, ng);
    const int mem = blockIdx.y;
    if (col < 0) return;
    const T *A = gan + (long)mem * nsp * ng + col;
    float *yr = y + (row0 + (long)mem * nsel + i) * (4L * nl);
    for (int c = 1; c <= nl; c++) {
        const long o = (long)(nl - c) * ng;
        yr[c - 1] = (float)A[o];                         // Tv change
        yr[nl + c - 1] = (float)A[3L * nl * ng + o];     // q change
        yr[2 * nl + c - 1] = (float)A[(long)nl * ng + o]; // u change
        yr[3 * nl + c - 1] = (float)A[2L * nl * ng + o];  // v change
    }
}

// Network outputs (normalised dT, dq, du, dv per level, top -> bottom) back to
// the physics grid fields; the column water after the change (pwat) for the mass
// fixer. Rows of MLP_CB columns are read as one coalesced block and transposed
// in LDS so that the level rows of the fields are written coalesced.
template <typename T>
__global__ __launch_bounds__(256) void k_mlp_apply(const float *__restrict__ y, const float *__restrict__ nrm,
                                                   const T *__restrict__ gsyn, const T *__restrict__ psg,
                                                   const T *__restrict__ ak, const T *__restrict__ bk,
                                                   T *__restrict__ gan, T *__restrict__ pwat_out,
                                                   T *__restrict__ precip_out, int nl, int nsyn, int nsp, long ng,
                                                   double grav) {
    extern __shared__ float tile[];  // MLP_CB rows x pitch
    __shared__ double pws[256 / MLP_CB][MLP_CB];
    const int nin = 4 * nl + 3, nout = 4 * nl, pitch = nout | 1;
    const float *my = nrm + 2 * nin, *sy = my + nout;
    const long c0 = (long)blockIdx.x * MLP_CB;
    const int mem = blockIdx.y;
    const int nrow = (int)min((long)MLP_CB, ng - c0);
    const float *yb = y + ((long)mem * ng + c0) * nout;
    for (int e = threadIdx.x; e < nrow * nout; e += blockDim.x) {
        const int rr = e / nout, f = e - rr * nout;
        tile[rr * pitch + f] = my[f] + sy[f] * yb[e];
    }
    __syncthreads();
    const int r = threadIdx.x % MLP_CB, grp = threadIdx.x / MLP_CB, ngrp = blockDim.x / MLP_CB;
    const long col = c0 + r;
    double pw = 0.0;
    if (r < nrow) {
        const T *Q = gsyn + (long)mem * nsyn * ng + 7L * nl * ng + col;
        T *A = gan + (long)mem * nsp * ng + col;
        const T ps = psg[(long)mem * ng + col];
        const float *tr = tile + r * pitch;
        for (int c = 1 + grp; c <= nl; c += ngrp) {
            const long o = (long)(nl - c) * ng;
            A[o] = (T)tr[c - 1];
            const T dq = (T)tr[nl + c - 1];
            A[3L * nl * ng + o] = dq;
            A[(long)nl * ng + o] = (T)tr[2 * nl + c - 1];
            A[2L * nl * ng + o] = (T)tr[3 * nl + c - 1];
            const double dp = (double)((ak[c] + bk[c] * ps) - (ak[c - 1] + bk[c - 1] * ps));
            pw += dp * (double)(dq + Q[o]);
        }
    }
    pws[grp][r] = pw;
    __syncthreads();
    if (grp == 0 && r < nrow) {
        double t = 0.0;
        for (int k = 0; k < ngrp; k++) t += pws[k][r];
        pwat_out[(long)mem * ng + col] = (T)(t / grav);
        precip_out[(long)mem * ng + col] = T(0);
    }
}

// judge: normalised squared difference between the network's and the plain
// physics' changes on the sampled columns (block partial sums)
template <typename T>
__global__ __launch_bounds__(256) void k_judge_partial(const T *__restrict__ gan, const T *__restrict__ ganj,
                                                       const float *__restrict__ nrm, int nl, int nsp, long ng,
                                                       ColSel cs, double *__restrict__ part) {
    // one (judged column, slot, level) value per thread and step of a grid-stride
    // loop, consecutive threads on consecutive judged columns: every CU reads
    const int mem = blockIdx.y;
    const long nsel = cs.stride > 0 ? ng / cs.stride : ng, total = nsel * 4L * nl;
    const int nin = 4 * nl + 3, nout = 4 * nl;
    const float *sy = nrm + 2 * nin + nout;
    double s = 0.0;
    for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (long)gridDim.x * blockDim.x) {
        const long i = t % nsel;
        const int e = (int)(t / nsel), sl = e / nl, c = e - sl * nl + 1;
        const long col = sel_col(cs, i, ng);
        // slot order in gan: Tv, u, v, q; target order: Tv, q, u, v
        const int ts = sl == 0 ? 0 : (sl == 1 ? 2 : (sl == 2 ? 3 : 1));
        const long o = (long)mem * nsp * ng + col + ((long)sl * nl + (nl - c)) * ng;
        const double d = ((double)gan[o] - (double)ganj[o]) / sy[ts * nl + c - 1];
        s += d * d;
    }
    __shared__ double red[256];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[(long)blockIdx.y * gridDim.x + blockIdx.x] = red[0];
}

// rms error in units of the targets' standard deviations; sets the fallback
// flag above the threshold; stats = [last error, fallbacks, judged steps]
__global__ __launch_bounds__(256) void k_judge_final(const double *__restrict__ part, int npart, double count,
                                                     double thr, int *__restrict__ flag,
                                                     double *__restrict__ stats) {
    __shared__ double red[256];
    double s = 0.0;
    for (int i = threadIdx.x; i < npart; i += 256) s += part[i];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const double err = sqrt(red[0] / count);
        const int fb = !(err <= thr);  // NaN falls back too
        flag[0] = fb;
        stats[0] = err;
        stats[1] += fb;
        stats[2] += 1.0;
    }
}

// per-feature mean and standard deviation of a row-major [n][nf] array (FP64
// sums, one block per feature); std floored at 1e-10
__global__ __launch_bounds__(256) void k_colstats(const float *__restrict__ a, long n, int nf,
                                                  float *__restrict__ mean, float *__restrict__ sd) {
    const int f = blockIdx.x;
    double s = 0.0, s2 = 0.0;
    for (long r = threadIdx.x; r < n; r += 256) {
        const double v = a[r * nf + f];
        s += v;
        s2 += v * v;
    }
    __shared__ double r1[256], r2[256];
    r1[threadIdx.x] = s;
    r2[threadIdx.x] = s2;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
            r1[threadIdx.x] += r1[threadIdx.x + w];
            r2[threadIdx.x] += r2[threadIdx.x + w];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const double m = r1[0] / n, var = fmax(r2[0] / n - m * m, 0.0);
        mean[f] = (float)m;
        sd[f] = (float)fmax(sqrt(var), 1e-10);
    }
}

// a normalised training batch: rows drawn uniformly (counter RNG) from [0, ntrain)
__global__ void k_mlp_batch(const float *__restrict__ dx, const float *__restrict__ dy, long ntrain, int nin,
                            int nout, const float *__restrict__ nrm, unsigned long long seed,
                            unsigned long long ctr, int nb, float *__restrict__ bx, float *__restrict__ by) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int nf = nin + nout;
    if (i >= (long)nb * nf) return;
    const int r = (int)(i / nf), f = (int)(i % nf);
    const long src = (long)(rng_mix(seed, ctr, (uint64_t)r) % (uint64_t)ntrain);
    if (f < nin)
        bx[(long)r * nin + f] = (dx[src * nin + f] - nrm[f]) / nrm[nin + f];
    else
        by[(long)r * nout + f - nin] = (dy[src * nout + f - nin] - nrm[2 * nin + f - nin]) / nrm[2 * nin + nout + f - nin];
}

// normalised rms error of predictions against targets (rows [0, n)) and of the
// mean predictor (the normalised targets themselves): partial sums
__global__ __launch_bounds__(256) void k_eval_partial(const float *__restrict__ yp, const float *__restrict__ dy,
                                                      long n, int nout, const float *__restrict__ nrm_y,
                                                      double *__restrict__ part) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    double e = 0.0, b = 0.0;
    if (i < n * nout) {
        const int f = (int)(i % nout);
        const double t = (dy[i] - nrm_y[f]) / nrm_y[nout + f];
        const double d = yp[i] - t;
        e = d * d;
        b = t * t;
    }
    __shared__ double r1[256], r2[256];
    r1[threadIdx.x] = e;
    r2[threadIdx.x] = b;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
            r1[threadIdx.x] += r1[threadIdx.x + w];
            r2[threadIdx.x] += r2[threadIdx.x + w];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = r1[0];
        part[2 * blockIdx.x + 1] = r2[0];
    }
}

// mass-fixer field of the simple physics: ln ps' + log(pcorr) with
// pcorr = (pdryini + g pwatg) / pmean (dyn_run.f90:618-631)
template <typename T>
__global__ __launch_bounds__(256) void k_massfix_field(const T *__restrict__ gsyn, T *__restrict__ gan,
                                                       const double *__restrict__ pdryini,
                                                       const double *__restrict__ pmean,
                                                       const double *__restrict__ pwsum, int nl, int ntr, int nsyn,
                                                       int nsp, long ng, double grav) {
    const long col = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int mem = blockIdx.y;
    if (col >= ng) return;
    const T *LNPS = gsyn + (long)mem * nsyn * ng + (7L + 3L * ntr) * nl * ng + col;
    gan[(long)mem * nsp * ng + 4L * nl * ng + col] =
        LNPS[0] + (T)log((pdryini[mem] + grav * pwsum[mem]) / pmean[mem]);
}

// AR(1) pattern advance (patterngenerator.f90:134-143 with getnoise 115-132):
// pat = phi pat + f var noise for nf independent patterns per member, one
// thread per (coefficient, member, pattern). Noise is Box-Muller on the counter
// RNG: seed + member, stream sbase + nf * (advance count) + pattern (the count
// read from the device counter so graph replays continue the stream), index
// 2k / 2k+1. sc = sqrt(normfact / ntrunc) with normfact = 2 pi.
template <typename T>
__global__ __launch_bounds__(256) void k_pattern_advance(cplx<T> *__restrict__ pat, const double *__restrict__ var,
                                                         const int2 *__restrict__ kmn, int nlm,
                                                         const unsigned long long *__restrict__ ctr,
                                                         unsigned long long seed, double phi, double f, double sc,
                                                         int nf, unsigned long long sbase) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    const int mem = blockIdx.y / nf, fld = blockIdx.y - mem * nf;
    if (k >= nlm) return;
    double nr = 0.0, ni = 0.0;
    if (k > 0) {
        const uint64_t stream = sbase + ctr[0] * (uint64_t)nf + (uint64_t)fld, sd = seed + (uint64_t)mem;
        const double u1 = (double)(rng_mix(sd, stream, 2ULL * k) >> 11) * 0x1p-53;
        const double u2 = (double)(rng_mix(sd, stream, 2ULL * k + 1) >> 11) * 0x1p-53;
        const double r = sqrt(-2.0 * log(1.0 - u1));
        const double gr = r * cos(2.0 * M_PI * u2), gi = r * sin(2.0 * M_PI * u2);
        const int2 mn = kmn[k];
        const double w = 1.0 / sqrt(2.0 * mn.y + 1.0);
        if (mn.x != 0) {
            nr = gr * w * sc;
            ni = gi * w * sc;
        } else {
            nr = sqrt(2.0) * gr * w * sc;
        }
    }
    cplx<T> *p = pat + ((long)mem * nf + fld) * nlm + k;
    const double v = f * var[k];
    *p = cplx<T>{(T)(phi * (double)p->x + v * nr), (T)(phi * (double)p->y + v * ni)};
}

__global__ void k_counter_inc(unsigned long long *ctr) {
    if (threadIdx.x == 0 && blockIdx.x == 0) ctr[0] += 1ULL;
}

// model clock: t = t + dt at the end of every step (run.f90:153)
__global__ void k_clock_add(double *clk, double dt) {
    if (threadIdx.x == 0 && blockIdx.x == 0) clk[0] += dt;
}

// sppt grid: the logit transform 2 / (1 + e^g) - 1 of run.f90:281
template <typename T> __global__ __launch_bounds__(256) void k_logit(T *__restrict__ g, long n) {
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        g[i] = T(2) / (T(1) + exp(g[i])) - T(1);
}

// getstochforcing inputs (stoch_data.f90:264-290), work layout w[group][member][level][nlm]:
// group 0 the streamfunction patterns, 1-2-1 filtered in the vertical when
// vfilt (one pass: the reference re-filters the unfiltered patterns on every
// pass; the end levels with the factor 1 + 1/3 of a default-real literal),
// group 1 -disspec vrt, group 2 -disspec div (the dissipation wind)
template <typename T>
__global__ __launch_bounds__(256) void k_an_prep(cplx<T> *__restrict__ w, const cplx<T> *__restrict__ psi,
                                                 const cplx<T> *__restrict__ spec, const T *__restrict__ disspec,
                                                 int nl, int nfs, int nm, int nlm, int vfilt, int diss) {
    const long tot = (long)nm * nl * nlm;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < tot; i += (long)gridDim.x * blockDim.x) {
        const int k = (int)(i % nlm);
        const long r = i / nlm;
        const int lev = (int)(r % nl), mem = (int)(r / nl);
        const cplx<T> *q = psi + i;
        cplx<T> o = *q;
        if (vfilt) {
            const T c = T(SGLF(1. + 1. / 3.));
            cplx<T> a;
            if (lev == 0)
                a = cplx<T>{c * q[nlm].x + T(2) * c * q[0].x, c * q[nlm].y + T(2) * c * q[0].y};
            else if (lev == nl - 1)
                a = cplx<T>{c * q[-nlm].x + T(2) * c * q[0].x, c * q[-nlm].y + T(2) * c * q[0].y};
            else
                a = cplx<T>{q[nlm].x + T(2) * q[0].x + q[-nlm].x, q[nlm].y + T(2) * q[0].y + q[-nlm].y};
            o = cplx<T>{T(0.25) * a.x, T(0.25) * a.y};
        }
        w[i] = o;
        if (diss) {
            const long s = (long)k * nfs * nm + (long)mem * nfs + lev;
            const T d = -disspec[k];
            const cplx<T> v = spec[s], dv = spec[s + nl];
            w[tot + i] = cplx<T>{d * v.x, d * v.y};
            w[2 * tot + i] = cplx<T>{d * dv.x, d * dv.y};
        }
    }
}

// smoothed-input field of getstochforcing :277-283 on the grid:
// sqrt(max(|u ud + v vd|, tiny)) into the ud slot (grid layout g[group][member][level][ng])
template <typename T>
__global__ __launch_bounds__(256) void k_an_kediss(T *__restrict__ g, const T *__restrict__ gsyn, int nl, int nsyn,
                                                   int nm, long ng) {
    const long tot = (long)nm * nl * ng;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < tot; i += (long)gridDim.x * blockDim.x) {
        const long col = i % ng, r = i / ng;
        const int lev = (int)(r % nl), mem = (int)(r / nl);
        const T *G = gsyn + (long)mem * nsyn * ng + col;
        const T d = fabs(G[(long)lev * ng] * g[i] + G[(long)(nl + lev) * ng] * g[tot + i]);
        const T tiny = (T)FLT_MIN;
        g[i] = sqrt(d < tiny ? tiny : d);
    }
}

// per-coefficient scaling of nf fields [field][nlm]: x *= f[k]
template <typename T>
__global__ __launch_bounds__(256) void k_spec_scale(cplx<T> *__restrict__ x, const T *__restrict__ f, long nf,
                                                    int nlm) {
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < nf * nlm; i += (long)gridDim.x * blockDim.x) {
        const T s = f[i % nlm];
        x[i] = cplx<T>{s * x[i].x, s * x[i].y};
    }
}

// modulated streamfunction forcing on the grid (:284-289): vfact psi (x the
// smoothed dissipation field with diss) into the group-0 slot
template <typename T>
__global__ __launch_bounds__(256) void k_an_modulate(T *__restrict__ g, const T *__restrict__ psig,
                                                     const T *__restrict__ sm, const T *__restrict__ vf, int nl, int nm,
                                                     long ng) {
    const long tot = (long)nm * nl * ng;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < tot; i += (long)gridDim.x * blockDim.x) {
        const int lev = (int)((i / ng) % nl);
        T v = vf[lev] * psig[i];
        if (sm) v *= sm[i];
        g[i] = v;
    }
}

// run.f90:541-552: vrt += dt lap / a^2 psif, or -dt sqrt(-lap) / a psif with
// kenorm (the temperature forcing is zero with addnoise_vrtonly)
template <typename T>
__global__ __launch_bounds__(256) void k_an_apply(cplx<T> *__restrict__ spec, const cplx<T> *__restrict__ psif,
                                                  const int *__restrict__ degree, int nl, int nfs, int nm, int nlm,
                                                  double dt, double rerth, int kenorm) {
    const long tot = (long)nm * nl * nlm;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < tot; i += (long)gridDim.x * blockDim.x) {
        const int k = (int)(i % nlm);
        const long r = i / nlm;
        const int lev = (int)(r % nl), mem = (int)(r / nl);
        const double n = degree[k], lap = -n * (n + 1.0);
        const T c = kenorm ? (T)(-dt * sqrt(-lap) / rerth) : (T)(dt * lap / (rerth * rerth));
        cplx<T> *o = spec + (long)k * nfs * nm + (long)mem * nfs + lev;
        const cplx<T> f = psif[i];
        *o = cplx<T>{o->x + c * f.x, o->y + c * f.y};
    }
}

// getiauforcing (iau_module.f90:84-115) at the clock's time t: zero outside
// [hrs[0], hrs[nf-1]] h, the first or last increment / dti at those end
// points, else ((1 - delt) inc[n] + delt inc[n-1]) / dti with n the first
// file later than t and delt = (hrs[n] - t/3600) / (hrs[n] - hrs[n-1]).
// Formed in FP64 (the reference's FP64 delt promotes it) and rounded to T.
// Every thread finds the weights itself from the clock: the kernel sits in
// the captured step and reads the time of the replay that runs it.
template <typename T>
__global__ __launch_bounds__(256) void k_iau_forcing(T *__restrict__ F, const T *__restrict__ inc,
                                                     const double *__restrict__ hrs, int nf, double dti,
                                                     const double *__restrict__ clk, long len) {
    const double t = clk[0];
    double whi = 0.0, wlo = 0.0;
    int n = 0;
    if (!(t < hrs[0] * 3600. || t > hrs[nf - 1] * 3600.)) {
        if (t == 3600. * hrs[nf - 1]) {
            n = nf - 1;
            whi = 1.0;
        } else if (t == 3600. * hrs[0]) {
            whi = 1.0;
        } else {
            for (n = 1; n < nf - 1; n++)
                if (hrs[n] * 3600. > t) break;
            const double delt = (hrs[n] - t / 3600.) / (hrs[n] - hrs[n - 1]);
            whi = 1. - delt;
            wlo = delt;
        }
    }
    const T *hi = inc + (long)n * len, *lo = n > 0 ? hi - len : hi;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < len; i += (long)gridDim.x * blockDim.x)
        F[i] = (T)((whi * (double)hi[i] + wlo * (double)lo[i]) / dti);
}

// y = a x + b y (b == 0: y = a x, whatever y held)
template <typename T>
__global__ __launch_bounds__(256) void k_axpby(T *__restrict__ y, const T *__restrict__ x, T a, T b, long n) {
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        y[i] = b == (T)0 ? a * x[i] : a * x[i] + b * y[i];
}

// temperature forcing pattern / tau on every level (vertical taper vf)
template <typename T>
__global__ void k_pattern_apply(cplx<T> *__restrict__ spec, const cplx<T> *__restrict__ pat, const T *__restrict__ vf,
                                int nl, int nfs, int nm, int nlm, T dt_tau) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long tot = (long)nlm * nm * nl;
    if (i >= tot) return;
    const int lev = (int)(i % nl);
    const long r = i / nl;
    const int mem = (int)(r % nm), k = (int)(r / nm);
    const cplx<T> q = pat[(long)mem * nlm + k];
    const T a = dt_tau * vf[lev];
    cplx<T> *o = spec + ((long)k * nm + mem) * nfs + 2 * nl + lev;
    *o = cplx<T>{o->x + a * q.x, o->y + a * q.y};
}

// Per-step diagnostics of run.f90:159-162 (spdmax, min/max ps, pstend) per member.
template <typename T>
__global__ __launch_bounds__(1024) void k_diag(const T *__restrict__ gsyn, const T *__restrict__ psg,
                                               const T *__restrict__ dlnpsdt, const double *__restrict__ areaw,
                                               double *__restrict__ out, int nl, int nsyn, long ng, int nlon) {
    const int mem = blockIdx.x;
    const T *U = gsyn + (long)mem * nsyn * ng, *V = U + (long)nl * ng;
    const T *P = psg + (long)mem * ng, *D = dlnpsdt + (long)mem * ng;
    double smax = 0, pmin = 1e300, pmax = -1e300, pst = 0;
    for (long i = threadIdx.x; i < (long)nl * ng; i += blockDim.x) {
        double s = sqrt((double)U[i] * U[i] + (double)V[i] * V[i]);
        smax = s > smax ? s : smax;
    }
    for (long i = threadIdx.x; i < ng; i += blockDim.x) {
        double p = P[i];
        pmin = p < pmin ? p : pmin;
        pmax = p > pmax ? p : pmax;
        double t = 36.0 * p * (double)D[i];
        pst += t * t * areaw[i / nlon];
    }
    __shared__ double r[4][1024];
    r[0][threadIdx.x] = smax;
    r[1][threadIdx.x] = pmin;
    r[2][threadIdx.x] = pmax;
    r[3][threadIdx.x] = pst;
    __syncthreads();
    for (int w = 512; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
            int a = threadIdx.x, b = threadIdx.x + w;
            r[0][a] = r[0][a] > r[0][b] ? r[0][a] : r[0][b];
            r[1][a] = r[1][a] < r[1][b] ? r[1][a] : r[1][b];
            r[2][a] = r[2][a] > r[2][b] ? r[2][a] : r[2][b];
            r[3][a] += r[3][b];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[4 * mem + 0] = r[0][0];
        out[4 * mem + 1] = r[1][0];
        out[4 * mem + 2] = r[2][0];
        out[4 * mem + 3] = sqrt(r[3][0]);
    }
}

// One stage of the explicit scheme for every spectral coefficient (run.f90:313-350,
// 374-417, 440-489 without the linear terms) and, after the last stage, the
// implicit damping (run.f90:493-502). One wavefront per (coefficient, member),
// lane = model level (bottom -> top).
template <typename T>
__global__ __launch_bounds__(256) void k_explicit_stage(
    cplx<T> *__restrict__ spec, const cplx<T> *__restrict__ spec0, const cplx<T> *__restrict__ ten0,
    const cplx<T> *__restrict__ ten1, const cplx<T> *__restrict__ ten2, const T *__restrict__ disspec,
    const T *__restrict__ diffp, const T *__restrict__ dmpp, int stage, Coeffs3 cf, int damp, int nl, int ntr, int nfs,
    int nm, int nlm, T dt) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const long item = (long)blockIdx.x * 4 + wave;  // (coefficient, member)
    if (item >= (long)nlm * nm) return;
    const int mem = (int)(item / nlm), k = (int)(item % nlm);
    const long base = (long)k * nfs * nm + (long)mem * nfs;
    const cplx<T> *tn[3] = {ten0, ten1, ten2};
    auto stepped = [&](long off) {
        cplx<T> acc{T(0), T(0)};
        for (int r = 0; r <= stage; r++) {
            const cplx<T> t = tn[r][off];
            acc.x += T(cf.a[r]) * t.x;
            acc.y += T(cf.a[r]) * t.y;
        }
        const cplx<T> o = spec0[off];
        return cplx<T>{o.x + dt * acc.x, o.y + dt * acc.y};
    };
    const T ds = disspec[k];
    for (int q = 0; q < 3 + ntr && lane < nl; q++) {  // vorticity, divergence, temperature, tracers
        const long off = base + (long)q * nl + lane;
        cplx<T> v = stepped(off);
        if (damp) {
            const T f = q < 2 ? T(1) - (ds * diffp[lane] - dmpp[lane]) * dt : T(1) - ds * diffp[lane] * dt;
            v = cplx<T>{v.x / f, v.y / f};
        }
        spec[off] = v;
    }
    const long ilp = base + (3L + ntr) * nl;
    if (lane == 0) spec[ilp] = stepped(ilp);
}

// One stage of the IMEX scheme (run.f90:313-350, 374-417, 440-489, damping 493-502) as
// batched matrix products on the matrix cores: a workgroup takes up to
// C = SiCfg<T>::C spectral coefficients of one total wavenumber n (each member's m = 0..n),
// i.e. 2 C real columns of level vectors, and every level operator
// (amhyb, bmhyb and d_hyb_m of degree n, all real) becomes one 64 x 64 x 64
// product Y = M X on MFMA 16x16x4 (wave w computes output levels 16w..16w+15).
// Real and imaginary parts are independent columns because all operators and
// coefficients are real. Level vectors stay in LDS between the products.
// Coefficients per workgroup: 8, the fewest that fill a 16-column MFMA block
// (2 C real columns, padded rows of LD values). The stage is bound by the
// latency of its load/product phases, not by the matrix cores, so the small
// tile's LDS (about 20 KB in FP32) and twice the workgroups per CU outrun 16
// coefficients per workgroup.
template <typename T> struct SiCfg {
    static constexpr int C = 8, W = 2 * C, LD = W + 4;
};
// MFMA 16x16x4 in the precision of the stage: A[i][k] from lane i + 16k,
// B[k][j] from lane j + 16k; accumulator element r of a lane is row 4 (lane/16)
// + r (f32) or lane/16 + 4 r (f64), column lane % 16.
template <typename T> struct SiMma;
template <> struct SiMma<float> {
    typedef float acc __attribute__((ext_vector_type(4)));
    __device__ static acc mma(float a, float b, acc c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
    __device__ static int row(int lane, int r) { return 4 * (lane >> 4) + r; }
};
template <> struct SiMma<double> {
    typedef double acc __attribute__((ext_vector_type(4)));
    __device__ static acc mma(double a, double b, acc c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
    __device__ static int row(int lane, int r) { return (lane >> 4) + 4 * r; }
};

// Rows that a product reads and writes: 32 of the 64 where the levels fit them
__device__ __forceinline__ int si_rows(int nl) { return nl <= 32 ? 32 : 64; }

// This lane's values of a level operator M, given transposed (Mt[k * nl + i] = M[i][k]),
// zero beyond nl levels: all loaded at once, one wait for the (cached) operator
template <typename T> struct SiOp {
    T a[16];
    template <int Q0, int Q1> __device__ __forceinline__ void part(const T *__restrict__ Mt, int nl, int i, int kq) {
#pragma unroll
        for (int q = Q0; q < Q1; q++) {
            const int k = 4 * q + kq;
            const T x = Mt[min(k, nl - 1) * nl + min(i, nl - 1)];
            a[q] = i < nl && k < nl ? x : T(0);
        }
    }
    __device__ __forceinline__ void load(const T *__restrict__ Mt, int nl, int wave, int lane) {
        const int i = wave * 16 + (lane & 15), kq = lane >> 4, nr = si_rows(nl);
        if (wave * 16 >= nr) return;
        part<0, 8>(Mt, nl, i, kq);
        if (nr > 32) part<8, 16>(Mt, nl, i, kq);
    }
};

// Y[i][col] = sum_k M[i][k] X[k][col] over the first si_rows(nl) rows, zero in X past nl
template <typename T, int NQ>
__device__ __forceinline__ void si_gemm_n(const SiOp<T> &M, const T (*X)[SiCfg<T>::LD], T (*Y)[SiCfg<T>::LD], int wave,
                                          int lane) {
    constexpr int NB = SiCfg<T>::W / 16;
    typename SiMma<T>::acc acc[NB];
#pragma unroll
    for (int b = 0; b < NB; b++) acc[b] = typename SiMma<T>::acc{T(0), T(0), T(0), T(0)};
#pragma unroll
    for (int q = 0; q < NQ; q++)
#pragma unroll
        for (int b = 0; b < NB; b++)
            acc[b] = SiMma<T>::mma(M.a[q], X[4 * q + (lane >> 4)][b * 16 + (lane & 15)], acc[b]);
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int r = 0; r < 4; r++) Y[wave * 16 + SiMma<T>::row(lane, r)][b * 16 + (lane & 15)] = acc[b][r];
}
template <typename T>
__device__ __forceinline__ void si_gemm(const SiOp<T> &M, int nl, const T (*X)[SiCfg<T>::LD], T (*Y)[SiCfg<T>::LD],
                                        int wave, int lane) {
    const int nr = si_rows(nl);
    if (wave * 16 >= nr) return;
    if (nr > 32)
        si_gemm_n<T, 16>(M, X, Y, wave, lane);
    else
        si_gemm_n<T, 8>(M, X, Y, wave, lane);
}

// by the last wavefront, which has no product where the levels fit 32 rows
template <typename T>
__device__ inline void si_colsum(const T *w, int nl, const T (*X)[SiCfg<T>::LD], T *out) {
    const int col = (int)threadIdx.x - 192;
    if (col >= 0 && col < SiCfg<T>::W) {
        T s = T(0);
#pragma unroll 8
        for (int l = 0; l < nl; l++) s += w[l] * X[l][col];
        out[col] = s;
    }
}

// What a later stage needs of an earlier one's tendency and linear term is one
// sum of the two, kept in their place (E1, E2); the initial state is kept by the
// stage that first reads it; the last stage keeps nothing. Per coefficient the
// three stages move 3154 instead of 4121 values a member at 64 levels (dry),
// the copy of the initial state included: T254L64 FP32 six steps 18.24 -> 17.96 ms.
// Bound by its chain of waits and barriers at small sizes, by memory (two thirds of
// the time of a copy of what it moves) at T254: T42 20 levels FP64 14.5 -> 11.0 us a stage
// with 32-row products where the levels fit, the coefficient's index computed instead
// of loaded, and the column sums on a wavefront of their own; T254 64 levels FP32 110 ->
// 105 us, 16 members at T126 393 -> 378 us. The operators and the combination's values
// loaded ahead of all else cost more in wavefronts (191 and 110 registers: T254 150 us).
// the tableau's column of a stage: its own coefficients, the next stage's and the one after's
struct SiNext {
    double a0, aa0, a1, aa1, a2, aa2;
};
template <typename T>
__global__ __launch_bounds__(256) void k_si_mfma(
    T *__restrict__ spec, T *__restrict__ spec0, const T *__restrict__ ten0, const T *__restrict__ ten1,
    const T *__restrict__ ten2, T *__restrict__ e1_, T *__restrict__ e2_,
    const T *__restrict__ At, const T *__restrict__ Bt, const T *__restrict__ Dt,
    const T *__restrict__ sv, const T *__restrict__ tor, const T *__restrict__ disspec,
    const T *__restrict__ diffp, const T *__restrict__ dmpp, const int2 *__restrict__ tiles, int stage, Coeffs3 cf,
    SiNext cn, T cimp, int do_implicit, int damp, int nl, int ntr, int nfs, int nm, int ntrunc, T dt,
    double *__restrict__ clock, double dtd) {
    constexpr int C = SiCfg<T>::C, W = SiCfg<T>::W, LD = SiCfg<T>::LD;
    typedef cplx<T> V2;
    __shared__ T S0[64][LD], S1[64][LD], S2[64][LD], S3[64][LD];
    __shared__ T lpin[W], lpc[W], csum[W];
    __shared__ long sbase[C], slbase[C];
    __shared__ int sk[C];
    __shared__ T svs[64], tors[64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (tid < nl) {
        svs[tid] = sv[tid];
        tors[tid] = tor[tid];
    }
    // tiles run in degree order, each XCD a contiguous range of them, so that
    // the tiles of one degree share its operators in one L2
    const int2 tl = tiles[xcd_tile(blockIdx.x, gridDim.x)];
    const int n = tl.x, i0 = tl.y, per = (n + 1) * nm;
    const int cnt = min(C, per - i0);
    const long NFS = (long)nfs * nm, nlin = 2L * nl + 1;
    if (tid < C) {
        long b = 0, lb = 0;
        int k = 0;
        if (tid < cnt) {
            const int item = i0 + tid, mem = item / (n + 1), m = item - mem * (n + 1);
            k = m * (2 * ntrunc + 3 - m) / 2 + n - m;
            b = (long)k * NFS + (long)mem * nfs;
            lb = (long)k * nlin * nm + (long)mem * nlin;
        }
        sbase[tid] = b;
        slbase[tid] = lb;
        sk[tid] = k;
    }
    __syncthreads();
    const T lap = -T(n) * T(n + 1);
    // the model clock moves with the last stage
    if (clock && stage == 2 && blockIdx.x == 0 && tid == 0) *clock += dtd;
    V2 *sp = (V2 *)spec;
    // stage 0 finds the step's initial state in spec, which it overwrites, and keeps it in spec0
    const V2 *sp0 = stage == 0 ? (const V2 *)spec : (const V2 *)spec0;
    const V2 *tn[3] = {(const V2 *)ten0, (const V2 *)ten1, (const V2 *)ten2};
    V2 *E1 = (V2 *)e1_, *E2 = (V2 *)e2_;
    // element e = c * nl + lev: one complex value (re, im) per element
    const int nel = cnt * nl;
    // the loads of the stage input (tv, div, ln ps) go out before those of the fields below
    constexpr int NI = 64 * C / 256;
    V2 tvi[NI], dvi[NI], lp0 = V2{T(0), T(0)};
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const int c = min((tid >> 6) + 4 * i, cnt - 1);
        const long b = sbase[c] + min(lane, nl - 1);
        tvi[i] = sp[b + 2L * nl];
        dvi[i] = sp[b + nl];
    }
    if (tid < cnt) lp0 = sp[sbase[tid] + 3L * nl + (long)ntr * nl];
    const V2 *Tn = tn[stage];
    const V2 *Ep = stage == 2 ? E2 : E1;
    // vorticity and tracers: always explicit (plus damping after the last stage)
    for (int e = tid; e < nel * (1 + ntr); e += 256) {
        const int fld = e / nel, r0 = e - fld * nel, c = r0 / nl, lev = r0 - c * nl;
        const long off = sbase[c] + (fld == 0 ? 0L : 3L * nl + (long)(fld - 1) * nl) + lev;
        V2 acc = V2{T(0), T(0)};
        for (int r = 0; r <= stage; r++) {
            const V2 t = tn[r][off];
            acc.x += cf.a[r] * t.x;
            acc.y += cf.a[r] * t.y;
        }
        const V2 o = sp0[off];
        if (stage == 0) ((V2 *)spec0)[off] = o;
        V2 v = V2{o.x + dt * acc.x, o.y + dt * acc.y};
        if (damp) {
            const T ds = disspec[sk[c]];
            const T f = (fld == 0) ? T(1) - (ds * diffp[lev] - dmpp[lev]) * dt : T(1) - ds * diffp[lev] * dt;
            v.x /= f;
            v.y /= f;
        }
        sp[off] = v;
    }
    // stage input: tv -> S0, div -> S1 (zero padded), ln ps -> lpin
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const int c = (tid >> 6) + 4 * i;
        const bool in = c < cnt && lane < nl;
        const V2 tv = in ? tvi[i] : V2{T(0), T(0)}, dv = in ? dvi[i] : V2{T(0), T(0)};
        if (stage == 0 && in) {
            ((V2 *)spec0)[sbase[c] + lane + 2L * nl] = tv;
            ((V2 *)spec0)[sbase[c] + lane + nl] = dv;
        }
        S0[lane][2 * c] = tv.x;
        S0[lane][2 * c + 1] = tv.y;
        S1[lane][2 * c] = dv.x;
        S1[lane][2 * c + 1] = dv.y;
    }
    if (tid < C) {
        if (stage == 0 && tid < cnt) ((V2 *)spec0)[sbase[tid] + 3L * nl + (long)ntr * nl] = lp0;
        lpin[2 * tid] = lp0.x;
        lpin[2 * tid + 1] = lp0.y;
    }
    __syncthreads();
    // linear terms of the stage input (run.f90:329-335)
    SiOp<T> op;
    op.load(At, nl, wave, lane);
    si_gemm<T>(op, nl, S0, S2, wave, lane);
    op.load(Bt, nl, wave, lane);
    si_gemm<T>(op, nl, S1, S3, wave, lane);
    si_colsum<T>(svs, nl, S1, csum);
    __syncthreads();
    // take them from this stage's tendency; explicit combination. A later stage
    // needs this one's tendency d and linear term l only as a d + aa l, so that is
    // what is kept: E1 for stage 1, E2 for stage 2
    // own contribution of (d, l), with the earlier stages' (e) from E; updates E for the
    // later ones (f: what E2 holds in stage 1)
    auto combine = [&](long lb, V2 d, V2 l, V2 e, V2 f) {
        auto mix = [&](double ca, double cl) { return V2{(T)(ca * d.x + cl * l.x), (T)(ca * d.y + cl * l.y)}; };
        const V2 a = mix(cn.a0, cn.aa0);
        if (stage == 0) {
            E1[lb] = mix(cn.a1, cn.aa1);
            E2[lb] = mix(cn.a2, cn.aa2);
            return a;
        }
        if (stage == 1) {
            const V2 m = mix(cn.a1, cn.aa1);
            E2[lb] = V2{f.x + m.x, f.y + m.y};
        }
        return V2{a.x + e.x, a.y + e.y};
    };
    for (int e = tid; e < nel; e += 256) {
        const int c = e / nl, lev = e - c * nl;
        const long lb = slbase[c] + lev, b = sbase[c] + lev;
        const V2 dd = Tn[b + nl], dT = Tn[b + 2L * nl], d0 = sp0[b + nl], t0 = sp0[b + 2L * nl];
        V2 e1{T(0), T(0)}, e2 = e1, f1 = e1, f2 = e1;
        if (stage > 0) {
            e1 = Ep[lb];
            e2 = Ep[lb + nl];
        }
        if (stage == 1) {
            f1 = E2[lb];
            f2 = E2[lb + nl];
        }
        V2 ddl, dtl;
        ddl.x = -lap * (S2[lev][2 * c] + tors[lev] * lpin[2 * c]);
        ddl.y = -lap * (S2[lev][2 * c + 1] + tors[lev] * lpin[2 * c + 1]);
        dtl.x = -S3[lev][2 * c];
        dtl.y = -S3[lev][2 * c + 1];
        const V2 a1 = combine(lb, V2{dd.x - ddl.x, dd.y - ddl.y}, ddl, e1, f1);
        const V2 a2 = combine(lb + nl, V2{dT.x - dtl.x, dT.y - dtl.y}, dtl, e2, f2);
        S1[lev][2 * c] = d0.x + dt * a1.x;  // dvc
        S1[lev][2 * c + 1] = d0.y + dt * a1.y;
        S0[lev][2 * c] = t0.x + dt * a2.x;  // tvc
        S0[lev][2 * c + 1] = t0.y + dt * a2.y;
    }
    if (tid < cnt) {
        const long b = sbase[tid] + 3L * nl + (long)ntr * nl;
        const long lb = slbase[tid] + 2L * nl;
        const V2 l{-csum[2 * tid], -csum[2 * tid + 1]}, d = Tn[b], p0 = sp0[b];
        const V2 zero{T(0), T(0)}, pe = stage > 0 ? Ep[lb] : zero, pf = stage == 1 ? E2[lb] : zero;
        const V2 a3 = combine(lb, V2{d.x - l.x, d.y - l.y}, l, pe, pf);
        lpc[2 * tid] = p0.x + dt * a3.x;
        lpc[2 * tid + 1] = p0.y + dt * a3.y;
    }
    __syncthreads();
    if (do_implicit) {
        // rhs, solve with d_hyb_m(:,:,n+1,stage) and back-substitution (run.f90:344-349)
        op.load(At, nl, wave, lane);
        si_gemm<T>(op, nl, S0, S2, wave, lane);
        __syncthreads();
        const int nrow = si_rows(nl);
        for (int e = tid; e < nrow * W; e += 256) {
            const int lev = e / W, col = e - lev * W;
            S3[lev][col] = (lev < nl) ? S1[lev][col] - cimp * lap * dt * (S2[lev][col] + tors[lev] * lpc[col]) : T(0);
        }
        __syncthreads();
        op.load(Dt + ((long)stage * (ntrunc + 1) + n) * nl * nl, nl, wave, lane);
        si_gemm<T>(op, nl, S3, S2, wave, lane);
        __syncthreads();
        op.load(Bt, nl, wave, lane);
        si_gemm<T>(op, nl, S2, S3, wave, lane);
        si_colsum<T>(svs, nl, S2, csum);
        __syncthreads();
        for (int e = tid; e < nl * W; e += 256) {
            const int lev = e / W, col = e - lev * W;
            S0[lev][col] -= cimp * dt * S3[lev][col];
            S1[lev][col] = S2[lev][col];
        }
        if (tid < W) lpc[tid] -= cimp * dt * csum[tid];
        __syncthreads();
    }
    for (int e = tid; e < nel; e += 256) {
        const int c = e / nl, lev = e - c * nl;
        const long b = sbase[c] + lev;
        V2 dv = V2{S1[lev][2 * c], S1[lev][2 * c + 1]}, tv = V2{S0[lev][2 * c], S0[lev][2 * c + 1]};
        if (damp) {
            const T ds = disspec[sk[c]];
            const T fv = T(1) - (ds * diffp[lev] - dmpp[lev]) * dt, ft = T(1) - ds * diffp[lev] * dt;
            dv.x /= fv;
            dv.y /= fv;
            tv.x /= ft;
            tv.y /= ft;
        }
        sp[b + nl] = dv;
        sp[b + 2L * nl] = tv;
    }
    if (tid < cnt) sp[sbase[tid] + 3L * nl + (long)ntr * nl] = V2{lpc[2 * tid], lpc[2 * tid + 1]};
}

// time-split physics update (run.f90:526-538)
template <typename T>
__global__ void k_phys_update(cplx<T> *__restrict__ spec, const cplx<T> *__restrict__ tp, int nl, int ntr, int nfs,
                              int nm, int nlm, T dt, int massfix) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    long nfst = (long)nfs * nm;
    if (i >= nfst * nlm) return;
    int f = (int)(i % nfst) % nfs;
    cplx<T> s = spec[i], t = tp[i];
    if (f < 3 * nl + ntr * nl) {
        spec[i] = cplx<T>{s.x + dt * t.x, s.y + dt * t.y};
    } else if (massfix) {
        // dlnpsspecdt = (workspec - lnpsspec)/dt; lnpsspec += dt*dlnpsspecdt, where
        // workspec = analysis of the deviation field + q_00 (the global mean, k = 0)
        if (i < nfst) t.x += s.x;
        cplx<T> d{(t.x - s.x) / dt, (t.y - s.y) / dt};
        spec[i] = cplx<T>{s.x + dt * d.x, s.y + dt * d.y};
    }
}

template <typename T> __global__ void k_copy(T *__restrict__ dst, const T *__restrict__ src, long n) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    long stride = (long)gridDim.x * blockDim.x;
    for (; i < n; i += stride) dst[i] = src[i];
}

// The fields of a state, by name, in the reference layout [member][field][nlm],
// each null where it is left out; off[i] is field run i's first field in a
// member's state fields, off[5] their number.
struct PackParts {
    const void *p[5];
    int off[6];
};
// reference layout <-> state layout spec[k][member * nfs + f]: 64 coefficients x 32
// (FP64: 16) state fields of whatever runs a tile are transposed through LDS, so
// that both sides move in runs of 256 bytes. One launch takes a whole state: a
// launch per field run with one element a thread, a field apart in the state,
// took 6.2 us for 64 levels at T126 (23 us at T254) and wrote a copy of each run.
constexpr int PACK_K = 64;
template <typename T> constexpr int PACK_F = sizeof(T) == 4 ? 32 : 16;
template <typename T>
__global__ __launch_bounds__(256) void k_pack(cplx<T> *__restrict__ spec, PackParts pp, int nfs, int nm, int nlm,
                                              int to_state) {
    constexpr int F = PACK_F<T>;
    __shared__ cplx<T> buf[F][PACK_K + 1];
    __shared__ cplx<T> *row[F];  // the reference row of each state field of the tile
    const int tid = threadIdx.x, k0 = blockIdx.x * PACK_K, c0 = blockIdx.y * F, NFS = nfs * nm;
    if (tid < F) {
        cplx<T> *r = nullptr;
        if (c0 + tid < NFS) {
            const int mem = (c0 + tid) / nfs, f = c0 + tid - mem * nfs;
#pragma unroll
            for (int i = 0; i < 5; i++)
                if (f >= pp.off[i] && f < pp.off[i + 1] && pp.p[i])
                    r = (cplx<T> *)const_cast<void *>(pp.p[i]) +
                        ((long)mem * (pp.off[i + 1] - pp.off[i]) + f - pp.off[i]) * nlm;
        }
        row[tid] = r;
    }
    __syncthreads();
    const int kl = tid % PACK_K, fl = tid % F;
    if (to_state) {
        cplx<T> v[F / 4];
#pragma unroll
        for (int i = 0; i < F / 4; i++) {
            const cplx<T> *r = row[4 * i + tid / PACK_K];
            if (r && k0 + kl < nlm) v[i] = r[k0 + kl];
        }
#pragma unroll
        for (int i = 0; i < F / 4; i++) buf[4 * i + tid / PACK_K][kl] = v[i];
        __syncthreads();
        if (row[fl])
            for (int k = tid / F; k < PACK_K && k0 + k < nlm; k += 256 / F)
                spec[(long)(k0 + k) * NFS + c0 + fl] = buf[fl][k];
    } else {
        if (row[fl])
#pragma unroll
            for (int i = 0; i < PACK_K * F / 256; i++) {
                const int k = tid / F + i * (256 / F);
                buf[fl][k] = spec[(long)min(k0 + k, nlm - 1) * NFS + c0 + fl];
            }
        __syncthreads();
        if (k0 + kl < nlm)
            for (int f = tid / PACK_K; f < F; f += 4)
                if (row[f]) row[f][k0 + kl] = buf[f][kl];
    }
}

// grid fields of a member-major field set -> caller layout
template <typename T>
__global__ void k_grid_gather(const T *__restrict__ src, long mstride, T *__restrict__ dst, long per_mem, int nm) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= per_mem * nm) return;
    long mem = i / per_mem, r = i % per_mem;
    dst[i] = src[mem * mstride + r];
}

// init_semimpdata's implicit operators on the device, in FP64
// (semimp_data.f90:238-251): for stage s and degree n, d_hyb_m(:,:,n+1,s) =
// inv(I + (c_s dt)^2 n (n+1) ym), c = (aa22, aa33, bb4). One workgroup per
// (n, s) runs Gauss-Jordan elimination with partial pivoting (the first row of
// largest magnitude, as LAPACK's dgetrf pivots) on the matrix and an identity
// in LDS. ym, d: column-major nl x nl; d holds (T+1) x 3 matrices, stage-major.
constexpr int SI_LD = MAXLEV + 1;  // LDS row pitch (odd, against bank conflicts)
__global__ __launch_bounds__(256) void k_semimp_inverse(const double *__restrict__ ym, double c0, double c1,
                                                        double c2, int nl, int ntrunc, double *__restrict__ d,
                                                        int *__restrict__ fail) {
    __shared__ double a[MAXLEV][SI_LD], b[MAXLEV][SI_LD];
    __shared__ double fr[MAXLEV];
    __shared__ int piv;
    const int n = blockIdx.x, st = blockIdx.y, tid = threadIdx.x;
    const double c = st == 0 ? c0 : st == 1 ? c1 : c2, f = c * c * (double)n * (n + 1);
    for (int e = tid; e < nl * nl; e += blockDim.x) {
        const int r = e % nl, j = e / nl;
        a[r][j] = (r == j ? 1.0 : 0.0) + f * ym[r + (long)j * nl];
        b[r][j] = r == j ? 1.0 : 0.0;
    }
    __syncthreads();
    for (int col = 0; col < nl; col++) {
        if (tid < 64) {
            // first row of largest |a(r, col)|, r >= col: wavefront argmax, ties to the lower row
            double v = -1.0;
            int r = nl;
            if (col + tid < nl) {
                v = fabs(a[col + tid][col]);
                r = col + tid;
            }
            for (int o = 32; o > 0; o >>= 1) {
                const double v2 = __shfl_down(v, o);
                const int r2 = __shfl_down(r, o);
                if (v2 > v || (v2 == v && r2 < r)) {
                    v = v2;
                    r = r2;
                }
            }
            if (tid == 0) {
                piv = r;
                if (!(v > 0.0)) *fail = 1;
            }
        }
        __syncthreads();
        const int p = piv;
        if (p != col)
            for (int j = tid; j < nl; j += blockDim.x) {
                double t = a[col][j];
                a[col][j] = a[p][j];
                a[p][j] = t;
                t = b[col][j];
                b[col][j] = b[p][j];
                b[p][j] = t;
            }
        __syncthreads();
        const double inv = 1.0 / a[col][col];
        __syncthreads();
        for (int j = tid; j < nl; j += blockDim.x) {
            a[col][j] *= inv;
            b[col][j] *= inv;
        }
        for (int r = tid; r < nl; r += blockDim.x) fr[r] = a[r][col];
        __syncthreads();
        for (int e = tid; e < nl * nl; e += blockDim.x) {
            const int r = e / nl, j = e % nl;
            if (r == col) continue;
            const double fq = fr[r];
            a[r][j] -= fq * a[col][j];
            b[r][j] -= fq * b[col][j];
        }
        __syncthreads();
    }
    double *D = d + ((long)st * (ntrunc + 1) + n) * nl * nl;
    for (int e = tid; e < nl * nl; e += blockDim.x) {
        const int r = e % nl, j = e / nl;
        D[r + (long)j * nl] = b[r][j];
    }
}

// solver operator layout: per (stage, degree) matrix, transposed and at precision T
template <typename T>
__global__ void k_semimp_pack(const double *__restrict__ d, T *__restrict__ dt3, int nl, long nmat) {
    const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= nmat * nl * nl) return;
    const long b = e / (nl * nl);
    const int q = (int)(e % (nl * nl)), i = q % nl, j = q / nl;
    dt3[b * nl * nl + (long)j * nl + i] = (T)d[b * nl * nl + i + (long)j * nl];
}

// ---------------------------------------------------------------------------
// host side

// gaussian_spect (patterngenerator.f90:145-177): sqrt(T exp(L^2 lap / 4a^2)),
// normalised so that the deterministic reference noise has unit variance
static std::vector<double> pattern_varspec(int T_, double L, double a) {
    std::vector<double> var((size_t)(T_ + 1) * (T_ + 2) / 2);
    const double twopi = 2.0 * M_PI;
    double v = 0.0;
    for (int m = 0, k = 0; m <= T_; m++)
        for (int n = m; n <= T_; n++, k++) {
            var[k] = std::sqrt(T_ * std::exp(L * L * (-(double)n * (n + 1.0)) / (4.0 * a * a)));
            double nz2 = (k == 0) ? 0.0 : 2.0 / (2.0 * n + 1.0) * (twopi / T_);
            v += (m != 0 ? 1.0 : 0.5) * var[k] * var[k] * nz2;
        }
    v /= twopi;
    for (double &x : var) x /= std::sqrt(v);
    return var;
}

template <typename T> static T *dalloc(size_t n) {
    T *p = nullptr;
    if (hipMalloc((void **)&p, sizeof(T) * (n ? n : 1)) != hipSuccess) return nullptr;
    return p;
}

template <typename T> static int dupload(void **d, const std::vector<T> &h, hipStream_t s) {
    *d = dalloc<T>(h.size());
    if (!*d) {
        set_error("device allocation failed");
        return GFSDC_ENOMEM;
    }
    GFSDC_CHECK(hipMemcpyAsync(*d, h.data(), sizeof(T) * h.size(), hipMemcpyHostToDevice, s));
    return 0;
}

template <typename T> static std::vector<T> castv(const std::vector<double> &v) {
    return std::vector<T>(v.begin(), v.end());
}

uint64_t rng_u64(uint64_t seed, uint64_t stream, uint64_t index) { return rng_mix(seed, stream, index); }

template <typename T> int Engine<T>::dyn_init() {
    const int nl = cfg.nlev, ntr = cfg.ntrac, nm = cfg.nmem, T_ = plan.ntrunc, nlm = plan.nlm;
    if (nl < 2 || nl > MAXLEV) {
        set_error("nlev must be in [2, 64]");
        return GFSDC_EINVAL;
    }
    if (ntr < 0) {
        set_error("ntrac must be >= 0");
        return GFSDC_EINVAL;
    }
    if (cfg.physics != GFSDC_PHYS_NONE && cfg.physics != GFSDC_PHYS_HS && cfg.physics != GFSDC_PHYS_SIMPLE) {
        set_error("physics must be GFSDC_PHYS_NONE, GFSDC_PHYS_HS or GFSDC_PHYS_SIMPLE");
        return GFSDC_EINVAL;
    }
    if (cfg.physics == GFSDC_PHYS_SIMPLE && ntr < 1) {
        set_error("simple moist physics needs ntrac >= 1 (tracer 1 is specific humidity)");
        return GFSDC_EINVAL;
    }
    if (cfg.simple_test < 0 || cfg.simple_test > 2) {
        set_error("simple_test must be 0, 1 or 2");
        return GFSDC_EINVAL;
    }
    DycoreBuffers *B = new DycoreBuffers();
    dyn = B;
    B->nl = nl;
    B->ntr = ntr;
    B->nm = nm;
    B->nfs = 3 * nl + ntr * nl + 1;
    B->nsyn = 7 * nl + 3 * ntr * nl + 3;
    B->nan = 4 * nl + 1 + ntr * nl;
    B->nhs = 3 * nl + 1;
    B->nsp = 4 * nl + 1;
    B->ng = (long)plan.nlat * plan.nlon;
    const long ng = B->ng, NFS = (long)B->nfs * nm;
    // ---- one-off operators in FP64 on the host (semimp_data.f90:127-256, dyn_init.f90:450-494)
    const double rd = cfg.rd, kappa = cfg.rd / cfg.cp, rerth = cfg.rerth;
    std::vector<double> dbk(nl), ck(nl), si(nl + 1);
    B->sl.resize(nl);
    for (int k = 1; k <= nl; k++) {
        dbk[k - 1] = bk[k] - bk[k - 1];
        ck[k - 1] = ak[k] * bk[k - 1] - ak[k - 1] * bk[k];
    }
    for (int k = 1; k <= nl + 1; k++) si[nl + 1 - k] = ak[k - 1] / SGLF(101300.0) + bk[k - 1];
    for (int k = 0; k < nl; k++) B->sl[k] = 0.5 * (si[k] + si[k + 1]);
    {
        const double tref = 300.0, pref = 800.e2;
        std::vector<double> pkref(nl + 1), dpkref(nl), alfaref(nl), yecm(nl * nl, 0.0), tecm(nl * nl, 0.0);
        for (int k = 0; k <= nl; k++) pkref[k] = ak[k] + bk[k] * pref;
        for (int k = 0; k < nl; k++) dpkref[k] = pkref[k + 1] - pkref[k];
        alfaref[0] = SGLF(0.69314718055994530942);
        for (int k = 2; k <= nl; k++)
            alfaref[k - 1] = 1.0 - (pkref[k - 1] / dpkref[k - 1]) * std::log(pkref[k] / pkref[k - 1]);
#define CM(A, i, j) A[((i) - 1) + (size_t)((j) - 1) * nl]
        for (int ir = 1; ir <= nl; ir++) {
            CM(yecm, ir, ir) = alfaref[ir - 1] * rd;
            for (int ic = ir + 1; ic <= nl; ic++) CM(yecm, ir, ic) = rd * std::log(pkref[ic] / pkref[ic - 1]);
            CM(tecm, ir, ir) = kappa * tref * alfaref[ir - 1];
            for (int ic = 1; ic <= ir - 1; ic++)
                CM(tecm, ir, ic) = (kappa * tref * dpkref[ic - 1] / dpkref[ir - 1]) * std::log(pkref[ir] / pkref[ir - 1]);
        }
        B->amhyb.assign(nl * nl, 0.0);
        B->bmhyb.assign(nl * nl, 0.0);
        B->svhyb.assign(nl, 0.0);
        B->tor_hyb.assign(nl, rd * tref / (rerth * rerth));
        for (int j = 1; j <= nl; j++) {
            B->svhyb[j - 1] = dpkref[nl - j] / pref;
            for (int k = 1; k <= nl; k++) {
                CM(B->amhyb, k, j) = CM(yecm, nl + 1 - k, nl + 1 - j) / (rerth * rerth);
                CM(B->bmhyb, k, j) = CM(tecm, nl + 1 - k, nl + 1 - j);
            }
        }
        std::vector<double> ym(nl * nl);
        for (int i = 1; i <= nl; i++)
            for (int j = 1; j <= nl; j++) {
                double s = B->tor_hyb[i - 1] * B->svhyb[j - 1];
                for (int k = 1; k <= nl; k++) s += CM(B->amhyb, i, k) * CM(B->bmhyb, k, j);
                CM(ym, i, j) = s;
            }
        B->ym = ym;
#undef CM
    }
    {  // setdampspec
        int ndiss = cfg.ndiss == 0 ? 8 : cfg.ndiss;
        double efold = cfg.efold, fshk = cfg.fshk, hf2 = cfg.hdif_fac2, hf = cfg.hdif_fac;
        if (efold <= 0) {
            if (T_ > 170)
                efold = 3600. / (hf2 * SGLF(std::pow((float)T_ / 170.f, 4)) * SGLF(1.1));
            else if (T_ == 126 || T_ == 170)
                efold = 1. / (hf2 * SGLF(12.E15) / std::pow(rerth, 4) * SGLF(80. * 81.) * SGLF(80. * 81.));
            else
                efold = 1. / (hf2 * SGLF(3.E15) / std::pow(rerth, 4) * SGLF(80. * 81.) * SGLF(80. * 81.));
            efold = 2. * efold;
        }
        if (fshk <= 0) {
            fshk = 1.0 * hf;
            if (T_ > 170) fshk = SGLF(2.2) * hf;
            if (T_ == 126) fshk = SGLF(1.5) * hf;
        }
        double slrd0 = SGLF(0.002), dmp1 = 1. / cfg.taustratdamp;
        B->diff_h.resize(nl);
        B->dmp_h.resize(nl);
        for (int k = 0; k < nl; k++) {
            B->dmp_h[k] = 0.0;
            B->diff_h[k] = std::pow(B->sl[k], std::log(1. / fshk));
            if (B->sl[k] < slrd0) B->dmp_h[k] = dmp1 * std::log(slrd0 / B->sl[k]);
        }
        B->disspec_h.resize(nlm);
        double minlap = -(double)T_ * (T_ + 1);
        int k = 0;
        for (int m = 0; m <= T_; m++)
            for (int n = m; n <= T_; n++, k++) {
                double r = (-(double)n * (n + 1)) / minlap, p = 1.0;
                for (int i = 0; i < ndiss / 2; i++) p *= r;
                B->disspec_h[k] = -(1. / efold) * p;
            }
    }
    // ---- device operators (transposed for the per-lane matvec)
    auto transp = [&](const std::vector<double> &cm, size_t off) {
        std::vector<T> t(nl * nl);
        for (int i = 0; i < nl; i++)
            for (int j = 0; j < nl; j++) t[j * nl + i] = (T)cm[off + i + (size_t)j * nl];
        return t;
    };
    int rc;
    if ((rc = dupload<T>(&B->at, transp(B->amhyb, 0), stream))) return rc;
    if ((rc = dupload<T>(&B->bt, transp(B->bmhyb, 0), stream))) return rc;
    {
        // the implicit operators, inverted in FP64 on the device (k_semimp_inverse),
        // then packed for the solver at precision T; the FP64 matrices are kept
        // on the host for gfsdc_get_semimp
        const size_t nmat = (size_t)(T_ + 1) * 3, nd = nmat * nl * nl;
        double *dym = nullptr, *dd = nullptr;
        int *dfail = nullptr;
        if ((rc = dupload<double>((void **)&dym, B->ym, stream))) return rc;
        dd = dalloc<double>(nd);
        dfail = dalloc<int>(1);
        B->dt3 = dalloc<T>(nd);
        if (!dd || !dfail || !B->dt3) {
            set_error("device allocation failed");
            return GFSDC_ENOMEM;
        }
        GFSDC_CHECK(hipMemsetAsync(dfail, 0, sizeof(int), stream));
        const double dt = cfg.dt;
        hipLaunchKernelGGL(k_semimp_inverse, dim3(T_ + 1, 3), dim3(256), 0, stream, dym, TAB_IMP[0] * dt,
                           TAB_IMP[1] * dt, TAB_IMP[2] * dt, nl, T_, dd, dfail);
        hipLaunchKernelGGL(k_semimp_pack<T>, dim3((unsigned)((nd + 255) / 256)), dim3(256), 0, stream,
                           (const double *)dd, (T *)B->dt3, nl, (long)nmat);
        GFSDC_CHECK(hipGetLastError());
        int fail = 0;
        B->d_hyb_m.resize(nd);
        GFSDC_CHECK(hipMemcpyAsync(B->d_hyb_m.data(), dd, sizeof(double) * nd, hipMemcpyDeviceToHost, stream));
        GFSDC_CHECK(hipMemcpyAsync(&fail, dfail, sizeof(int), hipMemcpyDeviceToHost, stream));
        GFSDC_CHECK(hipStreamSynchronize(stream));
        (void)hipFree(dym);
        (void)hipFree(dd);
        (void)hipFree(dfail);
        if (fail) {
            set_error("singular semi-implicit matrix");
            return GFSDC_EINVAL;
        }
    }
    if ((rc = dupload<T>(&B->sv, castv<T>(B->svhyb), stream))) return rc;
    if ((rc = dupload<T>(&B->tor, castv<T>(B->tor_hyb), stream))) return rc;
    if ((rc = dupload<T>(&B->disspec, castv<T>(B->disspec_h), stream))) return rc;
    if ((rc = dupload<T>(&B->diffp, castv<T>(B->diff_h), stream))) return rc;
    if ((rc = dupload<T>(&B->dmpp, castv<T>(B->dmp_h), stream))) return rc;
    if ((rc = dupload<T>(&B->ak, castv<T>(ak), stream))) return rc;
    if ((rc = dupload<T>(&B->bk, castv<T>(bk), stream))) return rc;
    if ((rc = dupload<T>(&B->ck, castv<T>(ck), stream))) return rc;
    if ((rc = dupload<T>(&B->dbk, castv<T>(dbk), stream))) return rc;
    {
        std::vector<double> dak(nl);
        for (int k = 0; k < nl; k++) dak[k] = ak[k + 1] - ak[k];
        if ((rc = dupload<T>(&B->dak, castv<T>(dak), stream))) return rc;
    }
    {
        std::vector<double> sl(plan.nlat), area(plan.nlat);
        double tot = 0;
        for (int j = 0; j < plan.nlat; j++) tot += plan.w[j] * plan.nlon;
        for (int j = 0; j < plan.nlat; j++) {
            sl[j] = plan.mu[j];  // sin(lat) = cos(colatitude)
            area[j] = plan.w[j] / tot;
        }
        if ((rc = dupload<T>(&B->sinlat, castv<T>(sl), stream))) return rc;
        if ((rc = dupload<double>(&B->areaw, area, stream))) return rc;
        std::vector<double> la(plan.nlat);
        for (int j = 0; j < plan.nlat; j++) la[j] = std::asin(plan.mu[j]);  // shtns.f90:127
        void *p;
        if ((rc = dupload<double>(&p, la, stream))) return rc;
        B->latd = (double *)p;
    }
    {
        std::vector<int> deg(nlm);
        int k = 0;
        for (int m = 0; m <= T_; m++)
            for (int n = m; n <= T_; n++) deg[k++] = n;
        void *p;
        if ((rc = dupload<int>(&p, deg, stream))) return rc;
        B->degree = (int *)p;
        std::vector<int2> tiles;
        for (int n = 0; n <= T_; n++)
            for (int i0 = 0; i0 < (n + 1) * nm; i0 += SiCfg<T>::C) tiles.push_back(make_int2(n, i0));
        if ((rc = dupload<int2>(&p, tiles, stream))) return rc;
        B->si_tiles = (int2 *)p;
        B->n_si_tiles = (int)tiles.size();
    }
    // ---- state and work buffers
    size_t nspec = (size_t)nlm * NFS;
    B->spec = dalloc<cplx<T>>(nspec);
    B->spec0 = dalloc<cplx<T>>(nspec);
    for (int s = 0; s < 3; s++) B->ten[s] = dalloc<cplx<T>>(nspec);
    if (!cfg.explicit_)
        for (int s = 0; s < 2; s++) B->mix[s] = dalloc<cplx<T>>((size_t)nlm * nm * (2 * nl + 1));
    B->tphys = dalloc<cplx<T>>(nspec);
    B->topo = dalloc<cplx<T>>((size_t)nlm * nm);
    B->gsyn = dalloc<T>((size_t)nm * B->nsyn * ng);
    B->gmean = dalloc<T>((size_t)nm * B->nsyn);
    B->gan = dalloc<T>((size_t)nm * B->nan * ng);
    B->etadot = dalloc<T>((size_t)nm * (nl + 1) * ng);
    B->dlnpdt = dalloc<T>((size_t)nm * nl * ng);
    B->psg = dalloc<T>((size_t)nm * ng);
    B->dlnpsdt = dalloc<T>((size_t)nm * ng);
    B->dphisdx = dalloc<T>((size_t)nm * ng);
    B->dphisdy = dalloc<T>((size_t)nm * ng);
    B->pdryini = dalloc<double>(nm);
    B->pmean = dalloc<double>(nm);
    B->pspart = dalloc<double>((size_t)nm * PS_BLOCKS * 4);
    B->psdone = dalloc<unsigned>(nm + 1);
    B->pwsum = dalloc<double>(nm);
    B->diag = dalloc<double>(4 * nm);
    B->clock = dalloc<double>(1);
    B->colq = dalloc<T>((size_t)nm * ng);
    B->pwat = dalloc<T>((size_t)nm * ng);
    B->precip = dalloc<T>((size_t)nm * ng);
    B->hsdyn = dalloc<int>(8);
    if (!cfg.explicit_ && (!B->mix[0] || !B->mix[1])) {
        set_error("device allocation failed for the dycore state");
        return GFSDC_ENOMEM;
    }
    void *ptrs[] = {B->spec, B->spec0, B->ten[0], B->ten[1], B->ten[2],
                    B->tphys, B->topo, B->gsyn, B->gan, B->etadot, B->dlnpdt, B->psg, B->dlnpsdt, B->dphisdx,
                    B->dphisdy, B->pdryini, B->pmean, B->diag, B->pspart, B->psdone, B->pwsum, B->colq, B->pwat,
                    B->precip, B->gmean, B->clock, B->hsdyn};
    for (void *p : ptrs)
        if (!p) {
            set_error("device allocation failed for the dycore state");
            return GFSDC_ENOMEM;
        }
    GFSDC_CHECK(hipMemsetAsync(B->spec, 0, sizeof(cplx<T>) * nspec, stream));
    GFSDC_CHECK(hipMemsetAsync(B->topo, 0, sizeof(cplx<T>) * nlm * nm, stream));
    GFSDC_CHECK(hipMemsetAsync(B->dphisdx, 0, sizeof(T) * nm * ng, stream));
    GFSDC_CHECK(hipMemsetAsync(B->dphisdy, 0, sizeof(T) * nm * ng, stream));
    GFSDC_CHECK(hipMemsetAsync(B->pdryini, 0, sizeof(double) * nm, stream));
    GFSDC_CHECK(hipMemsetAsync(B->clock, 0, sizeof(double), stream));
    GFSDC_CHECK(hipMemsetAsync(B->pwat, 0, sizeof(T) * nm * ng, stream));
    GFSDC_CHECK(hipMemsetAsync(B->precip, 0, sizeof(T) * nm * ng, stream));
    GFSDC_CHECK(hipMemsetAsync(B->pwsum, 0, sizeof(double) * nm, stream));
    GFSDC_CHECK(hipMemsetAsync(B->gmean, 0, sizeof(T) * nm * B->nsyn, stream));
    GFSDC_CHECK(hipMemsetAsync(B->hsdyn, 0, sizeof(int) * 8, stream));
    GFSDC_CHECK(hipMemsetAsync(B->psdone, 0, sizeof(unsigned) * (nm + 1), stream));
    Work<T> *W = new Work<T>();
    B->Work = W;
    if ((rc = work_alloc(*W, plan, nm * std::max(B->nsyn, B->nan)))) return rc;
    // ---- AR(1) temperature pattern (patterngenerator.f90:33-177, stoch_data.f90 spin-up)
    if (cfg.tpat_amp > 0) {
        if (!(cfg.tpat_tau > 0) || cfg.tpat_lscale < 0) {
            set_error("tpat_tau must be > 0 and tpat_lscale >= 0 when tpat_amp > 0");
            return GFSDC_EINVAL;
        }
        std::vector<double> var = pattern_varspec(T_, cfg.tpat_lscale, cfg.rerth), vf(nl);
        for (int k = 0; k < nl; k++) {
            const double sl = B->sl[k];
            vf[k] = 1.0;
            if (sl < 0.10 && sl > 0.05) vf[k] = (sl - 0.05) / (0.10 - 0.05);
            else if (sl <= 0.05) vf[k] = 0.0;
        }
        void *p;
        if ((rc = dupload<double>(&p, var, stream))) return rc;
        B->tpat_var = (double *)p;
        if ((rc = dupload<T>(&B->tpat_vf, castv<T>(vf), stream))) return rc;
        B->tpat = dalloc<cplx<T>>((size_t)nm * nlm);
        B->tpat_ctr = dalloc<unsigned long long>(1);
        if (!B->tpat || !B->tpat_ctr) {
            set_error("device allocation failed for the pattern");
            return GFSDC_ENOMEM;
        }
        GFSDC_CHECK(hipMemsetAsync(B->tpat, 0, sizeof(cplx<T>) * nm * nlm, stream));
        GFSDC_CHECK(hipMemsetAsync(B->tpat_ctr, 0, sizeof(unsigned long long), stream));
        B->tpat_phi = std::exp(-cfg.dt / cfg.tpat_tau);
        if ((rc = pattern_spinup())) return rc;
    }
    // ---- descriptors
    std::vector<SynthDesc> sd((size_t)nm * B->nsyn);
    std::vector<unsigned char> rs((size_t)nm * B->nsyn, 0), ra((size_t)nm * B->nan, 0), rh((size_t)nm * B->nan, 0);
    std::vector<AnalDesc> ad((size_t)nm * B->nfs), ah((size_t)nm * B->nfs), ap((size_t)nm * B->nfs);
    std::vector<AnalDesc> au((size_t)nm * B->nfs);
    std::vector<unsigned char> rp((size_t)nm * B->nsp, 0);
    const AnalDesc zero{AK_ZERO, -1, -1, 0.0, 0, 0, -1, 0.0};
    const double a = rerth, ra_ = 1.0 / rerth;
    for (int mem = 0; mem < nm; mem++) {
        SynthDesc *d = &sd[(size_t)mem * B->nsyn];
        unsigned char *r = &rs[(size_t)mem * B->nsyn];
        int s0 = mem * B->nfs;  // source field base of the member
        int vrt = s0, div = s0 + nl, tv = s0 + 2 * nl, tr = s0 + 3 * nl, lp = s0 + 3 * nl + ntr * nl;
        for (int k = 0; k < nl; k++) {
            d[k] = SynthDesc{SK_UHAT, vrt + k, div + k, a, a, 1, 1};           // ug (getuv)
            d[nl + k] = SynthDesc{SK_VHAT, vrt + k, div + k, a, a, 1, 1};      // vg
            d[2 * nl + k] = SynthDesc{SK_COPY, vrt + k, -1, 1.0, 0.0, 0, 0};   // vrtg
            d[3 * nl + k] = SynthDesc{SK_COPY, div + k, -1, 1.0, 0.0, 0, 0};   // divg
            d[4 * nl + k] = SynthDesc{SK_COPY_MEAN, tv + k, -1, 1.0, 0.0, 0, 0};  // virtempg
            d[5 * nl + k] = SynthDesc{SK_UHAT, -1, tv + k, 0.0, ra_, 0, 0};    // dvirtempdx (getgrad)
            d[6 * nl + k] = SynthDesc{SK_VHAT, -1, tv + k, 0.0, ra_, 0, 0};    // dvirtempdy
            r[k] = r[nl + k] = r[5 * nl + k] = r[6 * nl + k] = 1;
        }
        for (int k = 0; k < ntr * nl; k++) {
            d[7 * nl + k] = SynthDesc{SK_COPY, tr + k, -1, 1.0, 0.0, 0, 0};                   // tracerg
            d[7 * nl + ntr * nl + k] = SynthDesc{SK_UHAT, -1, tr + k, 0.0, ra_, 0, 0};       // dq/dx (getgrad)
            d[7 * nl + 2 * ntr * nl + k] = SynthDesc{SK_VHAT, -1, tr + k, 0.0, ra_, 0, 0};   // dq/dy
            r[7 * nl + ntr * nl + k] = r[7 * nl + 2 * ntr * nl + k] = 1;
        }
        int o = 7 * nl + 3 * ntr * nl;
        d[o] = SynthDesc{SK_COPY_DEV, lp, -1, 1.0, 0.0, 0, 0};  // lnpsg minus its global mean
        d[o + 1] = SynthDesc{SK_UHAT, -1, lp, 0.0, ra_, 0, 0};  // dlnpsdx
        d[o + 2] = SynthDesc{SK_VHAT, -1, lp, 0.0, ra_, 0, 0};  // dlnpsdy
        r[o + 1] = r[o + 2] = 1;
        // analysis: grid fields of the member (Tten, Fx, Fy, KE, dlnpsdt, dq) -> tendencies
        int g0 = mem * B->nan;
        AnalDesc *e = &ad[(size_t)mem * B->nfs];
        AnalDesc *hh = &ah[(size_t)mem * B->nfs];
        for (int k = 0; k < nl; k++) {
            // dyn_run.f90:250-252,268-271: getvrtdivspec(Fx,Fy,ddiv,dvrt); dvrt = -dvrt; ddiv -= lap/a^2 KE
            e[k] = AnalDesc{AK_DIV, g0 + nl + k, g0 + 2 * nl + k, -1.0, 0, 0, -1, 0.0};
            e[nl + k] = AnalDesc{AK_VRT, g0 + nl + k, g0 + 2 * nl + k, 1.0, 0, 0, g0 + 3 * nl + k,
                                 1.0 / (rerth * rerth)};
            e[2 * nl + k] = AnalDesc{AK_COPY, g0 + k, -1, 1.0, 0, 0, -1, 0.0};
            ra[g0 + nl + k] = ra[g0 + 2 * nl + k] = 1;
            // Held-Suarez forcing fields (hs_field): T forcing, vrt force, div force
            hh[k] = AnalDesc{AK_COPY, hs_field(nl, nm, mem, HS_VRT, k), -1, 1.0, 0, 0, -1, 0.0};
            hh[nl + k] = AnalDesc{AK_COPY, hs_field(nl, nm, mem, HS_DIV, k), -1, 1.0, 0, 0, -1, 0.0};
            hh[2 * nl + k] = AnalDesc{AK_COPY, hs_field(nl, nm, mem, HS_T, k), -1, 1.0, 0, 0, -1, 0.0};
        }
        for (int k = 0; k < ntr * nl; k++) {
            e[3 * nl + k] = AnalDesc{AK_COPY, g0 + 4 * nl + 1 + k, -1, 1.0, 0, 0, -1, 0.0};
            hh[3 * nl + k] = zero;  // Held-Suarez leaves tracers unchanged
        }
        e[3 * nl + ntr * nl] = AnalDesc{AK_COPY, g0 + 4 * nl, -1, 1.0, 0, 0, -1, 0.0};
        hh[3 * nl + ntr * nl] =
            cfg.massfix ? AnalDesc{AK_COPY, hs_field(nl, nm, mem, HS_T, nl), -1, 1.0, 0, 0, -1, 0.0} : zero;
        // the same outputs applied in place (run.f90:527-538): vrt, div, tv += dt
        // tendency, tracers unchanged, ln ps through the mass fixer
        AnalDesc *uu = &au[(size_t)mem * B->nfs];
        const AnalDesc keep{AK_ZERO, -1, -1, 0.0, 0, 1, -1, 0.0};
        for (int f = 0; f < B->nfs; f++) {
            uu[f] = hh[f].kind == AK_COPY ? hh[f] : keep;
            uu[f].scale = cfg.dt;
            uu[f].accum = 1;
        }
        if (cfg.massfix) uu[3 * nl + ntr * nl].kind = AK_MASSFIX;
        // simple physics (phy_run_simple.f90:160-171): grid changes / dt ->
        // tv, (vrt, div) = getvrtdivspec(du, dv), tracer 1; mass-fixer field
        int p0 = mem * B->nsp;
        AnalDesc *pp = &ap[(size_t)mem * B->nfs];
        const double rdt = 1.0 / cfg.dt;
        for (int k = 0; k < nl; k++) {
            pp[k] = AnalDesc{AK_VRT, p0 + nl + k, p0 + 2 * nl + k, rdt, 0, 0, -1, 0.0};
            pp[nl + k] = AnalDesc{AK_DIV, p0 + nl + k, p0 + 2 * nl + k, rdt, 0, 0, -1, 0.0};
            pp[2 * nl + k] = AnalDesc{AK_COPY, p0 + k, -1, rdt, 0, 0, -1, 0.0};
            rp[p0 + nl + k] = rp[p0 + 2 * nl + k] = 1;
        }
        for (int k = 0; k < ntr * nl; k++)
            pp[3 * nl + k] = k < nl ? AnalDesc{AK_COPY, p0 + 3 * nl + k, -1, rdt, 0, 0, -1, 0.0} : zero;
        pp[3 * nl + ntr * nl] = cfg.massfix ? AnalDesc{AK_COPY, p0 + 4 * nl, -1, 1.0, 0, 0, -1, 0.0} : zero;
    }
    {
        // grid fields the physics pass needs: u, v, vrt, div, tv (0..5nl), the
        // tracers (7nl..7nl+ntr nl) and ln ps with its gradient (last 3)
        // (member, grid field) pairs in transform order
        std::vector<std::pair<int, int>> keep, lean_a, lean_b;
        for (int mem = 0; mem < nm; mem++) {
            for (int f = 0; f < 5 * nl; f++) keep.push_back({mem, f});
            for (int f = 7 * nl; f < 7 * nl + ntr * nl; f++) keep.push_back({mem, f});
            for (int f = 7 * nl + 3 * ntr * nl; f < B->nsyn; f++) keep.push_back({mem, f});
            // the lean Held-Suarez pass: temperature (4nl..5nl) and ln ps, then
            for (int k = 0; k < nl; k++) lean_a.push_back({mem, 4 * nl + k});
            lean_a.push_back({mem, 7 * nl + 3 * ntr * nl});
        }
        // vorticity (2nl..3nl) and divergence (3nl..4nl) level-major from the lowest level
        for (int k = 0; k < nl; k++)
            for (int mem = 0; mem < nm; mem++) {
                lean_b.push_back({mem, 2 * nl + k});
                lean_b.push_back({mem, 3 * nl + k});
            }
        B->nph = (int)keep.size() / nm;
        B->nhla = (int)lean_a.size();
        B->nhlb = (int)lean_b.size();
        auto upload_subset = [&](const std::vector<std::pair<int, int>> &fs, SynthDesc **d, unsigned char **r,
                                 int **sl) {
            std::vector<SynthDesc> dsub;
            std::vector<unsigned char> rsub;
            std::vector<int> ssub;
            for (auto [mem, f] : fs) {
                dsub.push_back(sd[(size_t)mem * B->nsyn + f]);
                rsub.push_back(rs[(size_t)mem * B->nsyn + f]);
                ssub.push_back(mem * B->nsyn + f);
            }
            void *q;
            int e;
            if ((e = dupload<SynthDesc>(&q, dsub, stream))) return e;
            *d = (SynthDesc *)q;
            if ((e = dupload<unsigned char>(&q, rsub, stream))) return e;
            *r = (unsigned char *)q;
            if ((e = dupload<int>(&q, ssub, stream))) return e;
            *sl = (int *)q;
            return 0;
        };
        if ((rc = upload_subset(keep, &B->sdesc_ph, &B->rflag_ph, &B->slot_ph))) return rc;
        std::vector<std::pair<int, int>> lean = lean_a;
        lean.insert(lean.end(), lean_b.begin(), lean_b.end());
        if ((rc = upload_subset(lean, &B->sdesc_hl, &B->rflag_hl, &B->slot_hl))) return rc;
        // the first lean pass takes every level
        const int c0[8] = {0, 0, 0, B->nhla + B->nhlb, nl, 0, 0, 0};
        GFSDC_CHECK(hipMemcpyAsync(B->hsdyn, c0, sizeof(c0), hipMemcpyHostToDevice, stream));
        GFSDC_CHECK(hipStreamSynchronize(stream));
    }
    // the dynamics synthesis' Legendre fields and the map of its grid fields onto
    // them: runs of grid slots (u..tv, dtv/dx, dtv/dy, q, dq/dx, dq/dy, ln ps,
    // dlnps/dx, dlnps/dy) and the Legendre field each run starts at
    std::vector<SynthDesc> sdl;
    {
        const int T3 = ntr * nl, o = 7 * nl + 3 * T3, lo = 6 * nl + 2 * T3;
        const int st[9] = {0, 5 * nl, 6 * nl, 7 * nl, 7 * nl + T3, 7 * nl + 2 * T3, o, o + 1, o + 2};
        const int sr[9] = {0, 4 * nl, 5 * nl, 6 * nl, 6 * nl, 6 * nl + T3, lo, lo, lo + 1};
        const unsigned dxm = (1u << 1) | (1u << 4) | (1u << 7);
        FieldMap &M = B->fmap_dyn;
        M.nseg = 9;
        M.per_dst = B->nsyn;
        M.per_src = B->nleg = B->nsyn - nl - T3 - 1;
        M.dx = dxm;
        for (int i = 0; i < 9; i++) {
            M.start[i] = st[i];
            M.src[i] = sr[i];
        }
        fmap_set_divisor(M);
        if ((unsigned long long)nm * B->nsyn * B->nsyn >= ((unsigned long long)1 << 32)) {
            set_error("internal: dynamics synthesis map size");
            return GFSDC_EINVAL;
        }
        for (int mem = 0; mem < nm; mem++)
            for (int f = 0; f < B->nsyn; f++) {
                bool dx;
                const int l = fmap_field(M, mem * B->nsyn + f, dx) - mem * B->nleg;
                if (!dx) {
                    if (l != (int)sdl.size() - mem * B->nleg) {
                        set_error("internal: dynamics synthesis map");
                        return GFSDC_EINVAL;
                    }
                    sdl.push_back(sd[(size_t)mem * B->nsyn + f]);
                }
            }
        // every x-gradient is i m / a times the Legendre field of its own scalar
        for (int mem = 0; mem < nm; mem++)
            for (int f = 0; f < B->nsyn; f++) {
                bool dx;
                const int l = fmap_field(M, mem * B->nsyn + f, dx);
                const SynthDesc &g = sd[(size_t)mem * B->nsyn + f];
                if (dx && (g.kind != SK_UHAT || g.a >= 0 || g.sb != ra_ || g.inv_b || sdl[l].a != g.b ||
                           (sdl[l].kind != SK_COPY && sdl[l].kind != SK_COPY_DEV && sdl[l].kind != SK_COPY_MEAN))) {
                    set_error("internal: dynamics synthesis x-gradients");
                    return GFSDC_EINVAL;
                }
            }
    }
    void *p;
    if ((rc = dupload<SynthDesc>(&p, sdl, stream))) return rc;
    B->sdesc = (SynthDesc *)p;
    if ((rc = dupload<AnalDesc>(&p, ad, stream))) return rc;
    B->adesc_dyn = (AnalDesc *)p;
    if ((rc = dupload<AnalDesc>(&p, ah, stream))) return rc;
    B->adesc_hs = (AnalDesc *)p;
    if ((rc = dupload<AnalDesc>(&p, au, stream))) return rc;
    B->adesc_hsu = (AnalDesc *)p;
    if ((rc = dupload<AnalDesc>(&p, ap, stream))) return rc;
    B->adesc_sp = (AnalDesc *)p;
    if ((rc = dupload<unsigned char>(&p, rp, stream))) return rc;
    B->rflag_sp = (unsigned char *)p;
    if ((rc = dupload<unsigned char>(&p, rs, stream))) return rc;
    B->rflag_syn = (unsigned char *)p;
    if ((rc = dupload<unsigned char>(&p, ra, stream))) return rc;
    B->rflag_an = (unsigned char *)p;
    if ((rc = dupload<unsigned char>(&p, rh, stream))) return rc;
    B->rflag_hs = (unsigned char *)p;
    GFSDC_CHECK(hipStreamSynchronize(stream));
    return 0;
}

template <typename T> void Engine<T>::dyn_destroy() {
    DycoreBuffers *B = dyn;
    if (!B) return;
    drop_graph(B);
    for (auto e : B->ev) (void)hipEventDestroy(e);
    void *ptrs[] = {B->spec, B->spec0, B->ten[0], B->ten[1], B->ten[2], B->mix[0], B->mix[1],
                    B->tphys, B->gsyn, B->gan, B->etadot, B->dlnpdt, B->psg, B->dlnpsdt, B->dphisdx,
                    B->dphisdy, B->topo, B->at, B->bt, B->dt3, B->sv, B->tor, B->disspec, B->diffp, B->dmpp,
                    B->ak, B->bk, B->ck, B->dbk, B->sinlat, B->coslat, B->areaw, B->degree, B->si_tiles,
                    B->pdryini, B->pmean, B->pspart, B->psdone, B->diag, B->sdesc, B->adesc_dyn, B->adesc_hs, B->adesc_hsu,
                    B->rflag_syn,
                    B->rflag_an, B->rflag_hs, B->pwsum, B->colq, B->pwat, B->precip, B->latd,
                    B->adesc_sp, B->rflag_sp, B->tpat, B->tpat_var, B->tpat_vf, B->tpat_ctr, B->ds_x, B->ds_y,
                    B->nrm, B->xin, B->yout, B->tbx, B->tby, B->ganj, B->pwatj, B->precipj, B->jpart, B->jstat,
                    B->jflag, B->jctr, B->gmean, B->dak, B->sdesc_ph, B->rflag_ph, B->slot_ph, B->sdesc_hl,
                    B->rflag_hl, B->slot_hl, B->hsdyn,
                    B->clock, B->iau_hrs, B->iau_inc, B->iau_F, B->st_pat2, B->st_pat[3], B->st_var, B->st_vf,
                    B->st_ctr, B->st_grd, B->sd_pat, B->rf0, B->vcg, B->sd_vc, B->rf1, B->an_w, B->an_g,
                    B->an_sm, B->sd_an, B->ad_an, B->rf_an};
    if (B->mlp) mlp_destroy(B->mlp);
    for (void *q : ptrs)
        if (q) (void)hipFree(q);
    if (B->Work) {
        work_free(*(Work<T> *)B->Work);
        delete (Work<T> *)B->Work;
    }
    delete B;
    dyn = nullptr;
}

// ---- step pieces ------------------------------------------------------------

template <typename T> struct Step {
    Engine<T> &E;
    DycoreBuffers &B;
    Work<T> &W;
    hipStream_t s;
    bool lean = false;  // run the lean Held-Suarez physics pass (a step before an advance's last)
    bool grids = false; // the dynamics passes keep the omega / p and etadot grids (a getdyntend call)
    // the Held-Suarez forcing reads no grid that the lean pass leaves out; the
    // additive noise reads the winds of the physics pass
    bool lean_ok() const { return E.cfg.physics == GFSDC_PHYS_HS && !B.st_on[3]; }
    void mark(const char *name) {
        if (!B.profiling) return;
        hipEvent_t e;
        (void)hipEventCreate(&e);
        (void)hipEventRecord(e, s);
        B.ev.push_back(e);
        B.evname.push_back(name);
    }
    void synth_all() {
        const Plan<T> &p = E.plan;
        const int nlg = B.nm * B.nleg, nf = B.nm * B.nsyn;
        launch_synth_gather(p, (const cplx<T> *)B.spec, 1, (long)B.nfs * B.nm, B.sdesc, nlg, W.sx, W.ldc, 1.0, s,
                            (T *)B.gmean);
        mark("synth_gather");
        launch_leg_synth(p, W.sx, W.ldc, W.fs, W.ldc, 2 * nlg, s);
        mark("leg_synth");
        launch_fft_synth(p, W.fs, W.ldc, (T *)B.gsyn, B.ng, nf, B.rflag_syn, s, (const T *)B.gmean, nullptr, 0,
                         nullptr, &B.fmap_dyn, 1.0 / E.cfg.rerth);
        mark("fft_synth");
    }
    // the same chain for the physics pass, without the temperature and tracer
    // gradients (written to their grid slots through slot_ph)
    void synth_phys() {
        const Plan<T> &p = E.plan;
        int nf = B.nm * B.nph;
        launch_synth_gather(p, (const cplx<T> *)B.spec, 1, (long)B.nfs * B.nm, B.sdesc_ph, nf, W.sx, W.ldc, 1.0, s,
                            (T *)B.gmean);
        mark("synth_gather");
        launch_leg_synth(p, W.sx, W.ldc, W.fs, W.ldc, 2 * nf, s);
        mark("leg_synth");
        launch_fft_synth(p, W.fs, W.ldc, (T *)B.gsyn, B.ng, nf, B.rflag_ph, s, (const T *)B.gmean, B.slot_ph);
        mark("fft_synth");
    }
    // the lean Held-Suarez pass: temperature, ln ps and the vorticity and
    // divergence of the levels where the last lean pass found drag (and one
    // more) into their grid slots; ps as the column kernel forms it (k_area);
    // the levels where the drag can act now (with the area sums); and, only
    // where those reach past the first synthesis, the vorticity and divergence
    // of all of them
    void synth_hs_lean() {
        const Plan<T> &p = E.plan;
        const cplx<T> *spec = (const cplx<T> *)B.spec;
        const long sk = (long)B.nfs * B.nm;
        const int nf = B.nhla + B.nhlb, na = B.nhla;
        launch_synth_gather(p, spec, 1, sk, B.sdesc_hl, nf, W.sx, W.ldc, 1.0, s, (T *)B.gmean, B.hsdyn + 3);
        mark("synth_gather");
        launch_leg_synth(p, W.sx, W.ldc, W.fs, W.ldc, 2 * nf, s, B.hsdyn + 3);
        mark("leg_synth");
        launch_fft_synth(p, W.fs, W.ldc, (T *)B.gsyn, B.ng, nf, B.rflag_hl, s, (const T *)B.gmean, B.slot_hl, 0,
                         B.hsdyn + 3);
        mark("fft_synth");
        // ps, the global means of the forcing's mass fixer, and the drag's levels
        area<true>(nullptr, E.cfg.massfix ? B.pmean : (double *)nullptr, nullptr, nullptr);
        mark("psg");
        launch_synth_gather(p, spec, 1, sk, B.sdesc_hl + na, B.nhlb, W.sx, W.ldc, 1.0, s, (T *)nullptr, B.hsdyn);
        mark("synth_gather_more");
        launch_leg_synth(p, W.sx, W.ldc, W.fs, W.ldc, 2 * B.nhlb, s, B.hsdyn);
        mark("leg_synth_more");
        launch_fft_synth(p, W.fs, W.ldc, (T *)B.gsyn, B.ng, B.nhlb, B.rflag_hl + na, s, (const T *)nullptr,
                         B.slot_hl + na, 0, B.hsdyn);
        mark("fft_synth_more");
    }
    // dyn_run.f90:114-116: the vorticity gradient of vorticity confinement
    void synth_vc() {
        const Plan<T> &p = E.plan;
        const int nf = B.nm * 2 * B.nl;
        launch_synth_gather(p, (const cplx<T> *)B.spec, 1, (long)B.nfs * B.nm, B.sd_vc, nf, W.sx, W.ldc, 1.0, s);
        launch_leg_synth(p, W.sx, W.ldc, W.fs, W.ldc, 2 * nf, s);
        launch_fft_synth(p, W.fs, W.ldc, (T *)B.vcg, B.ng, nf, B.rf1, s);
        mark("synth_vc");
    }
    void columns(int inverse_only, bool colq = false) {
        const gfsdc_cfg &c = E.cfg;
        const bool vc = B.vc_on && !inverse_only;
        // the omega / p and etadot grids are stored where a caller sees them: by
        // the inverse pass of the physics, a getdyntend call, or with no physics
        // the dynamics passes themselves
        const int store = (inverse_only || grids || c.physics == GFSDC_PHYS_NONE) ? 1 : 0;
        if (vc) synth_vc();
        auto launch = [&](auto kern, unsigned nblk, unsigned nthr) {
            hipLaunchKernelGGL(kern, dim3(nblk, B.nm), dim3(nthr), 0, s, (const T *)B.gsyn, (T *)B.gan, (T *)B.etadot,
                           (T *)B.dlnpdt, (T *)B.psg, (T *)B.dlnpsdt, (const T *)B.dphisdx, (const T *)B.dphisdy,
                           (const T *)B.ak, (const T *)B.bk, (const T *)B.ck, (const T *)B.dbk,
                           (const T *)B.dak, (const T *)B.sinlat, B.nl, B.ntr, B.nsyn, B.nan, B.ng, E.plan.nlon, (T)c.rd,
                           (T)(c.rd / c.cp), (T)(c.cvap / c.cp - 1.0), (T)(2.0 * c.omega),
                           (const cplx<T> *)B.spec, B.nfs, colq ? (T *)B.colq : (T *)nullptr, (const T *)B.vcg,
                           B.st_on[0] ? (const T *)B.st_grd : (const T *)nullptr, (const T *)B.st_vf,
                           (T)B.sc.vcamp, store);
        };
        if (!inverse_only && columns_serial<T>(B.ng, B.nm, B.ntr, B.nl, grids)) {
            launch(vc ? k_columns_serial<T, true> : k_columns_serial<T, false>, (unsigned)((B.ng + 255) / 256), 256);
            mark("columns");
            return;
        }
        constexpr int NC = ColCfg<T>::NC, CH = ColCfg<T>::CH, LPC = MAXLEV / CH;
        const bool half = B.nl <= CH * LPC / 2;  // half the registers for the layers where they suffice
        auto pick = [&](auto mode, auto tr) {
            constexpr int M = decltype(mode)::value;
            constexpr bool TR = decltype(tr)::value;
            return half ? k_columns<T, M, LPC / 2, TR> : k_columns<T, M, LPC, TR>;
        };
        auto mode = [&](auto tr) {
            return vc ? pick(std::integral_constant<int, COL_VC>(), tr)
                      : inverse_only ? pick(std::integral_constant<int, COL_INV>(), tr)
                                     : pick(std::integral_constant<int, COL_DYN>(), tr);
        };
        launch(B.ntr > 0 ? mode(std::true_type()) : mode(std::false_type()), (unsigned)((B.ng + NC - 1) / NC), NC * CH);
        mark(inverse_only ? "columns_inverse" : "columns");
    }
    template <bool PSG> void area(const void *b, double *pmean, double *bsum, double *pdryini) {
        hipLaunchKernelGGL((k_area<T, PSG>), dim3(PS_BLOCKS, B.nm), dim3(256), 0, s, (T *)B.psg, (const T *)b,
                           (const double *)B.areaw, B.pspart, B.psdone, B.ng, E.plan.nlon, pmean, bsum, pdryini,
                           (const T *)B.ak, (const T *)B.bk, B.nl, B.hsdyn, (const T *)B.gsyn,
                           (const cplx<T> *)B.spec, B.ntr, B.nsyn, B.nfs);
    }
    // FP64 area sums: S(psg) -> pmean, S(b) -> bsum; pdryini = S(psg) - S(b) where 0
    void area_sums(const void *b, double *pmean, double *bsum, bool set_pdry) {
        area<false>(b, pmean, bsum, set_pdry ? B.pdryini : (double *)nullptr);
        mark("ps_mean");
    }
    // ngf grid fields of gan -> spectral fields of dst; with nfdyn only the
    // first *nfdyn grid fields (the others are zero on the grid)
    void analyse(const AnalDesc *desc, const unsigned char *rflag, int ngf, cplx<T> *dst,
                 const int *nfdyn = nullptr, bool massfix = false) {
        const Plan<T> &p = E.plan;
        launch_fft_anal(p, (const T *)B.gan, B.ng, ngf, rflag, W.fa, W.ldc, s, nfdyn);
        mark("fft_anal");
        launch_leg_anal(p, W.fa, W.ldc, W.sx, W.ldc, 2 * ngf, s, nfdyn);
        mark("leg_anal");
        launch_anal_scatter(p, W.sx, W.ldc, desc, B.nm * B.nfs, dst, 1, (long)B.nfs * B.nm, E.cfg.rerth, s,
                            nfdyn, massfix);
        mark("anal_scatter");
    }
    void getdyntend(int stage) {
        synth_all();
        columns(0, stage == 0 && B.ntr > 0);
        // dyn_run.f90:135-153 on this stage's psg (and column tracer mass)
        if (stage == 0) area_sums(B.ntr > 0 ? B.colq : nullptr, nullptr, nullptr, true);
        analyse(B.adesc_dyn, B.rflag_an, B.nm * B.nan, (cplx<T> *)B.ten[stage]);
        // run.f90:302-309,363-370,429-436: the IAU forcing joins every stage's
        // tendencies before the linear terms come off
        if (B.iau_n) {
            const long n = 2L * E.plan.nlm * B.nfs * B.nm;
            hipLaunchKernelGGL(k_axpby<T>, dim3(1024), dim3(256), 0, s, (T *)B.ten[stage], (const T *)B.iau_F,
                               (T)1, (T)1, n);
            mark("iau_add");
        }
    }
    // run.f90:250-258: the IAU forcing of this step, at the step's start time
    void iau_forcing() {
        const long len = 2L * E.plan.nlm * B.nfs * B.nm;
        hipLaunchKernelGGL(k_iau_forcing<T>, dim3(1024), dim3(256), 0, s, (T *)B.iau_F, (const T *)B.iau_inc,
                           (const double *)B.iau_hrs, B.iau_n, B.iau_dt, (const double *)B.clock, len);
        mark("iau_forcing");
    }
    bool si_mfma() const { return !E.cfg.explicit_; }
    void si_stage(int stage, bool damp) {
        const gfsdc_cfg &c = E.cfg;
        Coeffs3 cf;
        for (int r = 0; r < 3; r++) cf.a[r] = TAB_A[stage][r];
        if (si_mfma()) {
            const int do_imp = (stage < 2 || std::fabs(TAB_IMP[stage]) > 1.e-5) ? 1 : 0;
            auto ta = [&](int r) { return r < 3 ? TAB_A[r][stage] : 0.0; };
            auto taa = [&](int r) { return r < 3 ? TAB_AA[r][stage] : 0.0; };
            const SiNext cn{ta(stage), taa(stage), ta(stage + 1), taa(stage + 1), ta(stage + 2), taa(stage + 2)};
            hipLaunchKernelGGL(k_si_mfma<T>, dim3((unsigned)B.n_si_tiles), dim3(256), 0, s, (T *)B.spec,
                               (T *)B.spec0, (const T *)B.ten[0], (const T *)B.ten[1], (const T *)B.ten[2], (T *)B.mix[0],
                               (T *)B.mix[1], (const T *)B.at, (const T *)B.bt, (const T *)B.dt3,
                               (const T *)B.sv, (const T *)B.tor, (const T *)B.disspec, (const T *)B.diffp,
                               (const T *)B.dmpp, (const int2 *)B.si_tiles, stage, cf, cn,
                               (T)TAB_IMP[stage], do_imp, damp ? 1 : 0, B.nl, B.ntr, B.nfs, B.nm, E.plan.ntrunc,
                               (T)c.dt, B.clock, c.dt);
            mark("si_stage");
            return;
        }
        long items = (long)E.plan.nlm * B.nm;
        hipLaunchKernelGGL(k_explicit_stage<T>, dim3((unsigned)((items + 3) / 4)), dim3(256), 0, s, (cplx<T> *)B.spec,
                           (const cplx<T> *)B.spec0, (const cplx<T> *)B.ten[0], (const cplx<T> *)B.ten[1],
                           (const cplx<T> *)B.ten[2], (const T *)B.disspec, (const T *)B.diffp, (const T *)B.dmpp,
                           stage, cf, damp ? 1 : 0, B.nl, B.ntr, B.nfs, B.nm, E.plan.nlm, (T)c.dt);
        mark("si_stage");
    }
    void physics() {
        const gfsdc_cfg &c = E.cfg;
        const bool lean_pass = lean && lean_ok();
        if (lean_pass) {
            synth_hs_lean();
        } else {
            synth_phys();
            columns(1);
        }
        // run.f90:517-518: the additive noise forcing, before the physics
        if (B.st_on[3]) stoch_forcing();
        if (c.physics == GFSDC_PHYS_SIMPLE) {
            if (B.mlp_on)
                mlp_columns();
            else
                simple_columns();
            if (c.massfix) {
                area_sums(B.pwat, B.pmean, B.pwsum, false);
                dim3 g((unsigned)((B.ng + 255) / 256), B.nm);
                hipLaunchKernelGGL(k_massfix_field<T>, g, dim3(256), 0, s, (const T *)B.gsyn, (T *)B.gan,
                                   (const double *)B.pdryini, (const double *)B.pmean, (const double *)B.pwsum,
                                   B.nl, B.ntr, B.nsyn, B.nsp, B.ng, c.grav);
                mark("massfix_field");
            }
            analyse(B.adesc_sp, B.rflag_sp, B.nm * B.nsp, (cplx<T> *)B.tphys);
            phys_update();
        }
        if (c.physics == GFSDC_PHYS_HS) {
            if (!lean_pass) area_sums(nullptr, c.massfix ? B.pmean : (double *)nullptr, nullptr, false);
            dim3 g((unsigned)((B.ng + 255) / 256), B.nm * HS_LCH);
            // the lean pass forms and transforms the drag only where it can act (hs_level_drags)
            const int *cnt = lean_pass ? B.hsdyn : nullptr;
            hipLaunchKernelGGL(k_hs_columns<T>, g, dim3(256), 0, s, (const T *)B.gsyn, (const T *)B.psg, (T *)B.gan,
                               (const T *)B.ak, (const T *)B.bk, (const T *)B.sinlat, B.pdryini, B.pmean, B.nl,
                               B.ntr, B.nsyn, B.nm, B.ng, E.plan.nlon, (T)(c.rd / c.cp), c.massfix, cnt);
            mark("hs_columns");
            // HS fields per member: T, vrt, div forcing and the mass-fixer field,
            // analysed straight into the state (the scatter applies the update)
            analyse(B.adesc_hsu, B.rflag_hs, B.nm * B.nhs, (cplx<T> *)B.spec, cnt ? cnt + 1 : nullptr,
                    c.massfix != 0);
        }
        // run.f90:541-552: the streamfunction forcing into vorticity, after the physics
        if (B.st_on[3]) {
            const gfsdc_stoch_cfg &sc = B.sc;
            hipLaunchKernelGGL(k_an_apply<T>, dim3(1024), dim3(256), 0, s, (cplx<T> *)B.spec,
                               (const cplx<T> *)B.an_w, (const int *)B.degree, B.nl, B.nfs, B.nm, E.plan.nlm, c.dt,
                               c.rerth, (sc.addnoise_kenorm && sc.addnoise_vrtonly) ? 1 : 0);
            mark("stoch_apply");
        }
    }
    SimpleCfg simple_cfg() const {
        const gfsdc_cfg &c = E.cfg;
        SimpleCfg sc;
        sc.dt = c.dt;
        sc.fv = (double)(T)(c.rv / c.rd - 1.0);  // physcons.f90 con_fvirt
        sc.qmin = (double)1.e-10f;               // phy_run_simple.f90:37
        sc.grav = c.grav;
        sc.sst_mode = c.simple_test;
        sc.turbflux = c.turbflux;
        return sc;
    }
    // plain simple physics on all columns (or the selection cs) into (gan, pwat, precip)
    void simple_columns(ColSel cs = ColSel{0, nullptr, nullptr}, void *gan = nullptr, void *pwat = nullptr,
                        void *precip = nullptr, const char *name = "simple_columns") {
        const gfsdc_cfg &c = E.cfg;
        const long ncol = cs.stride > 0 ? B.ng / cs.stride : B.ng;
        dim3 g((unsigned)((ncol + SP_C - 1) / SP_C), B.nm);
        hipLaunchKernelGGL(k_simple_columns<T>, g, dim3(256), 0, s, (const T *)B.gsyn, (const T *)B.psg,
                           (T *)(gan ? gan : B.gan), (T *)(pwat ? pwat : B.pwat),
                           (T *)(precip ? precip : B.precip), (const T *)B.ak, (const T *)B.bk,
                           (const double *)B.latd, B.nl, B.ntr, B.nsyn, B.nsp, B.ng, E.plan.nlon, (T)(c.rd / c.cp),
                           simple_cfg(), cs);
        mark(name);
    }
    // learned column physics with the plain physics as judge on every
    // judge_stride-th column and as the fallback for the whole step
    void mlp_columns() {
        const gfsdc_cfg &c = E.cfg;
        const long rows = (long)B.nm * B.ng;
        dim3 g((unsigned)((B.ng + MLP_CB - 1) / MLP_CB), B.nm);
        const int nin = 4 * B.nl + 3, nout = 4 * B.nl;
        hipLaunchKernelGGL(k_mlp_features<T>, g, dim3(256), sizeof(float) * MLP_CB * (nin | 1), s, (const T *)B.gsyn,
                           (const T *)B.psg,
                           (const double *)B.latd, B.nl, B.nsyn, B.ng, E.plan.nlon, simple_cfg(),
                           ColSel{0, nullptr, nullptr}, B.ng, (const float *)B.nrm, B.xin, 0L);
        mark("mlp_features");
        mlp_forward(B.mlp, B.xin, nin, (int)rows, B.yout, nout, s);
        mark("mlp_forward");
        hipLaunchKernelGGL(k_mlp_apply<T>, g, dim3(256), sizeof(float) * MLP_CB * (nout | 1), s,
                           (const float *)B.yout, (const float *)B.nrm,
                           (const T *)B.gsyn, (const T *)B.psg, (const T *)B.ak, (const T *)B.bk, (T *)B.gan,
                           (T *)B.pwat, (T *)B.precip, B.nl, B.nsyn, B.nsp, B.ng, c.grav);
        mark("mlp_apply");
        const ColSel js{B.judge_stride, B.jctr, nullptr};
        simple_columns(js, B.ganj, B.pwatj, B.precipj, "judge_columns");
        const long nsel = B.ng / B.judge_stride;
        // partial sums fit the (ng / 256 + 2) per member of jpart
        dim3 gj((unsigned)std::min<long>(1024, B.ng / 256 + 2), B.nm);
        hipLaunchKernelGGL(k_judge_partial<T>, gj, dim3(256), 0, s, (const T *)B.gan, (const T *)B.ganj,
                           (const float *)B.nrm, B.nl, B.nsp, B.ng, js, B.jpart);
        hipLaunchKernelGGL(k_judge_final, dim3(1), dim3(256), 0, s, (const double *)B.jpart, (int)(gj.x * gj.y),
                           (double)nsel * B.nm * nout, B.judge_thr, B.jflag, B.jstat);
        hipLaunchKernelGGL(k_counter_inc, dim3(1), dim3(64), 0, s, B.jctr);
        mark("judge");
        simple_columns(ColSel{0, nullptr, B.jflag}, nullptr, nullptr, nullptr, "fallback_columns");
    }
    void phys_update() {
        const gfsdc_cfg &c = E.cfg;
        long n = (long)E.plan.nlm * B.nfs * B.nm;
        hipLaunchKernelGGL(k_phys_update<T>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, (cplx<T> *)B.spec,
                           (const cplx<T> *)B.tphys, B.nl, B.ntr, B.nfs, B.nm, E.plan.nlm, (T)c.dt, c.massfix);
        mark("phys_update");
    }
    // one AR(1) advance of every member's pattern (phi = 0 and f = amp start it)
    void pattern_advance(double phi, double f) {
        const Plan<T> &p = E.plan;
        hipLaunchKernelGGL(k_pattern_advance<T>, dim3((unsigned)((p.nlm + 255) / 256), B.nm), dim3(256), 0, s,
                           (cplx<T> *)B.tpat, (const double *)B.tpat_var, (const int2 *)p.kmn, p.nlm,
                           (const unsigned long long *)B.tpat_ctr,
                           (unsigned long long)(long long)E.cfg.tpat_seed, phi, f,
                           std::sqrt(2.0 * M_PI / p.ntrunc), 1, 1ULL << 40);
        hipLaunchKernelGGL(k_counter_inc, dim3(1), dim3(64), 0, s, B.tpat_ctr);
        mark("pattern_advance");
    }
    void pattern_apply() {
        long n = (long)E.plan.nlm * B.nm * B.nl;
        hipLaunchKernelGGL(k_pattern_apply<T>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, (cplx<T> *)B.spec,
                           (const cplx<T> *)B.tpat, (const T *)B.tpat_vf, B.nl, B.nfs, B.nm, E.plan.nlm,
                           (T)(E.cfg.dt / E.cfg.tpat_tau));
        mark("pattern_apply");
    }
    // one advance of stochastic pattern kind kd (phi = 0 and f = stdev start it)
    void stoch_advance(int kd, double phi, double f) {
        const Plan<T> &p = E.plan;
        hipLaunchKernelGGL(k_pattern_advance<T>, dim3((unsigned)((p.nlm + 255) / 256), B.nm * B.st_nf[kd]),
                           dim3(256), 0, s, (cplx<T> *)B.st_pat[kd], (const double *)B.st_var + (long)kd * p.nlm,
                           (const int2 *)p.kmn, p.nlm, (const unsigned long long *)B.st_ctr + kd, B.st_seed[kd], phi,
                           f, std::sqrt(2.0 * M_PI / p.ntrunc), B.st_nf[kd], (3ULL + kd) << 40);
        hipLaunchKernelGGL(k_counter_inc, dim3(1), dim3(64), 0, s, B.st_ctr + kd);
        mark("stoch_pattern");
    }
    // grids of the svc, sppt (logit transform) and shum patterns
    void stoch_grids() {
        const Plan<T> &p = E.plan;
        const int nf = 3 * B.nm;
        launch_synth_gather(p, (const cplx<T> *)B.st_pat2, p.nlm, 1, B.sd_pat, nf, W.sx, W.ldc, 1.0, s);
        launch_leg_synth(p, W.sx, W.ldc, W.fs, W.ldc, 2 * nf, s);
        launch_fft_synth(p, W.fs, W.ldc, (T *)B.st_grd, B.ng, nf, B.rf0, s);
        if (B.st_on[1])
            hipLaunchKernelGGL(k_logit<T>, dim3(512), dim3(256), 0, s, (T *)B.st_grd + (long)B.nm * B.ng,
                               (long)B.nm * B.ng);
        mark("stoch_grids");
    }
    // run.f90:272-292: the patterns used this step
    void stoch_patterns() {
        for (int kd = 0; kd < 4; kd++)
            if (B.st_on[kd])
                stoch_advance(kd, B.st_phi[kd], B.st_sd[kd] * std::sqrt(1.0 - B.st_phi[kd] * B.st_phi[kd]));
        if (B.st_on[0] || B.st_on[1] || B.st_on[2]) stoch_grids();
    }
    // getstochforcing (stoch_data.f90:254-354) on the physics pass's grid
    // fields: the streamfunction forcing into an_w group 0
    void stoch_forcing() {
        const Plan<T> &p = E.plan;
        const gfsdc_stoch_cfg &sc = B.sc;
        const int nf = B.nm * B.nl;
        const long tot = (long)nf * p.nlm, gtot = (long)nf * B.ng;
        cplx<T> *w = (cplx<T> *)B.an_w;
        T *g = (T *)B.an_g;
        const int diss = sc.addnoise_dissfact != 0;
        hipLaunchKernelGGL(k_an_prep<T>, dim3(1024), dim3(256), 0, s, w, (const cplx<T> *)B.st_pat[3],
                           (const cplx<T> *)B.spec, (const T *)B.disspec, B.nl, B.nfs, B.nm, p.nlm,
                           sc.addnoise_vfilt > 0 ? 1 : 0, diss);
        if (diss) {
            // the dissipation wind and the noise on the grid (groups 0, 1, 2)
            launch_synth_gather(p, w, p.nlm, 1, B.sd_an, 3 * nf, W.sx, W.ldc, 1.0, s);
            launch_leg_synth(p, W.sx, W.ldc, W.fs, W.ldc, 6 * nf, s);
            launch_fft_synth(p, W.fs, W.ldc, g, B.ng, 3 * nf, B.rf_an, s);
            hipLaunchKernelGGL(k_an_kediss<T>, dim3(2048), dim3(256), 0, s, g, (const T *)B.gsyn, B.nl, B.nsyn, B.nm,
                               B.ng);
            // spectral smoothing of sqrt(ke dissipation): group 0 grid -> group 1 spectral -> group 1 grid
            launch_fft_anal(p, g, B.ng, nf, B.rf0, W.fa, W.ldc, s);
            launch_leg_anal(p, W.fa, W.ldc, W.sx, W.ldc, 2 * nf, s);
            launch_anal_scatter(p, W.sx, W.ldc, B.ad_an, nf, w + tot, p.nlm, 1, E.cfg.rerth, s);
            hipLaunchKernelGGL(k_spec_scale<T>, dim3(1024), dim3(256), 0, s, w + tot, (const T *)B.an_sm, (long)nf,
                               p.nlm);
            launch_synth_gather(p, w, p.nlm, 1, B.sd_an + 3 * nf, nf, W.sx, W.ldc, 1.0, s);
            launch_leg_synth(p, W.sx, W.ldc, W.fs, W.ldc, 2 * nf, s);
            launch_fft_synth(p, W.fs, W.ldc, g + gtot, B.ng, nf, B.rf0, s);
        } else {
            launch_synth_gather(p, w, p.nlm, 1, B.sd_an + 4 * nf, nf, W.sx, W.ldc, 1.0, s);
            launch_leg_synth(p, W.sx, W.ldc, W.fs, W.ldc, 2 * nf, s);
            launch_fft_synth(p, W.fs, W.ldc, g + 2 * gtot, B.ng, nf, B.rf0, s);
        }
        hipLaunchKernelGGL(k_an_modulate<T>, dim3(2048), dim3(256), 0, s, g, (const T *)(g + 2 * gtot),
                           diss ? (const T *)(g + gtot) : (const T *)nullptr, (const T *)B.st_vf + 3L * B.nl, B.nl,
                           B.nm, B.ng);
        launch_fft_anal(p, g, B.ng, nf, B.rf0, W.fa, W.ldc, s);
        launch_leg_anal(p, W.fa, W.ldc, W.sx, W.ldc, 2 * nf, s);
        launch_anal_scatter(p, W.sx, W.ldc, B.ad_an, nf, w, p.nlm, 1, E.cfg.rerth, s);
        mark("stoch_forcing");
    }
    void step() {
        const bool pat = B.tpat != nullptr;
        if (B.iau_n) iau_forcing();
        // run.f90:272-292: the random patterns used this step
        if (pat) pattern_advance(B.tpat_phi, E.cfg.tpat_amp * std::sqrt(1.0 - B.tpat_phi * B.tpat_phi));
        stoch_patterns();
        // k_si_mfma keeps the initial state and moves the clock itself
        if (!si_mfma()) {
            long n = 2L * E.plan.nlm * B.nfs * B.nm;
            hipLaunchKernelGGL(k_copy<T>, dim3(2048), dim3(256), 0, s, (T *)B.spec0, (const T *)B.spec, n);
            mark("save_state");
        }
        for (int st = 0; st < 3; st++) {
            getdyntend(st);
            si_stage(st, st == 2);
        }
        if (E.cfg.physics != GFSDC_PHYS_NONE) physics();
        // stochastic temperature forcing, where run.f90:539-551 adds its tvforcing
        if (pat) pattern_apply();
        if (!si_mfma()) hipLaunchKernelGGL(k_clock_add, dim3(1), dim3(64), 0, s, B.clock, E.cfg.dt);
    }
};

// init_stochdata (stoch_data.f90): start from stdev * varspectrum * noise and
// spin up 5 e-folding times
template <typename T> int Engine<T>::pattern_spinup() {
    DycoreBuffers *B = dyn;
    Step<T> st{*this, *B, *(Work<T> *)B->Work, stream};
    st.pattern_advance(0.0, cfg.tpat_amp);
    const int nspinup = (int)(5.0 * cfg.tpat_tau / cfg.dt);
    for (int i = 0; i < nspinup; i++)
        st.pattern_advance(B->tpat_phi, cfg.tpat_amp * std::sqrt(1.0 - B->tpat_phi * B->tpat_phi));
    GFSDC_CHECK(hipGetLastError());
    return 0;
}

template <typename T> int Engine<T>::get_pattern(void *out, int dtype, int loc) {
    DycoreBuffers *B = dyn;
    if (!B || !B->tpat) {
        set_error("context has no stochastic pattern (tpat_amp == 0)");
        return GFSDC_ESTATE;
    }
    return output((const T *)B->tpat, out, (size_t)plan.nlm * B->nm * 2, dtype, loc, 1);
}

// ---- tile autotuner ----------------------------------------------------------
// Times the step's Fourier transforms (the synthesis of every grid field and
// the analysis of the dynamics tendencies) with 2, 4 and 8 fields per FFT
// workgroup on this context's own sizes and keeps the fastest, for the
// synthesis and the analysis separately. ms[c] is the synthesis plus analysis
// time of candidate c; best is the synthesis choice. Leaves the model state
// untouched; the next graph advance captures the new choice.
template <typename T> int Engine<T>::autotune(double *ms, int *best) {
    DycoreBuffers *B = dyn;
    if (!B) {
        set_error("autotune needs a dycore context");
        return GFSDC_ESTATE;
    }
    Work<T> &W = *(Work<T> *)B->Work;
    const int cand[3] = {2, 4, 8};
    hipEvent_t e0, e1, e2;
    GFSDC_CHECK(hipEventCreate(&e0));
    GFSDC_CHECK(hipEventCreate(&e1));
    GFSDC_CHECK(hipEventCreate(&e2));
    double best_syn = 1e300, best_an = 1e300;
    int nf_syn = plan.fft_nf, nf_an = plan.fft_nf_an;
    for (int c = 0; c < 3; c++) {
        plan.fft_nf = plan.fft_nf_an = cand[c];
        float ts = 0.f, ta = 0.f;
        for (int rep = 0; rep < 2; rep++) {  // first pass warms up
            GFSDC_CHECK(hipEventRecord(e0, stream));
            launch_fft_synth(plan, W.fs, W.ldc, (T *)B->gsyn, B->ng, B->nm * B->nsyn, B->rflag_syn, stream,
                             (const T *)B->gmean, nullptr, 0, nullptr, &B->fmap_dyn, 1.0 / cfg.rerth);
            GFSDC_CHECK(hipEventRecord(e1, stream));
            launch_fft_anal(plan, (const T *)B->gan, B->ng, B->nm * B->nan, B->rflag_an, W.fa, W.ldc, stream);
            GFSDC_CHECK(hipEventRecord(e2, stream));
            GFSDC_CHECK(hipEventSynchronize(e2));
            GFSDC_CHECK(hipEventElapsedTime(&ts, e0, e1));
            GFSDC_CHECK(hipEventElapsedTime(&ta, e1, e2));
        }
        if (ms) ms[c] = (double)ts + (double)ta;
        if (ts < best_syn) {
            best_syn = ts;
            nf_syn = cand[c];
        }
        if (ta < best_an) {
            best_an = ta;
            nf_an = cand[c];
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipEventDestroy(e2);
    plan.fft_nf = nf_syn;
    plan.fft_nf_an = nf_an;
    if (best) *best = nf_syn;
    drop_graph(B);
    return 0;
}

// ---- learned column physics: data, training, judge ---------------------------

__global__ void k_norm_rows(const float *__restrict__ src, long n, int nf, const float *__restrict__ mean,
                            const float *__restrict__ sd, float *__restrict__ dst) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n * nf) return;
    const int f = (int)(i % nf);
    dst[i] = (src[i] - mean[f]) / sd[f];
}

template <typename T> static int mlp_need(DycoreBuffers *B, bool norm) {
    if (!B || !B->mlp) {
        set_error("no column MLP: call gfsdc_mlp_init first");
        return GFSDC_ESTATE;
    }
    if (norm && !B->nrm_ready) {
        set_error("column MLP has no normalisation: collect data and call gfsdc_mlp_normalize first");
        return GFSDC_ESTATE;
    }
    return 0;
}

template <typename T>
int Engine<T>::mlp_init(int hidden, int nlayers, int maxbatch, long capacity, unsigned long long seed) {
    DycoreBuffers *B = dyn;
    if (!B || cfg.physics != GFSDC_PHYS_SIMPLE) {
        set_error("the column MLP needs a dycore context with physics = GFSDC_PHYS_SIMPLE (its teacher and judge)");
        return GFSDC_ESTATE;
    }
    if (B->mlp) {
        set_error("column MLP already initialised");
        return GFSDC_ESTATE;
    }
    if (capacity < 1 || maxbatch < 1) {
        set_error("capacity and maxbatch must be >= 1");
        return GFSDC_EINVAL;
    }
    const int nl = B->nl, nin = 4 * nl + 3, nout = 4 * nl, nm = B->nm;
    const long ng = B->ng;
    int rc = mlp_create(&B->mlp, nin, nout, hidden, nlayers, maxbatch, seed, stream);
    if (rc) return rc;
    B->ds_cap = capacity;
    B->ds_n = 0;
    B->ds_x = dalloc<float>((size_t)capacity * nin);
    B->ds_y = dalloc<float>((size_t)capacity * nout);
    B->nrm = dalloc<float>(2 * (size_t)(nin + nout));
    B->xin = dalloc<float>((size_t)nm * ng * nin);
    B->yout = dalloc<float>((size_t)nm * ng * nout);
    B->tbx = dalloc<float>((size_t)B->mlp->Bp * nin);
    B->tby = dalloc<float>((size_t)B->mlp->Bp * nout);
    B->ganj = dalloc<T>((size_t)nm * B->nsp * ng);
    B->pwatj = dalloc<T>((size_t)nm * ng);
    B->precipj = dalloc<T>((size_t)nm * ng);
    B->jpart = dalloc<double>((size_t)nm * (ng / 256 + 2));
    B->jstat = dalloc<double>(3);
    B->jflag = dalloc<int>(1);
    B->jctr = dalloc<unsigned long long>(1);
    void *ptrs[] = {B->ds_x, B->ds_y, B->nrm, B->xin, B->yout, B->tbx, B->tby, B->ganj, B->pwatj,
                    B->precipj, B->jpart, B->jstat, B->jflag, B->jctr};
    for (void *q : ptrs)
        if (!q) {
            set_error("device allocation failed for the column MLP");
            return GFSDC_ENOMEM;
        }
    GFSDC_CHECK(hipMemsetAsync(B->jstat, 0, sizeof(double) * 3, stream));
    GFSDC_CHECK(hipMemsetAsync(B->jflag, 0, sizeof(int), stream));
    GFSDC_CHECK(hipMemsetAsync(B->jctr, 0, sizeof(unsigned long long), stream));
    GFSDC_CHECK(hipStreamSynchronize(stream));
    return 0;
}

template <typename T> int Engine<T>::mlp_collect(int nsteps, int stride, long *ncollected) {
    DycoreBuffers *B = dyn;
    int rc = mlp_need<T>(B, false);
    if (rc) return rc;
    if (stride < 1) {
        set_error("stride must be >= 1");
        return GFSDC_EINVAL;
    }
    const bool was_on = B->mlp_on;
    B->mlp_on = false;  // the plain physics produces the training data
    Step<T> st{*this, *B, *(Work<T> *)B->Work, stream};
    const long nsel = B->ng / stride, per = nsel * B->nm;
    for (int i = 0; i < nsteps && B->ds_n + per <= B->ds_cap; i++) {
        st.step();
        const ColSel cs{stride, B->jctr, nullptr};
        dim3 g((unsigned)((nsel + 255) / 256), B->nm);
        dim3 gf((unsigned)((nsel + MLP_CB - 1) / MLP_CB), B->nm);
        hipLaunchKernelGGL(k_mlp_features<T>, gf, dim3(256), sizeof(float) * MLP_CB * ((4 * B->nl + 3) | 1), stream,
                           (const T *)B->gsyn, (const T *)B->psg, (const double *)B->latd, B->nl, B->nsyn, B->ng,
                           plan.nlon, st.simple_cfg(), cs, nsel, (const float *)nullptr, B->ds_x, B->ds_n);
        hipLaunchKernelGGL(k_mlp_targets<T>, g, dim3(256), 0, stream, (const T *)B->gan, B->nl, B->nsp, B->ng, cs,
                           nsel, B->ds_y, B->ds_n);
        hipLaunchKernelGGL(k_counter_inc, dim3(1), dim3(64), 0, stream, B->jctr);
        GFSDC_CHECK(hipGetLastError());
        B->ds_n += per;
    }
    GFSDC_CHECK(hipStreamSynchronize(stream));
    B->mlp_on = was_on;
    if (ncollected) *ncollected = B->ds_n;
    return 0;
}

template <typename T> int Engine<T>::mlp_normalize() {
    DycoreBuffers *B = dyn;
    int rc = mlp_need<T>(B, false);
    if (rc) return rc;
    if (B->ds_n < 2) {
        set_error("collect at least two columns before gfsdc_mlp_normalize");
        return GFSDC_ESTATE;
    }
    const int nin = B->mlp->nin, nout = B->mlp->nout;
    hipLaunchKernelGGL(k_colstats, dim3(nin), dim3(256), 0, stream, (const float *)B->ds_x, B->ds_n, nin, B->nrm,
                       B->nrm + nin);
    hipLaunchKernelGGL(k_colstats, dim3(nout), dim3(256), 0, stream, (const float *)B->ds_y, B->ds_n, nout,
                       B->nrm + 2 * nin, B->nrm + 2 * nin + nout);
    GFSDC_CHECK(hipGetLastError());
    GFSDC_CHECK(hipStreamSynchronize(stream));
    B->nrm_ready = true;
    return 0;
}

template <typename T>
int Engine<T>::mlp_train(int nsteps, int batch, double lr, double wd, long ntrain, double *losses) {
    DycoreBuffers *B = dyn;
    int rc = mlp_need<T>(B, true);
    if (rc) return rc;
    if (ntrain <= 0 || ntrain > B->ds_n) ntrain = B->ds_n;
    if (batch < 1 || batch > B->mlp->Bp) {
        set_error("batch must be in [1, maxbatch]");
        return GFSDC_EINVAL;
    }
    const int nin = B->mlp->nin, nout = B->mlp->nout;
    double *dl = dalloc<double>(nsteps > 0 ? nsteps : 1);
    if (!dl) {
        set_error("device allocation failed");
        return GFSDC_ENOMEM;
    }
    const long nb = (long)batch * (nin + nout);
    for (int it = 0; it < nsteps; it++) {
        hipLaunchKernelGGL(k_mlp_batch, dim3((unsigned)((nb + 255) / 256)), dim3(256), 0, stream,
                           (const float *)B->ds_x, (const float *)B->ds_y, ntrain, nin, nout, (const float *)B->nrm,
                           (unsigned long long)B->mlp->seed ^ 0xBA7C4ULL, B->bctr++, batch, B->tbx, B->tby);
        if ((rc = mlp_backward(B->mlp, B->tbx, nin, B->tby, nout, batch, stream))) break;
        if ((rc = mlp_adamw(B->mlp, lr, wd, nullptr, stream))) break;
        GFSDC_CHECK(hipMemcpyAsync(dl + it, mlp_loss_dev(B->mlp), sizeof(double), hipMemcpyDeviceToDevice, stream));
    }
    if (!rc && losses && nsteps > 0)
        GFSDC_CHECK(hipMemcpyAsync(losses, dl, sizeof(double) * nsteps, hipMemcpyDeviceToHost, stream));
    GFSDC_CHECK(hipStreamSynchronize(stream));
    (void)hipFree(dl);
    return rc;
}

template <typename T> int Engine<T>::mlp_eval(long first, long count, double *err, double *base) {
    DycoreBuffers *B = dyn;
    int rc = mlp_need<T>(B, true);
    if (rc) return rc;
    if (first < 0 || count < 1 || first + count > B->ds_n) {
        set_error("eval rows outside the collected data");
        return GFSDC_EINVAL;
    }
    const int nin = B->mlp->nin, nout = B->mlp->nout;
    const long cap = (long)B->nm * B->ng;  // rows of the inference buffers
    double se = 0.0, sb = 0.0;
    std::vector<double> part;
    for (long r0 = first; r0 < first + count; r0 += cap) {
        const long n = std::min(cap, first + count - r0);
        hipLaunchKernelGGL(k_norm_rows, dim3((unsigned)((n * nin + 255) / 256)), dim3(256), 0, stream,
                           (const float *)B->ds_x + r0 * nin, n, nin, (const float *)B->nrm,
                           (const float *)B->nrm + nin, B->xin);
        if ((rc = mlp_forward(B->mlp, B->xin, nin, (int)n, B->yout, nout, stream))) return rc;
        const long nblk = (n * nout + 255) / 256;
        double *dp = (double *)B->jpart;  // reuse when large enough, else a temporary
        bool tmp = (size_t)(2 * nblk) > (size_t)B->nm * (B->ng / 256 + 2);
        if (tmp) dp = dalloc<double>(2 * nblk);
        if (!dp) {
            set_error("device allocation failed");
            return GFSDC_ENOMEM;
        }
        hipLaunchKernelGGL(k_eval_partial, dim3((unsigned)nblk), dim3(256), 0, stream, (const float *)B->yout,
                           (const float *)B->ds_y + r0 * nout, n, nout, (const float *)B->nrm + 2 * nin, dp);
        part.resize(2 * nblk);
        GFSDC_CHECK(hipMemcpyAsync(part.data(), dp, sizeof(double) * 2 * nblk, hipMemcpyDeviceToHost, stream));
        GFSDC_CHECK(hipStreamSynchronize(stream));
        if (tmp) (void)hipFree(dp);
        for (long i = 0; i < nblk; i++) {
            se += part[2 * i];
            sb += part[2 * i + 1];
        }
    }
    if (err) *err = std::sqrt(se / ((double)count * nout));
    if (base) *base = std::sqrt(sb / ((double)count * nout));
    return 0;
}

template <typename T> int Engine<T>::mlp_enable(int on, int judge_stride, double threshold) {
    DycoreBuffers *B = dyn;
    int rc = mlp_need<T>(B, on != 0);
    if (rc) return rc;
    if (judge_stride < 1 || judge_stride > B->ng) {
        set_error("judge_stride must be in [1, nlon*nlat]");
        return GFSDC_EINVAL;
    }
    B->mlp_on = on != 0;
    B->judge_stride = judge_stride;
    B->judge_thr = threshold;
    GFSDC_CHECK(hipMemsetAsync(B->jstat, 0, sizeof(double) * 3, stream));
    GFSDC_CHECK(hipStreamSynchronize(stream));
    // the captured step changes: capture again on the next graph advance
    drop_graph(B);
    return 0;
}

template <typename T> int Engine<T>::mlp_judge_stats(double *out) {
    DycoreBuffers *B = dyn;
    int rc = mlp_need<T>(B, false);
    if (rc) return rc;
    GFSDC_CHECK(hipMemcpyAsync(out, B->jstat, sizeof(double) * 3, hipMemcpyDeviceToHost, stream));
    GFSDC_CHECK(hipStreamSynchronize(stream));
    return 0;
}

template <typename T> long Engine<T>::mlp_nparams() {
    DycoreBuffers *B = dyn;
    return (B && B->mlp) ? (long)gfsdc::mlp_nparams(B->mlp) : 0;
}

template <typename T> int Engine<T>::mlp_params(float *get, const float *set) {
    DycoreBuffers *B = dyn;
    int rc = mlp_need<T>(B, false);
    if (rc) return rc;
    if (set && (rc = mlp_set_params(B->mlp, set, stream))) return rc;
    if (get && (rc = mlp_get_params(B->mlp, get, stream))) return rc;
    return 0;
}

template <typename T> int Engine<T>::mlp_norm(float *get, const float *set) {
    DycoreBuffers *B = dyn;
    int rc = mlp_need<T>(B, false);
    if (rc) return rc;
    const int nin = B->mlp->nin, nout = B->mlp->nout, n = 2 * (nin + nout);
    if (set) {
        // means finite, spreads positive and finite (the features divide by them)
        for (int i = 0; i < n; i++) {
            const bool spread = (i >= nin && i < 2 * nin) || i >= 2 * nin + nout;
            if (!std::isfinite(set[i]) || (spread && !(set[i] > 0.f))) {
                set_error("gfsdc_mlp_norm: entry " + std::to_string(i) + " is not a finite mean or a positive spread");
                return GFSDC_EINVAL;
            }
        }
        GFSDC_CHECK(hipMemcpyAsync(B->nrm, set, sizeof(float) * n, hipMemcpyHostToDevice, stream));
        GFSDC_CHECK(hipStreamSynchronize(stream));
        B->nrm_ready = true;
        drop_graph(B);  // a captured step holds no copy, but keep captures in step with the network state
    }
    if (get) {
        if (!B->nrm_ready) {
            set_error("column MLP has no normalisation: collect data and call gfsdc_mlp_normalize first");
            return GFSDC_ESTATE;
        }
        GFSDC_CHECK(hipMemcpyAsync(get, B->nrm, sizeof(float) * n, hipMemcpyDeviceToHost, stream));
        GFSDC_CHECK(hipStreamSynchronize(stream));
    }
    return 0;
}

template <typename T> int Engine<T>::mlp_forward_host(const float *x, long n, float *y) {
    DycoreBuffers *B = dyn;
    int rc = mlp_need<T>(B, false);
    if (rc) return rc;
    const int nin = B->mlp->nin, nout = B->mlp->nout;
    float *dx = dalloc<float>((size_t)n * nin), *dy = dalloc<float>((size_t)n * nout);
    if (!dx || !dy) {
        if (dx) (void)hipFree(dx);
        if (dy) (void)hipFree(dy);
        set_error("device allocation failed");
        return GFSDC_ENOMEM;
    }
    GFSDC_CHECK(hipMemcpyAsync(dx, x, sizeof(float) * n * nin, hipMemcpyHostToDevice, stream));
    rc = mlp_forward(B->mlp, dx, nin, (int)n, dy, nout, stream);
    if (!rc) GFSDC_CHECK(hipMemcpyAsync(y, dy, sizeof(float) * n * nout, hipMemcpyDeviceToHost, stream));
    GFSDC_CHECK(hipStreamSynchronize(stream));
    (void)hipFree(dx);
    (void)hipFree(dy);
    return rc;
}

template <typename T> int Engine<T>::mlp_grad_host(const float *x, const float *t, int n, float *grad, double *loss) {
    DycoreBuffers *B = dyn;
    int rc = mlp_need<T>(B, false);
    if (rc) return rc;
    const int nin = B->mlp->nin, nout = B->mlp->nout;
    if (n < 1 || n > B->mlp->Bp) {
        set_error("n must be in [1, maxbatch]");
        return GFSDC_EINVAL;
    }
    GFSDC_CHECK(hipMemcpyAsync(B->tbx, x, sizeof(float) * n * nin, hipMemcpyHostToDevice, stream));
    GFSDC_CHECK(hipMemcpyAsync(B->tby, t, sizeof(float) * n * nout, hipMemcpyHostToDevice, stream));
    if ((rc = mlp_backward(B->mlp, B->tbx, nin, B->tby, nout, n, stream))) return rc;
    if (loss) GFSDC_CHECK(hipMemcpyAsync(loss, mlp_loss_dev(B->mlp), sizeof(double), hipMemcpyDeviceToHost, stream));
    GFSDC_CHECK(hipStreamSynchronize(stream));
    if (grad && (rc = mlp_get_grad(B->mlp, grad, stream))) return rc;
    return 0;
}

template <typename T> int Engine<T>::mlp_adamw_host(const float *grad, double lr, double wd) {
    DycoreBuffers *B = dyn;
    int rc = mlp_need<T>(B, false);
    if (rc) return rc;
    rc = mlp_adamw(B->mlp, lr, wd, grad, stream);
    GFSDC_CHECK(hipStreamSynchronize(stream));
    return rc;
}

template <typename T> static PackParts pack_parts(const DycoreBuffers *B, const void *const (&p)[5]) {
    const int nl = B->nl, t = B->ntr * nl;
    PackParts pp{{p[0], p[1], p[2], p[3], p[4]}, {0, nl, 2 * nl, 3 * nl, 3 * nl + t, 3 * nl + t + 1}};
    return pp;
}

template <typename T> static void launch_pack(const Plan<T> &p, const DycoreBuffers *B, cplx<T> *spec, const PackParts &pp,
                                              bool to_state, hipStream_t s) {
    dim3 g((unsigned)((p.nlm + PACK_K - 1) / PACK_K), (unsigned)((B->nfs * B->nm + PACK_F<T> - 1) / PACK_F<T>));
    hipLaunchKernelGGL(k_pack<T>, g, dim3(256), 0, s, spec, pp, B->nfs, B->nm, p.nlm, to_state ? 1 : 0);
}

// caller's vrt, div, tv, tracers, ln ps (null: left alone) -> state layout
template <typename T> int Engine<T>::pack_in(void *spec, const void *const (&p)[5], int dtype, int loc) {
    DycoreBuffers *B = dyn;
    const PackParts all = pack_parts<T>(B, p);
    PackParts dir = all;
    for (int i = 0; i < 5; i++) {
        const int nfr = all.off[i + 1] - all.off[i];
        if (!p[i] || nfr == 0 || is_direct<T>(dtype, loc)) continue;
        dir.p[i] = nullptr;
        const T *in;
        int rc = input(p[i], (size_t)nfr * B->nm * plan.nlm * 2, dtype, loc, 0, &in);
        if (rc) return rc;
        PackParts one = all;
        for (int j = 0; j < 5; j++) one.p[j] = j == i ? in : nullptr;
        launch_pack(plan, B, (cplx<T> *)spec, one, true, stream);
    }
    if (is_direct<T>(dtype, loc)) launch_pack(plan, B, (cplx<T> *)spec, dir, true, stream);
    GFSDC_CHECK(hipGetLastError());
    return 0;
}

// state layout -> the caller's buffers (null: not wanted)
template <typename T> int Engine<T>::pack_out(const void *spec, void *const (&p)[5], int dtype, int loc) {
    DycoreBuffers *B = dyn;
    const void *cp[5] = {p[0], p[1], p[2], p[3], p[4]};
    const PackParts all = pack_parts<T>(B, cp);
    cplx<T> *sp = (cplx<T> *)const_cast<void *>(spec);
    if (is_direct<T>(dtype, loc)) {
        launch_pack(plan, B, sp, all, false, stream);
        GFSDC_CHECK(hipGetLastError());
        return 0;
    }
    for (int i = 0; i < 5; i++) {
        const int nfr = all.off[i + 1] - all.off[i];
        if (!p[i] || nfr == 0) continue;
        const size_t n = (size_t)nfr * B->nm * plan.nlm;
        int rc = ensure_stage(3, n * sizeof(cplx<T>));
        if (rc) return rc;
        PackParts one = all;
        for (int j = 0; j < 5; j++) one.p[j] = j == i ? stage[3] : nullptr;
        launch_pack(plan, B, sp, one, false, stream);
        GFSDC_CHECK(hipGetLastError());
        if ((rc = output((const T *)stage[3], p[i], n * 2, dtype, loc, 1))) return rc;
    }
    return 0;
}

template <typename T>
int Engine<T>::set_state(const void *vrt, const void *div, const void *tv, const void *trac, const void *lnps,
                         int dtype, int loc) {
    DycoreBuffers *B = dyn;
    if (!B) {
        set_error("context has no dycore (nlev == 0)");
        return GFSDC_ESTATE;
    }
    const void *const parts[5] = {vrt, div, tv, trac, lnps};
    int rc = pack_in(B->spec, parts, dtype, loc);
    if (rc) return rc;
    GFSDC_CHECK(hipStreamSynchronize(stream));
    return 0;
}

template <typename T>
int Engine<T>::get_state(void *vrt, void *div, void *tv, void *trac, void *lnps, int dtype, int loc) {
    DycoreBuffers *B = dyn;
    if (!B) {
        set_error("context has no dycore (nlev == 0)");
        return GFSDC_ESTATE;
    }
    void *const parts[5] = {vrt, div, tv, trac, lnps};
    return pack_out(B->spec, parts, dtype, loc);
}

template <typename T> int Engine<T>::set_topo(const void *topo, int dtype, int loc) {
    DycoreBuffers *B = dyn;
    if (!B) {
        set_error("context has no dycore");
        return GFSDC_ESTATE;
    }
    const int nlm = plan.nlm, nm = B->nm;
    const T *in;
    int rc = input(topo, (size_t)nlm * nm * 2, dtype, loc, 0, &in);
    if (rc) return rc;
    // dyn_init.f90:84 getgrad(grav*topospec) -> dphisdx, dphisdy
    Work<T> &W = *(Work<T> *)B->Work;
    std::vector<SynthDesc> sd(2 * nm);
    double g = cfg.grav / cfg.rerth;
    for (int mem = 0; mem < nm; mem++) {
        sd[mem] = SynthDesc{SK_UHAT, -1, mem, 0.0, g, 0, 0};
        sd[nm + mem] = SynthDesc{SK_VHAT, -1, mem, 0.0, g, 0, 0};
    }
    if ((rc = upload_descs(sd, std::vector<unsigned char>(2 * nm, 1)))) return rc;
    GFSDC_CHECK(hipMemcpyAsync(B->topo, in, sizeof(cplx<T>) * nlm * nm, hipMemcpyDeviceToDevice, stream));
    launch_synth_gather(plan, (const cplx<T> *)B->topo, nlm, 1, d_sdesc, 2 * nm, W.sx, W.ldc, 1.0, stream);
    launch_leg_synth(plan, W.sx, W.ldc, W.fs, W.ldc, 4 * nm, stream);
    // dphisdx then dphisdy are contiguous (nm fields each)
    launch_fft_synth(plan, W.fs, W.ldc, (T *)B->dphisdx, B->ng, nm, d_rflag, stream);
    GFSDC_CHECK(hipGetLastError());
    // second half of the fields (dphisdy): Fourier fields nm..2 nm - 1
    launch_fft_synth(plan, W.fs, W.ldc, (T *)B->dphisdy, B->ng, nm, d_rflag + nm, stream, (const T *)nullptr,
                     (const int *)nullptr, nm);
    GFSDC_CHECK(hipGetLastError());
    GFSDC_CHECK(hipStreamSynchronize(stream));
    return 0;
}

template <typename T>
int Engine<T>::getdyntend(int rkstage, int inverse_only, void *dvrt, void *ddiv, void *dtv, void *dtrac,
                          void *dlnps, int dtype, int loc) {
    DycoreBuffers *B = dyn;
    if (!B) {
        set_error("context has no dycore");
        return GFSDC_ESTATE;
    }
    if (rkstage < 1 || rkstage > 3) {
        set_error("rkstage must be 1, 2 or 3");
        return GFSDC_EINVAL;
    }
    Step<T> st{*this, *B, *(Work<T> *)B->Work, stream};
    st.grids = true;
    B->grids_partial = false;
    if (inverse_only) {
        st.synth_all();
        st.columns(1, rkstage == 1 && B->ntr > 0);
        if (rkstage == 1) st.area_sums(B->ntr > 0 ? B->colq : nullptr, nullptr, nullptr, true);
        GFSDC_CHECK(hipGetLastError());
        GFSDC_CHECK(hipStreamSynchronize(stream));
        return 0;
    }
    st.synth_all();
    st.columns(0, rkstage == 1 && B->ntr > 0);
    // dyn_run.f90:135-153
    if (rkstage == 1) st.area_sums(B->ntr > 0 ? B->colq : nullptr, nullptr, nullptr, true);
    st.analyse(B->adesc_dyn, B->rflag_an, B->nm * B->nan, (cplx<T> *)B->ten[0]);
    GFSDC_CHECK(hipGetLastError());
    void *const parts[5] = {dvrt, ddiv, dtv, dtrac, dlnps};
    return pack_out(B->ten[0], parts, dtype, loc);
}

template <typename T> int Engine<T>::advance(int nsteps, int use_graph) {
    DycoreBuffers *B = dyn;
    if (!B) {
        set_error("context has no dycore");
        return GFSDC_ESTATE;
    }
    Step<T> st{*this, *B, *(Work<T> *)B->Work, stream};
    // every step but the last may run the lean physics pass: only the last
    // step's grids are seen by callers (get_grid, step_diag)
    const bool lean = st.lean_ok() && nsteps > 1;
    if (nsteps > 0) B->grids_partial = false;
    if (!use_graph) {
        for (int i = 0; i < nsteps; i++) {
            st.lean = lean && i < nsteps - 1;
            st.step();
        }
        GFSDC_CHECK(hipGetLastError());
        return 0;
    }
    auto capture = [&](bool ln, hipGraph_t *g, hipGraphExec_t *x) -> int {
        st.lean = ln;
        GFSDC_CHECK(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
        st.step();
        GFSDC_CHECK(hipStreamEndCapture(stream, g));
        GFSDC_CHECK(hipGraphInstantiate(x, *g, nullptr, nullptr, 0));
        return 0;
    };
    int rc;
    if (!B->gexec && (rc = capture(false, &B->graph, &B->gexec))) return rc;
    if (lean && !B->gexec_lean && (rc = capture(true, &B->graph_lean, &B->gexec_lean))) return rc;
    for (int i = 0; i < nsteps; i++)
        GFSDC_CHECK(hipGraphLaunch(lean && i < nsteps - 1 ? B->gexec_lean : B->gexec, stream));
    return 0;
}


// run.f90:53 t = tstart (params.f90: tstart = fhour of the initial file, in s)
template <typename T> int Engine<T>::set_time(double t) {
    DycoreBuffers *B = dyn;
    if (!B) {
        set_error("context has no dycore");
        return GFSDC_ESTATE;
    }
    GFSDC_CHECK(hipMemcpyAsync(B->clock, &t, sizeof(double), hipMemcpyHostToDevice, stream));
    GFSDC_CHECK(hipStreamSynchronize(stream));
    return 0;
}

template <typename T> int Engine<T>::get_time(double *t) {
    DycoreBuffers *B = dyn;
    if (!B || !t) {
        set_error(!B ? "context has no dycore" : "null argument");
        return !B ? GFSDC_ESTATE : GFSDC_EINVAL;
    }
    GFSDC_CHECK(hipMemcpyAsync(t, B->clock, sizeof(double), hipMemcpyDeviceToHost, stream));
    GFSDC_CHECK(hipStreamSynchronize(stream));
    return 0;
}

template <typename T> int Engine<T>::hs_drag_levels(int *n) {
    DycoreBuffers *B = dyn;
    if (!B || !n) {
        set_error(!B ? "context has no dycore" : "null argument");
        return !B ? GFSDC_ESTATE : GFSDC_EINVAL;
    }
    GFSDC_CHECK(hipMemcpyAsync(n, B->hsdyn + 2, sizeof(int), hipMemcpyDeviceToHost, stream));
    GFSDC_CHECK(hipStreamSynchronize(stream));
    return 0;
}

// init_iau (iau_module.f90:20-81) with the increments already formed by the
// caller (analysis - first guess); each field has a trailing nfiles dimension
// after the set_state layout. nfiles = 0 switches the forcing off.
template <typename T>
int Engine<T>::iau_set(int nfiles, const double *fhrs, double delthrs, const void *vrt, const void *div,
                       const void *tv, const void *trac, const void *lnps, int dtype, int loc) {
    DycoreBuffers *B = dyn;
    if (!B) {
        set_error("context has no dycore");
        return GFSDC_ESTATE;
    }
    void *old[] = {B->iau_hrs, B->iau_inc, B->iau_F};
    GFSDC_CHECK(hipStreamSynchronize(stream));
    for (void *q : old)
        if (q) (void)hipFree(q);
    B->iau_hrs = nullptr;
    B->iau_inc = B->iau_F = nullptr;
    B->iau_n = 0;
    drop_graph(B);
    if (nfiles == 0) return 0;
    // iau_module.f90:38-51: two or more files at a constant spacing
    if (nfiles < 2 || !fhrs) {
        set_error("iau needs at least two increment times");
        return GFSDC_EINVAL;
    }
    for (int n = 1; n < nfiles; n++)
        if (!(fhrs[n] > fhrs[n - 1]) || fhrs[n] - fhrs[n - 1] != fhrs[1] - fhrs[0]) {
            set_error("iau increment times must increase at a constant spacing");
            return GFSDC_EINVAL;
        }
    if (!(delthrs > 0)) {
        set_error("iau_delthrs must be > 0");
        return GFSDC_EINVAL;
    }
    if (!vrt || !div || !tv || !lnps || (B->ntr > 0 && !trac)) {
        set_error("iau increments need vrt, div, tv, lnps (and trac when ntrac > 0)");
        return GFSDC_EINVAL;
    }
    const int nl = B->nl, nlm = plan.nlm, nm = B->nm;
    const long len = (long)nlm * B->nfs * nm;  // complex values per state
    int rc;
    if ((rc = dupload<double>((void **)&B->iau_hrs, std::vector<double>(fhrs, fhrs + nfiles), stream))) return rc;
    B->iau_inc = dalloc<cplx<T>>((size_t)len * nfiles);
    B->iau_F = dalloc<cplx<T>>((size_t)len);
    if (!B->iau_inc || !B->iau_F) {
        set_error("device allocation failed for the iau increments");
        return GFSDC_ENOMEM;
    }
    const size_t esz = dtype == GFSDC_DT_F32 ? 4 : 8;
    const void *const parts[5] = {vrt, div, tv, B->ntr ? trac : nullptr, lnps};
    const int nfr[5] = {nl, nl, nl, B->ntr * nl, 1};
    for (int f = 0; f < nfiles; f++) {
        const void *at[5];
        for (int i = 0; i < 5; i++) {
            if (nfr[i] && !parts[i]) {
                set_error("null buffer");
                return GFSDC_EINVAL;
            }
            at[i] = nfr[i] ? (const char *)parts[i] + (size_t)f * nfr[i] * nm * nlm * 2 * esz : nullptr;
        }
        if ((rc = pack_in((cplx<T> *)B->iau_inc + (long)f * len, at, dtype, loc))) return rc;
        GFSDC_CHECK(hipStreamSynchronize(stream));
    }
    B->iau_n = nfiles;
    B->iau_dt = delthrs * 3600.;
    return 0;
}

// set_dfi_wts (run.f90:567-587): Lanczos-windowed sinc over the 2 N + 1
// states of the window, normalised to sum 1 (pi the default-real acos(-1.))
static std::vector<double> dfi_weights(int N) {
    const double pi = (double)(float)M_PI;
    std::vector<double> w(2 * N + 1, 1.0);
    double tot = 0.0;
    for (int k = 0; k <= 2 * N; k++) {
        if (k != N) {
            const double sx = pi * (k - N) / N, wx = pi * (k - N) / (N + 1);
            w[k] = std::sin(wx) / wx * std::sin(sx) / sx;
        }
        tot += w[k];
    }
    for (double &x : w) x /= tot;
    return w;
}

// Digital filter initialisation, run.f90:58-145: 2 ntdfi steps with the
// weighted average of the window's 2 ntdfi + 1 states accumulated on the
// device, the state replaced by it and the clock set to the window's middle.
template <typename T> int Engine<T>::dfi(int ntdfi, int use_graph) {
    DycoreBuffers *B = dyn;
    if (!B) {
        set_error("context has no dycore");
        return GFSDC_ESTATE;
    }
    if (ntdfi < 1) {
        set_error("ntdfi must be >= 1");
        return GFSDC_EINVAL;
    }
    const std::vector<double> w = dfi_weights(ntdfi);
    const long n = 2L * plan.nlm * B->nfs * B->nm;
    double t0;
    int rc;
    if ((rc = get_time(&t0))) return rc;
    T *acc = dalloc<T>((size_t)n);
    if (!acc) {
        set_error("device allocation failed for the dfi average");
        return GFSDC_ENOMEM;
    }
    hipLaunchKernelGGL(k_axpby<T>, dim3(1024), dim3(256), 0, stream, acc, (const T *)B->spec, (T)w[0], (T)0, n);
    for (int nt = 1; nt <= 2 * ntdfi && !rc; nt++) {
        rc = advance(1, use_graph);
        hipLaunchKernelGGL(k_axpby<T>, dim3(1024), dim3(256), 0, stream, acc, (const T *)B->spec, (T)w[nt], (T)1,
                           n);
    }
    if (!rc) {
        hipLaunchKernelGGL(k_copy<T>, dim3(2048), dim3(256), 0, stream, (T *)B->spec, (const T *)acc, n);
        if (hipGetLastError() != hipSuccess) rc = GFSDC_EHIP;
    }
    (void)hipStreamSynchronize(stream);
    (void)hipFree(acc);
    if (rc) {
        if (rc == GFSDC_EHIP) set_error("dfi kernel launch failed");
        return rc;
    }
    return set_time(t0 + ntdfi * cfg.dt);
}

// ---- stochastic physics (stoch_data.f90:37-238 init_stochdata) -----------------
// vertical factors: the sigma 0.10 -> 0.05 taper (svc :63-71, sppt :85-93,
// addnoise :128-136) and exp((sl - 1) / 0.2) for shum (:103-106)
static std::vector<double> stoch_vfact(int kd, const std::vector<double> &sl) {
    std::vector<double> vf(sl.size());
    const double b = SGLF(0.10), t = SGLF(0.05);
    for (size_t k = 0; k < sl.size(); k++) {
        if (kd == 2) {
            vf[k] = std::exp((sl[k] - 1.) / SGLF(0.2));
            continue;
        }
        vf[k] = 1.0;
        if (sl[k] < b && sl[k] > t) vf[k] = (sl[k] - t) / (b - t);
        else if (sl[k] <= t) vf[k] = 0.0;
    }
    return vf;
}

template <typename T> int Engine<T>::stoch_init(const gfsdc_stoch_cfg *sc) {
    DycoreBuffers *B = dyn;
    if (!B || !sc) {
        set_error(!B ? "context has no dycore" : "null argument");
        return !B ? GFSDC_ESTATE : GFSDC_EINVAL;
    }
    const double amp[4] = {sc->svc, sc->sppt, sc->shum, sc->addnoise};
    const double tau[4] = {sc->svc_tau, sc->sppt_tau, sc->shum_tau, sc->addnoise_tau};
    const double lsc[4] = {sc->svc_lscale, sc->sppt_lscale, sc->shum_lscale, sc->addnoise_lscale};
    const int seed[4] = {sc->iseed_svc, sc->iseed_sppt, sc->iseed_shum, sc->iseed_addnoise};
    for (int kd = 0; kd < 4; kd++)
        if (amp[kd] > FLT_MIN && (!(tau[kd] > 0) || lsc[kd] < 0)) {
            set_error("a stochastic scheme with amplitude > 0 needs tau > 0 and lscale >= 0");
            return GFSDC_EINVAL;
        }
    if (sc->addnoise > FLT_MIN && !sc->addnoise_vrtonly) {
        set_error("addnoise_vrtonly = 0 needs the GSI balance operator file (berror_stats), which is not supported");
        return GFSDC_EINVAL;
    }
    if (sc->addnoise > FLT_MIN && sc->addnoise_dissfact && !(sc->addnoise_lscale > 0)) {
        set_error("addnoise_dissfact needs addnoise_lscale > 0");
        return GFSDC_EINVAL;
    }
    GFSDC_CHECK(hipStreamSynchronize(stream));
    void *old[] = {B->st_pat2, B->st_pat[3], B->st_var, B->st_vf, B->st_ctr, B->st_grd, B->sd_pat, B->rf0,
                   B->vcg, B->sd_vc, B->rf1, B->an_w, B->an_g, B->an_sm, B->sd_an, B->ad_an, B->rf_an};
    for (void *q : old)
        if (q) (void)hipFree(q);
    B->st_pat2 = B->st_pat[0] = B->st_pat[1] = B->st_pat[2] = B->st_pat[3] = nullptr;
    B->st_var = nullptr;
    B->st_vf = B->st_grd = B->vcg = B->an_w = B->an_g = B->an_sm = nullptr;
    B->st_ctr = nullptr;
    B->sd_pat = B->sd_vc = B->sd_an = nullptr;
    B->ad_an = nullptr;
    B->rf0 = B->rf1 = B->rf_an = nullptr;
    B->vc_on = false;
    for (int kd = 0; kd < 4; kd++) B->st_on[kd] = 0;
    drop_graph(B);
    B->sc = *sc;
    const int nl = B->nl, nm = B->nm, nlm = plan.nlm, T_ = plan.ntrunc;
    const long ng = B->ng;
    bool any = false;
    for (int kd = 0; kd < 4; kd++) {
        B->st_on[kd] = amp[kd] > FLT_MIN;
        any = any || B->st_on[kd];
    }
    B->vc_on = sc->vcamp > FLT_MIN || sc->svc > FLT_MIN;
    const int nf = nm * nl;
    int rc;
    if (any) {
        std::vector<double> var(4 * (size_t)nlm, 0.0), vf(4 * (size_t)nl, 0.0);
        for (int kd = 0; kd < 4; kd++) {
            if (!B->st_on[kd]) continue;
            const std::vector<double> v = pattern_varspec(T_, lsc[kd], cfg.rerth), f = stoch_vfact(kd, B->sl);
            std::copy(v.begin(), v.end(), var.begin() + (long)kd * nlm);
            std::copy(f.begin(), f.end(), vf.begin() + (long)kd * nl);
            B->st_nf[kd] = kd == 3 ? nl : 1;
            B->st_phi[kd] = std::exp(-cfg.dt / tau[kd]);
            B->st_sd[kd] = amp[kd];
            B->st_seed[kd] = (unsigned long long)(long long)seed[kd];
        }
        void *pv;
        if ((rc = dupload<double>(&pv, var, stream))) return rc;
        B->st_var = (double *)pv;
        if ((rc = dupload<T>(&B->st_vf, castv<T>(vf), stream))) return rc;
        B->st_pat2 = dalloc<cplx<T>>(3 * (size_t)nm * nlm);
        B->st_ctr = dalloc<unsigned long long>(4);
        B->st_grd = dalloc<T>(3 * (size_t)nm * ng);
        std::vector<SynthDesc> sd(3 * (size_t)nm);
        for (int i = 0; i < 3 * nm; i++) sd[i] = SynthDesc{SK_COPY, i, -1, 1.0, 0.0, 0, 0};
        if ((rc = dupload<SynthDesc>(&pv, sd, stream))) return rc;
        B->sd_pat = (SynthDesc *)pv;
        if ((rc = dupload<unsigned char>(&pv, std::vector<unsigned char>(std::max(3 * nm, 3 * nf), 0), stream)))
            return rc;
        B->rf0 = (unsigned char *)pv;
        if (!B->st_pat2 || !B->st_ctr || !B->st_grd) {
            set_error("device allocation failed for the stochastic patterns");
            return GFSDC_ENOMEM;
        }
        GFSDC_CHECK(hipMemsetAsync(B->st_pat2, 0, sizeof(cplx<T>) * 3 * nm * nlm, stream));
        GFSDC_CHECK(hipMemsetAsync(B->st_ctr, 0, 4 * sizeof(unsigned long long), stream));
        for (int kd = 0; kd < 3; kd++) B->st_pat[kd] = (cplx<T> *)B->st_pat2 + (long)kd * nm * nlm;
    }
    if (B->st_on[3]) {
        B->st_pat[3] = dalloc<cplx<T>>((size_t)nf * nlm);
        B->an_w = dalloc<cplx<T>>(3 * (size_t)nf * nlm);
        B->an_g = dalloc<T>(3 * (size_t)nf * ng);
        if (!B->st_pat[3] || !B->an_w || !B->an_g) {
            set_error("device allocation failed for the additive noise");
            return GFSDC_ENOMEM;
        }
        GFSDC_CHECK(hipMemsetAsync(B->st_pat[3], 0, sizeof(cplx<T>) * nf * nlm, stream));
        GFSDC_CHECK(hipMemsetAsync(B->an_w, 0, sizeof(cplx<T>) * 3 * nf * nlm, stream));
        // getstochforcing :269-276: Gaussian smoothing at three times the noise scale
        std::vector<double> sm(nlm, 1.0);
        if (sc->addnoise_dissfact) {
            const double rnn1 = 2. * cfg.rerth / (3. * sc->addnoise_lscale), rnn0 = rnn1 * (rnn1 + 1.);
            for (int m = 0, k = 0; m <= T_; m++)
                for (int n = m; n <= T_; n++, k++) sm[k] = std::exp(-(n * (n + 1.) / rnn0));
        }
        if ((rc = dupload<T>(&B->an_sm, castv<T>(sm), stream))) return rc;
        // descriptors: [ud, vd, psi] grids of the wind of (-disspec vrt, -disspec div)
        // and of the noise, then group-1 and group-0 copies
        std::vector<SynthDesc> d(5 * (size_t)nf);
        std::vector<unsigned char> rf(3 * (size_t)nf, 0);
        std::vector<AnalDesc> ad(nf);
        const double a = cfg.rerth;
        for (int i = 0; i < nf; i++) {
            d[i] = SynthDesc{SK_UHAT, nf + i, 2 * nf + i, a, a, 1, 1};   // getuv (stoch_data.f90:280)
            d[nf + i] = SynthDesc{SK_VHAT, nf + i, 2 * nf + i, a, a, 1, 1};
            d[2 * nf + i] = SynthDesc{SK_COPY, i, -1, 1.0, 0.0, 0, 0};
            d[3 * nf + i] = SynthDesc{SK_COPY, nf + i, -1, 1.0, 0.0, 0, 0};
            d[4 * nf + i] = SynthDesc{SK_COPY, i, -1, 1.0, 0.0, 0, 0};
            rf[i] = rf[nf + i] = 1;
            ad[i] = AnalDesc{AK_COPY, i, -1, 1.0, 0, 0, -1, 0.0};
        }
        void *pv;
        if ((rc = dupload<SynthDesc>(&pv, d, stream))) return rc;
        B->sd_an = (SynthDesc *)pv;
        if ((rc = dupload<AnalDesc>(&pv, ad, stream))) return rc;
        B->ad_an = (AnalDesc *)pv;
        if ((rc = dupload<unsigned char>(&pv, rf, stream))) return rc;
        B->rf_an = (unsigned char *)pv;
    }
    if (B->vc_on) {
        B->vcg = dalloc<T>(2 * (size_t)nf * ng);
        if (!B->vcg) {
            set_error("device allocation failed for the vorticity gradient");
            return GFSDC_ENOMEM;
        }
        // getgrad(vrtspec) of each level: sphtor_to_spat(0, vrt) / a
        std::vector<SynthDesc> d(2 * (size_t)nf);
        for (int mem = 0; mem < nm; mem++)
            for (int k = 0; k < nl; k++) {
                d[(size_t)mem * 2 * nl + k] = SynthDesc{SK_UHAT, -1, mem * B->nfs + k, 0.0, 1.0 / cfg.rerth, 0, 0};
                d[(size_t)mem * 2 * nl + nl + k] = SynthDesc{SK_VHAT, -1, mem * B->nfs + k, 0.0, 1.0 / cfg.rerth, 0, 0};
            }
        void *pv;
        if ((rc = dupload<SynthDesc>(&pv, d, stream))) return rc;
        B->sd_vc = (SynthDesc *)pv;
        if ((rc = dupload<unsigned char>(&pv, std::vector<unsigned char>(2 * (size_t)nf, 1), stream))) return rc;
        B->rf1 = (unsigned char *)pv;
    }
    if (any) {
        // stdev x varspectrum x noise, then 5 e-folding times of spin-up, and the grids
        Step<T> st{*this, *B, *(Work<T> *)B->Work, stream};
        for (int kd = 0; kd < 4; kd++) {
            if (!B->st_on[kd]) continue;
            st.stoch_advance(kd, 0.0, B->st_sd[kd]);
            const int nspinup = (int)(5.0 * tau[kd] / cfg.dt);
            for (int i = 0; i < nspinup; i++)
                st.stoch_advance(kd, B->st_phi[kd], B->st_sd[kd] * std::sqrt(1.0 - B->st_phi[kd] * B->st_phi[kd]));
        }
        st.stoch_grids();
    }
    GFSDC_CHECK(hipGetLastError());
    GFSDC_CHECK(hipStreamSynchronize(stream));
    return 0;
}

template <typename T> int Engine<T>::get_stoch(int which, void *out, int dtype, int loc) {
    DycoreBuffers *B = dyn;
    if (!B) {
        set_error("context has no dycore");
        return GFSDC_ESTATE;
    }
    const int kd = which < 3 ? which : which < 6 ? which - 3 : 3;
    if (which < 0 || which > 7 || !B->st_on[kd]) {
        set_error("no such stochastic field, or its scheme is off");
        return GFSDC_EINVAL;
    }
    const size_t nm = B->nm, nlm = plan.nlm, nl = B->nl;
    if (which < 3) return output((const T *)B->st_grd + (long)which * nm * B->ng, out, nm * B->ng, dtype, loc, 1);
    if (which < 6) return output((const T *)B->st_pat[kd], out, 2 * nm * nlm, dtype, loc, 1);
    return output((const T *)(which == 6 ? B->st_pat[3] : B->an_w), out, 2 * nm * nl * nlm, dtype, loc, 1);
}

// ---- checkpoint / resume ----------------------------------------------------
// One contiguous image of everything the next steps read that the caller did
// not configure: the spectral state, orography, pdryini, the clock, the
// stochastic pattern and its counter, the judge counter. Operators, the iau
// increments and learned weights are configuration and are not included.
namespace {
struct CkptHeader {
    char magic[8];
    int32_t version, esz, nlm, nfs, nm, nl, ntr, has_pattern, has_judge, stoch_mask;
    double time;
    uint64_t tpat_ctr, jctr, bctr;
    char pad[128 - 8 - 11 * 4 - 8 - 3 * 8];
};
static_assert(sizeof(CkptHeader) == 128, "checkpoint header is 128 bytes");
const char CKPT_MAGIC[8] = {'G', 'F', 'S', 'D', 'C', 'C', 'K', '1'};
}  // namespace

static int stoch_mask(const DycoreBuffers *B) {
    int m = 0;
    for (int kd = 0; kd < 4; kd++)
        if (B->st_on[kd]) m |= 1 << kd;
    return m;
}

template <typename T> size_t Engine<T>::checkpoint_size() {
    DycoreBuffers *B = dyn;
    if (!B) return 0;
    const size_t c = sizeof(cplx<T>), nlm = plan.nlm, nm = B->nm;
    size_t n = sizeof(CkptHeader) + c * nlm * B->nfs * nm + c * nlm * nm + 8 * nm + (B->tpat ? c * nlm * nm : 0);
    for (int kd = 0; kd < 4; kd++)
        if (B->st_on[kd]) n += c * nlm * nm * B->st_nf[kd];
    return n + (stoch_mask(B) ? 4 * 8 : 0);
}

template <typename T> int Engine<T>::checkpoint_save(void *buf, size_t nbytes, int loc) {
    DycoreBuffers *B = dyn;
    if (!B) {
        set_error("context has no dycore");
        return GFSDC_ESTATE;
    }
    if (!buf || nbytes < checkpoint_size()) {
        set_error("checkpoint buffer is smaller than gfsdc_checkpoint_size()");
        return GFSDC_EINVAL;
    }
    CkptHeader h;
    std::memset(&h, 0, sizeof(h));
    std::memcpy(h.magic, CKPT_MAGIC, 8);
    h.version = 1;
    h.esz = (int32_t)sizeof(T);
    h.nlm = plan.nlm;
    h.nfs = B->nfs;
    h.nm = B->nm;
    h.nl = B->nl;
    h.ntr = B->ntr;
    h.has_pattern = B->tpat ? 1 : 0;
    h.has_judge = B->jctr ? 1 : 0;
    h.stoch_mask = stoch_mask(B);
    h.bctr = B->bctr;
    GFSDC_CHECK(hipMemcpyAsync(&h.time, B->clock, sizeof(double), hipMemcpyDeviceToHost, stream));
    if (B->tpat_ctr)
        GFSDC_CHECK(hipMemcpyAsync(&h.tpat_ctr, B->tpat_ctr, 8, hipMemcpyDeviceToHost, stream));
    if (B->jctr) GFSDC_CHECK(hipMemcpyAsync(&h.jctr, B->jctr, 8, hipMemcpyDeviceToHost, stream));
    GFSDC_CHECK(hipStreamSynchronize(stream));
    const hipMemcpyKind k = loc == GFSDC_DEVICE ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost;
    char *o = (char *)buf;
    GFSDC_CHECK(hipMemcpyAsync(o, &h, sizeof(h), loc == GFSDC_DEVICE ? hipMemcpyHostToDevice : hipMemcpyHostToHost,
                               stream));
    o += sizeof(h);
    const size_t c = sizeof(cplx<T>), nlm = plan.nlm, nm = B->nm;
    struct Sec {
        const void *p;
        size_t n;
    } secs[] = {{B->spec, c * nlm * B->nfs * nm}, {B->topo, c * nlm * nm}, {B->pdryini, 8 * nm},
                {B->tpat, B->tpat ? c * nlm * nm : 0},
                {B->st_pat[0], B->st_on[0] ? c * nlm * nm : 0}, {B->st_pat[1], B->st_on[1] ? c * nlm * nm : 0},
                {B->st_pat[2], B->st_on[2] ? c * nlm * nm : 0},
                {B->st_pat[3], B->st_on[3] ? c * nlm * nm * (size_t)B->nl : 0}, {B->st_ctr, h.stoch_mask ? (size_t)32 : (size_t)0}};
    for (auto &sc : secs) {
        if (!sc.n) continue;
        GFSDC_CHECK(hipMemcpyAsync(o, sc.p, sc.n, k, stream));
        o += sc.n;
    }
    GFSDC_CHECK(hipStreamSynchronize(stream));
    return 0;
}

template <typename T> int Engine<T>::checkpoint_load(const void *buf, size_t nbytes, int loc) {
    DycoreBuffers *B = dyn;
    if (!B) {
        set_error("context has no dycore");
        return GFSDC_ESTATE;
    }
    CkptHeader h;
    if (!buf || nbytes < sizeof(h)) {
        set_error("checkpoint buffer too small");
        return GFSDC_EINVAL;
    }
    GFSDC_CHECK(hipMemcpyAsync(&h, buf, sizeof(h), loc == GFSDC_DEVICE ? hipMemcpyDeviceToHost : hipMemcpyHostToHost,
                               stream));
    GFSDC_CHECK(hipStreamSynchronize(stream));
    if (std::memcmp(h.magic, CKPT_MAGIC, 8) != 0 || h.version != 1) {
        set_error("not a gfsdc checkpoint (bad magic or version)");
        return GFSDC_EINVAL;
    }
    if (h.esz != (int32_t)sizeof(T) || h.nlm != plan.nlm || h.nfs != B->nfs || h.nm != B->nm || h.nl != B->nl ||
        h.ntr != B->ntr || h.has_pattern != (B->tpat ? 1 : 0) || h.stoch_mask != stoch_mask(B)) {
        set_error("checkpoint was written by a context of another precision, grid, level count, tracer "
                  "count, member count or pattern setting");
        return GFSDC_EINVAL;
    }
    if (nbytes < checkpoint_size()) {
        set_error("checkpoint buffer is shorter than its header says");
        return GFSDC_EINVAL;
    }
    const hipMemcpyKind k = loc == GFSDC_DEVICE ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice;
    const char *o = (const char *)buf + sizeof(h);
    const size_t c = sizeof(cplx<T>), nlm = plan.nlm, nm = B->nm;
    int rc = ensure_stage(2, c * nlm * nm);
    if (rc) return rc;
    struct Sec {
        void *p;
        size_t n;
    } secs[] = {{B->spec, c * nlm * B->nfs * nm}, {stage[2], c * nlm * nm}, {B->pdryini, 8 * nm},
                {B->tpat, B->tpat ? c * nlm * nm : 0},
                {B->st_pat[0], B->st_on[0] ? c * nlm * nm : 0}, {B->st_pat[1], B->st_on[1] ? c * nlm * nm : 0},
                {B->st_pat[2], B->st_on[2] ? c * nlm * nm : 0},
                {B->st_pat[3], B->st_on[3] ? c * nlm * nm * (size_t)B->nl : 0}, {B->st_ctr, h.stoch_mask ? (size_t)32 : (size_t)0}};
    for (auto &sc : secs) {
        if (!sc.n) continue;
        GFSDC_CHECK(hipMemcpyAsync(sc.p, o, sc.n, k, stream));
        o += sc.n;
    }
    GFSDC_CHECK(hipMemcpyAsync(B->clock, &h.time, sizeof(double), hipMemcpyHostToDevice, stream));
    if (B->tpat_ctr) GFSDC_CHECK(hipMemcpyAsync(B->tpat_ctr, &h.tpat_ctr, 8, hipMemcpyHostToDevice, stream));
    if (B->jctr && h.has_judge) GFSDC_CHECK(hipMemcpyAsync(B->jctr, &h.jctr, 8, hipMemcpyHostToDevice, stream));
    B->bctr = h.bctr;
    GFSDC_CHECK(hipStreamSynchronize(stream));
    // orography and its gradient (dyn_init.f90:84)
    return set_topo(stage[2], sizeof(T) == 8 ? GFSDC_DT_F64 : GFSDC_DT_F32, GFSDC_DEVICE);
}

// tendencies of a physics package on the current grid fields, without the
// state update; tphys in the state layout -> caller buffers
template <typename T>
int Engine<T>::pack_tphys(void *dvrt, void *ddiv, void *dtv, void *dtrac, int dtype, int loc) {
    DycoreBuffers *B = dyn;
    GFSDC_CHECK(hipGetLastError());
    void *const parts[5] = {dvrt, ddiv, dtv, dtrac, nullptr};
    return pack_out(B->tphys, parts, dtype, loc);
}

template <typename T> int Engine<T>::hs_phytend(void *dvrt, void *ddiv, void *dtv, int dtype, int loc) {
    DycoreBuffers *B = dyn;
    if (!B) {
        set_error("context has no dycore");
        return GFSDC_ESTATE;
    }
    Step<T> st{*this, *B, *(Work<T> *)B->Work, stream};
    dim3 g((unsigned)((B->ng + 255) / 256), B->nm * HS_LCH);
    hipLaunchKernelGGL(k_hs_columns<T>, g, dim3(256), 0, stream, (const T *)B->gsyn, (const T *)B->psg,
                       (T *)B->gan, (const T *)B->ak, (const T *)B->bk, (const T *)B->sinlat, B->pdryini, B->pmean,
                       B->nl, B->ntr, B->nsyn, B->nm, B->ng, plan.nlon, (T)(cfg.rd / cfg.cp), 0,
                       (const int *)nullptr);
    st.analyse(B->adesc_hs, B->rflag_hs, B->nm * B->nhs, (cplx<T> *)B->tphys);
    return pack_tphys(dvrt, ddiv, dtv, nullptr, dtype, loc);
}

template <typename T>
int Engine<T>::simple_phytend(void *dvrt, void *ddiv, void *dtv, void *dtrac, int dtype, int loc) {
    DycoreBuffers *B = dyn;
    if (!B) {
        set_error("context has no dycore");
        return GFSDC_ESTATE;
    }
    if (cfg.physics != GFSDC_PHYS_SIMPLE) {
        set_error("simple_phytend needs a context created with physics = GFSDC_PHYS_SIMPLE");
        return GFSDC_ESTATE;
    }
    Step<T> st{*this, *B, *(Work<T> *)B->Work, stream};
    st.simple_columns();
    st.analyse(B->adesc_sp, B->rflag_sp, B->nm * B->nsp, (cplx<T> *)B->tphys);
    return pack_tphys(dvrt, ddiv, dtv, dtrac, dtype, loc);
}

template <typename T> int Engine<T>::get_grid(int which, void *out, int dtype, int loc) {
    DycoreBuffers *B = dyn;
    if (!B) {
        set_error("context has no dycore");
        return GFSDC_ESTATE;
    }
    if (B->grids_partial) {
        set_error("the last step ran the lean Held-Suarez physics pass (profile_step), which keeps only the "
                  "grids its forcing reads: advance or getdyntend first");
        return GFSDC_ESTATE;
    }
    const int nl = B->nl, nm = B->nm;
    const long ng = B->ng;
    const T *src = nullptr;
    long per = 0, mstride = 0;
    switch (which) {
    case GF_UG: src = (const T *)B->gsyn; per = nl * ng; mstride = (long)B->nsyn * ng; break;
    case GF_VG: src = (const T *)B->gsyn + nl * ng; per = nl * ng; mstride = (long)B->nsyn * ng; break;
    case GF_VRT: src = (const T *)B->gsyn + 2 * nl * ng; per = nl * ng; mstride = (long)B->nsyn * ng; break;
    case GF_DIV: src = (const T *)B->gsyn + 3 * nl * ng; per = nl * ng; mstride = (long)B->nsyn * ng; break;
    case GF_TV: src = (const T *)B->gsyn + 4 * nl * ng; per = nl * ng; mstride = (long)B->nsyn * ng; break;
    case GF_DLNPDT: src = (const T *)B->dlnpdt; per = nl * ng; mstride = per; break;
    case GF_ETADOT: src = (const T *)B->etadot; per = (nl + 1) * ng; mstride = per; break;
    case GF_PSG: src = (const T *)B->psg; per = ng; mstride = ng; break;
    case GF_DLNPSDT: src = (const T *)B->dlnpsdt; per = ng; mstride = ng; break;
    case GF_DLNPSDX: src = (const T *)B->gsyn + (7L + 3L * B->ntr) * nl * ng + ng; per = ng; mstride = (long)B->nsyn * ng; break;
    case GF_DLNPSDY: src = (const T *)B->gsyn + (7L + 3L * B->ntr) * nl * ng + 2 * ng; per = ng; mstride = (long)B->nsyn * ng; break;
    case GF_TRACER:
        if (B->ntr == 0) {
            set_error("no tracers (ntrac == 0)");
            return GFSDC_EINVAL;
        }
        src = (const T *)B->gsyn + 7L * nl * ng; per = (long)B->ntr * nl * ng; mstride = (long)B->nsyn * ng; break;
    case GF_PRECIP: src = (const T *)B->precip; per = ng; mstride = ng; break;
    case GF_PWAT: src = (const T *)B->pwat; per = ng; mstride = ng; break;
    default:
        set_error("unknown grid field");
        return GFSDC_EINVAL;
    }
    int rc = ensure_stage(3, sizeof(T) * per * nm);
    if (rc) return rc;
    hipLaunchKernelGGL(k_grid_gather<T>, dim3((unsigned)((per * nm + 255) / 256)), dim3(256), 0, stream, src,
                       mstride, (T *)stage[3], per, nm);
    GFSDC_CHECK(hipGetLastError());
    return output((const T *)stage[3], out, (size_t)per * nm, dtype, loc, 1);
}

template <typename T>
int Engine<T>::get_semimp(double *a, double *b, double *sv, double *tor, double *d) {
    DycoreBuffers *B = dyn;
    if (!B) {
        set_error("context has no dycore");
        return GFSDC_ESTATE;
    }
    if (a) std::copy(B->amhyb.begin(), B->amhyb.end(), a);
    if (b) std::copy(B->bmhyb.begin(), B->bmhyb.end(), b);
    if (sv) std::copy(B->svhyb.begin(), B->svhyb.end(), sv);
    if (tor) std::copy(B->tor_hyb.begin(), B->tor_hyb.end(), tor);
    if (d) std::copy(B->d_hyb_m.begin(), B->d_hyb_m.end(), d);
    return 0;
}

template <typename T> int Engine<T>::get_damp(double *ds, double *df, double *dm) {
    DycoreBuffers *B = dyn;
    if (!B) {
        set_error("context has no dycore");
        return GFSDC_ESTATE;
    }
    if (ds) std::copy(B->disspec_h.begin(), B->disspec_h.end(), ds);
    if (df) std::copy(B->diff_h.begin(), B->diff_h.end(), df);
    if (dm) std::copy(B->dmp_h.begin(), B->dmp_h.end(), dm);
    return 0;
}

template <typename T> int Engine<T>::step_diag(double *out) {
    DycoreBuffers *B = dyn;
    if (!B) {
        set_error("context has no dycore");
        return GFSDC_ESTATE;
    }
    if (B->grids_partial) {
        set_error("the last step ran the lean Held-Suarez physics pass (profile_step), which keeps only the "
                  "grids its forcing reads: advance or getdyntend first");
        return GFSDC_ESTATE;
    }
    hipLaunchKernelGGL(k_diag<T>, dim3(B->nm), dim3(1024), 0, stream, (const T *)B->gsyn, (const T *)B->psg,
                       (const T *)B->dlnpsdt, (const double *)B->areaw, B->diag, B->nl, B->nsyn, B->ng, plan.nlon);
    GFSDC_CHECK(hipGetLastError());
    GFSDC_CHECK(hipMemcpyAsync(out, B->diag, sizeof(double) * 4 * B->nm, hipMemcpyDeviceToHost, stream));
    GFSDC_CHECK(hipStreamSynchronize(stream));
    return 0;
}

template <typename T> int Engine<T>::set_pdryini(const double *p) {
    if (!dyn) {
        set_error("context has no dycore");
        return GFSDC_ESTATE;
    }
    GFSDC_CHECK(hipMemcpyAsync(dyn->pdryini, p, sizeof(double) * dyn->nm, hipMemcpyHostToDevice, stream));
    GFSDC_CHECK(hipStreamSynchronize(stream));
    return 0;
}

template <typename T> int Engine<T>::get_pdryini(double *p) {
    if (!dyn) {
        set_error("context has no dycore");
        return GFSDC_ESTATE;
    }
    GFSDC_CHECK(hipMemcpyAsync(p, dyn->pdryini, sizeof(double) * dyn->nm, hipMemcpyDeviceToHost, stream));
    GFSDC_CHECK(hipStreamSynchronize(stream));
    return 0;
}

// Resting isothermal state plus random vorticity (counter-based RNG, stream =
// level, index = spectral coefficient; member i uses seed + i).
template <typename T>
int Engine<T>::init_rest_state(double t0, double ps0, double vort_rms, int nmin, int nmax, unsigned long long seed) {
    DycoreBuffers *B = dyn;
    if (!B) {
        set_error("context has no dycore");
        return GFSDC_ESTATE;
    }
    const int nl = B->nl, nm = B->nm, nlm = plan.nlm, T_ = plan.ntrunc;
    const double sq4pi = std::sqrt(4.0 * M_PI);
    std::vector<double> vrt((size_t)nm * nl * nlm * 2, 0.0), tv((size_t)nm * nl * nlm * 2, 0.0),
        lp((size_t)nm * nlm * 2, 0.0), zero((size_t)nm * nl * nlm * 2, 0.0);
    for (int mem = 0; mem < nm; mem++) {
        for (int l = 0; l < nl; l++) {
            double *v = &vrt[((size_t)mem * nl + l) * nlm * 2];
            double ss = 0.0;
            int k = 0;
            for (int m = 0; m <= T_; m++)
                for (int n = m; n <= T_; n++, k++) {
                    if (n < nmin || n > nmax) continue;
                    double u = (double)(rng_u64(seed + mem, (uint64_t)l, (uint64_t)k) >> 11) * 0x1p-53;
                    double th = 2.0 * M_PI * u;
                    v[2 * k] = std::cos(th);
                    v[2 * k + 1] = (m == 0) ? 0.0 : std::sin(th);
                    ss += (m == 0 ? 1.0 : 2.0) * (v[2 * k] * v[2 * k] + v[2 * k + 1] * v[2 * k + 1]);
                }
            double rms = std::sqrt(ss / (4.0 * M_PI));
            double sc = rms > 0 ? vort_rms / rms : 0.0;
            for (int i = 0; i < nlm * 2; i++) v[i] *= sc;
            tv[((size_t)mem * nl + l) * nlm * 2] = t0 * sq4pi;
        }
        lp[(size_t)mem * nlm * 2] = std::log(ps0) * sq4pi;
    }
    int rc = set_state(vrt.data(), zero.data(), tv.data(), nullptr, lp.data(), GFSDC_DT_F64, GFSDC_HOST);
    if (rc) return rc;
    std::vector<double> z(nm, 0.0);
    return set_pdryini(z.data());
}

template <typename T> int Engine<T>::profile_step(char names[][48], double *ms, int nmax) {
    DycoreBuffers *B = dyn;
    if (!B) {
        set_error("context has no dycore");
        return GFSDC_ESTATE;
    }
    for (auto e : B->ev) (void)hipEventDestroy(e);
    B->ev.clear();
    B->evname.clear();
    B->profiling = true;
    Step<T> st{*this, *B, *(Work<T> *)B->Work, stream};
    // the step as advance runs all but its last (lean physics pass where it applies)
    st.lean = st.lean_ok();
    B->grids_partial = st.lean;
    st.mark("start");
    st.step();
    B->profiling = false;
    GFSDC_CHECK(hipStreamSynchronize(stream));
    int n = 0;
    for (size_t i = 1; i < B->ev.size() && n < nmax; i++, n++) {
        float t = 0;
        GFSDC_CHECK(hipEventElapsedTime(&t, B->ev[i - 1], B->ev[i]));
        std::strncpy(names[n], B->evname[i].c_str(), 47);
        names[n][47] = 0;
        ms[n] = t;
    }
    return n;
}

template struct Engine<float>;
template struct Engine<double>;

}  // namespace gfsdc
