// Device-resident Krylov solvers: the Ritz extreme eigenvalue (RitzSolver.cpp:92-297) of one vector and
// the multi-shift CG of the Zolotarev sign (OverlapU.cpp:5-149).  Every scalar of the recurrences lives
// in device memory: a kernel that needs one sums the partial results of the kernel before it (a fixed
// order, the same in every workgroup), so an iteration is a handful of dependent launches and the host
// only looks for the end of the iteration once per batch.
//
// A single vector has a layout of its own, [comp][site] (comp = spin * Nc + colour) with links
// [mu][i][j][site]: consecutive lanes are consecutive sites and nothing is padded to a mode block.
//
// What bounds them is latency: a vector of 8^3 SU(2) is 64 KB, and every phase of an iteration needs
// the sum of the one before.  Measured on MI355X against host scalars and 16-mode fields (a launch of
// two kernels, a copy and a synchronisation per inner product, 124 us per CG iteration and 360 us per
// Ritz iteration): single-mode overlap operator on 12^3 SU(2) 6.22 -> 1.35 ms (four launches of 3.3 - 5.5 us
// per iteration, batches of eight as a graph), Zolotarev step of 16 modes on 8^3 SU(2) with its Ritz bounds 348
// -> 27 ms (five launches of 4.3 - 5.3 us per pair of Ritz iterations, batches of twenty as a graph),
// single-mode Wilson operator on 24^3 SU(3) 627 -> 545 us (stencil 37 -> 6 us; the rest is the 11.3 MB of
// host arrays).
#include "ovl_internal.hpp"

#include <algorithm>

namespace ovl {

namespace {

constexpr int TPB1 = 128;        // threads per workgroup of the single-vector kernels: 64 sites of the stencil
constexpr int POINT_BLOCKS = 256;  // most workgroups (and partial results) of a pointwise kernel
constexpr int PART = 4;          // doubles per partial result

__device__ __forceinline__ double wave_add(double v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// sum of NV values over the workgroup, in every thread (fixed order; called by all threads)
template <int NV> __device__ __forceinline__ void block_sum(double *v)
{
    __shared__ double sh[TPB1 / 64][NV];
    const int w = threadIdx.x / 64;
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k] = wave_add(v[k]);
    __syncthreads();
    if (threadIdx.x % 64 == 0)
#pragma unroll
        for (int k = 0; k < NV; ++k) sh[w][k] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        double r = sh[0][k];
#pragma unroll
        for (int j = 1; j < TPB1 / 64; ++j) r += sh[j][k];
        v[k] = r;
    }
}

template <int NV> __device__ __forceinline__ void put_partial(double *part, double *v)
{
    block_sum<NV>(v);
    if (threadIdx.x == 0)
#pragma unroll
        for (int k = 0; k < NV; ++k) part[(size_t)blockIdx.x * PART + k] = v[k];
}

template <int NV> __device__ __forceinline__ void sum_partials(const double *part, int n, double *v)
{
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k] = 0.0;
    for (int b = threadIdx.x; b < n; b += TPB1)
#pragma unroll
        for (int k = 0; k < NV; ++k) v[k] += part[(size_t)b * PART + k];
    block_sum<NV>(v);
}

// ---------------------------------------------------------------------------------------------
// h_W of one vector.  Two lanes share a site, one per upper spin component sp: after the spin
// projection the two components never mix, so a lane projects, transports and keeps one of them
// (half the loads and half the arithmetic) and the two exchange three complex numbers at the end:
// the terms that sigma_x and sigma_y carry into the other lane's lower component.  Bound by latency
// (one vector of a 24^3 SU(3) lattice is 2.7 MB), so the split is for lanes in flight.
// ---------------------------------------------------------------------------------------------
struct Lat1 {
    int n0, n1, n2, V;
    FastDiv dv_n01, dv_n0;
    double amass;
};

__device__ __forceinline__ unsigned div_by(unsigned n, const FastDiv &f)
{
    return f.d <= 1 ? n : (__umulhi(n, f.mul) >> f.shift);
}

template <int NC, int K, int SG>
__device__ __forceinline__ void hop1_dir(const double2 *__restrict__ in, const double2 *__restrict__ lk, int V, int q,
                                         int sl, int sp, double t, double2 *xu, double2 *xl, double2 *xo)
{
    // q: neighbour site, sl: site of the link; upper component sp, lower partner 1 - sp (sigma_x,
    // sigma_y) or sp (sigma_z); t = +1 (sp = 0) or -1
    const int lp = 2 + (K == 2 ? sp : 1 - sp);
    double2 h[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const double2 u = in[(size_t)(sp * NC + c) * V + q], l = in[(size_t)(lp * NC + c) * V + q];
        if constexpr (K == 0) h[c] = make_double2(u.x - SG * l.y, u.y + SG * l.x);
        else if constexpr (K == 1) h[c] = make_double2(u.x + SG * t * l.x, u.y + SG * t * l.y);
        else h[c] = make_double2(u.x - SG * t * l.y, u.y + SG * t * l.x);
    }
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        double ar = 0, ai = 0;
#pragma unroll
        for (int j = 0; j < NC; ++j) {
            const double2 u = lk[(size_t)(SG > 0 ? i * NC + j : j * NC + i) * V + sl];
            const double ui = SG > 0 ? u.y : -u.y;
            ar = __builtin_fma(u.x, h[j].x, ar);
            ar = __builtin_fma(-ui, h[j].y, ar);
            ai = __builtin_fma(u.x, h[j].y, ai);
            ai = __builtin_fma(ui, h[j].x, ai);
        }
        xu[i].x -= ar;
        xu[i].y -= ai;
        if constexpr (K == 0) { xo[i].x -= SG * ai; xo[i].y += SG * ar; }
        else if constexpr (K == 1) { xo[i].x -= SG * t * ar; xo[i].y -= SG * t * ai; }
        else { xl[i].x -= SG * t * ai; xl[i].y += SG * t * ar; }
    }
}

// components u = h_W(in)[sp], l = h_W(in)[2 + sp] at site s (all lanes of the wavefront take part)
template <int NC>
__device__ __forceinline__ void hop1_site(const double2 *__restrict__ in, const double2 *__restrict__ links,
                                          const Lat1 &g, int s, int sp, double2 *u, double2 *l)
{
    constexpr int NN = NC * NC;
    const int V = g.V;
    const int z = (int)div_by((unsigned)s, g.dv_n01), rem = s - z * g.n0 * g.n1;
    const int y = (int)div_by((unsigned)rem, g.dv_n0), x = rem - y * g.n0;
    const double t = sp ? -1.0 : 1.0;
    double2 xo[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const double2 a = in[(size_t)(sp * NC + c) * V + s], b = in[(size_t)((2 + sp) * NC + c) * V + s];
        u[c] = make_double2(g.amass * a.x, g.amass * a.y);
        l[c] = make_double2(g.amass * b.x, g.amass * b.y);
        xo[c] = make_double2(0.0, 0.0);
    }
    const int xp = s + (x + 1 == g.n0 ? 1 - g.n0 : 1), xm = s + (x == 0 ? g.n0 - 1 : -1);
    const int yp = s + (y + 1 == g.n1 ? (1 - g.n1) * g.n0 : g.n0), ym = s + (y == 0 ? (g.n1 - 1) * g.n0 : -g.n0);
    const int n01 = g.n0 * g.n1;
    const int zp = s + (z + 1 == g.n2 ? (1 - g.n2) * n01 : n01), zm = s + (z == 0 ? (g.n2 - 1) * n01 : -n01);
    const double2 *lx = links, *ly = links + (size_t)NN * V, *lz = links + (size_t)2 * NN * V;
    hop1_dir<NC, 0, 1>(in, lx, V, xp, s, sp, t, u, l, xo);
    hop1_dir<NC, 0, -1>(in, lx, V, xm, xm, sp, t, u, l, xo);
    hop1_dir<NC, 1, 1>(in, ly, V, yp, s, sp, t, u, l, xo);
    hop1_dir<NC, 1, -1>(in, ly, V, ym, ym, sp, t, u, l, xo);
    hop1_dir<NC, 2, 1>(in, lz, V, zp, s, sp, t, u, l, xo);
    hop1_dir<NC, 2, -1>(in, lz, V, zm, zm, sp, t, u, l, xo);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        l[c].x += __shfl_xor(xo[c].x, 32, 64);
        l[c].y += __shfl_xor(xo[c].y, 32, 64);
        u[c].x *= 0.5;
        u[c].y *= 0.5;
        l[c].x *= -0.5;
        l[c].y *= -0.5;
    }
}

// lane -> (site, upper component): a wavefront is 32 consecutive sites, sp = 0 then sp = 1
__device__ __forceinline__ bool site1(int V, int &s, int &sp)
{
    const int lane = threadIdx.x % 64;
    s = (blockIdx.x * (TPB1 / 64) + threadIdx.x / 64) * 32 + lane % 32;
    sp = lane / 32;
    const bool ok = s < V;
    if (!ok) s = V - 1;
    return ok;
}

__device__ __forceinline__ double2 cxmul(double ar, double ai, double2 b)
{
    return make_double2(ar * b.x - ai * b.y, ar * b.y + ai * b.x);
}

// out = sh h_W(in) + sx G(x), G = gamma0 when x_gamma0 (x null: no second term)
template <int NC>
__global__ __launch_bounds__(TPB1) void k_hop1(const double2 *__restrict__ in, double2 *__restrict__ out,
                                               const double2 *__restrict__ links, Lat1 g, double sh_r, double sh_i,
                                               const double2 *__restrict__ x, double sx_r, double sx_i, int x_gamma0)
{
    int s, sp;
    const bool ok = site1(g.V, s, sp);
    double2 u[NC], l[NC];
    hop1_site<NC>(in, links, g, s, sp, u, l);
    if (!ok) return;
    const double gl = x_gamma0 ? -1.0 : 1.0;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const size_t iu = (size_t)(sp * NC + c) * g.V + s, il = (size_t)((2 + sp) * NC + c) * g.V + s;
        double2 a = cxmul(sh_r, sh_i, u[c]), b = cxmul(sh_r, sh_i, l[c]);
        if (x) {
            const double2 p = cxmul(sx_r, sx_i, x[iu]), q = cxmul(gl * sx_r, gl * sx_i, x[il]);
            a.x += p.x; a.y += p.y;
            b.x += q.x; b.y += q.y;
        }
        out[iu] = a;
        out[il] = b;
    }
}

// ---------------------------------------------------------------------------------------------
// layouts of one vector and of its links
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ bool not_finite(double2 v)
{
    const unsigned long long a = (unsigned long long)__double_as_longlong(v.x), b = (unsigned long long)__double_as_longlong(v.y);
    return (a >> 52 & 0x7ff) == 0x7ff || (b >> 52 & 0x7ff) == 0x7ff;
}

// links [mu][site][i][j] -> [mu][i][j][site]; bad[0] = 1 when an entry is Inf or NaN (bad may be null)
__global__ __launch_bounds__(256) void k_links1(const double2 *__restrict__ src, double2 *__restrict__ dst, int V, int nn,
                                                int *bad)
{
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= 3l * V * nn) return;
    const int s = (int)(i % V);
    const int r = (int)(i / V), e = r % nn, mu = r / nn;
    const double2 v = src[((size_t)mu * V + s) * nn + e];
    dst[i] = v;
    if (bad && not_finite(v)) *bad = 1;
}

// one mode: host AoS [site][colour][spin] <-> [spin][colour][site]
__global__ __launch_bounds__(256) void k_vec1_in(const double2 *__restrict__ aos, double2 *__restrict__ f, int V, int nc,
                                                 int *bad)
{
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= 4l * nc * V) return;
    const int s = (int)(i % V), r = (int)(i / V), sp = r / nc, c = r % nc;
    const double2 v = aos[((size_t)s * nc + c) * 4 + sp];
    f[i] = v;
    if (bad && not_finite(v)) *bad = 1;
}

__global__ __launch_bounds__(256) void k_vec1_out(const double2 *__restrict__ f, double2 *__restrict__ aos, int V, int nc)
{
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= 4l * nc * V) return;
    const int sp = (int)(i % 4), r = (int)(i / 4), c = r % nc, s = r / nc;
    aos[i] = f[(size_t)(sp * nc + c) * V + s];
}

// ---------------------------------------------------------------------------------------------
// Ritz.  blockIdx.y = solve: independent vectors x, y, z, g, p, w (RITZ_VECS fields apart), signs,
// partial results and state.  The state of inner iteration i is st[i & 1]; its last kernel writes
// st[(i + 1) & 1], so that no workgroup reads what another one of the same launch writes.
// ---------------------------------------------------------------------------------------------
enum { RX = 0, RY, RZ_, RG, RP, RW };
// partial results of a solve: PP |p|^2 (one array per parity, as the state); PZ {Re<p,z>, Re<x,z>};
// XX {|x|^2, <x,y>}; GG {|g|^2, <x,p>}
enum { Q_PP = 0, Q_PZ = 2, Q_XX, Q_GG, Q_KINDS };
static_assert(Q_KINDS == RITZ_PARTS, "host allocation");

struct RitzArgs {
    double2 *vec;   // [solve][RITZ_VECS][n]
    double *part;   // [solve][Q_KINDS][nbmax][PART]
    RitzState *st;  // [solve][2]
    const double2 *links;
    Lat1 g;
    long n;         // complex entries of one vector
    int nb_hop, nb_pt, nbmax, par;
    double sign[RITZ_SOLVES], delitr;
    int nitlz;
};

struct RitzView {
    double2 *x, *y, *z, *g, *p, *w;
    double *part[Q_KINDS];
    RitzState *st;
    const RitzState *cur;
    double sign;
};

__device__ __forceinline__ RitzView ritz_view(const RitzArgs &a)
{
    RitzView v;
    const int q = blockIdx.y;
    double2 *b = a.vec + (size_t)q * RITZ_VECS * a.n;
    v.x = b + RX * a.n; v.y = b + RY * a.n; v.z = b + RZ_ * a.n;
    v.g = b + RG * a.n; v.p = b + RP * a.n; v.w = b + RW * a.n;
#pragma unroll
    for (int k = 0; k < Q_KINDS; ++k) v.part[k] = a.part + ((size_t)q * Q_KINDS + k) * a.nbmax * PART;
    v.st = a.st + 2 * q;
    v.cur = v.st + a.par;
    v.sign = q ? a.sign[1] : a.sign[0];
    return v;
}

// |x|^2 of the start vector (x unnormalised) into XX
__global__ __launch_bounds__(TPB1) void k_ritz_start(RitzArgs a)
{
    const RitzView v = ritz_view(a);
    double s[1] = {0.0};
    for (long i = (long)blockIdx.x * TPB1 + threadIdx.x; i < a.n; i += (long)gridDim.x * TPB1)
        s[0] += v.x[i].x * v.x[i].x + v.x[i].y * v.x[i].y;
    put_partial<1>(v.part[Q_XX], s);
}
// x <- x / |x|
__global__ __launch_bounds__(TPB1) void k_ritz_normalise(RitzArgs a)
{
    const RitzView v = ritz_view(a);
    double s[1];
    sum_partials<1>(v.part[Q_XX], a.nb_pt, s);
    const double f = 1.0 / sqrt(s[0]);
    for (long i = (long)blockIdx.x * TPB1 + threadIdx.x; i < a.n; i += (long)gridDim.x * TPB1)
        v.x[i] = make_double2(f * v.x[i].x, f * v.x[i].y);
}

// w = h_W of x (RESTART) or of p / |p|
template <int NC, bool RESTART> __global__ __launch_bounds__(TPB1) void k_ritz_hop(RitzArgs a)
{
    const RitzView v = ritz_view(a);
    if (v.cur->done) return;
    double f = 1.0;
    if (!RESTART) {
        double s[1];
        sum_partials<1>(v.part[Q_PP + a.par], a.nb_pt, s);
        f = 1.0 / sqrt(s[0]);
    }
    int s, sp;
    const bool ok = site1(a.g.V, s, sp);
    double2 u[NC], l[NC];
    hop1_site<NC>(RESTART ? v.x : v.p, a.links, a.g, s, sp, u, l);
    if (!ok) return;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        v.w[(size_t)(sp * NC + c) * a.g.V + s] = make_double2(f * u[c].x, f * u[c].y);
        v.w[(size_t)((2 + sp) * NC + c) * a.g.V + s] = make_double2(f * l[c].x, f * l[c].y);
    }
}

// RESTART: y = sign h_W w, partial <x, y>; else z = sign h_W w, partial {Re<p, z>, Re<x, z>} (p as stored,
// not normalised)
template <int NC, bool RESTART> __global__ __launch_bounds__(TPB1) void k_ritz_hop2(RitzArgs a)
{
    const RitzView v = ritz_view(a);
    if (v.cur->done) return;
    int s, sp;
    const bool ok = site1(a.g.V, s, sp);
    double2 r[2][NC];
    hop1_site<NC>(v.w, a.links, a.g, s, sp, r[0], r[1]);
    double2 *out = RESTART ? v.y : v.z;
    double t[3] = {0.0, 0.0, 0.0};
    if (ok)
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const size_t i = (size_t)((2 * k + sp) * NC + c) * a.g.V + s;
                const double2 q = make_double2(v.sign * r[k][c].x, v.sign * r[k][c].y);
                out[i] = q;
                const double2 x = v.x[i];
                if (RESTART) {
                    t[1] += x.x * q.x + x.y * q.y;
                    t[2] += x.x * q.y - x.y * q.x;
                } else {
                    const double2 p = v.p[i];
                    t[0] += p.x * q.x + p.y * q.y;
                    t[1] += x.x * q.x + x.y * q.y;
                }
            }
    if (RESTART) put_partial<3>(v.part[Q_XX], t);
    else put_partial<2>(v.part[Q_PZ], t);
}

// restart: g = y - <x,y> x, p = g, partial |g|^2
__global__ __launch_bounds__(TPB1) void k_ritz_restart(RitzArgs a)
{
    const RitzView v = ritz_view(a);
    if (v.cur->done) return;
    double d[3];
    sum_partials<3>(v.part[Q_XX], a.nb_hop, d);
    const double cr = d[1], ci = d[2];
    double s[1] = {0.0};
    for (long i = (long)blockIdx.x * TPB1 + threadIdx.x; i < a.n; i += (long)gridDim.x * TPB1) {
        const double2 x = v.x[i], y = v.y[i];
        const double2 q = make_double2(y.x - (cr * x.x - ci * x.y), y.y - (cr * x.y + ci * x.x));
        v.g[i] = q;
        v.p[i] = q;
        s[0] += q.x * q.x + q.y * q.y;
    }
    put_partial<1>(v.part[Q_PP + a.par], s);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        RitzState *w = v.st + a.par;  // no other thread of this launch reads these fields
        w->xy_r = cr;
        w->xy_i = ci;
        w->fresh = 1;
    }
}

// the rotation of (x, p) that extremises the Rayleigh quotient (RitzSolver.cpp:186-222)
__device__ __forceinline__ void ritz_rotation(double amb, double ccc, double &ct, double &st)
{
    const double cox = 2.0 * ccc / amb;
    const double sig1 = -copysign(1.0, amb);
    const double sig2 = copysign(1.0, cox) * sig1;
    const double cox2 = cox * cox;
    if (cox2 <= 1.0e-3) {
        // series of RitzSolver.cpp:199-200
        const double sqp = 1.0 - 0.125 * cox2 + 0.0859375 * cox2 * cox2 - 0.0673828125 * cox2 * cox2 * cox2 +
                           0.0562439 * cox2 * cox2 * cox2 * cox2 + 0.0487 * cox2 * cox2 * cox2 * cox2 * cox2;
        const double sqm = 0.5 * sig1 * sig2 * cox *
                           (1.0 - 0.375 * cox2 + 0.2421875 * cox2 * cox2 - 0.182617875 * cox2 * cox2 * cox2 +
                            0.1482849 * cox2 * cox2 * cox2 * cox2 - 0.12575 * cox2 * cox2 * cox2 * cox2 * cox2 +
                            0.1097 * cox2 * cox2 * cox2 * cox2 * cox2 * cox2);
        if (sig1 < 0.0) { ct = sqm; st = sig2 * sqp; }
        else { ct = sqp; st = sig2 * sqm; }
    } else {
        const double sox = sig1 / sqrt(1.0 + cox2);
        ct = sqrt((1.0 + sox) * 0.5);
        st = sqrt((1.0 - sox) * 0.5) * sig2;
    }
}

// x = ct x + st p/|p|, y = ct y + st z; partial {|x|^2, <x, y>}
__global__ __launch_bounds__(TPB1) void k_ritz_rotate(RitzArgs a)
{
    const RitzView v = ritz_view(a);
    if (v.cur->done) return;
    double pp[1], pz[2];
    sum_partials<1>(v.part[Q_PP + a.par], a.nb_pt, pp);
    sum_partials<2>(v.part[Q_PZ], a.nb_hop, pz);
    const double ps = 1.0 / sqrt(pp[0]);
    double ct, st;
    ritz_rotation(v.cur->xy_r - ps * pz[0], pz[1], ct, st);
    const double sp = st * ps;
    double t[3] = {0.0, 0.0, 0.0};
    for (long i = (long)blockIdx.x * TPB1 + threadIdx.x; i < a.n; i += (long)gridDim.x * TPB1) {
        double2 x = v.x[i], y = v.y[i];
        const double2 p = v.p[i], z = v.z[i];
        x = make_double2(ct * x.x + sp * p.x, ct * x.y + sp * p.y);
        y = make_double2(ct * y.x + st * z.x, ct * y.y + st * z.y);
        v.x[i] = x;
        v.y[i] = y;
        t[0] += x.x * x.x + x.y * x.y;
        t[1] += x.x * y.x + x.y * y.y;
        t[2] += x.x * y.y - x.y * y.x;
    }
    put_partial<3>(v.part[Q_XX], t);
}

// x <- x / |x|, xy = <x, y> / |x| (both vectors as left by the rotation, RitzSolver.cpp:226-236),
// g = y - xy x; partial {|g|^2, <x, p/|p|>}
__global__ __launch_bounds__(TPB1) void k_ritz_gradient(RitzArgs a)
{
    const RitzView v = ritz_view(a);
    if (v.cur->done) return;
    double d[3], pp[1];
    sum_partials<3>(v.part[Q_XX], a.nb_pt, d);
    sum_partials<1>(v.part[Q_PP + a.par], a.nb_pt, pp);
    const double xn = 1.0 / sqrt(d[0]), ps = 1.0 / sqrt(pp[0]);
    const double cr = d[1] * xn, ci = d[2] * xn;
    double t[3] = {0.0, 0.0, 0.0};
    for (long i = (long)blockIdx.x * TPB1 + threadIdx.x; i < a.n; i += (long)gridDim.x * TPB1) {
        const double2 o = v.x[i], y = v.y[i], p = v.p[i];
        const double2 x = make_double2(xn * o.x, xn * o.y);
        const double2 q = make_double2(y.x - (cr * x.x - ci * x.y), y.y - (cr * x.y + ci * x.x));
        v.x[i] = x;
        v.g[i] = q;
        t[0] += q.x * q.x + q.y * q.y;
        t[1] += ps * (x.x * p.x + x.y * p.y);
        t[2] += ps * (x.x * p.y - x.y * p.x);
    }
    put_partial<3>(v.part[Q_GG], t);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        RitzState *w = v.st + a.par;  // read by the next launch only
        w->xyn_r = cr;
        w->xyn_i = ci;
    }
}

// the stopping tests of RitzSolver.cpp:246-262 and p = g + beta (p/|p| - <x,p> x); partial |p|^2
__global__ __launch_bounds__(TPB1) void k_ritz_direction(RitzArgs a)
{
    const RitzView v = ritz_view(a);
    const RitzState c = *v.cur;
    RitzState *nx = v.st + (1 - a.par);
    const bool first = blockIdx.x == 0 && threadIdx.x == 0;
    if (c.done) {
        if (first) *nx = c;
        return;
    }
    double d[3], pp[1];
    sum_partials<3>(v.part[Q_GG], a.nb_pt, d);
    sum_partials<1>(v.part[Q_PP + a.par], a.nb_pt, pp);
    const double pnorm = sqrt(pp[0]), ps = 1.0 / pnorm;
    const double gnorm = d[0];
    const double gnormim = c.fresh ? pp[0] : c.gnormim;  // after a restart p = g
    RitzState n = c;
    n.iters = c.iters + 1;
    n.xy_r = c.xyn_r;
    n.xy_i = c.xyn_i;
    n.gnormim = gnorm;
    n.fresh = 0;
    const bool stop = c.xyn_r > c.xy_r || gnorm < a.delitr * v.sign * c.xyn_r;
    n.done = stop || n.iters >= a.nitlz;
    if (!stop) {
        const double beta = gnorm / gnormim * pnorm;
        const double bp = beta * ps, xr = beta * d[1], xi = beta * d[2];
        double t[1] = {0.0};
        for (long i = (long)blockIdx.x * TPB1 + threadIdx.x; i < a.n; i += (long)gridDim.x * TPB1) {
            const double2 x = v.x[i], p = v.p[i], g = v.g[i];
            const double2 q = make_double2(bp * p.x - (xr * x.x - xi * x.y) + g.x, bp * p.y - (xr * x.y + xi * x.x) + g.y);
            v.p[i] = q;
            t[0] += q.x * q.x + q.y * q.y;
        }
        put_partial<1>(v.part[Q_PP + 1 - a.par], t);
    }
    if (first) *nx = n;
}


// ---------------------------------------------------------------------------------------------
// multi-shift CG (OverlapU.cpp:5-149): chi = sum_k bz_k (h_W^2 + dz_k)^{-1} in
// ---------------------------------------------------------------------------------------------
// the scalar recurrences of one mode after r was updated (rr = |r|^2, al0 the step length of shift 0),
// one lane per shift k; z and gc of the lane go from the old to the new values; coef = {bz beta_k,
// alpha_k, zeta_k}
__device__ __forceinline__ void cg_shift_scalars(double rn, double a0_old, double betam, const CgShifts &sh, int k,
                                                 double al0, double rr, double &z, double &gc, double *coef)
{
    double be = al0;
    if (k > 0) {
        const double dr = al0 * a0_old * (1.0 - z) + betam * (1.0 + (sh.dz[k] - sh.dz[0]) * al0);
        z = betam / dr;
        be = al0 * z;
    }
    const double a0 = rr / rn;
    gc = gc * z;
    coef[0] = sh.bz[k] * be;
    coef[1] = a0 * z * be / al0;
    coef[2] = gc;
}

__device__ __forceinline__ bool cg_goes_on(double rr, double bn, int it, double tol, int cap)
{
    return rr > tol * bn && it < cap;
}

struct Cg1Args {
    double2 *ps;    // [CG_SHIFTS][n]
    double2 *chi, *r, *q, *w;
    const double2 *in, *links;
    double *part;   // {|r|^2 or Re<p,q>}: [2][nbmax][PART], PQ then RR
    CgMode *st;     // [2], by parity as the Ritz state
    Lat1 g;
    long n;
    int nb_hop, nb_pt, nbmax, par;
    const CgShifts *sh;
    double tol;
    int cap;
};

__global__ __launch_bounds__(TPB1) void k_cg1_start(Cg1Args a)
{
    double s[1] = {0.0};
    for (long i = (long)blockIdx.x * TPB1 + threadIdx.x; i < a.n; i += (long)gridDim.x * TPB1) {
        const double2 v = a.in[i];
        a.r[i] = v;
        a.chi[i] = make_double2(0.0, 0.0);
        for (int k = 0; k < CG_SHIFTS; ++k) a.ps[(size_t)k * a.n + i] = v;
        s[0] += v.x * v.x + v.y * v.y;
    }
    put_partial<1>(a.part + (size_t)a.nbmax * PART, s);
}

__global__ __launch_bounds__(TPB1) void k_cg1_begin(Cg1Args a)
{
    double s[1];
    sum_partials<1>(a.part + (size_t)a.nbmax * PART, a.nb_pt, s);
    const int k = threadIdx.x;
    if (k < CG_SHIFTS) a.st[0].z[k] = a.st[0].gc[k] = 1.0;
    if (k == 0) {
        a.st[0].rn = s[0];
        a.st[0].bn = sqrt(s[0]);
        a.st[0].a0 = 0.0;
        a.st[0].betam = 1.0;
        a.st[0].it = 0;
        a.st[0].act = s[0] > a.tol * sqrt(s[0]);
    }
}

// SECOND: q = h_W w + dz_0 p, partial Re<p, q>; else w = h_W p (p: shift 0)
template <int NC, bool SECOND> __global__ __launch_bounds__(TPB1) void k_cg1_hop(Cg1Args a)
{
    if (!a.st[a.par].act) return;
    int s, sp;
    const bool ok = site1(a.g.V, s, sp);
    double2 r[2][NC];
    hop1_site<NC>(SECOND ? a.w : a.ps, a.links, a.g, s, sp, r[0], r[1]);
    const double dz0 = a.sh->dz[0];
    double t[1] = {0.0};
    if (ok)
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const size_t i = (size_t)((2 * k + sp) * NC + c) * a.g.V + s;
                double2 v = r[k][c];
                if (SECOND) {
                    const double2 p = a.ps[i];
                    v.x += dz0 * p.x;
                    v.y += dz0 * p.y;
                    a.q[i] = v;
                    t[0] += p.x * v.x + p.y * v.y;
                } else {
                    a.w[i] = v;
                }
            }
    if (SECOND) put_partial<1>(a.part, t);
}

// r -= (rn / <p,q>) q, partial |r|^2
__global__ __launch_bounds__(TPB1) void k_cg1_residual(Cg1Args a)
{
    const CgMode &o = a.st[a.par];
    if (!o.act) return;
    double pq[1];
    sum_partials<1>(a.part, a.nb_hop, pq);
    const double al = o.rn / pq[0];
    double t[1] = {0.0};
    for (long i = (long)blockIdx.x * TPB1 + threadIdx.x; i < a.n; i += (long)gridDim.x * TPB1) {
        double2 r = a.r[i];
        const double2 q = a.q[i];
        r.x -= al * q.x;
        r.y -= al * q.y;
        a.r[i] = r;
        t[0] += r.x * r.x + r.y * r.y;
    }
    put_partial<1>(a.part + (size_t)a.nbmax * PART, t);
}

// the scalars (every workgroup computes the same ones, the first keeps them), chi += bz beta_k p_k and
// p_k = alpha_k p_k + zeta_k r.  All shifts' loads of an element are independent: unrolled, so that a
// lane has them in flight together.
__global__ __launch_bounds__(TPB1) void k_cg1_shifts(Cg1Args a)
{
    const CgMode &o = a.st[a.par];
    CgMode *nx = a.st + (1 - a.par);
    const int k = threadIdx.x;
    if (!o.act) {
        if (blockIdx.x == 0 && k == 0) {
            nx->act = 0;
            nx->it = o.it;
            nx->rn = o.rn;
            nx->bn = o.bn;
        }
        return;
    }
    double pq[1], rr[1];
    sum_partials<1>(a.part, a.nb_hop, pq);
    sum_partials<1>(a.part + (size_t)a.nbmax * PART, a.nb_pt, rr);
    const double al0 = o.rn / pq[0];
    __shared__ double cf[CG_SHIFTS][3];
    if (k < CG_SHIFTS) {
        double z = o.z[k], gc = o.gc[k], f[3];
        cg_shift_scalars(o.rn, o.a0, o.betam, *a.sh, k, al0, rr[0], z, gc, f);
        cf[k][0] = f[0];
        cf[k][1] = f[1];
        cf[k][2] = f[2];
        if (blockIdx.x == 0) {
            nx->z[k] = z;
            nx->gc[k] = gc;
            if (k == 0) {
                nx->rn = rr[0];
                nx->bn = o.bn;
                nx->a0 = rr[0] / o.rn;
                nx->betam = al0;
                nx->it = o.it + 1;
                nx->act = cg_goes_on(rr[0], o.bn, o.it + 1, a.tol, a.cap);
            }
        }
    }
    __syncthreads();
    for (long i = (long)blockIdx.x * TPB1 + threadIdx.x; i < a.n; i += (long)gridDim.x * TPB1) {
        const double2 r = a.r[i];
        double2 x = a.chi[i];
        double2 p[CG_SHIFTS];
#pragma unroll
        for (int j = 0; j < CG_SHIFTS; ++j) p[j] = a.ps[(size_t)j * a.n + i];
#pragma unroll
        for (int j = 0; j < CG_SHIFTS; ++j) {
            x.x += cf[j][0] * p[j].x;
            x.y += cf[j][0] * p[j].y;
            a.ps[(size_t)j * a.n + i] = make_double2(cf[j][1] * p[j].x + cf[j][2] * r.x, cf[j][1] * p[j].y + cf[j][2] * r.y);
        }
        a.chi[i] = x;
    }
}

// ---- many modes (mode-block layout): one wavefront per mode works out that mode's scalars ----
__device__ __forceinline__ double mode_sum(const double2 *part, int chunks, int nmodes, int mode)
{
    double v = 0.0;
    for (int c = threadIdx.x; c < chunks; c += 64) v += part[(size_t)c * nmodes + mode].x;
    return wave_add(v);
}

__global__ __launch_bounds__(64) void k_cgm_begin(const double2 *part, int chunks, int nmodes, CgMode *st, int *act, double tol)
{
    const int mode = blockIdx.x, k = threadIdx.x;
    const double rn = mode_sum(part, chunks, nmodes, mode);
    CgMode &m = st[mode];
    if (k < CG_SHIFTS) m.z[k] = m.gc[k] = 1.0;
    if (k == 0) {
        m.rn = rn;
        m.bn = sqrt(rn);
        m.a0 = 0.0;
        m.betam = 1.0;
        m.it = 0;
        act[mode] = rn > tol * sqrt(rn);
    }
}

__global__ __launch_bounds__(64) void k_cgm_alpha(const double2 *part, int chunks, int nmodes, CgMode *st, const int *act)
{
    const int mode = blockIdx.x;
    const double pq = mode_sum(part, chunks, nmodes, mode);
    if (threadIdx.x == 0) st[mode].alpha = act[mode] ? st[mode].rn / pq : 0.0;
}

// r -= alpha q and the partial |r|^2 per mode, one pass (the reads and the order of k_mode_dot)
template <int MB>
__global__ __launch_bounds__(256) void k_cgm_residual(double2 *__restrict__ r, const double2 *__restrict__ q,
                                                      const CgMode *__restrict__ st, const int *__restrict__ act,
                                                      double2 *__restrict__ part, long nel, int nblk)
{
    constexpr int LPM = 256 / MB;
    const int m = threadIdx.x % MB, lane = threadIdx.x / MB, blk = blockIdx.y, mode = blk * MB + m;
    const double al = st[mode].alpha;
    double s = 0.0;
    if (act[mode])
        for (long e = (long)blockIdx.x * LPM + lane; e < nel; e += (long)gridDim.x * LPM) {
            const size_t i = ((size_t)blk * nel + e) * MB + m;
            double2 v = r[i];
            const double2 b = q[i];
            v.x -= al * b.x;
            v.y -= al * b.y;
            r[i] = v;
            s += v.x * v.x + v.y * v.y;
        }
    __shared__ double sh[256];
    sh[threadIdx.x] = s;
    __syncthreads();
    if (lane == 0) {
        double t = 0.0;
        for (int l = 0; l < LPM; ++l) t += sh[l * MB + m];
        part[(size_t)blockIdx.x * nblk * MB + mode] = make_double2(t, 0.0);
    }
}

__global__ __launch_bounds__(64) void k_cgm_scalars(const double2 *part, int chunks, int nmodes, CgMode *st, const int *act,
                                                    int *act_next, double *coef, CgShifts sh, double tol, int cap)
{
    const int mode = blockIdx.x, k = threadIdx.x;
    if (!act[mode]) {
        if (k == 0) act_next[mode] = 0;
        return;
    }
    const double rr = mode_sum(part, chunks, nmodes, mode);
    CgMode &m = st[mode];
    const double rn = m.rn, bn = m.bn, a0 = m.a0, betam = m.betam, alpha = m.alpha;
    const int it = m.it + 1;
    __syncthreads();  // every lane holds the old scalars before the first one is overwritten
    if (k < CG_SHIFTS) {
        double z = m.z[k], gc = m.gc[k];
        cg_shift_scalars(rn, a0, betam, sh, k, alpha, rr, z, gc, coef + ((size_t)mode * CG_SHIFTS + k) * 3);
        m.z[k] = z;
        m.gc[k] = gc;
    }
    if (k == 0) {
        m.rn = rr;
        m.a0 = rr / rn;
        m.betam = alpha;
        m.it = it;
        act_next[mode] = cg_goes_on(rr, bn, it, tol, cap);
    }
}

// flat host order (s + V (spin + 4 colour)) -> [spin][colour][site]
__global__ __launch_bounds__(256) void k_vec1_flat(const double2 *__restrict__ src, double2 *__restrict__ dst, int V, int nc)
{
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= 4l * nc * V) return;
    const int s = (int)(i % V), r = (int)(i / V), sp = r / nc, c = r % nc;
    dst[i] = src[(size_t)(sp + 4 * c) * V + s];
}

Lat1 lat1(const Geom &g, double amass)
{
    Lat1 l;
    l.n0 = g.n0; l.n1 = g.n1; l.n2 = g.n2; l.V = g.V;
    l.dv_n01 = make_fastdiv((unsigned)(g.n0 * g.n1));
    l.dv_n0 = make_fastdiv((unsigned)g.n0);
    l.amass = amass;
    return l;
}

int hop_blocks(const Geom &g) { return (g.V + TPB1 / 2 - 1) / (TPB1 / 2); }
int point_blocks(long n) { return (int)std::min<long>(POINT_BLOCKS, (n + TPB1 - 1) / TPB1); }
unsigned blocks256(long n) { return (unsigned)((n + 255) / 256); }

RitzArgs ritz_args(const Geom &g, const RitzCall &c)
{
    RitzArgs a{};
    a.vec = (double2 *)c.vec;
    a.part = c.part;
    a.st = (RitzState *)c.state;
    a.links = (const double2 *)c.links;
    a.g = lat1(g, c.amass);
    a.n = 4l * g.nc * g.V;
    a.nb_hop = hop_blocks(g);
    a.nb_pt = point_blocks(a.n);
    a.nbmax = std::max(a.nb_hop, a.nb_pt);
    a.sign[0] = c.sign[0];
    a.sign[1] = c.sign[1];
    a.delitr = c.delitr;
    a.nitlz = c.nitlz;
    return a;
}

Cg1Args cg1_args(const Geom &g, const Cg1Call &c)
{
    Cg1Args a{};
    const long n = 4l * g.nc * g.V;
    double2 *b = (double2 *)c.work;
    a.ps = b;
    a.chi = b + (size_t)CG_SHIFTS * n;
    a.r = a.chi + n;
    a.q = a.r + n;
    a.w = a.q + n;
    a.in = (const double2 *)c.in;
    a.links = (const double2 *)c.links;
    a.part = c.part;
    a.st = (CgMode *)c.state;
    a.g = lat1(g, c.amass);
    a.n = n;
    a.nb_hop = hop_blocks(g);
    a.nb_pt = point_blocks(n);
    a.nbmax = std::max(a.nb_hop, a.nb_pt);
    a.sh = (const CgShifts *)c.shifts;
    a.tol = c.tol;
    a.cap = c.cap;
    return a;
}

}  // namespace

// ---------------------------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------------------------
size_t single_partial_len(const Geom &g)
{
    const size_t nb = (size_t)std::max(hop_blocks(g), point_blocks(4l * g.nc * g.V));
    return std::max((size_t)RITZ_SOLVES * RITZ_PARTS, (size_t)2) * nb * PART;
}

hipError_t launch_links1(const Geom &g, const void *links, void *out, int *bad, hipStream_t st)
{
    const int nn = g.nc * g.nc;
    k_links1<<<blocks256(3l * g.V * nn), 256, 0, st>>>((const double2 *)links, (double2 *)out, g.V, nn, bad);
    return hipGetLastError();
}
hipError_t launch_vec1_in(const Geom &g, const double *aos, void *out, int *bad, hipStream_t st)
{
    k_vec1_in<<<blocks256(4l * g.nc * g.V), 256, 0, st>>>((const double2 *)aos, (double2 *)out, g.V, g.nc, bad);
    return hipGetLastError();
}
hipError_t launch_vec1_out(const Geom &g, const void *f, double *aos, hipStream_t st)
{
    k_vec1_out<<<blocks256(4l * g.nc * g.V), 256, 0, st>>>((const double2 *)f, (double2 *)aos, g.V, g.nc);
    return hipGetLastError();
}
hipError_t launch_vec1_flat(const Geom &g, const double *flat, void *out, hipStream_t st)
{
    k_vec1_flat<<<blocks256(4l * g.nc * g.V), 256, 0, st>>>((const double2 *)flat, (double2 *)out, g.V, g.nc);
    return hipGetLastError();
}

hipError_t launch_hop1(const Geom &g, double amass, const void *in, void *out, const void *links, double sh_r, double sh_i,
                       const void *x, double sx_r, double sx_i, int x_gamma0, hipStream_t st)
{
    const unsigned nb = (unsigned)hop_blocks(g);
    if (g.nc == 2)
        k_hop1<2><<<nb, TPB1, 0, st>>>((const double2 *)in, (double2 *)out, (const double2 *)links, lat1(g, amass), sh_r,
                                       sh_i, (const double2 *)x, sx_r, sx_i, x_gamma0);
    else
        k_hop1<3><<<nb, TPB1, 0, st>>>((const double2 *)in, (double2 *)out, (const double2 *)links, lat1(g, amass), sh_r,
                                       sh_i, (const double2 *)x, sx_r, sx_i, x_gamma0);
    return hipGetLastError();
}

hipError_t launch_ritz_start(const Geom &g, const RitzCall &c, hipStream_t st)
{
    const RitzArgs a = ritz_args(g, c);
    const dim3 pt(a.nb_pt, c.solves);
    k_ritz_start<<<pt, TPB1, 0, st>>>(a);
    k_ritz_normalise<<<pt, TPB1, 0, st>>>(a);
    return hipGetLastError();
}

template <int NC, bool RESTART> static void ritz_hops_nc(const RitzArgs &a, int solves, hipStream_t st)
{
    const dim3 hp(a.nb_hop, solves);
    k_ritz_hop<NC, RESTART><<<hp, TPB1, 0, st>>>(a);
    k_ritz_hop2<NC, RESTART><<<hp, TPB1, 0, st>>>(a);
}

hipError_t launch_ritz_hops(const Geom &g, const RitzCall &c, int iter, bool restart, hipStream_t st)
{
    RitzArgs a = ritz_args(g, c);
    a.par = iter & 1;
    if (g.nc == 2) restart ? ritz_hops_nc<2, true>(a, c.solves, st) : ritz_hops_nc<2, false>(a, c.solves, st);
    else restart ? ritz_hops_nc<3, true>(a, c.solves, st) : ritz_hops_nc<3, false>(a, c.solves, st);
    return hipGetLastError();
}

hipError_t launch_ritz_rest(const Geom &g, const RitzCall &c, int iter, bool restart, hipStream_t st)
{
    RitzArgs a = ritz_args(g, c);
    a.par = iter & 1;
    const dim3 pt(a.nb_pt, c.solves);
    if (restart) {
        k_ritz_restart<<<pt, TPB1, 0, st>>>(a);
    } else {
        k_ritz_rotate<<<pt, TPB1, 0, st>>>(a);
        k_ritz_gradient<<<pt, TPB1, 0, st>>>(a);
        k_ritz_direction<<<pt, TPB1, 0, st>>>(a);
    }
    return hipGetLastError();
}

hipError_t launch_cg1_start(const Geom &g, const Cg1Call &c, hipStream_t st)
{
    const Cg1Args a = cg1_args(g, c);
    k_cg1_start<<<a.nb_pt, TPB1, 0, st>>>(a);
    k_cg1_begin<<<1, TPB1, 0, st>>>(a);
    return hipGetLastError();
}

hipError_t launch_cg1_iteration(const Geom &g, const Cg1Call &c, int iter, hipStream_t st)
{
    Cg1Args a = cg1_args(g, c);
    a.par = iter & 1;
    if (g.nc == 2) {
        k_cg1_hop<2, false><<<a.nb_hop, TPB1, 0, st>>>(a);
        k_cg1_hop<2, true><<<a.nb_hop, TPB1, 0, st>>>(a);
    } else {
        k_cg1_hop<3, false><<<a.nb_hop, TPB1, 0, st>>>(a);
        k_cg1_hop<3, true><<<a.nb_hop, TPB1, 0, st>>>(a);
    }
    k_cg1_residual<<<a.nb_pt, TPB1, 0, st>>>(a);
    k_cg1_shifts<<<a.nb_pt, TPB1, 0, st>>>(a);
    return hipGetLastError();
}
void *cg1_chi(const Geom &g, void *work) { return (double2 *)work + (size_t)CG_SHIFTS * 4 * g.nc * g.V; }

hipError_t launch_cgm_begin(const Geom &g, const double *part, int chunks, CgMode *modes, int *act, double tol, hipStream_t st)
{
    const int nm = g.nblk * g.mb;
    k_cgm_begin<<<nm, 64, 0, st>>>((const double2 *)part, chunks, nm, modes, act, tol);
    return hipGetLastError();
}
hipError_t launch_cgm_alpha(const Geom &g, const double *part, int chunks, CgMode *modes, const int *act, hipStream_t st)
{
    const int nm = g.nblk * g.mb;
    k_cgm_alpha<<<nm, 64, 0, st>>>((const double2 *)part, chunks, nm, modes, act);
    return hipGetLastError();
}
hipError_t launch_cgm_residual(const Geom &g, void *r, const void *q, const CgMode *modes, const int *act, double *part,
                               int chunks, hipStream_t st)
{
    const dim3 grid(chunks, g.nblk);
    const long nel = 4l * g.nc * g.V;
    const auto R = (double2 *)r;
    const auto Q = (const double2 *)q;
    const auto P = (double2 *)part;
    if (g.mb == 16) k_cgm_residual<16><<<grid, 256, 0, st>>>(R, Q, modes, act, P, nel, g.nblk);
    else if (g.mb == 32) k_cgm_residual<32><<<grid, 256, 0, st>>>(R, Q, modes, act, P, nel, g.nblk);
    else if (g.mb == 64) k_cgm_residual<64><<<grid, 256, 0, st>>>(R, Q, modes, act, P, nel, g.nblk);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}
hipError_t launch_cgm_scalars(const Geom &g, const double *part, int chunks, CgMode *modes, const int *act, int *act_next,
                              double *coef, const CgShifts &sh, double tol, int cap, hipStream_t st)
{
    const int nm = g.nblk * g.mb;
    k_cgm_scalars<<<nm, 64, 0, st>>>((const double2 *)part, chunks, nm, modes, act, act_next, coef, sh, tol, cap);
    return hipGetLastError();
}

}  // namespace ovl
