// gfx950 kernels of the OVERLAP fermion hot path.
//
// All spinor kernels are HBM-bandwidth bound: one lane owns one (site, mode) pair, a wavefront
// covers 64 consecutive (mode, site) lanes of one mode block, so every 16-byte load of a spinor
// component is one contiguous MB*16-byte segment.  Links are shared by all modes of a site and
// read once per wavefront (MB = 64) or once per MB-lane group.
#include "../../include/ovl.h"
#include "ovl_internal.hpp"

#include <algorithm>
#include <cmath>
#include <mutex>
#include <type_traits>
#include <unordered_set>

namespace ovl {

namespace {

constexpr int TPB = STENCIL_TPB;  // threads per block for the streaming kernels

// 48-bit storage of a double: its top 48 bits (sign, exponent, 36 mantissa bits) after rounding
// the dropped 16 bits to nearest.  Only a tag for the templates: the bits live in 16-byte units.
struct f48 { unsigned short h[3]; };
static_assert(sizeof(f48) == 6, "f48 tag size selects the 48-bit layout");

// storage type -> arithmetic type (C) and stencil link type (L).  FP16 storage computes in FP32
// with the FP32 links, 48-bit storage in FP64 with the FP64 links.
template <typename T> struct Vec;
template <> struct Vec<double> { using C = double; using L = double2; };
template <> struct Vec<float> { using C = float; using L = float2; };
template <> struct Vec<_Float16> { using C = float; using L = float2; };
template <> struct Vec<f48> { using C = double; using L = double2; };

// 16 bytes of FP16 storage: 4 complex numbers
typedef _Float16 h8v __attribute__((ext_vector_type(8)));
typedef unsigned u4v __attribute__((ext_vector_type(4)));

// 48-bit units: 4 complex (v0..v7 = re0, im0, .., re3, im3) take three 16-byte units holding
// six 64-bit words W0..W5 (W0, W1 | W2, W3 | W4, W5).  W_i (i < 6) is v_i's sign, exponent and top
// 36 mantissa bits in bits 16..63 and one 16-bit piece of v6 (W0..W2) or v7 (W3..W5) in bits 0..15:
// the piece of W_i, read as the low mantissa bits of v_i, is accounted for when v_i's top bits are
// rounded, so W_i read as a double IS v_i to within 2^-37 (no decoding).  v6 and v7 are their top
// 48 bits (rounded to nearest) reassembled from the three pieces.
__device__ __forceinline__ unsigned long long r48(double v)
{
    // top 48 bits rounded to nearest (+2^15 then truncation, on the sign-magnitude pattern)
    return ((unsigned long long)__double_as_longlong(v) + 0x8000ull) & ~0xffffull;
}
__device__ __forceinline__ unsigned long long w48(double v, unsigned long long piece)
{
    // top 48 bits t of v such that t | piece is the nearest such pattern to v's magnitude
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const unsigned long long sgn = b & 0x8000000000000000ull, mag = b ^ sgn;
    const unsigned long long t = (mag < 0x10000ull) ? 0ull : ((mag - piece + 0x8000ull) & ~0xffffull);
    return sgn | t | piece;
}
__device__ __forceinline__ double w_as_double(unsigned lo, unsigned hi)
{
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
// v6 / v7 from the low 16 bits of the three words that carry its pieces
__device__ __forceinline__ double pieces_as_double(unsigned w0, unsigned w1, unsigned w2)
{
    // high word: low half of w1 below low half of w2, one byte permute
    return w_as_double(w0 << 16, __builtin_amdgcn_perm(w2, w1, 0x05040100u));
}
// TRUNC: the six words keep their top 48 bits as they are (v_i's low 16 bits are replaced by the
// piece: within 2^-36 instead of 2^-37) and v6 / v7 are truncated to 48 bits; two instructions per
// word instead of about twelve.  Used for the intermediate w = h b of a Clenshaw step.
template <bool TRUNC = false, typename C>
__device__ __forceinline__ void pack48(const C *re, const C *im, int u, u4v &A, u4v &B, u4v &M)
{
    double v[8];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        v[2 * j] = (double)re[4 * u + j];
        v[2 * j + 1] = (double)im[4 * u + j];
    }
    unsigned long long w[6];
    if constexpr (TRUNC) {
        const unsigned long long r6 = (unsigned long long)__double_as_longlong(v[6]);
        const unsigned long long r7 = (unsigned long long)__double_as_longlong(v[7]);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            w[i] = ((unsigned long long)__double_as_longlong(v[i]) & ~0xffffull) | ((r6 >> (16 * (i + 1))) & 0xffffull);
            w[i + 3] =
                ((unsigned long long)__double_as_longlong(v[i + 3]) & ~0xffffull) | ((r7 >> (16 * (i + 1))) & 0xffffull);
        }
    } else {
        const unsigned long long r6 = r48(v[6]), r7 = r48(v[7]);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            w[i] = w48(v[i], (r6 >> (16 * (i + 1))) & 0xffffull);
            w[i + 3] = w48(v[i + 3], (r7 >> (16 * (i + 1))) & 0xffffull);
        }
    }
    A = {(unsigned)w[0], (unsigned)(w[0] >> 32), (unsigned)w[1], (unsigned)(w[1] >> 32)};
    B = {(unsigned)w[2], (unsigned)(w[2] >> 32), (unsigned)w[3], (unsigned)(w[3] >> 32)};
    M = {(unsigned)w[4], (unsigned)(w[4] >> 32), (unsigned)w[5], (unsigned)(w[5] >> 32)};
}
template <typename C>
__device__ __forceinline__ void unpack48(const u4v &A, const u4v &B, const u4v &M, int u, C *re, C *im)
{
    re[4 * u + 0] = w_as_double(A.x, A.y);
    im[4 * u + 0] = w_as_double(A.z, A.w);
    re[4 * u + 1] = w_as_double(B.x, B.y);
    im[4 * u + 1] = w_as_double(B.z, B.w);
    re[4 * u + 2] = w_as_double(M.x, M.y);
    im[4 * u + 2] = w_as_double(M.z, M.w);
    re[4 * u + 3] = pieces_as_double(A.x, A.z, B.x);
    im[4 * u + 3] = pieces_as_double(B.z, M.x, M.z);
}

// ---------------------------------------------------------------------------------------------
// spinor load / store for one lane
// ---------------------------------------------------------------------------------------------
// FP16 layout: 16-byte units of 4 complex, (blk, site, comp/4, m) at ((blk*V + site)*NCOMP/4 + comp/4)*MB + m
// 48-bit layout: three 16-byte units j = A, B, M per 4 complex at
//   (((blk*V + site)*NCOMP/4 + comp/4)*3 + j)*MB + m
template <int NC, int MB, typename T, typename C>
__device__ __forceinline__ void load_sp(const void *__restrict__ base, int V, int blk, int s, int m, C *re, C *im)
{
    constexpr int NCOMP = 4 * NC;
    if constexpr (sizeof(T) == 6) {
        const u4v *p = reinterpret_cast<const u4v *>(base) + ((size_t)(blk * V + s) * (NCOMP / 4)) * 3 * MB + m;
#pragma unroll
        for (int u = 0; u < NCOMP / 4; ++u) {
            const u4v A = p[(size_t)(3 * u) * MB], B = p[(size_t)(3 * u + 1) * MB], M = p[(size_t)(3 * u + 2) * MB];
            unpack48(A, B, M, u, re, im);
        }
    } else if constexpr (sizeof(T) == 2) {
        const h8v *p = reinterpret_cast<const h8v *>(base) + ((size_t)(blk * V + s) * (NCOMP / 4)) * MB + m;
#pragma unroll
        for (int u = 0; u < NCOMP / 4; ++u) {
            const h8v t = p[(size_t)u * MB];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                re[4 * u + j] = (C)t[2 * j];
                im[4 * u + j] = (C)t[2 * j + 1];
            }
        }
    } else if constexpr (sizeof(T) == 8) {
        const double2 *p = reinterpret_cast<const double2 *>(base) + ((size_t)(blk * V + s) * NCOMP) * MB + m;
#pragma unroll
        for (int c = 0; c < NCOMP; ++c) {
            double2 t = p[(size_t)c * MB];
            re[c] = t.x;
            im[c] = t.y;
        }
    } else {
        const float4 *p = reinterpret_cast<const float4 *>(base) + ((size_t)(blk * V + s) * (NCOMP / 2)) * MB + m;
#pragma unroll
        for (int c = 0; c < NCOMP / 2; ++c) {
            float4 t = p[(size_t)c * MB];
            re[2 * c] = t.x;
            im[2 * c] = t.y;
            re[2 * c + 1] = t.z;
            im[2 * c + 1] = t.w;
        }
    }
}

// streaming (non-temporal) variants for operands read or written exactly once per launch, so that
// they do not evict the stencil input whose neighbours are re-read from L2
typedef double d2v __attribute__((ext_vector_type(2)));
typedef float f4v __attribute__((ext_vector_type(4)));

template <int NC, int MB, typename T, typename C>
__device__ __forceinline__ void load_sp_nt(const void *__restrict__ base, int V, int blk, int s, int m, C *re, C *im)
{
    constexpr int NCOMP = 4 * NC;
    if constexpr (sizeof(T) == 6) {
        const u4v *p = reinterpret_cast<const u4v *>(base) + ((size_t)(blk * V + s) * (NCOMP / 4)) * 3 * MB + m;
#pragma unroll
        for (int u = 0; u < NCOMP / 4; ++u) {
            const u4v A = __builtin_nontemporal_load(p + (size_t)(3 * u) * MB);
            const u4v B = __builtin_nontemporal_load(p + (size_t)(3 * u + 1) * MB);
            const u4v M = __builtin_nontemporal_load(p + (size_t)(3 * u + 2) * MB);
            unpack48(A, B, M, u, re, im);
        }
    } else if constexpr (sizeof(T) == 2) {
        const h8v *p = reinterpret_cast<const h8v *>(base) + ((size_t)(blk * V + s) * (NCOMP / 4)) * MB + m;
#pragma unroll
        for (int u = 0; u < NCOMP / 4; ++u) {
            const h8v t = __builtin_nontemporal_load(p + (size_t)u * MB);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                re[4 * u + j] = (C)t[2 * j];
                im[4 * u + j] = (C)t[2 * j + 1];
            }
        }
    } else if constexpr (sizeof(T) == 8) {
        const d2v *p = reinterpret_cast<const d2v *>(base) + ((size_t)(blk * V + s) * NCOMP) * MB + m;
#pragma unroll
        for (int c = 0; c < NCOMP; ++c) {
            const d2v t = __builtin_nontemporal_load(p + (size_t)c * MB);
            re[c] = t.x;
            im[c] = t.y;
        }
    } else {
        const f4v *p = reinterpret_cast<const f4v *>(base) + ((size_t)(blk * V + s) * (NCOMP / 2)) * MB + m;
#pragma unroll
        for (int c = 0; c < NCOMP / 2; ++c) {
            const f4v t = __builtin_nontemporal_load(p + (size_t)c * MB);
            re[2 * c] = t.x;
            im[2 * c] = t.y;
            re[2 * c + 1] = t.z;
            im[2 * c + 1] = t.w;
        }
    }
}

// the output is read by the very next launch, so it is stored normally (it may stay in the MALL)
template <int NC, int MB, typename T, typename C>
__device__ __forceinline__ h8v pack_h8(const C *re, const C *im, int u)
{
    h8v v;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        v[2 * j] = (_Float16)re[4 * u + j];
        v[2 * j + 1] = (_Float16)im[4 * u + j];
    }
    return v;
}

template <int NC, int MB, typename T, bool TRUNC = false, typename C>
__device__ __forceinline__ void store_sp(void *__restrict__ base, int V, int blk, int s, int m, const C *re,
                                         const C *im)
{
    constexpr int NCOMP = 4 * NC;
    if constexpr (sizeof(T) == 6) {
        u4v *p = reinterpret_cast<u4v *>(base) + ((size_t)(blk * V + s) * (NCOMP / 4)) * 3 * MB + m;
#pragma unroll
        for (int u = 0; u < NCOMP / 4; ++u) {
            u4v A, B, M;
            pack48<TRUNC>(re, im, u, A, B, M);
            p[(size_t)(3 * u) * MB] = A;
            p[(size_t)(3 * u + 1) * MB] = B;
            p[(size_t)(3 * u + 2) * MB] = M;
        }
    } else if constexpr (sizeof(T) == 2) {
        h8v *p = reinterpret_cast<h8v *>(base) + ((size_t)(blk * V + s) * (NCOMP / 4)) * MB + m;
#pragma unroll
        for (int u = 0; u < NCOMP / 4; ++u) p[(size_t)u * MB] = pack_h8<NC, MB, T>(re, im, u);
    } else if constexpr (sizeof(T) == 8) {
        double2 *p = reinterpret_cast<double2 *>(base) + ((size_t)(blk * V + s) * NCOMP) * MB + m;
#pragma unroll
        for (int c = 0; c < NCOMP; ++c) p[(size_t)c * MB] = make_double2(re[c], im[c]);
    } else {
        float4 *p = reinterpret_cast<float4 *>(base) + ((size_t)(blk * V + s) * (NCOMP / 2)) * MB + m;
#pragma unroll
        for (int c = 0; c < NCOMP / 2; ++c)
            p[(size_t)c * MB] = make_float4(re[2 * c], im[2 * c], re[2 * c + 1], im[2 * c + 1]);
    }
}

// streaming store of an output that the launch never reads back (keeps L2 for the stencil input)
template <int NC, int MB, typename T, bool TRUNC = false, typename C>
__device__ __forceinline__ void store_sp_nt(void *__restrict__ base, int V, int blk, int s, int m, const C *re,
                                            const C *im)
{
    constexpr int NCOMP = 4 * NC;
    if constexpr (sizeof(T) == 6) {
        u4v *p = reinterpret_cast<u4v *>(base) + ((size_t)(blk * V + s) * (NCOMP / 4)) * 3 * MB + m;
#pragma unroll
        for (int u = 0; u < NCOMP / 4; ++u) {
            u4v A, B, M;
            pack48<TRUNC>(re, im, u, A, B, M);
            __builtin_nontemporal_store(A, p + (size_t)(3 * u) * MB);
            __builtin_nontemporal_store(B, p + (size_t)(3 * u + 1) * MB);
            __builtin_nontemporal_store(M, p + (size_t)(3 * u + 2) * MB);
        }
    } else if constexpr (sizeof(T) == 2) {
        h8v *p = reinterpret_cast<h8v *>(base) + ((size_t)(blk * V + s) * (NCOMP / 4)) * MB + m;
#pragma unroll
        for (int u = 0; u < NCOMP / 4; ++u) __builtin_nontemporal_store(pack_h8<NC, MB, T>(re, im, u), p + (size_t)u * MB);
    } else if constexpr (sizeof(T) == 8) {
        d2v *p = reinterpret_cast<d2v *>(base) + ((size_t)(blk * V + s) * NCOMP) * MB + m;
#pragma unroll
        for (int c = 0; c < NCOMP; ++c) {
            d2v v = {re[c], im[c]};
            __builtin_nontemporal_store(v, p + (size_t)c * MB);
        }
    } else {
        f4v *p = reinterpret_cast<f4v *>(base) + ((size_t)(blk * V + s) * (NCOMP / 2)) * MB + m;
#pragma unroll
        for (int c = 0; c < NCOMP / 2; ++c) {
            f4v v = {re[2 * c], im[2 * c], re[2 * c + 1], im[2 * c + 1]};
            __builtin_nontemporal_store(v, p + (size_t)c * MB);
        }
    }
}

// Lane -> (mode m, site s, block blk) for the three traversals (TRAV_*).  The hardware hands
// workgroup b to XCD b % 8; the XCD traversals undo that round-robin so that XCD k runs the
// contiguous k-th eighth of the logical workgroups (the grid is rounded up to whole eighths):
//   TRAV_BOXES: the eighth is XCD k's spatial box of sites (order[k V/8 .. (k+1) V/8)), every
//     mode block in turn, so x/y/z neighbours are re-read from that XCD's L2 except at the box
//     faces;
//   TRAV_MODES: the eighth is a contiguous range of (mode block, site-order position) in block-major order --
//     whole mode blocks where their number divides by eight, else runs that begin and end anywhere in a
//     block's site order -- with sites in the order of `order` (y slabs, z-major) or lexicographic, so few
//     sites are fetched by two XCDs and the z-neighbour planes of a slab stay in L2.
__device__ __forceinline__ unsigned fdiv(unsigned n, const FastDiv &f)
{
    return f.d <= 1 ? n : (__umulhi(n, f.mul) >> f.shift);
}

struct Site {
    int s, x, y, z;
};
template <int MB>
__device__ __forceinline__ bool lane_coords(const HopArgs &a, unsigned wg, unsigned wgs, int n0, int n1, int V, int &m,
                                            Site &p, int &blk)
{
    // workgroup wg of the wgs of the stencil
    const unsigned total = (unsigned)a.nblk * (unsigned)V * MB;  // < 2^31, checked by the launcher
    unsigned lb = wg;
    if (a.trav != TRAV_LEX) lb = (wg % NUM_XCD) * (wgs / NUM_XCD) + wg / NUM_XCD;
    const unsigned gl = lb * TPB + threadIdx.x;
    if (gl >= total) return false;
    m = (int)(gl % MB);
    unsigned r = gl / MB;
    if constexpr (MB == 64) r = __builtin_amdgcn_readfirstlane(r);  // one site per wavefront
    int s;
    if (a.trav == TRAV_BOXES) {
        const unsigned xc = fdiv(r, a.dv_per);  // XCD of the traversal slot (nblk V / 8 slots each)
        const unsigned rr = r - xc * a.dv_per.d;
        const unsigned b = fdiv(rr, a.dv_v8);
        const unsigned i = rr - b * a.dv_v8.d;
        blk = (int)b;
        if (!a.order) {
            // whole boxes: the site follows from the slot, without a table in memory.  Neither way wins throughout
            // (96 degrees, computed and from a table: SU(2) 32^3, 32 modes FP64 17.2 and 17.7 ms, SU(3) 32^3, 32 modes
            // FP32 14.38 and 14.58, SU(3) 24^3, 64 modes 11.25 and 11.23, 12^3, 64 modes 2.02 and 1.98).
            const unsigned slow = fdiv(i, a.box.dv_plane), ip = i - slow * a.box.dv_plane.d;
            const unsigned mid = fdiv(ip, a.box.dv_x);
            const unsigned kx = xc & ((1u << a.box.lx) - 1), ky = (xc >> a.box.lx) & ((1u << a.box.ly) - 1);
            const unsigned kz = xc >> (a.box.lx + a.box.ly);
            p.x = (int)(kx * a.box.dv_x.d + (ip - mid * a.box.dv_x.d));
            p.y = (int)(ky * a.box.by + (a.box.y_mid ? mid : slow));
            p.z = (int)(kz * a.box.bz + (a.box.y_mid ? slow : mid));
            p.s = p.x + n0 * (p.y + n1 * p.z);
            return true;
        }
        s = a.order[xc * a.dv_v8.d + i];
    } else {
        const unsigned b = fdiv(r, a.dv_V);
        const unsigned i = r - b * (unsigned)V;
        blk = (int)b;
        s = (a.trav == TRAV_MODES && a.order) ? a.order[i] : (int)i;
    }
    if constexpr (MB == 64) s = __builtin_amdgcn_readfirstlane(s);
    p.s = s;
    p.z = (int)fdiv((unsigned)s, a.dv_n01);
    const int rem = s - p.z * (int)a.dv_n01.d;
    p.y = (int)fdiv((unsigned)rem, a.dv_n0);
    p.x = rem - p.y * n0;
    return true;
}

// ---------------------------------------------------------------------------------------------
// one direction of the Wilson hopping term (spin-projected):
//   forward  (sg=+1): h = u + i sigma_k l,  v = U h,      X_u -= v, X_l += i sigma_k v
//   backward (sg=-1): g = u - i sigma_k l,  v = U^+ g,    X_u -= v, X_l -= i sigma_k v
// which is -(1 +- i gamma_k) U phi  in the Dirac basis of DiracAlgebra.cpp:5-9.
// ---------------------------------------------------------------------------------------------
// a * b + c rounded once: the complex multiply-accumulates of the colour mat-vec as two FMAs per
// real part (the compiler does not contract a sum of two products into a running sum by itself)
__device__ __forceinline__ double fmac(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fmac(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// u + S l (S = +-1) rounded once in T.  Operands read from FP16 storage are widened inside one
// mixed-precision FMA, u * one + S l with one = 1 held in a register the compiler cannot see
// through (a literal 1 turns the FMA back into an add of two separately widened values): the same
// value, without the two conversion instructions.
template <int S, typename T, typename TP>
__device__ __forceinline__ T padd(TP u, TP l, float one)
{
    if constexpr (std::is_same<TP, _Float16>::value)
        return S > 0 ? __builtin_fmaf((float)u, one, (float)l) : __builtin_fmaf((float)u, one, -(float)l);
    else
        return u + S * l;
}
__device__ __forceinline__ float opaque_one()
{
    float one;
    asm("s_mov_b32 %0, 1.0" : "=s"(one));
    return one;
}

// TP: element type of the input spinor as loaded (the storage type for FP16, else T)
template <int NC, int K, int SG, typename TP, typename T, typename LT>
__device__ __forceinline__ void hop_dir(const TP *pr, const TP *pi, const LT *__restrict__ U, T *xr, T *xi)
{
    // spinor component index: spin*NC + colour; u = spins 0,1, l = spins 2,3
    T hr[2][NC], hi[2][NC];
    const float one = std::is_same<TP, _Float16>::value ? opaque_one() : 1.0f;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const TP u0r = pr[0 * NC + c], u0i = pi[0 * NC + c];
        const TP u1r = pr[1 * NC + c], u1i = pi[1 * NC + c];
        const TP l0r = pr[2 * NC + c], l0i = pi[2 * NC + c];
        const TP l1r = pr[3 * NC + c], l1i = pi[3 * NC + c];
        if constexpr (K == 0) {  // i sigma_x l = (i l1, i l0)
            hr[0][c] = padd<-SG, T>(u0r, l1i, one); hi[0][c] = padd<SG, T>(u0i, l1r, one);
            hr[1][c] = padd<-SG, T>(u1r, l0i, one); hi[1][c] = padd<SG, T>(u1i, l0r, one);
        } else if constexpr (K == 1) {  // i sigma_y l = (l1, -l0)
            hr[0][c] = padd<SG, T>(u0r, l1r, one); hi[0][c] = padd<SG, T>(u0i, l1i, one);
            hr[1][c] = padd<-SG, T>(u1r, l0r, one); hi[1][c] = padd<-SG, T>(u1i, l0i, one);
        } else {  // i sigma_z l = (i l0, -i l1)
            hr[0][c] = padd<-SG, T>(u0r, l0i, one); hi[0][c] = padd<SG, T>(u0i, l0r, one);
            hr[1][c] = padd<SG, T>(u1r, l1i, one); hi[1][c] = padd<-SG, T>(u1i, l1r, one);
        }
    }
    T vr[2][NC], vi[2][NC];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            T ar = 0, ai = 0;
#pragma unroll
            for (int j = 0; j < NC; ++j) {
                if constexpr (SG > 0) {
                    const LT u = U[i * NC + j];
                    const T ur = (T)u.x, ui = (T)u.y;
                    ar = fmac(ur, hr[s][j], ar);
                    ar = fmac(-ui, hi[s][j], ar);
                    ai = fmac(ur, hi[s][j], ai);
                    ai = fmac(ui, hr[s][j], ai);
                } else {
                    const LT u = U[j * NC + i];  // (U^+)_{ij} = conj(U_{ji})
                    const T ur = (T)u.x, ui = (T)u.y;
                    ar = fmac(ur, hr[s][j], ar);
                    ar = fmac(ui, hi[s][j], ar);
                    ai = fmac(ur, hi[s][j], ai);
                    ai = fmac(-ui, hr[s][j], ai);
                }
            }
            vr[s][i] = ar;
            vi[s][i] = ai;
        }
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        xr[0 * NC + c] -= vr[0][c]; xi[0 * NC + c] -= vi[0][c];
        xr[1 * NC + c] -= vr[1][c]; xi[1 * NC + c] -= vi[1][c];
        // X_l += SG * i sigma_k v
        if constexpr (K == 0) {  // (i v1, i v0)
            xr[2 * NC + c] -= SG * vi[1][c]; xi[2 * NC + c] += SG * vr[1][c];
            xr[3 * NC + c] -= SG * vi[0][c]; xi[3 * NC + c] += SG * vr[0][c];
        } else if constexpr (K == 1) {  // (v1, -v0)
            xr[2 * NC + c] += SG * vr[1][c]; xi[2 * NC + c] += SG * vi[1][c];
            xr[3 * NC + c] -= SG * vr[0][c]; xi[3 * NC + c] -= SG * vi[0][c];
        } else {  // (i v0, -i v1)
            xr[2 * NC + c] -= SG * vi[0][c]; xi[2 * NC + c] += SG * vr[0][c];
            xr[3 * NC + c] += SG * vi[1][c]; xi[3 * NC + c] -= SG * vr[1][c];
        }
    }
}

// One (site, mode) lane of the stencil: out = sh*h_W(in) + sx*G(x) + s1*b1 + s2*b2 + st*tgt,
// h_W = (1/2) gamma0 [A in - sum_k (1+i gamma_k) U in(x+k) + (1-i gamma_k) U^+ in(x-k)]
// (WilsonOperator.cpp:30-114 computes -i h_W of one mode; here every mode of every block).
// The site s lives on an n0 x n1 x n2 lattice; its spinors are site-block q0 + s of the fields
// (q0 = first site-block of this lane's mode block), its links start at site index l0.
// Kinds of launch, known at compile time so that a launch carries no arguments, tests or products of
// terms it does not have (a complex factor with a zero part costs two instructions per real part more):
//   EPI_PURE      out = sh h_W(in), sh real: w of a Clenshaw step
//   EPI_ANY       every term, each present if its pointer is
//   EPI_CLENSHAW  out = sh h_W(in) + sx x + s1 b1 + s2 b2, all factors real
//   EPI_AXPY      out = i sh h_W(in) + tgt: a leapfrog step
// The products and sums of the last two round as EPI_ANY's do (the zero parts only add zeros).
enum { EPI_PURE = 0, EPI_ANY = 1, EPI_CLENSHAW = 2, EPI_AXPY = 3 };

// an operand of the epilogue as loaded: FP16 stays in halves until the product widens it
template <typename T> using OpT = typename std::conditional<std::is_same<T, _Float16>::value, _Float16, typename Vec<T>::C>::type;

// -0 in a register the compiler cannot see through: f * v + (-0) is the rounded product, as one
// mixed-precision FMA when v is a half (no conversion)
__device__ __forceinline__ float opaque_minus_zero()
{
    float z;
    asm("s_mov_b32 %0, 0x80000000" : "=s"(z));
    return z;
}
// acc + f * v with two roundings, as the complex form with a zero imaginary factor has
template <typename T>
__device__ __forceinline__ typename Vec<T>::C add_scaled(typename Vec<T>::C acc, typename Vec<T>::C f, OpT<T> v, float mz)
{
#pragma clang fp contract(off)
    if constexpr (std::is_same<T, _Float16>::value) return acc + __builtin_fmaf((float)v, f, mz);
    else return acc + f * v;
}

template <int NC, typename TI, typename TO, int MB, int EPI = EPI_ANY>
__device__ __forceinline__ void hop_site(const HopArgs &a, int n0, int n1, int n2, const Site &p, int q0, int l0, int m)
{
    constexpr int NCOMP = 4 * NC;
    using LT = typename Vec<TI>::L;
    using CI = typename Vec<TI>::C;  // arithmetic type of the stencil
    using CO = typename Vec<TO>::C;  // arithmetic type of the epilogue
    const int V = n0 * n1 * n2, s = p.s;

    const LT *__restrict__ L = reinterpret_cast<const LT *>(a.links) + (size_t)l0 * NC * NC;
    constexpr int NN = NC * NC;

    // FP16 input stays in FP16 registers until the arithmetic widens it (hop_dir's projection)
    using PT = typename std::conditional<std::is_same<TI, _Float16>::value, _Float16, CI>::type;
    CI xr[NCOMP], xi[NCOMP];
    PT pr[NCOMP], pi[NCOMP];
    load_sp<NC, MB, TI>(a.in, 0, 0, q0 + s, m, pr, pi);
    const CI am = (CI)a.amass;
#pragma unroll
    for (int c = 0; c < NCOMP; ++c) { xr[c] = am * (CI)pr[c]; xi[c] = am * (CI)pi[c]; }

    {  // x direction
        const int sp = s + ((p.x + 1 == n0) ? 1 - n0 : 1);
        const int sm = s + ((p.x == 0) ? n0 - 1 : -1);
        load_sp<NC, MB, TI>(a.in, 0, 0, q0 + sp, m, pr, pi);
        hop_dir<NC, 0, 1>(pr, pi, L + ((size_t)0 * V + s) * NN, xr, xi);
        load_sp<NC, MB, TI>(a.in, 0, 0, q0 + sm, m, pr, pi);
        hop_dir<NC, 0, -1>(pr, pi, L + ((size_t)0 * V + sm) * NN, xr, xi);
    }
    {  // y direction
        const int sp = s + ((p.y + 1 == n1) ? (1 - n1) * n0 : n0);
        const int sm = s + ((p.y == 0) ? (n1 - 1) * n0 : -n0);
        load_sp<NC, MB, TI>(a.in, 0, 0, q0 + sp, m, pr, pi);
        hop_dir<NC, 1, 1>(pr, pi, L + ((size_t)1 * V + s) * NN, xr, xi);
        load_sp<NC, MB, TI>(a.in, 0, 0, q0 + sm, m, pr, pi);
        hop_dir<NC, 1, -1>(pr, pi, L + ((size_t)1 * V + sm) * NN, xr, xi);
    }
    {  // z direction
        const int sp = s + ((p.z + 1 == n2) ? (1 - n2) * n0 * n1 : n0 * n1);
        const int sm = s + ((p.z == 0) ? (n2 - 1) * n0 * n1 : -n0 * n1);
        load_sp<NC, MB, TI>(a.in, 0, 0, q0 + sp, m, pr, pi);
        hop_dir<NC, 2, 1>(pr, pi, L + ((size_t)2 * V + s) * NN, xr, xi);
        load_sp<NC, MB, TI>(a.in, 0, 0, q0 + sm, m, pr, pi);
        hop_dir<NC, 2, -1>(pr, pi, L + ((size_t)2 * V + sm) * NN, xr, xi);
    }

    // h_W = (1/2) gamma0 X, then the epilogue in the output precision
    const int q = q0 + s;
    CO orr[NCOMP], oi[NCOMP];
    if constexpr (EPI == EPI_PURE || EPI == EPI_CLENSHAW) {
        const CO f = (CO)0.5 * (CO)a.sh_r;
#pragma unroll
        for (int c = 0; c < NCOMP; ++c) {
            const CO g = (c < 2 * NC) ? f : -f;
            orr[c] = g * (CO)xr[c];
            oi[c] = g * (CO)xi[c];
        }
    }
    if constexpr (EPI == EPI_CLENSHAW) {
        OpT<TO> tr[NCOMP], ti[NCOMP];
        const float mz = std::is_same<TO, _Float16>::value ? opaque_minus_zero() : -0.0f;
        auto term = [&](const void *v, double factor) {
            load_sp_nt<NC, MB, TO>(v, 0, 0, q, m, tr, ti);
            const CO f = (CO)factor;
#pragma unroll
            for (int c = 0; c < NCOMP; ++c) {
                orr[c] = add_scaled<TO>(orr[c], f, tr[c], mz);
                oi[c] = add_scaled<TO>(oi[c], f, ti[c], mz);
            }
        };
        term(a.x, a.sx_r);
        term(a.b1, a.s1_r);
        term(a.b2, a.s2_r);
    }
    if constexpr (EPI == EPI_AXPY) {
        CO tr[NCOMP], ti[NCOMP];
        load_sp_nt<NC, MB, TO>(a.tgt, 0, 0, q, m, tr, ti);
        const CO f = (CO)0.5 * (CO)a.sh_i;
#pragma unroll
        for (int c = 0; c < NCOMP; ++c) {
            const CO g = (c < 2 * NC) ? f : -f;
            orr[c] = add_scaled<TO>(tr[c], -g, (CO)xi[c], -0.0f);
            oi[c] = add_scaled<TO>(ti[c], g, (CO)xr[c], -0.0f);
        }
    }
    if constexpr (EPI == EPI_ANY) {
    const CO shr = (CO)a.sh_r, shi = (CO)a.sh_i;
#pragma unroll
    for (int c = 0; c < NCOMP; ++c) {
        const CO g = (c < 2 * NC) ? (CO)0.5 : (CO)-0.5;
        const CO hr = g * (CO)xr[c], hi = g * (CO)xi[c];
        orr[c] = shr * hr - shi * hi;
        oi[c] = shr * hi + shi * hr;
    }
    CO tr[NCOMP], ti[NCOMP];
    if (a.x) {
        load_sp_nt<NC, MB, TO>(a.x, 0, 0, q, m, tr, ti);
        const CO cr = (CO)a.sx_r, ci = (CO)a.sx_i;
#pragma unroll
        for (int c = 0; c < NCOMP; ++c) {
            const CO g = (a.x_gamma0 && c >= 2 * NC) ? (CO)-1 : (CO)1;
            const CO vr = g * tr[c], vi = g * ti[c];
            orr[c] += cr * vr - ci * vi;
            oi[c] += cr * vi + ci * vr;
        }
    }
    if (a.out2) {  // sh*h_W(in) + sx*G(x) alone, times out2_scale (the overlap term of a leapfrog axpy)
        CO ur[NCOMP], ui[NCOMP];
        const CO f = (CO)a.out2_scale;
#pragma unroll
        for (int c = 0; c < NCOMP; ++c) { ur[c] = f * orr[c]; ui[c] = f * oi[c]; }
        store_sp<NC, MB, TO>(a.out2, 0, 0, q, m, ur, ui);
    }
    if (a.b1) {
        load_sp_nt<NC, MB, TO>(a.b1, 0, 0, q, m, tr, ti);
        const CO cr = (CO)a.s1_r, ci = (CO)a.s1_i;
#pragma unroll
        for (int c = 0; c < NCOMP; ++c) { orr[c] += cr * tr[c] - ci * ti[c]; oi[c] += cr * ti[c] + ci * tr[c]; }
    }
    if (a.b2) {
        load_sp_nt<NC, MB, TO>(a.b2, 0, 0, q, m, tr, ti);
        const CO cr = (CO)a.s2_r, ci = (CO)a.s2_i;
#pragma unroll
        for (int c = 0; c < NCOMP; ++c) { orr[c] += cr * tr[c] - ci * ti[c]; oi[c] += cr * ti[c] + ci * tr[c]; }
    }
    if (a.tgt) {
        load_sp_nt<NC, MB, TO>(a.tgt, 0, 0, q, m, tr, ti);
        const CO cr = (CO)a.st_r, ci = (CO)a.st_i;
#pragma unroll
        for (int c = 0; c < NCOMP; ++c) { orr[c] += cr * tr[c] - ci * ti[c]; oi[c] += cr * ti[c] + ci * tr[c]; }
    }
    }
    // the pure launch's output w is an intermediate of the step: 48-bit storage truncates it
    constexpr bool TRUNC = EPI == EPI_PURE;
    if (a.nt_out) store_sp_nt<NC, MB, TO, TRUNC>(a.out, 0, 0, q, m, orr, oi);
    else store_sp<NC, MB, TO, TRUNC>(a.out, 0, 0, q, m, orr, oi);
}

// WPE: minimum waves per SIMD the register allocation must allow (1 = compiler's choice); the
// stencil hoists its neighbour loads, so this trades memory-level parallelism per wave against
// waves in flight.  The host picks the variant per problem shape (autotune).
template <int NC, typename TI, typename TO, int MB, int WPE, int EPI>
__global__ __launch_bounds__(TPB) __attribute__((amdgpu_waves_per_eu(WPE))) void k_hop(HopArgs a, int n0, int n1,
                                                                                       int n2)
{
    const int V = n0 * n1 * n2;
    int m, blk;
    Site p;
    // 64-mode blocks have one site per wavefront: site and block are wave-uniform there, so that the links
    // (shared by all modes of the site) come through scalar loads instead of 64 identical vector lanes
    if (!lane_coords<MB>(a, blockIdx.x, gridDim.x, n0, n1, V, m, p, blk)) return;
    hop_site<NC, TI, TO, MB, EPI>(a, n0, n1, n2, p, blk * V, 0, m);
}

// Ensemble launch: many independent lattices of different sizes in one grid.  One tile = TPB lanes
// of one system: workgroup w.y of system w.x (lanes (site, mode) in block-major order, as k_hop's
// lexicographic traversal).
template <int NC, typename TI, typename TO, int MB, int EPI>
__device__ __forceinline__ void hop_ens_tile(const HopArgs &a, int2 w)
{
    const SysDesc d = a.ens_sys[w.x];
    const unsigned gl = (unsigned)w.y * TPB + threadIdx.x;  // lane within the system
    if (gl >= (unsigned)(d.V * d.nblk * MB)) return;
    const int m = (int)(gl % MB);
    unsigned r = gl / MB;
    if constexpr (MB == 64) r = __builtin_amdgcn_readfirstlane(r);  // one site per wavefront
    const int blk = (int)fdiv(r, d.dv_V);
    const int s = (int)r - blk * d.V;
    const int z = (int)fdiv((unsigned)s, d.dv_n01);
    const int rem = s - z * d.n0 * d.n1;
    const int y = (int)fdiv((unsigned)rem, d.dv_n0);
    hop_site<NC, TI, TO, MB, EPI>(a, d.n0, d.n1, d.n2, Site{s, rem - y * d.n0, y, z}, d.q0 + blk * d.V, d.l0, m);
}

// Static table (ens_qctr null): workgroup b runs tile ens_work[b]; the host cuts the tiles of all systems,
// system by system, into eight equal runs, one per XCD.
// Work queues (ens_qctr set): a persistent grid; workgroup b claims ens_per tiles at a time from the
// queue of XCD b % 8 until it is empty, so the tiles of an XCD's systems go to whichever of its
// workgroups is free.  Every workgroup leaves when its queue is exhausted (no workgroup waits on
// another); the last one of each queue to leave resets the queue's counters for the next launch.
template <int NC, typename TI, typename TO, int MB, int WPE, int EPI>
__global__ __launch_bounds__(TPB) __attribute__((amdgpu_waves_per_eu(WPE))) void k_hop_ens(HopArgs a)
{
    if (!a.ens_qctr) {
        const int2 w = a.ens_work[blockIdx.x];
        if (w.x >= 0) hop_ens_tile<NC, TI, TO, MB, EPI>(a, w);
        return;
    }
    const int q = (int)(blockIdx.x % NUM_XCD);
    const int beg = a.ens_qoff[q], len = a.ens_qoff[q + 1] - beg;
    __shared__ int claim;
    for (;;) {
        if (threadIdx.x == 0) claim = atomicAdd(&a.ens_qctr[q], 1);
        __syncthreads();
        const int t0 = claim * a.ens_per;
        __syncthreads();  // every lane has read `claim` before the next claim overwrites it
        if (t0 >= len) break;
        const int t1 = min(len, t0 + a.ens_per);
        for (int t = t0; t < t1; ++t) hop_ens_tile<NC, TI, TO, MB, EPI>(a, a.ens_qwork[beg + t]);
    }
    if (threadIdx.x == 0) {
        const int wgs = (int)(gridDim.x / NUM_XCD);
        if (atomicAdd(&a.ens_qctr[NUM_XCD + q], 1) == wgs - 1) {
            atomicExch(&a.ens_qctr[q], 0);
            atomicExch(&a.ens_qctr[NUM_XCD + q], 0);
        }
    }
}

// ---------------------------------------------------------------------------------------------
// pointwise kernels
// ---------------------------------------------------------------------------------------------
// precision conversion between the FP64 (double2) and FP32 (float4) layouts
// precision conversions between the field layouts, dst = scale * src.  A FP32 unit (float4) holds
// complex pairs 2r, 2r+1 and a FP16 unit (8 halves) complex 4r..4r+3 of the FP64 layout, where
// r = unit index / MB; the mode index is unit index % MB in all three.
__global__ __launch_bounds__(TPB) void k_d2f(const double2 *__restrict__ src, float4 *__restrict__ dst, long npairs,
                                             int mb, double scale)
{
    long i = (long)blockIdx.x * TPB + threadIdx.x;
    if (i >= npairs) return;
    const long m = i % mb, q = i / mb;
    const double2 a = src[(2 * q) * mb + m], b = src[(2 * q + 1) * mb + m];
    dst[i] = make_float4((float)(scale * a.x), (float)(scale * a.y), (float)(scale * b.x), (float)(scale * b.y));
}
__global__ __launch_bounds__(TPB) void k_f2d(const float4 *__restrict__ src, double2 *__restrict__ dst, long npairs,
                                             int mb, double scale)
{
    long i = (long)blockIdx.x * TPB + threadIdx.x;
    if (i >= npairs) return;
    const long m = i % mb, q = i / mb;
    const float4 t = src[i];
    dst[(2 * q) * mb + m] = make_double2(scale * t.x, scale * t.y);
    dst[(2 * q + 1) * mb + m] = make_double2(scale * t.z, scale * t.w);
}
__global__ __launch_bounds__(TPB) void k_d2h(const double2 *__restrict__ src, h8v *__restrict__ dst, long nunits,
                                             int mb, double scale)
{
    long i = (long)blockIdx.x * TPB + threadIdx.x;
    if (i >= nunits) return;
    const long m = i % mb, q = i / mb;
    h8v v;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const double2 a = src[(4 * q + j) * mb + m];
        v[2 * j] = (_Float16)(float)(scale * a.x);
        v[2 * j + 1] = (_Float16)(float)(scale * a.y);
    }
    dst[i] = v;
}
__global__ __launch_bounds__(TPB) void k_h2f(const h8v *__restrict__ src, float4 *__restrict__ dst, long nunits,
                                             int mb, float scale)
{
    long i = (long)blockIdx.x * TPB + threadIdx.x;
    if (i >= nunits) return;
    const long m = i % mb, q = i / mb;
    const h8v t = src[i];
    dst[(2 * q) * mb + m] = make_float4(scale * (float)t[0], scale * (float)t[1], scale * (float)t[2], scale * (float)t[3]);
    dst[(2 * q + 1) * mb + m] =
        make_float4(scale * (float)t[4], scale * (float)t[5], scale * (float)t[6], scale * (float)t[7]);
}

// one group of 4 complex numbers (group q of the FP64 numbering: complex 4q..4q+3 of a mode
// block's (site, comp) sequence, mode m) in any of the four layouts, as doubles
template <typename T>
__device__ __forceinline__ void load_group(const void *__restrict__ base, long q, long m, int mb, double *re, double *im)
{
    if constexpr (sizeof(T) == 6) {
        const u4v *p = reinterpret_cast<const u4v *>(base);
        unpack48(p[(3 * q) * mb + m], p[(3 * q + 1) * mb + m], p[(3 * q + 2) * mb + m], 0, re, im);
    } else if constexpr (sizeof(T) == 8) {
        const double2 *p = reinterpret_cast<const double2 *>(base);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const double2 t = p[(4 * q + j) * mb + m];
            re[j] = t.x;
            im[j] = t.y;
        }
    } else if constexpr (sizeof(T) == 4) {
        const float4 *p = reinterpret_cast<const float4 *>(base);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const float4 t = p[(2 * q + j) * mb + m];
            re[2 * j] = t.x;
            im[2 * j] = t.y;
            re[2 * j + 1] = t.z;
            im[2 * j + 1] = t.w;
        }
    } else {
        const h8v t = reinterpret_cast<const h8v *>(base)[q * mb + m];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            re[j] = (double)t[2 * j];
            im[j] = (double)t[2 * j + 1];
        }
    }
}
template <typename T>
__device__ __forceinline__ void store_group(void *__restrict__ base, long q, long m, int mb, const double *re,
                                            const double *im)
{
    if constexpr (sizeof(T) == 6) {
        u4v A, B, M;
        pack48(re, im, 0, A, B, M);
        u4v *p = reinterpret_cast<u4v *>(base);
        p[(3 * q) * mb + m] = A;
        p[(3 * q + 1) * mb + m] = B;
        p[(3 * q + 2) * mb + m] = M;
    } else if constexpr (sizeof(T) == 8) {
        double2 *p = reinterpret_cast<double2 *>(base);
#pragma unroll
        for (int j = 0; j < 4; ++j) p[(4 * q + j) * mb + m] = make_double2(re[j], im[j]);
    } else if constexpr (sizeof(T) == 4) {
        float4 *p = reinterpret_cast<float4 *>(base);
#pragma unroll
        for (int j = 0; j < 2; ++j)
            p[(2 * q + j) * mb + m] =
                make_float4((float)re[2 * j], (float)im[2 * j], (float)re[2 * j + 1], (float)im[2 * j + 1]);
    } else {
        h8v v;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            v[2 * j] = (_Float16)re[j];
            v[2 * j + 1] = (_Float16)im[j];
        }
        reinterpret_cast<h8v *>(base)[q * mb + m] = v;
    }
}
// dst = scale * src, one (group, mode) per lane (the conversions to and from the 48-bit layout)
template <typename TS, typename TD>
__global__ __launch_bounds__(TPB) void k_convert(const void *__restrict__ src, void *__restrict__ dst, long nlanes,
                                                 int mb, double scale)
{
    const long i = (long)blockIdx.x * TPB + threadIdx.x;
    if (i >= nlanes) return;
    const long m = i % mb, q = i / mb;
    double re[4], im[4];
    load_group<TS>(src, q, m, mb, re, im);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        re[j] *= scale;
        im[j] *= scale;
    }
    store_group<TD>(dst, q, m, mb, re, im);
}

template <typename T>
__global__ __launch_bounds__(TPB) void k_lincomb(T *__restrict__ out, const T *__restrict__ a, double car, double cai,
                                                 const T *__restrict__ b, double cbr, double cbi, long ncplx)
{
    long i = (long)blockIdx.x * TPB + threadIdx.x;
    if (i >= ncplx) return;
    const T ar = a[2 * i], ai = a[2 * i + 1];
    T r = (T)car * ar - (T)cai * ai, im = (T)car * ai + (T)cai * ar;
    if (b) {
        const T br = b[2 * i], bi = b[2 * i + 1];
        r += (T)cbr * br - (T)cbi * bi;
        im += (T)cbr * bi + (T)cbi * br;
    }
    out[2 * i] = r;
    out[2 * i + 1] = im;
}

// host AoS (count modes starting at `first`) <-> device SoA FP64
__global__ __launch_bounds__(TPB) void k_aos_to_soa(const double2 *__restrict__ aos, double2 *__restrict__ f, int first,
                                                    int count, int V, int ncomp, int mb)
{
    long i = (long)blockIdx.x * TPB + threadIdx.x;
    long tot = (long)count * V * ncomp;
    if (i >= tot) return;
    // host AoS component = colour*4 + spin; device component = spin*Nc + colour
    const int ca = (int)(i % ncomp);
    const int c = (ca % 4) * (ncomp / 4) + ca / 4;
    const long q = i / ncomp;
    const int s = (int)(q % V);
    const int k = (int)(q / V);
    const int mode = first + k, blk = mode / mb, m = mode % mb;
    f[((size_t)(blk * V + s) * ncomp + c) * mb + m] = aos[i];
}

__global__ __launch_bounds__(TPB) void k_soa_to_aos(const double2 *__restrict__ f, double2 *__restrict__ aos, int first,
                                                    int count, int V, int ncomp, int mb)
{
    long i = (long)blockIdx.x * TPB + threadIdx.x;
    long tot = (long)count * V * ncomp;
    if (i >= tot) return;
    // host AoS component = colour*4 + spin; device component = spin*Nc + colour
    const int ca = (int)(i % ncomp);
    const int c = (ca % 4) * (ncomp / 4) + ca / 4;
    const long q = i / ncomp;
    const int s = (int)(q % V);
    const int k = (int)(q / V);
    const int mode = first + k, blk = mode / mb, m = mode % mb;
    aos[i] = f[((size_t)(blk * V + s) * ncomp + c) * mb + m];
}

// ---------------------------------------------------------------------------------------------
// gauge-link algebra (FP64)
// ---------------------------------------------------------------------------------------------
struct cd { double r, i; };
__device__ __forceinline__ cd cmul(cd a, cd b) { return {a.r * b.r - a.i * b.i, a.r * b.i + a.i * b.r}; }
__device__ __forceinline__ cd cadd(cd a, cd b) { return {a.r + b.r, a.i + b.i}; }

template <int NC> struct Mat { cd e[NC * NC]; };

template <int NC> __device__ __forceinline__ Mat<NC> mmul(const Mat<NC> &a, const Mat<NC> &b)
{
    Mat<NC> c;
#pragma unroll
    for (int i = 0; i < NC; ++i)
#pragma unroll
        for (int j = 0; j < NC; ++j) {
            cd s = {0, 0};
#pragma unroll
            for (int k = 0; k < NC; ++k) s = cadd(s, cmul(a.e[i * NC + k], b.e[k * NC + j]));
            c.e[i * NC + j] = s;
        }
    return c;
}

template <int NC> __device__ __forceinline__ Mat<NC> mdag(const Mat<NC> &a)
{
    Mat<NC> c;
#pragma unroll
    for (int i = 0; i < NC; ++i)
#pragma unroll
        for (int j = 0; j < NC; ++j) c.e[i * NC + j] = {a.e[j * NC + i].r, -a.e[j * NC + i].i};
    return c;
}

template <int NC> __device__ __forceinline__ Mat<NC> mid()
{
    Mat<NC> c;
#pragma unroll
    for (int i = 0; i < NC * NC; ++i) c.e[i] = {0, 0};
#pragma unroll
    for (int i = 0; i < NC; ++i) c.e[i * NC + i] = {1, 0};
    return c;
}

// first double of link (s, mu) in the reference format.  54 doubles a site in SU(3): a 32-bit product overflows from
// 2^31 / 54 = 39.8 million sites on
template <int NC> __host__ __device__ constexpr size_t link_at(int s, int mu)
{
    return (size_t)(NC == 2 ? 4 : 18) * (mu + 3 * (size_t)s);
}
static_assert(link_at<3>(OVL_NOALLOC_MAX_SITES - 1, 2) + 18 == 54ull * OVL_NOALLOC_MAX_SITES &&
                  link_at<2>(OVL_NOALLOC_MAX_SITES - 1, 2) + 4 == 12ull * OVL_NOALLOC_MAX_SITES,
              "the last link of the largest lattice");

// master link (reference format) -> row-major matrix
template <int NC> __device__ __forceinline__ Mat<NC> get_link(const double *__restrict__ links, int s, int mu)
{
    Mat<NC> m;
    if constexpr (NC == 2) {
        const double *u = links + link_at<2>(s, mu);  // GetMatrix, SU2/GroupOperations.cpp:213-225
        m.e[0] = {u[3], u[2]};
        m.e[1] = {u[1], u[0]};
        m.e[2] = {-u[1], u[0]};
        m.e[3] = {u[3], -u[2]};
    } else {
        const double *u = links + link_at<3>(s, mu);
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) m.e[i * 3 + j] = {u[2 * (i + 3 * j)], u[2 * (i + 3 * j) + 1]};
    }
    return m;
}

// generators t^a as (row, col, value) entries; value = (re, im) times 1/2 (SU(3): lambda_8/(2 sqrt 3))
template <int NC> __device__ __forceinline__ Mat<NC> alg_to_mat(const double *alpha)
{
    Mat<NC> m;
    if constexpr (NC == 2) {  // alpha_a sigma_a / 2
        m.e[0] = {0.5 * alpha[2], 0};
        m.e[3] = {-0.5 * alpha[2], 0};
        m.e[1] = {0.5 * alpha[0], -0.5 * alpha[1]};
        m.e[2] = {0.5 * alpha[0], 0.5 * alpha[1]};
    } else {  // alpha_a lambda_a / 2
        const double r3 = 0.5 / sqrt(3.0);
        m.e[0] = {__builtin_fma(r3, alpha[7], 0.5 * alpha[2]), 0};
        m.e[4] = {__builtin_fma(r3, alpha[7], -0.5 * alpha[2]), 0};
        m.e[8] = {-2.0 * r3 * alpha[7], 0};
        m.e[1] = {0.5 * alpha[0], -0.5 * alpha[1]};
        m.e[3] = {0.5 * alpha[0], 0.5 * alpha[1]};
        m.e[2] = {0.5 * alpha[3], -0.5 * alpha[4]};
        m.e[6] = {0.5 * alpha[3], 0.5 * alpha[4]};
        m.e[5] = {0.5 * alpha[5], -0.5 * alpha[6]};
        m.e[7] = {0.5 * alpha[5], 0.5 * alpha[6]};
    }
    return m;
}

// ReTr(i t^a V) = retr_factor(a) * out[a] for all generators: tr(t^a V) = sum_ij t_ij V_ji, ReTr(i X) = -Im tr X
template <int NC> __device__ __forceinline__ void retr_sums(const Mat<NC> &v, double *out)
{
    if constexpr (NC == 2) {
        // t0: (0,1)=(1,0)=1/2 -> tr = (V10 + V01)/2
        out[0] = v.e[2].i + v.e[1].i;
        // t1: (0,1)=-i/2, (1,0)=i/2 -> tr = (-i V10 + i V01)/2 ; Im = (V01.r - V10.r)/2
        out[1] = v.e[1].r - v.e[2].r;
        out[2] = v.e[0].i - v.e[3].i;
    } else {
        out[0] = v.e[3].i + v.e[1].i;
        out[1] = v.e[1].r - v.e[3].r;
        out[2] = v.e[0].i - v.e[4].i;
        out[3] = v.e[6].i + v.e[2].i;
        out[4] = v.e[2].r - v.e[6].r;
        out[5] = v.e[7].i + v.e[5].i;
        out[6] = v.e[5].r - v.e[7].r;
        out[7] = v.e[0].i + v.e[4].i - 2.0 * v.e[8].i;
    }
}
__device__ __forceinline__ double retr_factor(int a) { return a == 7 ? -0.5 / sqrt(3.0) : -0.5; }
template <int NC> __device__ __forceinline__ void retr_it(const Mat<NC> &v, double *out)
{
    retr_sums<NC>(v, out);
#pragma unroll
    for (int a = 0; a < NC * NC - 1; ++a) out[a] *= retr_factor(a);
}

// column `col` of A B from A and the column of B: the sums of mmul, each complex product with two roundings
// per part in a fixed form (AR: the imaginary part rounds a.i b.r first, else a.r b.i), so that a link does
// not depend on how the compiler contracts the expression around it (an FP32 evolution amplifies the
// last bit of a link to the size of its own rounding)
template <bool AR> __device__ __forceinline__ void mcol(const Mat<3> &a, cd *b)
{
    cd r[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        cd s = {0, 0};
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const cd x = a.e[i * 3 + k], y = b[k];
            s = cadd(s, {__builtin_fma(x.r, y.r, -(x.i * y.i)),
                         AR ? __builtin_fma(x.r, y.i, x.i * y.r) : __builtin_fma(x.i, y.r, x.r * y.i)});
        }
        r[i] = s;
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) b[i] = r[i];
}

// the matrix whose columns the lanes 4 q .. 4 q + 2 of a wavefront hold
__device__ __forceinline__ Mat<3> gather_columns(const cd *c)
{
    Mat<3> m;
    const int base = (int)(threadIdx.x & 60);
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int i = 0; i < 3; ++i) m.e[i * 3 + j] = {__shfl(c[i].r, base + j, 64), __shfl(c[i].i, base + j, 64)};
    return m;
}

// the same from one lane's three columns
__device__ __forceinline__ Mat<3> from_columns(const cd (&c)[3][3])
{
    Mat<3> m;
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int i = 0; i < 3; ++i) m.e[i * 3 + j] = c[j][i];
    return m;
}

// 1/k of the Taylor series (a division would be as long as the product it scales)
__device__ const double inverse_of[21] = {0.0,      1.0,      1.0 / 2,  1.0 / 3,  1.0 / 4,  1.0 / 5,  1.0 / 6,
                                          1.0 / 7,  1.0 / 8,  1.0 / 9,  1.0 / 10, 1.0 / 11, 1.0 / 12, 1.0 / 13,
                                          1.0 / 14, 1.0 / 15, 1.0 / 16, 1.0 / 17, 1.0 / 18, 1.0 / 19, 1.0 / 20};

// exp(i c alpha^a t^a) by scaling and squaring of the Taylor series (FP64): the scaled matrix and the number of
// squarings
__device__ __forceinline__ int iexp_scale(double c, const double *alpha, Mat<3> &a)
{
    a = alg_to_mat<3>(alpha);
    double nrm = 0;
#pragma unroll
    for (int i = 0; i < 9; ++i) {
        a.e[i] = {-c * a.e[i].i, c * a.e[i].r};  // i c A
        nrm += a.e[i].r * a.e[i].r + a.e[i].i * a.e[i].i;
    }
    nrm = sqrt(nrm);
    int sq = 0;
    while (nrm > 0.25 && sq < 64) { nrm *= 0.5; ++sq; }
    const double sc = ldexp(1.0, -sq);
#pragma unroll
    for (int i = 0; i < 9; ++i) { a.e[i].r *= sc; a.e[i].i *= sc; }
    return sq;
}
// column `col` of the series, Horner: I + a(1 + a/2(1 + a/3(...))).  The columns are independent.
__device__ __forceinline__ void iexp_series(const Mat<3> &a, int col, cd *r)
{
    const double one[3] = {col == 0 ? 1.0 : 0.0, col == 1 ? 1.0 : 0.0, col == 2 ? 1.0 : 0.0};
#pragma unroll
    for (int i = 0; i < 3; ++i) r[i] = {one[i], 0.0};
    for (int k = 20; k >= 1; --k) {
        mcol<true>(a, r);
        const double f = inverse_of[k];
#pragma unroll
        for (int i = 0; i < 3; ++i) r[i] = {__builtin_fma(f, r[i].r, one[i]), f * r[i].i};
    }
}

// project onto SU(3): the unitary polar factor P = V (V^+ V)^{-1/2} (the U(3) matrix closest to V,
// of largest Re Tr(P^+ V)) by the Newton iteration X <- (X + X^{-+})/2, quadratically convergent
// from any nonsingular V (Higham 1986; six steps take a drift of 1e-3 far below rounding), then
// P det(P)^{-1/3} with the principal cube root so that det = 1.  The reference's SU(3)
// MaxTraceProjection (SU3/GroupOperations.cpp:510-533, Cabibbo-Marinari sweeps over SU(3)) agrees
// to second order in the distance of V from the group.
__device__ __forceinline__ cd cdiv(cd a, cd b)
{
    const double d = 1.0 / (b.r * b.r + b.i * b.i);
    return {(a.r * b.r + a.i * b.i) * d, (a.i * b.r - a.r * b.i) * d};
}
__device__ __forceinline__ cd csub(cd a, cd b) { return {a.r - b.r, a.i - b.i}; }

__device__ Mat<3> reunit3(Mat<3> x)
{
    for (int it = 0; it < 6; ++it) {
        const cd *a = x.e;
        const cd c00 = csub(cmul(a[4], a[8]), cmul(a[5], a[7]));
        const cd c01 = csub(cmul(a[5], a[6]), cmul(a[3], a[8]));
        const cd c02 = csub(cmul(a[3], a[7]), cmul(a[4], a[6]));
        const cd det = cadd(cadd(cmul(a[0], c00), cmul(a[1], c01)), cmul(a[2], c02));
        Mat<3> inv;  // row-major inverse: adjugate / det
        inv.e[0] = cdiv(c00, det);
        inv.e[3] = cdiv(c01, det);
        inv.e[6] = cdiv(c02, det);
        inv.e[1] = cdiv(csub(cmul(a[2], a[7]), cmul(a[1], a[8])), det);
        inv.e[4] = cdiv(csub(cmul(a[0], a[8]), cmul(a[2], a[6])), det);
        inv.e[7] = cdiv(csub(cmul(a[1], a[6]), cmul(a[0], a[7])), det);
        inv.e[2] = cdiv(csub(cmul(a[1], a[5]), cmul(a[2], a[4])), det);
        inv.e[5] = cdiv(csub(cmul(a[2], a[3]), cmul(a[0], a[5])), det);
        inv.e[8] = cdiv(csub(cmul(a[0], a[4]), cmul(a[1], a[3])), det);
        Mat<3> nx;
        for (int i = 0; i < 3; ++i)
            for (int j = 0; j < 3; ++j) {  // (X^{-+})_{ij} = conj((X^{-1})_{ji})
                const cd v = x.e[i * 3 + j], w = inv.e[j * 3 + i];
                nx.e[i * 3 + j] = {0.5 * (v.r + w.r), 0.5 * (v.i - w.i)};
            }
        x = nx;
    }
    const cd *a = x.e;
    const cd det = cadd(cadd(cmul(a[0], csub(cmul(a[4], a[8]), cmul(a[5], a[7]))),
                             cmul(a[1], csub(cmul(a[5], a[6]), cmul(a[3], a[8])))),
                        cmul(a[2], csub(cmul(a[3], a[7]), cmul(a[4], a[6]))));
    const double ph = -atan2(det.i, det.r) / 3.0;
    const cd f = {cos(ph), sin(ph)};
    for (int k = 0; k < 9; ++k) x.e[k] = cmul(x.e[k], f);
    return x;
}

// one entry of the stencil links (ConvertGaugeLinks, OverlapEvolutionOperator.cpp:23-51, with the QED
// phase folded in).  The products round in a fixed form, so that every kernel that writes a stencil link
// writes the same bits: PI: the imaginary part rounds ph.i m.r first, else ph.r m.i
template <bool PI>
__device__ __forceinline__ void put_stencil_entry(cd ph, cd m, double2 *__restrict__ u64, float2 *__restrict__ u32, size_t k)
{
    const cd v = {__builtin_fma(ph.r, m.r, -(ph.i * m.i)),
                  PI ? __builtin_fma(ph.r, m.i, ph.i * m.r) : __builtin_fma(ph.i, m.r, ph.r * m.i)};
    u64[k] = make_double2(v.r, v.i);
    u32[k] = make_float2((float)v.r, (float)v.i);
}
__device__ __forceinline__ cd phase_of(const double2 *__restrict__ phase, int i)
{
    if (!phase) return {1, 0};
    return {phase[i].x, phase[i].y};
}

template <int NC>
__global__ __launch_bounds__(TPB) void k_link_setup(const double *__restrict__ links, const double2 *__restrict__ phase,
                                                    double2 *__restrict__ u64, float2 *__restrict__ u32, int V)
{
    const int i = blockIdx.x * TPB + threadIdx.x;
    if (i >= 3 * V) return;
    const int mu = i / V, s = i - mu * V;
    const Mat<NC> m = get_link<NC>(links, s, mu);
    const cd ph = phase_of(phase, i);
#pragma unroll
    for (int k = 0; k < NC * NC; ++k) {
        if (NC == 2 && (k == 1 || k == 2)) put_stencil_entry<true>(ph, m.e[k], u64, u32, (size_t)i * NC * NC + k);
        else put_stencil_entry<false>(ph, m.e[k], u64, u32, (size_t)i * NC * NC + k);
    }
}

// stencil links from a host-layout u_cc array (already in [mu*V+s][i][j] order)
__global__ __launch_bounds__(TPB) void k_ucc_setup(const double2 *__restrict__ ucc, double2 *__restrict__ u64,
                                                   float2 *__restrict__ u32, long n)
{
    const long i = (long)blockIdx.x * TPB + threadIdx.x;
    if (i >= n) return;
    const double2 v = ucc[i];
    u64[i] = v;
    u32[i] = make_float2((float)v.x, (float)v.y);
}

// Dynamics.cpp:97-138: U <- exp(i cU E) U with cU = -dt.  With u64 the new stencil links are written in the
// same pass (the leapfrog's half step: one launch instead of two, and the links are not read again).
// A workgroup is one wavefront, so that a small lattice spreads over the CUs.  SU(3): LPL = 4 lanes per
// link, the first three a column each: a third of the chain of 20 matrix products per lane.  With a lane per
// link and the stencil links apart: 11.1 + 4.8 us on 15 x 12 x 10 (the serial chain in 22 workgroups) and
// 14.1 + 7.5 us on 24^3 SU(3); so 5.7 and 15.7 us (24^3: 25 MB read and written in 144-byte strides).  LPL = 1, the
// same sums in one lane, does not pay for the fourth lane and the exchanges of the others: ovl_update_links with
// LPL = 4 and 1, 24^3 23.1 and 23.5 us, 32^3 33.2 and 31.8, 40^3 54.5 and 44.1, 56^3 123 and 96.
constexpr int LINK_TPB = 64;
template <int NC, int LPL>
__device__ __forceinline__ void link_update_lane(unsigned lane, double *__restrict__ links, const double *__restrict__ e,
                                                 double dt, int V, int reunit, const double2 *__restrict__ phase,
                                                 double2 *__restrict__ u64, float2 *__restrict__ u32)
{
    const int i = (int)(lane / LPL);
    if (i >= 3 * V) return;  // the lanes of a link leave together
    const int s = i / 3, mu = i - 3 * s;  // link (s, mu) at index mu + 3 s
    constexpr int NG = NC * NC - 1;
    double al[NG];
#pragma unroll
    for (int a = 0; a < NG; ++a) al[a] = e[(size_t)NG * i + a];
    const double c = -dt;
    if constexpr (NC == 2) {
        // MatrixIExp (SU2/AlgebraOperations.cpp:37-55) and UU (SU2/GroupOperations.cpp:103-110)
        const double d = sqrt((c * al[0]) * (c * al[0]) + (c * al[1]) * (c * al[1]) + (c * al[2]) * (c * al[2]));
        double up[4];
        if (d != 0) {
            const double mm = c * sin(0.5 * d) / d;
            up[0] = mm * al[0]; up[1] = mm * al[1]; up[2] = mm * al[2]; up[3] = cos(0.5 * d);
        } else {
            up[0] = up[1] = up[2] = 0; up[3] = 1;
        }
        double *u = links + 4 * (size_t)i;
        const double o0 = u[0], o1 = u[1], o2 = u[2], o3 = u[3];
        double n0 = up[3] * o0 + up[0] * o3 - (up[1] * o2 - up[2] * o1);
        double n1 = up[3] * o1 + up[1] * o3 + (up[0] * o2 - up[2] * o0);
        double n2 = up[3] * o2 + up[2] * o3 - (up[0] * o1 - up[1] * o0);
        double n3 = up[3] * o3 - up[0] * o0 - up[1] * o1 - up[2] * o2;
        if (reunit) {  // MaxTraceProjection (SU2/GroupOperations.cpp:261-270)
            const double nn = sqrt(n0 * n0 + n1 * n1 + n2 * n2 + n3 * n3);
            n0 /= nn; n1 /= nn; n2 /= nn; n3 /= nn;
        }
        u[0] = n0; u[1] = n1; u[2] = n2; u[3] = n3;
        if (u64) {
            const int iu = mu * V + s;
            const cd ph = phase_of(phase, iu);
            put_stencil_entry<false>(ph, cd{n3, n2}, u64, u32, (size_t)iu * 4);
            put_stencil_entry<true>(ph, cd{n1, n0}, u64, u32, (size_t)iu * 4 + 1);
            put_stencil_entry<true>(ph, cd{-n1, n0}, u64, u32, (size_t)iu * 4 + 2);
            put_stencil_entry<false>(ph, cd{n3, -n2}, u64, u32, (size_t)iu * 4 + 3);
        }
    } else if constexpr (LPL == 1) {
        double *u = links + 18 * (size_t)i;
        Mat<3> a;
        const int sq = iexp_scale(c, al, a);
        cd r[3][3];
#pragma unroll
        for (int j = 0; j < 3; ++j) iexp_series(a, j, r[j]);
        for (int k = 0; k < sq; ++k) {
            a = from_columns(r);
#pragma unroll
            for (int j = 0; j < 3; ++j) mcol<true>(a, r[j]);
        }
        a = from_columns(r);
#pragma unroll
        for (int j = 0; j < 3; ++j) {
#pragma unroll
            for (int k = 0; k < 3; ++k) r[j][k] = {u[6 * j + 2 * k], u[6 * j + 2 * k + 1]};
            mcol<false>(a, r[j]);
        }
        a = from_columns(r);
        if (reunit) a = reunit3(a);
#pragma unroll
        for (int j = 0; j < 3; ++j)
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                u[6 * j + 2 * k] = a.e[3 * k + j].r;
                u[6 * j + 2 * k + 1] = a.e[3 * k + j].i;
            }
        if (u64) {
            const int iu = mu * V + s;
            const cd ph = phase_of(phase, iu);
#pragma unroll
            for (int k = 0; k < 9; ++k) put_stencil_entry<false>(ph, a.e[k], u64, u32, (size_t)iu * 9 + k);
        }
    } else {
        const int col = threadIdx.x % 4 < 3 ? threadIdx.x % 4 : 0;  // the fourth lane repeats the first
        double *u = links + 18 * (size_t)i + 6 * col;
        Mat<3> a;
        const int sq = iexp_scale(c, al, a);
        cd ex[3], r[3];
        iexp_series(a, col, ex);
        for (int k = 0; k < sq; ++k) {  // sq is the same in the four lanes of a link
            const Mat<3> m = gather_columns(ex);
            mcol<true>(m, ex);
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) r[k] = {u[2 * k], u[2 * k + 1]};
        mcol<false>(gather_columns(ex), r);
        if (reunit) {
            const Mat<3> m = reunit3(gather_columns(r));
#pragma unroll
            for (int k = 0; k < 3; ++k) r[k] = col == 0 ? m.e[3 * k] : (col == 1 ? m.e[3 * k + 1] : m.e[3 * k + 2]);
        }
        if (threadIdx.x % 4 == 3) return;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            u[2 * k] = r[k].r;
            u[2 * k + 1] = r[k].i;
        }
        if (u64) {
            const int iu = mu * V + s;
            const cd ph = phase_of(phase, iu);
#pragma unroll
            for (int k = 0; k < 3; ++k) put_stencil_entry<false>(ph, r[k], u64, u32, (size_t)iu * 9 + 3 * k + col);
        }
    }
}
template <int NC, int LPL>
__global__ __launch_bounds__(LINK_TPB) void k_link_update(GaugeHalf g)
{
    link_update_lane<NC, LPL>(blockIdx.x * LINK_TPB + threadIdx.x, g.links, g.efield, g.dt, g.V, g.reunit,
                         (const double2 *)g.phase, (double2 *)g.ul64, (float2 *)g.ul32);
}

__device__ __forceinline__ int nbr(int s, int dmu, int step, int n0, int n1, int n2)
{
    int z = s / (n0 * n1), rem = s - z * n0 * n1, y = rem / n0, x = rem - y * n0;
    if (dmu == 0) { x = (x + step) % n0; if (x < 0) x += n0; }
    else if (dmu == 1) { y = (y + step) % n1; if (y < 0) y += n1; }
    else { z = (z + step) % n2; if (z < 0) z += n2; }
    return x + n0 * (y + n1 * z);
}

// E_mu(x) += dt * (-2) sum_{nu != mu} [ReTr(i t^a U_{mu nu}(x)) + ReTr(i t^a U_{mu,-nu}(x))]
// (Hamilton's equation of H = 1/2 E^2 + 2 sum ReTr(1 - U_plaq) for U' = -i E U; the
// reference's plaquette macros used by Dynamics.cpp:145-197 are absent)
// Four lanes per link (LPL = 4), one plaquette each (two planes, forward and backward), their components summed
// from the four lanes: a lane's chain is three matrix products instead of twelve (SU(3): 14.1 -> 7.3 us on
// 15 x 12 x 10, where a lane per link left most CUs without a wave, 17.8 -> 15.3 us on 24^3, where the
// matrices' strided loads bound it).  The lanes of a wavefront then walk both the forward and the backward
// products; with LPL = 1, one lane and the same sums, none does: ovl_update_efield
// with LPL = 4 and 1, SU(2) 16^3 14.8 and 15.5 us, 24^3 17.3 and 15.9, 32^3 21.3 and 17.9, 64^3 72 and 46 (48^3 29.2
// and 64^3 43.2 in workgroups of one wavefront, 28.4 and 42.1 in workgroups of four).  SU(3)
// has four lanes throughout: in one lane 24^3 takes 24.5 us instead of 23.7, 48^3 97.6 instead of 88.4.

// sums of ReTr(i t^a U_plaq) (retr_sums) of plaquette j of link (s, mu): plane (mu, the j/2-th other direction), j odd:
// the backward one
template <int NC>
__device__ __forceinline__ void plaquette_sums(const double *__restrict__ links, int s, int mu, int j, int n0, int n1, int n2,
                                               double *f)
{
    const int nu = j < 2 ? (mu == 0 ? 1 : 0) : (mu == 2 ? 1 : 2);  // the two other directions, ascending
    const bool back = j & 1;
    const int sp = nbr(s, mu, 1, n0, n1, n2);
    // forward:  U_mu(x) U_nu(x+mu) U_mu(x+nu)^+ U_nu(x)^+
    // backward: U_mu(x) U_nu(x+mu-nu)^+ U_mu(x-nu)^+ U_nu(x-nu)
    Mat<NC> p = get_link<NC>(links, s, mu);
    if (back) {
        const int sn = nbr(s, nu, -1, n0, n1, n2);
        p = mmul<NC>(p, mdag<NC>(get_link<NC>(links, nbr(sp, nu, -1, n0, n1, n2), nu)));
        p = mmul<NC>(p, mdag<NC>(get_link<NC>(links, sn, mu)));
        p = mmul<NC>(p, get_link<NC>(links, sn, nu));
    } else {
        p = mmul<NC>(p, get_link<NC>(links, sp, nu));
        p = mmul<NC>(p, mdag<NC>(get_link<NC>(links, nbr(s, nu, 1, n0, n1, n2), mu)));
        p = mmul<NC>(p, mdag<NC>(get_link<NC>(links, s, nu)));
    }
    retr_sums<NC>(p, f);
}
template <int NC, int LPL>
__device__ __forceinline__ void efield_update_lane(unsigned lane, const double *__restrict__ links, double *__restrict__ e,
                                                   double dt, int n0, int n1, int n2)
{
    const int V = n0 * n1 * n2;
    const int i = (int)(lane / LPL);
    constexpr int NG = NC * NC - 1;
    if constexpr (LPL == 1) {
        if (i >= 3 * V) return;
        const int s = i / 3, mu = i - 3 * s;
        double t[NG];
#pragma unroll
        for (int k = 0; k < NG; ++k) t[k] = 0;
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            double f[NG];
            plaquette_sums<NC>(links, s, mu, l, n0, n1, n2, f);
#pragma unroll
            for (int k = 0; k < NG; ++k) t[k] = __builtin_fma(retr_factor(k), f[k], t[k]);
        }
        double *o = e + (size_t)NG * i;
#pragma unroll
        for (int k = 0; k < NG; ++k) o[k] += -2.0 * dt * t[k];
    } else {
        const int j = threadIdx.x % 4;
        const bool ok = i < 3 * V;
        const int il = ok ? i : 3 * V - 1;
        const int s = il / 3, mu = il - 3 * s;
        double f[NG];
        plaquette_sums<NC>(links, s, mu, j, n0, n1, n2, f);
        const int base = (int)(threadIdx.x & 60);
#pragma unroll
        for (int k = 0; k < NG; ++k) {  // in the order of the planes
            double t = 0;
#pragma unroll
            for (int l = 0; l < 4; ++l) t = __builtin_fma(retr_factor(k), __shfl(f[k], base + l, 64), t);
            f[k] = t;
        }
        if (!ok) return;
        double *o = e + (size_t)NG * i;
#pragma unroll
        for (int k = 0; k < NG; ++k)
            if (k % 4 == j) o[k] += -2.0 * dt * f[k];
    }
}
template <int NC, int LPL, int NT> __global__ __launch_bounds__(NT) void k_efield_update(GaugeHalf g)
{
    efield_update_lane<NC, LPL>(blockIdx.x * NT + threadIdx.x, g.links, g.efield, g.dt, g.n0, g.n1, g.n2);
}

// A Wilson half step and a gauge half step in one launch: the first gauge.blocks workgroups (a multiple of the
// XCDs, so that the others keep theirs) update the links (into other stencil links than the ones being
// read) or the E field, the rest are the stencil's.  The two do not depend on each other, and on small
// lattices each is a launch that leaves most of the chip idle.  The stencil keeps its registers (VGPRs, 16/32- and
// 64-mode blocks, as k_hop and here: SU(2) FP64 234, 162 and 236, 164; FP32 124, 82 and 126, 122; SU(3) FP64 398, 244 and
// 396, 246; FP32 203, 125 and 204, 127), so only SU(2) in FP32 with 64-mode blocks has fewer waves, four instead of
// five per SIMD.
template <int NC, typename T, int MB>
__global__ __launch_bounds__(TPB) void k_hop_gauge(HopArgs a, GaugeHalf g, int n0, int n1, int n2)
{
    if (blockIdx.x < (unsigned)g.blocks) {
        const unsigned lane = blockIdx.x * TPB + threadIdx.x;
        if (g.what == GAUGE_LINKS_HALF)
            link_update_lane<NC, NC == 2 ? 1 : 4>(lane, g.links, g.efield, g.dt, g.V, g.reunit, (const double2 *)g.phase,
                                                  (double2 *)g.ul64, (float2 *)g.ul32);
        else if (NC == 2 && g.lpl == 1) efield_update_lane<NC, NC == 2 ? 1 : 4>(lane, g.links, g.efield, g.dt, n0, n1, n2);
        else efield_update_lane<NC, 4>(lane, g.links, g.efield, g.dt, n0, n1, n2);
        return;
    }
    const int V = n0 * n1 * n2;
    int m, blk;
    Site p;
    if (!lane_coords<MB>(a, blockIdx.x - g.blocks, gridDim.x - g.blocks, n0, n1, V, m, p, blk)) return;
    hop_site<NC, T, T, MB, EPI_AXPY>(a, n0, n1, n2, p, blk * V, 0, m);
}

// ---------------------------------------------------------------------------------------------
// deterministic reductions: fixed grid, per-block partials, one fixed-order final pass
// ---------------------------------------------------------------------------------------------
constexpr int RED_BLOCKS = 512;

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
__device__ __forceinline__ double wave_max(double v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    return v;
}

// block reduction of NV values (sum or max per value; those of `mask`) in a workgroup of NT threads; result
// valid in thread 0
template <int NV, int NT = TPB>
__device__ __forceinline__ void block_reduce(double *v, const int *is_max, unsigned mask = (1u << NV) - 1)
{
    __shared__ double sh[NT / 64][NV];
    const int w = threadIdx.x / 64, l = threadIdx.x % 64;
#pragma unroll
    for (int k = 0; k < NV; ++k)
        if (mask >> k & 1) v[k] = is_max[k] ? wave_max(v[k]) : wave_sum(v[k]);
    if (l == 0)
#pragma unroll
        for (int k = 0; k < NV; ++k) sh[w][k] = v[k];
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            double r = sh[0][k];
            for (int j = 1; j < NT / 64; ++j) r = is_max[k] ? fmax(r, sh[j][k]) : r + sh[j][k];
            v[k] = r;
        }
    }
}

// components X^a = 2 tr(t^a X) of a Hermitian traceless matrix, via ReTr(i t^a (-i X))
template <int NC> __device__ __forceinline__ void alg_components(const Mat<NC> &X, double *out)
{
    Mat<NC> mx;
#pragma unroll
    for (int k = 0; k < NC * NC; ++k) mx.e[k] = {X.e[k].i, -X.e[k].r};
    retr_it<NC>(mx, out);
#pragma unroll
    for (int a = 0; a < NC * NC - 1; ++a) out[a] *= 2.0;
}

// The site-local observables in one pass, four lanes per site (lane mu < 3 has direction mu, the plane
// (mu + 1, mu + 2) and the link (s, mu); lane 3 idles):
//   (1/2) sum E^2 and (1/2) sum_planes 4 ReTr(1 - U_plaq)     (BulkObservables.cpp:29-31,84-86)
//   max |G^a| and sum G^2 of G(x) = sum_mu E_mu(x) - U_mu(x-mu)^+ E_mu(x-mu) U_mu(x-mu)
//                                                             (GaussLawViolation.cpp:13-61)
//   max and sum of the squares of ||U U^+ - 1||               (UnitarityViolation.cpp:13-51)
// `what` (a sum of OBS_ENERGY, OBS_GAUSS, OBS_UNITARITY) leaves out the others; each quantity is the same sums
// either way.  g (optional): G^a(x) stored as [site][a].  24^3 SU(3): 9.7 us for all where three kernels and
// their finishing passes took 37 us.  Up to LOC_BLOCKS workgroups of 64 sites: see there.
enum { LOC_EEL = 0, LOC_EMAG, LOC_GMAX, LOC_GSUM, LOC_UMAX, LOC_USUM, LOC_COUNT };
// the LOC_* values (bits) that the observables `what` have
constexpr unsigned loc_mask(int what)
{
    return (what & OBS_ENERGY ? 3u << LOC_EEL : 0) | (what & OBS_GAUSS ? 3u << LOC_GMAX : 0) |
           (what & OBS_UNITARITY ? 3u << LOC_UMAX : 0);
}
template <int NC, int WHAT, int NT>
__device__ __forceinline__ void obs_local(int wg, int wgs, const double *__restrict__ links,
                                          const double *__restrict__ e, double *partial, double *__restrict__ g, int n0,
                                          int n1, int n2)
{
    const int V = n0 * n1 * n2;
    constexpr int NG = NC * NC - 1;
    double v[LOC_COUNT] = {0, 0, 0, 0, 0, 0};
    const int mu = threadIdx.x % 4;
    const bool dir = mu < 3;
    const int stride = wgs * (TPB / 4);
    // the four lanes of a site share the loop condition; threads beyond TPB only join the reduction
    for (int s = threadIdx.x < TPB ? wg * (TPB / 4) + (int)threadIdx.x / 4 : V; s < V; s += stride) {
        double comp[NG];
#pragma unroll
        for (int a = 0; a < NG; ++a) comp[a] = 0;
        if (dir) {
            if constexpr (WHAT & OBS_GAUSS) {
                const int sm = nbr(s, mu, -1, n0, n1, n2);
                const Mat<NC> e0 = alg_to_mat<NC>(e + (size_t)NG * (mu + 3 * (size_t)s));
                const Mat<NC> e1 = alg_to_mat<NC>(e + (size_t)NG * (mu + 3 * (size_t)sm));
                const Mat<NC> ub = get_link<NC>(links, sm, mu);
                Mat<NC> t = mmul<NC>(mmul<NC>(mdag<NC>(ub), e1), ub);
#pragma unroll
                for (int k = 0; k < NC * NC; ++k) t.e[k] = {e0.e[k].r - t.e[k].r, e0.e[k].i - t.e[k].i};
                alg_components<NC>(t, comp);
            }
            if constexpr (WHAT & OBS_ENERGY) {
                for (int a = 0; a < NG; ++a) {
                    const double q = e[(size_t)NG * (mu + 3 * (size_t)s) + a];
                    v[LOC_EEL] += q * q;
                }
                const int a = (mu + 1) % 3, b = (mu + 2) % 3;
                Mat<NC> p = mmul<NC>(get_link<NC>(links, s, a), get_link<NC>(links, nbr(s, a, 1, n0, n1, n2), b));
                p = mmul<NC>(p, mdag<NC>(get_link<NC>(links, nbr(s, b, 1, n0, n1, n2), a)));
                p = mmul<NC>(p, mdag<NC>(get_link<NC>(links, s, b)));
                double tr = 0;
#pragma unroll
                for (int i = 0; i < NC; ++i) tr += 1.0 - p.e[i * NC + i].r;
                v[LOC_EMAG] += 4.0 * tr;
            }
            if constexpr (WHAT & OBS_UNITARITY) {
                double nrm;
                if constexpr (NC == 2) {  // UnitarityNorm (SU2/GroupOperations.cpp:172-184)
                    const double *u = links + link_at<2>(s, mu);
                    const double c3 = u[3] * u[3] + u[0] * u[0] + u[1] * u[1] + u[2] * u[2];
                    nrm = fabs(c3 - 1.0);
                } else {
                    const Mat<3> u = get_link<3>(links, s, mu);
                    const Mat<3> q = mmul<3>(u, mdag<3>(u));
                    nrm = 0;
                    for (int i = 0; i < 3; ++i)
                        for (int k = 0; k < 3; ++k) {
                            const double re = q.e[i * 3 + k].r - (i == k ? 1.0 : 0.0), im = q.e[i * 3 + k].i;
                            nrm += re * re + im * im;
                        }
                    nrm = sqrt(nrm);
                }
                v[LOC_UMAX] = fmax(v[LOC_UMAX], nrm);
                v[LOC_USUM] += nrm * nrm;
            }
        }
        if constexpr (WHAT & OBS_GAUSS)
#pragma unroll
            for (int a = 0; a < NG; ++a) {
                comp[a] += __shfl_xor(comp[a], 1, 64);
                comp[a] += __shfl_xor(comp[a], 2, 64);
                if (a % 4 == mu) {  // every lane of the site holds G^a: each keeps its share
                    if (g) g[(size_t)NG * s + a] = comp[a];
                    const double q = fabs(comp[a]);
                    v[LOC_GMAX] = fmax(v[LOC_GMAX], q);
                    v[LOC_GSUM] += q * q;
                }
            }
    }
    v[LOC_EEL] *= 0.5;
    v[LOC_EMAG] *= 0.5;
    const int ism[LOC_COUNT] = {0, 0, 1, 0, 1, 0};
    block_reduce<LOC_COUNT, NT>(v, ism, loc_mask(WHAT));
    if (threadIdx.x == 0)
#pragma unroll
        for (int k = 0; k < LOC_COUNT; ++k)
            if (loc_mask(WHAT) >> k & 1) partial[(size_t)wg * LOC_COUNT + k] = v[k];
}
template <int NC, int WHAT>
__global__ __launch_bounds__(TPB) void k_obs_local(const double *__restrict__ links, const double *__restrict__ e,
                                                   double *partial, double *__restrict__ g, int n0, int n1, int n2)
{
    obs_local<NC, WHAT, TPB>((int)blockIdx.x, (int)gridDim.x, links, e, partial, g, n0, n1, n2);
}

// the partial results of the local observables of WHAT (nl workgroups') and of E.B (ne, with OBS_EDOTB), summed in
// a fixed order: out[0 .. LOC_COUNT) and out[LOC_COUNT]; `derived` (optional, with all of them): the
// quantities of ovl_system_observables from them
template <int WHAT>
__global__ __launch_bounds__(TPB) void k_obs_finish(const double *__restrict__ local, int nl,
                                                    const double *__restrict__ edotb, int ne, double *out,
                                                    double *derived, double n_adj_v, double three_v)
{
    constexpr unsigned MASK = loc_mask(WHAT) | (WHAT & OBS_EDOTB ? 1u << LOC_COUNT : 0);
    const int ism[LOC_COUNT + 1] = {0, 0, 1, 0, 1, 0, 0};
    double v[LOC_COUNT + 1] = {0, 0, 0, 0, 0, 0, 0};
    if constexpr (loc_mask(WHAT) != 0)
        for (int b = threadIdx.x; b < nl; b += TPB)
#pragma unroll
            for (int k = 0; k < LOC_COUNT; ++k)
                if (MASK >> k & 1) {
                    const double p = local[(size_t)b * LOC_COUNT + k];
                    v[k] = ism[k] ? fmax(v[k], p) : v[k] + p;
                }
    if constexpr ((WHAT & OBS_EDOTB) != 0)
        for (int b = threadIdx.x; b < ne; b += TPB) v[LOC_COUNT] += edotb[b];
    block_reduce<LOC_COUNT + 1>(v, ism, MASK);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k <= LOC_COUNT; ++k)
            if (MASK >> k & 1) out[k] = v[k];
        if (derived) {
            derived[OVL_OBS_E_EL] = v[RAW_EEL];
            derived[OVL_OBS_E_MAG] = v[RAW_EMAG];
            derived[OVL_OBS_GAUSS_MAX] = v[RAW_GMAX];
            derived[OVL_OBS_GAUSS_RMS] = sqrt(v[RAW_GSUM] / n_adj_v);
            derived[OVL_OBS_UNIT_MAX] = v[RAW_UMAX];
            derived[OVL_OBS_UNIT_RMS] = sqrt(v[RAW_USUM] / three_v);
            derived[OVL_OBS_NCS_DOT] = 0.125 * v[RAW_EDOTB] / (M_PI * M_PI);  // ChernSimonsDerivative.cpp:47
        }
    }
}

// one relaxation step of GaussLawRestoration::UpdateElectricFields (GaussRestore.cpp:74-112):
//   E_mu(x) -= gamma (G(x) - U_mu(x) G(x+mu) U_mu(x)^+)
// i.e. gradient descent on (1/2) sum_x G(x)^2 in E
template <int NC>
__global__ __launch_bounds__(TPB) void k_gauss_restore(const double *__restrict__ links, const double *__restrict__ g,
                                                       double *__restrict__ e, double gamma, int n0, int n1, int n2)
{
    const int V = n0 * n1 * n2;
    constexpr int NG = NC * NC - 1;
    const int i = blockIdx.x * TPB + threadIdx.x;
    if (i >= 3 * V) return;
    const int s = i / 3, mu = i - 3 * s;
    const int sp = nbr(s, mu, 1, n0, n1, n2);
    const Mat<NC> u = get_link<NC>(links, s, mu);
    const Mat<NC> t = mmul<NC>(mmul<NC>(u, alg_to_mat<NC>(g + (size_t)NG * sp)), mdag<NC>(u));
    double up[NG];
    alg_components<NC>(t, up);
#pragma unroll
    for (int a = 0; a < NG; ++a) e[(size_t)NG * (mu + 3 * s) + a] -= gamma * (g[(size_t)NG * s + a] - up[a]);
}

// improved sum_x E.B (ChernSimonsOperators.cpp:228-439): per site and direction mu, with (a, b) the plane
// across mu,
//   E = 7/12 E(0) - 1/12 U E(1) U^+ + 7/12 U(-1)^+ E(-1) U(-1) - 1/12 (..)^+ E(-2) (..)
//   B = 5/12 sum of the four plaquettes at the site - 1/24 sum of the eight 2 x 1 rectangles
// with every loop and E transported to the site; the sum is 4 sum_c ReTr(t^c E) ReTr(i t^c B) =
// 4 ReTr(i E' B) with E' the traceless Hermitian half of E.
//
// A lane holds one row of one quadrant's loops (a plaquette and two rectangles) or of E and walks it
// along their links, a row times a matrix per link; loops that share their first or last links are added
// before the shared ones (10 or 17 products per quadrant instead of 16 and 24).  A wavefront is one
// quadrant (or E) of 64 / Nc (site, mu) pairs, so its lanes run the same products; the five wavefronts
// of a workgroup meet in LDS.  FP64 issue bounds it on large lattices (62 products of about 80
// instructions per Nc lanes), the chain of 17 on small ones.  One lane per site making 675 matrix
// products took 328 us on 24^3 SU(3) and 94 us on 8^3 SU(2); this form 55 and 5 us.
template <int NC, bool DAG>
__device__ __forceinline__ void row_step(cd *v, const double *__restrict__ links, int s, int mu)
{
    const Mat<NC> m = get_link<NC>(links, s, mu);
    cd r[NC];
#pragma unroll
    for (int j = 0; j < NC; ++j) {
        cd t = {0, 0};
#pragma unroll
        for (int k = 0; k < NC; ++k)
            t = cadd(t, DAG ? cmul(v[k], cd{m.e[j * NC + k].r, -m.e[j * NC + k].i}) : cmul(v[k], m.e[k * NC + j]));
        r[j] = t;
    }
#pragma unroll
    for (int j = 0; j < NC; ++j) v[j] = r[j];
}

// v <- v E of the site's field e[0 .. Nc^2 - 1)
template <int NC> __device__ __forceinline__ void row_field(cd *v, const double *__restrict__ e)
{
    const Mat<NC> m = alg_to_mat<NC>(e);
    cd r[NC];
#pragma unroll
    for (int j = 0; j < NC; ++j) {
        cd t = {0, 0};
#pragma unroll
        for (int k = 0; k < NC; ++k) t = cadd(t, cmul(v[k], m.e[k * NC + j]));
        r[j] = t;
    }
#pragma unroll
    for (int j = 0; j < NC; ++j) v[j] = r[j];
}

template <int NC> struct Row {
    cd e[NC];
};
template <int NC> __device__ __forceinline__ Row<NC> row_add(const Row<NC> &x, double wx, const Row<NC> &y, double wy)
{
    Row<NC> r;
#pragma unroll
    for (int k = 0; k < NC; ++k) r.e[k] = {wx * x.e[k].r + wy * y.e[k].r, wx * x.e[k].i + wy * y.e[k].i};
    return r;
}

__device__ __forceinline__ int wrap(int c, int n) { return c < 0 ? c + n : (c >= n ? c - n : c); }  // |offset| <= 2 < n

constexpr int EB_TPB = 5 * 64;  // four quadrants and E
// two waves per SIMD for SU(3): three or four spill (24^3: 65, 119 and 136 us)
template <int NC> constexpr int EB_WPE = NC == 3 ? 2 : 4;
template <int NC>
__device__ __forceinline__ void edotb(int wg, int wgs, const double *__restrict__ links, const double *__restrict__ e,
                                      double *partial, int n0, int n1, int n2)
{
    constexpr int NG = NC * NC - 1, PAIRS = 64 / NC;
    constexpr double W4 = 5.0 / 12.0, W6 = -1.0 / 24.0;
    __shared__ cd er[PAIRS][NC][NC];
    const int V = n0 * n1 * n2;
    const int part = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
    const bool used = lane < PAIRS * NC;
    const int pair = used ? lane / NC : PAIRS - 1, row = used ? lane % NC : 0;
    double acc[1] = {0.0};
    const int npairs = 3 * V;
    for (int base = wg * PAIRS; base < npairs; base += wgs * PAIRS) {
        const int gi = base + pair;
        const int gc = gi < npairs ? gi : npairs - 1;  // spare lanes repeat the last pair's work
        const bool ok = used && gi < npairs;
        const int s = gc / 3, mu = gc - 3 * s;
        const int z = s / (n0 * n1), rem = s - z * n0 * n1, y = rem / n0, x = rem - y * n0;
        const int a = mu == 2 ? 0 : mu + 1, b = mu == 0 ? 2 : mu - 1;
        auto pick = [](int d, int v0, int v1, int v2) { return d == 0 ? v0 : (d == 1 ? v1 : v2); };
        const int ca = pick(a, x, y, z), na = pick(a, n0, n1, n2), sa = pick(a, 1, n0, n0 * n1);
        const int cb = pick(b, x, y, z), nb = pick(b, n0, n1, n2), sb = pick(b, 1, n0, n0 * n1);
        const int origin = s - ca * sa - cb * sb;
        auto at = [&](int i, int j) { return origin + wrap(ca + i, na) * sa + wrap(cb + j, nb) * sb; };
        Row<NC> v;
#pragma unroll
        for (int k = 0; k < NC; ++k) v.e[k] = {k == row ? 1.0 : 0.0, 0.0};
        // v <- v U, v U^+ for the links A (direction a) and B at the offsets (i, j)
        auto A = [&](Row<NC> &r, int i, int j) { row_step<NC, false>(r.e, links, at(i, j), a); };
        auto Ad = [&](Row<NC> &r, int i, int j) { row_step<NC, true>(r.e, links, at(i, j), a); };
        auto B = [&](Row<NC> &r, int i, int j) { row_step<NC, false>(r.e, links, at(i, j), b); };
        auto Bd = [&](Row<NC> &r, int i, int j) { row_step<NC, true>(r.e, links, at(i, j), b); };
        if (part == 0) {  // quadrant (+a, +b)
            A(v, 0, 0);
            Row<NC> t = v, q = v;
            B(t, 1, 0);
            A(q, 1, 0); B(q, 2, 0); Ad(q, 1, 1);
            q = row_add<NC>(t, W4, q, W6);
            Ad(q, 0, 1);
            B(t, 1, 1); Ad(t, 0, 2); Bd(t, 0, 1);
            v = row_add<NC>(q, 1.0, t, W6);
            Bd(v, 0, 0);
        } else if (part == 1) {  // quadrant (-a, +b), transported along a
            Ad(v, -1, 0);
            Row<NC> q = v;
            A(v, -1, 0); B(v, 0, 0);
            Row<NC> t = v;
            Ad(v, -1, 1);
            B(t, 0, 1); Ad(t, -1, 2); Bd(t, -1, 1);
            v = row_add<NC>(v, W4, t, W6);
            Bd(v, -1, 0);
            Ad(q, -2, 0); A(q, -2, 0); A(q, -1, 0); B(q, 0, 0); Ad(q, -1, 1); Ad(q, -2, 1); Bd(q, -2, 0); A(q, -2, 0);
            v = row_add<NC>(v, 1.0, q, W6);
            A(v, -1, 0);
        } else if (part == 2) {  // quadrant (-a, -b)
            Ad(v, -1, 0);
            Row<NC> t = v, q = v;
            Bd(t, -1, -1);
            Ad(q, -2, 0); Bd(q, -2, -1); A(q, -2, -1);
            q = row_add<NC>(t, W4, q, W6);
            A(q, -1, -1);
            Bd(t, -1, -2); A(t, -1, -2); B(t, 0, -2);
            v = row_add<NC>(q, 1.0, t, W6);
            B(v, 0, -1);
        } else if (part == 3) {  // quadrant (+a, -b), transported along b
            Bd(v, 0, -1);
            Row<NC> q = v;
            A(v, 0, -1);
            Row<NC> t = v;
            B(v, 1, -1);
            A(t, 1, -1); B(t, 2, -1); Ad(t, 1, 0);
            v = row_add<NC>(v, W4, t, W6);
            Ad(v, 0, 0); Bd(v, 0, -1);
            Bd(q, 0, -2); A(q, 0, -2); B(q, 1, -2); B(q, 1, -1); Ad(q, 0, 0); Bd(q, 0, -1); Bd(q, 0, -2); B(q, 0, -2);
            v = row_add<NC>(v, 1.0, q, W6);
            B(v, 0, -1);
        } else {
            const int cm = pick(mu, x, y, z), nm = pick(mu, n0, n1, n2), sm = pick(mu, 1, n0, n0 * n1);
            const int line = s - cm * sm;
            const int sp = line + wrap(cm + 1, nm) * sm, s1 = line + wrap(cm - 1, nm) * sm, s2 = line + wrap(cm - 2, nm) * sm;
            auto E = [&](Row<NC> &r, int site) { row_field<NC>(r.e, e + (size_t)NG * (mu + 3 * (size_t)site)); };
            Row<NC> t = v, q = v;
            E(v, s);
            row_step<NC, false>(t.e, links, s, mu);
            E(t, sp);
            row_step<NC, true>(t.e, links, s, mu);
            v = row_add<NC>(v, 7.0 / 12.0, t, -1.0 / 12.0);
            row_step<NC, true>(q.e, links, s1, mu);
            t = q;
            E(q, s1);
            row_step<NC, true>(t.e, links, s2, mu);
            E(t, s2);
            row_step<NC, false>(t.e, links, s2, mu);
            q = row_add<NC>(q, 7.0 / 12.0, t, -1.0 / 12.0);
            row_step<NC, false>(q.e, links, s1, mu);
            v = row_add<NC>(v, 1.0, q, 1.0);
            if (used)
#pragma unroll
                for (int k = 0; k < NC; ++k) er[pair][row][k] = v.e[k];
        }
        __syncthreads();
        if (ok && part < 4) {
            double tr = 0, im = 0;
            for (int k = 0; k < NC; ++k) tr += er[pair][k][k].r;
#pragma unroll
            for (int k = 0; k < NC; ++k) {  // Im of (B E')_{row,row}
                const cd p = er[pair][k][row], q = er[pair][row][k];
                const cd h = {0.25 * (p.r + q.r) - (k == row ? 0.5 * tr / NC : 0.0), 0.25 * (p.i - q.i)};
                im += cmul(v.e[k], h).i;
            }
            acc[0] -= 4.0 * im;
        }
        __syncthreads();
    }
    const int ism[1] = {0};
    block_reduce<1, EB_TPB>(acc, ism);
    if (threadIdx.x == 0) partial[wg] = acc[0];
}
template <int NC>
__global__ __launch_bounds__(EB_TPB) __attribute__((amdgpu_waves_per_eu(EB_WPE<NC>))) void k_edotb(
    const double *__restrict__ links, const double *__restrict__ e, double *partial, int n0, int n1, int n2)
{
    edotb<NC>((int)blockIdx.x, (int)gridDim.x, links, e, partial, n0, n1, n2);
}

// The local observables (the first nb workgroups, their fifth wavefront idle, take the nl shares of k_obs_local in
// turn, so that the sums are its sums) and E.B in one launch: small lattices are bound by the launches.  All
// seven observables queued, in four launches and in two with k_obs_finish: 14.0 and 8.2 us on 8^3 SU(2), 19.8 and
// 11.4 us on 8^3 SU(3), 67.3 and 64.5 us on 24^3 SU(3).  More than OBS_BLOCKS workgroups only displace those of E.B
// (a workgroup for each of up to 1020 shares: SU(2) 48^3 93 -> 102 us, SU(3) 32^3 134 -> 140 us).
constexpr int OBS_BLOCKS = 256;
template <int NC>
__global__ __launch_bounds__(EB_TPB) __attribute__((amdgpu_waves_per_eu(EB_WPE<NC>))) void k_observables(
    const double *__restrict__ links, const double *__restrict__ e, double *local, int nl, int nb, double *eb,
    double *__restrict__ g, int n0, int n1, int n2)
{
    const int wg = (int)blockIdx.x;
    if (wg < nb)
        for (int w = wg; w < nl; w += nb) {
            obs_local<NC, OBS_LOCAL, EB_TPB>(w, nl, links, e, local, g, n0, n1, n2);
            __syncthreads();  // the reduction's LDS is free again
        }
    else edotb<NC>(wg - nb, (int)gridDim.x - nb, links, e, eb, n0, n1, n2);
}

// per-mode inner products: partial[chunk][mode] then a fixed-order sum over chunks
constexpr int DOT_CHUNKS = 128;

template <int NC, int MB>
__global__ __launch_bounds__(TPB) void k_mode_dot(const double2 *__restrict__ a, const double2 *__restrict__ b,
                                                  double2 *__restrict__ partial, int V, int nblk)
{
    // grid: (DOT_CHUNKS, nblk); each thread: one mode (m) and a strided subset of (site, comp)
    constexpr int NCOMP = 4 * NC;
    constexpr int LPM = TPB / MB;  // lanes per mode inside the block
    const int m = threadIdx.x % MB, lane = threadIdx.x / MB;
    const int blk = blockIdx.y;
    const long nel = (long)V * NCOMP;
    double sr = 0, si = 0;
    for (long q = (long)blockIdx.x * LPM + lane; q < nel; q += (long)DOT_CHUNKS * LPM) {
        const size_t idx = ((size_t)blk * nel + q) * MB + m;
        const double2 x = a[idx], y = b[idx];
        sr += x.x * y.x + x.y * y.y;
        si += x.x * y.y - x.y * y.x;
    }
    __shared__ double2 sh[TPB];
    sh[threadIdx.x] = make_double2(sr, si);
    __syncthreads();
    if (lane == 0) {
        double rr = 0, ii = 0;
        for (int l = 0; l < LPM; ++l) { rr += sh[l * MB + m].x; ii += sh[l * MB + m].y; }
        partial[((size_t)blockIdx.x) * nblk * MB + (size_t)blk * MB + m] = make_double2(rr, ii);
    }
}

// sum over the chunks in their order, one wavefront per mode: the lanes fetch the partial results together
// (a lane that walked them itself waited for 128 loads, 10 us), two lanes add the real and imaginary parts.
// The order is part of the results: the FP16 scales of the mixed sign are the norms' next power of two,
// and norms of one sit on the edge of it.
__global__ __launch_bounds__(64) void k_mode_dot_finish(const double2 *__restrict__ partial, double2 *__restrict__ out,
                                                        int nmodes_pad)
{
    __shared__ double sh[2][DOT_CHUNKS];
    const int i = blockIdx.x;
    for (int c = threadIdx.x; c < DOT_CHUNKS; c += 64) {
        const double2 p = partial[(size_t)c * nmodes_pad + i];
        sh[0][c] = p.x;
        sh[1][c] = p.y;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        double r = 0;
#pragma unroll 16
        for (int c = 0; c < DOT_CHUNKS; ++c) r += sh[threadIdx.x][c];
        reinterpret_cast<double *>(out)[2 * i + threadIdx.x] = r;
    }
}

// currents (OverlapCurrents.cpp:137-228), per (site, mode) bilinears summed over the modes of a block.
// gam: [kind][mu][a][b] complex, kind 0 = g0 g^mu, 1 = g0 g^mu g5, 2 = -(i/2) g0 g^mu g0,
// 3 = -(i/2) g0 g^mu g5 g0 (built on the host from the Dirac matrices as the reference does)
template <int NC, int MB>
__global__ __launch_bounds__(TPB) void k_currents(const double2 *__restrict__ psi, const double2 *__restrict__ hpsi,
                                                  const double2 *__restrict__ gam, double *__restrict__ partial, int V,
                                                  int nblk, int first_mode)
{
    constexpr int SPB = TPB / MB;
    const int m = threadIdx.x % MB, sl = threadIdx.x / MB;
    const long site_g = (long)blockIdx.x * SPB + sl;  // over nblk * V
    const bool ok = site_g < (long)nblk * V;
    const int blk = ok ? (int)(site_g / V) : 0, s = ok ? (int)(site_g % V) : 0;
    double j[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (ok) {
        const double w = (((blk * MB + m) + first_mode) % 2 == 0) ? 1.0 : -1.0;
        for (int c = 0; c < NC; ++c) {
            double2 p[4], h[4];
            for (int sp = 0; sp < 4; ++sp) {
                const size_t idx = ((size_t)(blk * V + s) * 4 * NC + sp * NC + c) * MB + m;
                p[sp] = psi[idx];
                h[sp] = hpsi[idx];
            }
            for (int mu = 0; mu < 4; ++mu)
                for (int a = 0; a < 4; ++a)
                    for (int b = 0; b < 4; ++b) {
                        // conj(p_a) p_b and conj(p_a) h_b
                        const double ppr = p[a].x * p[b].x + p[a].y * p[b].y, ppi = p[a].x * p[b].y - p[a].y * p[b].x;
                        const double phr = p[a].x * h[b].x + p[a].y * h[b].y, phi = p[a].x * h[b].y - p[a].y * h[b].x;
                        const double2 gv = gam[((0 * 4 + mu) * 4 + a) * 4 + b], ga = gam[((1 * 4 + mu) * 4 + a) * 4 + b];
                        const double2 gv2 = gam[((2 * 4 + mu) * 4 + a) * 4 + b], ga2 = gam[((3 * 4 + mu) * 4 + a) * 4 + b];
                        j[mu] += w * (gv.x * ppr - gv.y * ppi + gv2.x * phr - gv2.y * phi);
                        j[4 + mu] += w * (ga.x * ppr - ga.y * ppi + ga2.x * phr - ga2.y * phi);
                    }
        }
    }
    // sum over the MB modes of this site (lanes of one site are contiguous), fixed order
    __shared__ double sh[TPB][8];
    for (int k = 0; k < 8; ++k) sh[threadIdx.x][k] = j[k];
    __syncthreads();
    if (m == 0 && ok) {
        double t[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        for (int q = 0; q < MB; ++q)
            for (int k = 0; k < 8; ++k) t[k] += sh[sl * MB + q][k];
        for (int k = 0; k < 8; ++k) partial[((size_t)blk * V + s) * 8 + k] = t[k];
    }
}

__global__ __launch_bounds__(TPB) void k_currents_finish(const double *__restrict__ partial, double *jv, double *ja,
                                                         int V, int nblk, double pre)
{
    const int s = blockIdx.x * TPB + threadIdx.x;
    if (s >= V) return;
    double t[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int b = 0; b < nblk; ++b)
        for (int k = 0; k < 8; ++k) t[k] += partial[((size_t)b * V + s) * 8 + k];
    for (int k = 0; k < 4; ++k) { jv[4 * s + k] = pre * t[k]; ja[4 * s + k] = pre * t[4 + k]; }
}

// multi-shift CG vector update (OverlapU.cpp:164-177), with chi += bz_k beta_k p_k accumulated
// directly:  for each shift k: chi += cw_k p_k ; p_k = a_k p_k + g_k r   (per-mode coefficients)
__global__ __launch_bounds__(TPB) void k_mscg_update2(int nshift, double2 *__restrict__ ps, double2 *__restrict__ chi,
                                                      const double2 *__restrict__ r, const double *__restrict__ coef,
                                                      const int *__restrict__ active, long per_blk, int nblk, int mb)
{
    // element i = (blk, q, m) with per_blk = V*NCOMP elements per mode block
    const long i = (long)blockIdx.x * TPB + threadIdx.x;
    const long nel = per_blk * nblk * mb;
    if (i >= nel) return;
    const int m = (int)(i % mb);
    const int blk = (int)(i / ((long)per_blk * mb));
    const int mode = blk * mb + m;
    if (!active[mode]) return;
    const double *c = coef + (size_t)mode * 3 * nshift;
    const double2 rv = r[i];
    double2 x = chi[i];
    for (int k = 0; k < nshift; ++k) {
        double2 p = ps[(size_t)k * nel + i];
        x.x += c[3 * k] * p.x;
        x.y += c[3 * k] * p.y;
        p.x = c[3 * k + 1] * p.x + c[3 * k + 2] * rv.x;
        p.y = c[3 * k + 1] * p.y + c[3 * k + 2] * rv.y;
        ps[(size_t)k * nel + i] = p;
    }
    chi[i] = x;
}

inline unsigned nblocks(long n) { return (unsigned)((n + TPB - 1) / TPB); }

// occupancy variant 5: the wpe = 1 kernel with an LDS reservation it does not use, larger than
// half of a CU's 160 KiB, so that one workgroup (one wave per SIMD) runs per CU: fewer sites in
// flight per XCD, so the neighbour planes of the stencil input fit in L2 beside them
constexpr unsigned LDS_ONE_WG = 96 * 1024;
hipError_t reserve_lds(const void *kernel)
{
    static std::mutex mu;
    static std::unordered_set<const void *> done;
    std::lock_guard<std::mutex> lock(mu);
    if (!done.insert(kernel).second) return hipSuccess;
    return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LDS_ONE_WG);
}

template <int NC, typename TI, typename TO, int MB, int EPI>
void hop_wpe_epi(const HopArgs &b, unsigned nb, int wpe, const Geom &g, hipStream_t st)
{
    switch (wpe) {
    case 2: k_hop<NC, TI, TO, MB, 2, EPI><<<nb, TPB, 0, st>>>(b, g.n0, g.n1, g.n2); break;
    case 3: k_hop<NC, TI, TO, MB, 3, EPI><<<nb, TPB, 0, st>>>(b, g.n0, g.n1, g.n2); break;
    case 4: k_hop<NC, TI, TO, MB, 4, EPI><<<nb, TPB, 0, st>>>(b, g.n0, g.n1, g.n2); break;
    case 5:
        (void)reserve_lds(reinterpret_cast<const void *>(k_hop<NC, TI, TO, MB, 1, EPI>));
        k_hop<NC, TI, TO, MB, 1, EPI><<<nb, TPB, LDS_ONE_WG, st>>>(b, g.n0, g.n1, g.n2);
        break;
    default: k_hop<NC, TI, TO, MB, 1, EPI><<<nb, TPB, 0, st>>>(b, g.n0, g.n1, g.n2); break;
    }
}

// the kind of launch (EPI_*) that a set of operands and factors is
int epi_kind(const HopArgs &b)
{
    const bool none = !b.x && !b.b1 && !b.b2 && !b.out2;
    if (none && !b.tgt && b.sh_i == 0.0) return EPI_PURE;
    if (none && b.tgt && b.sh_r == 0.0 && b.st_r == 1.0 && b.st_i == 0.0) return EPI_AXPY;
    if (b.x && b.b1 && b.b2 && !b.tgt && !b.out2 && !b.x_gamma0 && b.sh_i == 0.0 && b.sx_i == 0.0 && b.s1_i == 0.0 &&
        b.s2_i == 0.0)
        return EPI_CLENSHAW;
    return EPI_ANY;
}

template <int NC, typename TI, typename TO, int MB>
void hop_wpe(const HopArgs &b, unsigned nb, int wpe, const Geom &g, hipStream_t st)
{
    if constexpr (std::is_same<TI, TO>::value) {
        switch (epi_kind(b)) {
        case EPI_PURE: return hop_wpe_epi<NC, TI, TO, MB, EPI_PURE>(b, nb, wpe, g, st);
        case EPI_CLENSHAW: return hop_wpe_epi<NC, TI, TO, MB, EPI_CLENSHAW>(b, nb, wpe, g, st);
        case EPI_AXPY:
            // the leapfrog's fields are FP64 or FP32
            if constexpr (sizeof(TI) == 8 || sizeof(TI) == 4) return hop_wpe_epi<NC, TI, TO, MB, EPI_AXPY>(b, nb, wpe, g, st);
            break;
        default: break;
        }
    }
    hop_wpe_epi<NC, TI, TO, MB, EPI_ANY>(b, nb, wpe, g, st);
}

template <int NC, typename TI, typename TO, int MB, int EPI>
void hop_ens_wpe_epi(const HopArgs &b, int wpe, hipStream_t st)
{
    unsigned nb = (unsigned)b.ens_grid;
    if (b.ens_qctr) {
        // persistent grid: the resident workgroups of the variant on every CU, a multiple of the XCDs
        int dev = 0, cus = 0, per_cu = 0;
        (void)hipGetDevice(&dev);
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = 256;
        const void *f = wpe == 2 ? reinterpret_cast<const void *>(k_hop_ens<NC, TI, TO, MB, 2, EPI>)
                      : wpe == 3 ? reinterpret_cast<const void *>(k_hop_ens<NC, TI, TO, MB, 3, EPI>)
                      : wpe == 4 ? reinterpret_cast<const void *>(k_hop_ens<NC, TI, TO, MB, 4, EPI>)
                                 : reinterpret_cast<const void *>(k_hop_ens<NC, TI, TO, MB, 1, EPI>);
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, f, TPB, wpe == 5 ? LDS_ONE_WG : 0) != hipSuccess ||
            per_cu < 1)
            per_cu = 1;
        nb = (unsigned)std::max(NUM_XCD, (cus * per_cu) / NUM_XCD * NUM_XCD);
    }
    switch (wpe) {
    case 2: k_hop_ens<NC, TI, TO, MB, 2, EPI><<<nb, TPB, 0, st>>>(b); break;
    case 3: k_hop_ens<NC, TI, TO, MB, 3, EPI><<<nb, TPB, 0, st>>>(b); break;
    case 4: k_hop_ens<NC, TI, TO, MB, 4, EPI><<<nb, TPB, 0, st>>>(b); break;
    case 5:
        (void)reserve_lds(reinterpret_cast<const void *>(k_hop_ens<NC, TI, TO, MB, 1, EPI>));
        k_hop_ens<NC, TI, TO, MB, 1, EPI><<<nb, TPB, LDS_ONE_WG, st>>>(b);
        break;
    default: k_hop_ens<NC, TI, TO, MB, 1, EPI><<<nb, TPB, 0, st>>>(b); break;
    }
}
template <int NC, typename TI, typename TO, int MB>
void hop_ens_wpe(const HopArgs &b, int wpe, hipStream_t st)
{
    if constexpr (std::is_same<TI, TO>::value) {
        switch (epi_kind(b)) {
        case EPI_PURE: return hop_ens_wpe_epi<NC, TI, TO, MB, EPI_PURE>(b, wpe, st);
        case EPI_CLENSHAW: return hop_ens_wpe_epi<NC, TI, TO, MB, EPI_CLENSHAW>(b, wpe, st);
        case EPI_AXPY:
            if constexpr (sizeof(TI) == 8 || sizeof(TI) == 4) return hop_ens_wpe_epi<NC, TI, TO, MB, EPI_AXPY>(b, wpe, st);
            break;
        default: break;
        }
    }
    hop_ens_wpe_epi<NC, TI, TO, MB, EPI_ANY>(b, wpe, st);
}

// the launch arguments of one lattice: lane coordinates and traversal; false when the lanes exceed 32 bits
bool lattice_args(const Geom &g, const HopArgs &a, HopArgs &b, unsigned &nb)
{
    const long total = (long)a.nblk * g.V * g.mb;
    if (total >= (1l << 31)) return false;
    nb = nblocks(total);
    b = a;
    b.dv_V = make_fastdiv((unsigned)g.V);
    b.dv_per = make_fastdiv((unsigned)((long)a.nblk * g.V / NUM_XCD));
    b.dv_v8 = make_fastdiv((unsigned)(g.V / NUM_XCD));
    b.dv_n01 = make_fastdiv((unsigned)(g.n0 * g.n1));
    b.dv_n0 = make_fastdiv((unsigned)g.n0);
    // The XCD traversals give each XCD an eighth of the workgroups: the grid is rounded up to whole eighths
    // (the last ones find no lanes).  A box of sites needs eight equal boxes.
    if (b.trav == TRAV_BOXES && (g.V % NUM_XCD != 0 || (!b.order && b.box.dv_x.d == 0))) b.trav = TRAV_MODES;
    if (b.trav != TRAV_LEX) nb = (nb + NUM_XCD - 1) / NUM_XCD * NUM_XCD;
    return true;
}

template <int NC, typename TI, typename TO>
hipError_t hop_mb(const Geom &g, const HopArgs &a, int wpe, hipStream_t st)
{
    if (a.ens_sys) {
        if (a.ens_grid <= 0) return hipErrorInvalidValue;
        switch (g.mb) {
        case 16: hop_ens_wpe<NC, TI, TO, 16>(a, wpe, st); break;
        case 32: hop_ens_wpe<NC, TI, TO, 32>(a, wpe, st); break;
        case 64: hop_ens_wpe<NC, TI, TO, 64>(a, wpe, st); break;
        default: return hipErrorInvalidValue;
        }
        return hipGetLastError();
    }
    HopArgs b;
    unsigned nb;
    if (!lattice_args(g, a, b, nb)) return hipErrorInvalidValue;
    switch (g.mb) {
    case 16: hop_wpe<NC, TI, TO, 16>(b, nb, wpe, g, st); break;
    case 32: hop_wpe<NC, TI, TO, 32>(b, nb, wpe, g, st); break;
    case 64: hop_wpe<NC, TI, TO, 64>(b, nb, wpe, g, st); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}
template <int NC, typename T>
hipError_t hop_gauge_mb(const Geom &g, const HopArgs &a, const GaugeHalf &h, hipStream_t st)
{
    HopArgs b;
    unsigned nb;
    if (!lattice_args(g, a, b, nb) || h.blocks % NUM_XCD != 0) return hipErrorInvalidValue;
    nb += (unsigned)h.blocks;
    switch (g.mb) {
    case 16: k_hop_gauge<NC, T, 16><<<nb, TPB, 0, st>>>(b, h, g.n0, g.n1, g.n2); break;
    case 32: k_hop_gauge<NC, T, 32><<<nb, TPB, 0, st>>>(b, h, g.n0, g.n1, g.n2); break;
    case 64: k_hop_gauge<NC, T, 64><<<nb, TPB, 0, st>>>(b, h, g.n0, g.n1, g.n2); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------
// QED eigenbasis: unit sources, z-momentum blocks and their checks
// ---------------------------------------------------------------------------------------------
// One batch of unit sources in a zeroed FP64 field: mode mm < cnt gets a 1 at source src = k0 + mm,
// i.e. colour 0, spin src % 4 at site src / 4 of the z = 0 plane when src < dz, else colour 1,
// spin src - dz at site 0.
template <int NC, int MB>
__global__ __launch_bounds__(TPB) void k_eig_sources(double2 *field, int V, long k0, int cnt, long dz)
{
    constexpr int NCOMP = 4 * NC;
    const int mm = blockIdx.x * TPB + threadIdx.x;
    if (mm >= cnt) return;
    const long src = k0 + mm;
    const int blk = mm / MB, m = mm - blk * MB;
    const long site = src < dz ? src / 4 : 0;
    const int comp = src < dz ? (int)(src % 4) * NC : (int)(src - dz) * NC + 1;
    field[(((size_t)blk * V + site) * NCOMP + comp) * MB + m] = make_double2(1.0, 0.0);
}

// A[j dz^2 + (k0 + mm) dz + row] = out[blk][j ncol + (xy NCOMP + sp NC) MB + m] for row = 4 xy + sp
// and the first nsb modes mm (blk = mm / MB, m = mm % MB) of a batch; `out` holds per mode block
// the n2 z-momentum planes of ncol = plane NCOMP MB entries each
template <int NC, int MB>
__global__ __launch_bounds__(TPB) void k_eig_gather(const double2 *__restrict__ out, double2 *__restrict__ A,
                                                    long plane, int n2, long k0, int nsb)
{
    constexpr int NCOMP = 4 * NC;
    const long dz = 4 * plane, ncol = plane * NCOMP * MB;
    const long total = (long)n2 * nsb * dz;
    for (long i = (long)blockIdx.x * TPB + threadIdx.x; i < total; i += (long)gridDim.x * TPB) {
        const long row = i % dz, r2 = i / dz;
        const int mm = (int)(r2 % nsb), j = (int)(r2 / nsb);
        const int blk = mm / MB, m = mm - blk * MB;
        const long xy = row / 4;
        const int sp = (int)(row % 4);
        A[(size_t)j * dz * dz + (size_t)(k0 + mm) * dz + row] =
            out[((size_t)blk * n2 + j) * ncol + (size_t)(xy * NCOMP + sp * NC) * MB + m];
    }
}

__device__ __forceinline__ double abs_or_inf(double2 x)
{
    const double a = sqrt(x.x * x.x + x.y * x.y);
    return (a <= 1.7976931348623157e308) ? a : __builtin_inf();  // NaN and inf count as inf
}

// largest |entry| of colours >= 1 among the first nvalid modes of an FP64 field (non-finite entries
// count as inf); one partial maximum per workgroup
template <int NC, int MB>
__global__ __launch_bounds__(TPB) void k_eig_leak(const double2 *__restrict__ f, int V, int nblk, int nvalid,
                                                  double *partial)
{
    constexpr int NCOMP = 4 * NC;
    double v[1] = {0.0};
    const long total = (long)nblk * V * NCOMP * MB;
    for (long i = (long)blockIdx.x * TPB + threadIdx.x; i < total; i += (long)gridDim.x * TPB) {
        const int m = (int)(i % MB);
        const long r = i / MB;
        const int comp = (int)(r % NCOMP), blk = (int)(r / NCOMP / V);
        if (comp % NC == 0 || blk * MB + m >= nvalid) continue;
        v[0] = fmax(v[0], abs_or_inf(f[i]));
    }
    const int ism[1] = {1};
    block_reduce<1>(v, ism);
    if (threadIdx.x == 0) partial[blockIdx.x] = v[0];
}

// Hermitian part of each of the n2 column-major dz x dz blocks, in place: the pair (row, col),
// (col, row) with row >= col is handled by one thread.  partial[2 b] = largest |A_rc - conj(A_cr)|,
// partial[2 b + 1] = 1 when an entry is not finite.
__global__ __launch_bounds__(TPB) void k_eig_hermitize(double2 *A, long dz, int n2, double *partial)
{
    double v[2] = {0.0, 0.0};
    const long total = (long)n2 * dz * dz;
    for (long i = (long)blockIdx.x * TPB + threadIdx.x; i < total; i += (long)gridDim.x * TPB) {
        const long row = i % dz, r2 = i / dz;
        const long col = r2 % dz, j = r2 / dz;
        if (row < col) continue;
        double2 *b = A + (size_t)j * dz * dz;
        const double2 x = b[(size_t)col * dz + row], y = b[(size_t)row * dz + col];
        const double2 d = make_double2(x.x - y.x, x.y + y.y);  // x - conj(y)
        const double a = abs_or_inf(d);
        if (a > 1.7976931348623157e308 || abs_or_inf(x) > 1.7976931348623157e308 ||
            abs_or_inf(y) > 1.7976931348623157e308)
            v[1] = 1.0;
        else
            v[0] = fmax(v[0], a);
        const double2 h = make_double2(0.5 * (x.x + y.x), 0.5 * (x.y - y.y));
        b[(size_t)col * dz + row] = h;
        b[(size_t)row * dz + col] = make_double2(h.x, -h.y);
    }
    const int ism[2] = {1, 1};
    block_reduce<2>(v, ism);
    if (threadIdx.x == 0) {
        partial[2 * blockIdx.x] = v[0];
        partial[2 * blockIdx.x + 1] = v[1];
    }
}

// Psi and PsiMid of the requested modes, every entry of both fields (modes >= nm are zero): mode
// e.blk >= 0 is f conj(tw[e.blk n2 + z]) A[e.blk dz^2 + e.idx dz + 4 xy + spin] on colour 0 (site =
// z plane + xy), mode e.blk = -1 is e.v at site e.idx, colour e.col; PsiMid = Psi rot
template <int NC, int MB>
__global__ __launch_bounds__(TPB) void k_eig_modes(const EigMode *__restrict__ modes, int nm,
                                                   const double2 *__restrict__ A, const double2 *__restrict__ tw,
                                                   double f, int V, long plane, int n2, int nblk,
                                                   double2 *__restrict__ psi, double2 *__restrict__ mid)
{
    constexpr int NCOMP = 4 * NC;
    const long dz = 4 * plane;
    const long total = (long)nblk * V * NCOMP * MB;
    for (long i = (long)blockIdx.x * TPB + threadIdx.x; i < total; i += (long)gridDim.x * TPB) {
        const int m = (int)(i % MB);
        const long r = i / MB;
        const int comp = (int)(r % NCOMP);
        const long r2 = r / NCOMP;
        const int site = (int)(r2 % V), blk = (int)(r2 / V);
        const int mode = blk * MB + m, sp = comp / NC, colour = comp - sp * NC;
        double vr = 0.0, vi = 0.0, rr = 0.0, ri = 0.0;
        if (mode < nm) {
            const EigMode &e = modes[mode];
            rr = e.rot_r;
            ri = e.rot_i;
            if (e.blk >= 0) {
                if (colour == 0) {
                    const long z = site / plane, xy = site - z * plane;
                    const double2 t = tw[(size_t)e.blk * n2 + z];
                    const double ph_r = f * t.x, ph_i = -(f * t.y);
                    const double2 a = A[(size_t)e.blk * dz * dz + (size_t)e.idx * dz + xy * 4 + sp];
                    vr = ph_r * a.x - ph_i * a.y;
                    vi = ph_r * a.y + ph_i * a.x;
                }
            } else if (site == e.idx && colour == e.col) {
                vr = e.v[2 * sp];
                vi = e.v[2 * sp + 1];
            }
        }
        psi[i] = make_double2(vr, vi);
        mid[i] = make_double2(vr * rr - vi * ri, vr * ri + vi * rr);
    }
}

// Inf or NaN: the 11 exponent bits all set (read from the high word of each double)
__device__ __forceinline__ unsigned nonfinite_bits(d2v v)
{
    const unsigned hx = (unsigned)((unsigned long long)__double_as_longlong(v.x) >> 32);
    const unsigned hy = (unsigned)((unsigned long long)__double_as_longlong(v.y) >> 32);
    return (unsigned)((hx & 0x7ff00000u) == 0x7ff00000u) | (unsigned)((hy & 0x7ff00000u) == 0x7ff00000u);
}

// 1 in partial[blockIdx.x] when one of the n doubles of a, or of b (when given), is not finite.  A
// streaming pass over one index range (b's 16-byte units follow a's): four 16-byte loads in flight
// per lane, read once (non-temporal).
__global__ __launch_bounds__(TPB) void k_nonfinite(const double *__restrict__ a, const double *__restrict__ b, long n,
                                                   double *partial)
{
    constexpr int U = 4;
    const long n2 = n / 2;                // whole double2 units per array
    const long total = b ? 2 * n2 : n2;   // units of a, then of b
    const d2v *__restrict__ a2 = reinterpret_cast<const d2v *>(a);
    const d2v *__restrict__ b2 = reinterpret_cast<const d2v *>(b);
    const long stride = (long)gridDim.x * TPB;
    long i = (long)blockIdx.x * TPB + threadIdx.x;
    unsigned bad = 0;
    for (; i + (U - 1) * stride < total; i += U * stride) {
        d2v v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const long j = i + u * stride;
            v[u] = __builtin_nontemporal_load(j < n2 ? a2 + j : b2 + (j - n2));
        }
#pragma unroll
        for (int u = 0; u < U; ++u) bad |= nonfinite_bits(v[u]);
    }
    for (; i < total; i += stride) bad |= nonfinite_bits(i < n2 ? a2[i] : b2[i - n2]);
    if ((n & 1) && blockIdx.x == 0 && threadIdx.x == 0) {  // an odd last double of each array
        bad |= nonfinite_bits(d2v{a[n - 1], 0.0});
        if (b) bad |= nonfinite_bits(d2v{b[n - 1], 0.0});
    }
    double v[1] = {bad ? 1.0 : 0.0};
    const int ism[1] = {1};
    block_reduce<1>(v, ism);
    if (threadIdx.x == 0) partial[blockIdx.x] = v[0];
}

}  // namespace

// ---------------------------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------------------------
hipError_t launch_hop(const Geom &g, int pin, int pout, const HopArgs &a, int wpe, hipStream_t st)
{
    if (g.nc == 2) {
        if (pin == P64 && pout == P64) return hop_mb<2, double, double>(g, a, wpe, st);
        if (pin == P32 && pout == P32) return hop_mb<2, float, float>(g, a, wpe, st);
        if (pin == P32 && pout == P64) return hop_mb<2, float, double>(g, a, wpe, st);
        if (pin == P16 && pout == P16) return hop_mb<2, _Float16, _Float16>(g, a, wpe, st);
        if (pin == P48 && pout == P48) return hop_mb<2, f48, f48>(g, a, wpe, st);
    } else if (g.nc == 3) {
        if (pin == P64 && pout == P64) return hop_mb<3, double, double>(g, a, wpe, st);
        if (pin == P32 && pout == P32) return hop_mb<3, float, float>(g, a, wpe, st);
        if (pin == P32 && pout == P64) return hop_mb<3, float, double>(g, a, wpe, st);
        if (pin == P16 && pout == P16) return hop_mb<3, _Float16, _Float16>(g, a, wpe, st);
        if (pin == P48 && pout == P48) return hop_mb<3, f48, f48>(g, a, wpe, st);
    }
    return hipErrorInvalidValue;
}

hipError_t launch_convert(const Geom &g, int nblk, const void *src, int psrc, void *dst, int pdst, hipStream_t st,
                          double scale)
{
    const long npairs = (long)nblk * g.V * (4 * g.nc / 2) * g.mb;
    const long nunits = npairs / 2;
    if (psrc == P64 && pdst == P32)
        k_d2f<<<nblocks(npairs), TPB, 0, st>>>((const double2 *)src, (float4 *)dst, npairs, g.mb, scale);
    else if (psrc == P32 && pdst == P64)
        k_f2d<<<nblocks(npairs), TPB, 0, st>>>((const float4 *)src, (double2 *)dst, npairs, g.mb, scale);
    else if (psrc == P64 && pdst == P16)
        k_d2h<<<nblocks(nunits), TPB, 0, st>>>((const double2 *)src, (h8v *)dst, nunits, g.mb, scale);
    else if (psrc == P16 && pdst == P32)
        k_h2f<<<nblocks(nunits), TPB, 0, st>>>((const h8v *)src, (float4 *)dst, nunits, g.mb, (float)scale);
    else if (psrc == P64 && pdst == P48)
        k_convert<double, f48><<<nblocks(nunits), TPB, 0, st>>>(src, dst, nunits, g.mb, scale);
    else if (psrc == P32 && pdst == P48)
        k_convert<float, f48><<<nblocks(nunits), TPB, 0, st>>>(src, dst, nunits, g.mb, scale);
    else if (psrc == P48 && pdst == P64)
        k_convert<f48, double><<<nblocks(nunits), TPB, 0, st>>>(src, dst, nunits, g.mb, scale);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launch_lincomb(const Geom &g, int nblk, int p, void *out, const void *a, double car, double cai,
                          const void *b, double cbr, double cbi, hipStream_t st)
{
    const long ncplx = (long)nblk * g.V * 4 * g.nc * g.mb;
    if (p == P64)
        k_lincomb<double><<<nblocks(ncplx), TPB, 0, st>>>((double *)out, (const double *)a, car, cai, (const double *)b,
                                                          cbr, cbi, ncplx);
    else
        k_lincomb<float><<<nblocks(ncplx), TPB, 0, st>>>((float *)out, (const float *)a, car, cai, (const float *)b, cbr,
                                                         cbi, ncplx);
    return hipGetLastError();
}

hipError_t launch_aos_to_soa(const Geom &g, const double *aos, int first, int count, void *field, hipStream_t st)
{
    const long tot = (long)count * g.V * 4 * g.nc;
    k_aos_to_soa<<<nblocks(tot), TPB, 0, st>>>((const double2 *)aos, (double2 *)field, first, count, g.V, 4 * g.nc, g.mb);
    return hipGetLastError();
}

hipError_t launch_soa_to_aos(const Geom &g, const void *field, int first, int count, double *aos, hipStream_t st)
{
    const long tot = (long)count * g.V * 4 * g.nc;
    k_soa_to_aos<<<nblocks(tot), TPB, 0, st>>>((const double2 *)field, (double2 *)aos, first, count, g.V, 4 * g.nc, g.mb);
    return hipGetLastError();
}

hipError_t launch_link_setup(const Geom &g, const double *links, const double *phase, double *ul64, float *ul32,
                             hipStream_t st)
{
    const unsigned nb = nblocks(3L * g.V);
    if (g.nc == 2)
        k_link_setup<2><<<nb, TPB, 0, st>>>(links, (const double2 *)phase, (double2 *)ul64, (float2 *)ul32, g.V);
    else
        k_link_setup<3><<<nb, TPB, 0, st>>>(links, (const double2 *)phase, (double2 *)ul64, (float2 *)ul32, g.V);
    return hipGetLastError();
}

hipError_t launch_ucc_to_links(const Geom &g, const double *ucc, double *ul64, float *ul32, hipStream_t st)
{
    const long n = 3L * g.V * g.nc * g.nc;
    k_ucc_setup<<<nblocks(n), TPB, 0, st>>>((const double2 *)ucc, (double2 *)ul64, (float2 *)ul32, n);
    return hipGetLastError();
}

// Lanes per link of a gauge half step: four while they are needed to fill the chip, else one (link_update_lane,
// efield_update_lane; SU(2) links are always one).  The lines lie where the two cross: SU(2) E fields between 16^3
// and 18^3 (18^3: 15.8 and 15.7 us), SU(3) links alone at 32^3, with the stencil links, whose stores are better
// spread over four lanes, between 40^3 and 44^3 (a Wilson step of one FP32 mode with E moving: 40^3 335 and 333 us,
// 36^3 242 and 247, 44^3 449 and 446).
constexpr long ONE_LANE_EFIELD_SU2 = 16384, ONE_LANE_LINKS_SU3 = 90000, ONE_LANE_STENCIL_SU3 = 200000;
static int lanes_per_link(const Geom &g, int what, bool stencil)
{
    const long links = 3L * g.V;
    if (g.nc == 2) return what == GAUGE_LINKS_HALF || links > ONE_LANE_EFIELD_SU2 ? 1 : 4;
    return what == GAUGE_LINKS_HALF && links > (stencil ? ONE_LANE_STENCIL_SU3 : ONE_LANE_LINKS_SU3) ? 1 : 4;
}

GaugeHalf gauge_half_args(const Geom &g, int what, double *links, double *efield, double dt, int reunit, const double *phase,
                          double *ul64, float *ul32)
{
    return GaugeHalf{links, efield, phase, ul64, ul32, dt, reunit, g.n0, g.n1, g.n2, g.V, what, lanes_per_link(g, what, ul64 != nullptr), 0};
}

hipError_t launch_gauge_half(const Geom &g, const GaugeHalf &h, hipStream_t st)
{
    const unsigned nb = (unsigned)((3L * g.V * h.lpl + LINK_TPB - 1) / LINK_TPB);
    if (h.what == GAUGE_LINKS_HALF) {
        if (g.nc == 2) k_link_update<2, 1><<<nb, LINK_TPB, 0, st>>>(h);
        else if (h.lpl == 1) k_link_update<3, 1><<<nb, LINK_TPB, 0, st>>>(h);
        else k_link_update<3, 4><<<nb, LINK_TPB, 0, st>>>(h);
    } else {
        // one lane per link fills the chip with workgroups of any size: the larger ones start sooner
        if (g.nc == 3) k_efield_update<3, 4, LINK_TPB><<<nb, LINK_TPB, 0, st>>>(h);
        else if (h.lpl == 1) k_efield_update<2, 1, TPB><<<(unsigned)((3L * g.V + TPB - 1) / TPB), TPB, 0, st>>>(h);
        else k_efield_update<2, 4, LINK_TPB><<<nb, LINK_TPB, 0, st>>>(h);
    }
    return hipGetLastError();
}

hipError_t launch_hop_gauge(const Geom &g, int prec, const HopArgs &a, const GaugeHalf &half, hipStream_t st)
{
    if (a.ens_sys || epi_kind(a) != EPI_AXPY) return hipErrorInvalidValue;
    GaugeHalf h = half;
    if (g.nc == 3) h.lpl = 4;  // the exponential in one lane would take the stencil's registers
    const long nb = (3L * g.V * h.lpl + TPB - 1) / TPB;
    h.blocks = (int)((nb + NUM_XCD - 1) / NUM_XCD * NUM_XCD);
    if (g.nc == 2) return prec == P64 ? hop_gauge_mb<2, double>(g, a, h, st) : hop_gauge_mb<2, float>(g, a, h, st);
    return prec == P64 ? hop_gauge_mb<3, double>(g, a, h, st) : hop_gauge_mb<3, float>(g, a, h, st);
}

size_t mode_dot_partial_len(const Geom &g) { return (size_t)DOT_CHUNKS * g.nblk * g.mb * 2; }

int mode_dot_chunks() { return DOT_CHUNKS; }

hipError_t launch_mode_dot_partial(const Geom &g, const void *a, const void *b, double *partial, hipStream_t st)
{
    dim3 grid(DOT_CHUNKS, g.nblk);
    const auto A = (const double2 *)a;
    const auto B = (const double2 *)b;
    const auto P = (double2 *)partial;
#define DOT(NC, MB) k_mode_dot<NC, MB><<<grid, TPB, 0, st>>>(A, B, P, g.V, g.nblk)
    if (g.nc == 2) {
        if (g.mb == 16) DOT(2, 16); else if (g.mb == 32) DOT(2, 32); else DOT(2, 64);
    } else {
        if (g.mb == 16) DOT(3, 16); else if (g.mb == 32) DOT(3, 32); else DOT(3, 64);
    }
#undef DOT
    return hipGetLastError();
}

hipError_t launch_mode_dot(const Geom &g, const void *a, const void *b, double *partial, double *out, hipStream_t st)
{
    const hipError_t e = launch_mode_dot_partial(g, a, b, partial, st);
    if (e != hipSuccess) return e;
    const int np = g.nblk * g.mb;
    k_mode_dot_finish<<<np, 64, 0, st>>>((const double2 *)partial, (double2 *)out, np);
    return hipGetLastError();
}

// partial results of the observables: LOC_BLOCKS x LOC_COUNT of the local ones, then EB_BLOCKS of E.B
// (fixed upper limits: the static scratch of ovl_observables_noalloc holds them too).  A workgroup of the local ones
// has 64 sites at a time; with 256 of them at most, lattices from 32^3 on left the chip half empty (SU(2) 64^3, a
// call with its synchronisation: energy 62.8 us and Gauss law 48.4 us; with 1024 workgroups and nothing
// else computed 37.3 and 38.8; the unitarity norm 61.7 and 27.0).
constexpr int LOC_BLOCKS = 1024, EB_BLOCKS = 2048;
static_assert(LOC_COUNT + 1 == OBS_RAW, "raw observables");
size_t reduce_partial_len(const Geom &) { return (size_t)LOC_BLOCKS * LOC_COUNT + EB_BLOCKS; }

template <int NC, int WHAT>
static hipError_t observables(const Geom &g, const double *links, const double *efield, double *gfield, double *partial,
                              double *out, double *derived, hipStream_t st)
{
    const int nl = (int)std::min<long>(LOC_BLOCKS, (4L * g.V + TPB - 1) / TPB);
    const int nb = std::min(nl, OBS_BLOCKS);
    const int ne = (int)std::min<long>(EB_BLOCKS, (3L * g.V + 64 / NC - 1) / (64 / NC));
    double *pe = partial + (size_t)LOC_BLOCKS * LOC_COUNT;
    if constexpr (WHAT == OBS_ALL)
        k_observables<NC><<<nb + ne, EB_TPB, 0, st>>>(links, efield, partial, nl, nb, pe, gfield, g.n0, g.n1, g.n2);
    else if constexpr (WHAT == OBS_EDOTB) k_edotb<NC><<<ne, EB_TPB, 0, st>>>(links, efield, pe, g.n0, g.n1, g.n2);
    else k_obs_local<NC, WHAT><<<nl, TPB, 0, st>>>(links, efield, partial, gfield, g.n0, g.n1, g.n2);
    if (out)
        k_obs_finish<WHAT><<<1, TPB, 0, st>>>(partial, nl, pe, ne, out, derived, (double)(NC * NC - 1) * (double)g.V,
                                              3.0 * (double)g.V);
    return hipGetLastError();
}

template <int NC>
static hipError_t observables_nc(const Geom &g, const double *links, const double *efield, int what, double *gfield,
                                 double *partial, double *out, double *derived, hipStream_t st)
{
    switch (what) {
    case OBS_ENERGY: return observables<NC, OBS_ENERGY>(g, links, efield, gfield, partial, out, nullptr, st);
    case OBS_GAUSS: return observables<NC, OBS_GAUSS>(g, links, efield, gfield, partial, out, nullptr, st);
    case OBS_UNITARITY: return observables<NC, OBS_UNITARITY>(g, links, efield, gfield, partial, out, nullptr, st);
    case OBS_EDOTB: return observables<NC, OBS_EDOTB>(g, links, efield, gfield, partial, out, nullptr, st);
    case OBS_ALL: return observables<NC, OBS_ALL>(g, links, efield, gfield, partial, out, derived, st);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_observables(const Geom &g, const double *links, const double *efield, int what, double *gfield,
                              double *partial, double *out, hipStream_t st, double *derived)
{
    if (derived && !(what == OBS_ALL && out)) return hipErrorInvalidValue;
    return g.nc == 2 ? observables_nc<2>(g, links, efield, what, gfield, partial, out, derived, st)
                     : observables_nc<3>(g, links, efield, what, gfield, partial, out, derived, st);
}

hipError_t launch_gauss_restore(const Geom &g, const double *links, const double *gfield, double *efield, double gamma,
                                hipStream_t st)
{
    const unsigned nb = nblocks(3L * g.V);
    if (g.nc == 2) k_gauss_restore<2><<<nb, TPB, 0, st>>>(links, gfield, efield, gamma, g.n0, g.n1, g.n2);
    else k_gauss_restore<3><<<nb, TPB, 0, st>>>(links, gfield, efield, gamma, g.n0, g.n1, g.n2);
    return hipGetLastError();
}

size_t currents_partial_len(const Geom &g) { return (size_t)g.nblk * g.V * 8; }

hipError_t launch_currents(const Geom &g, const void *psi, const void *hpsi, const double *gam, int first_mode,
                           double *partial, double *jv, double *ja, hipStream_t st)
{
    const long nsites = (long)g.nblk * g.V;
    const auto P = (const double2 *)psi;
    const auto H = (const double2 *)hpsi;
#define CUR(NC, MB) k_currents<NC, MB><<<(unsigned)((nsites + TPB / MB - 1) / (TPB / MB)), TPB, 0, st>>>(P, H, (const double2 *)gam, partial, g.V, g.nblk, first_mode)
    if (g.nc == 2) {
        if (g.mb == 16) CUR(2, 16); else if (g.mb == 32) CUR(2, 32); else CUR(2, 64);
    } else {
        if (g.mb == 16) CUR(3, 16); else if (g.mb == 32) CUR(3, 32); else CUR(3, 64);
    }
#undef CUR
    k_currents_finish<<<nblocks(g.V), TPB, 0, st>>>(partial, jv, ja, g.V, g.nblk, 1.0 / (2.0 * g.V));
    return hipGetLastError();
}

hipError_t launch_mscg_update(const Geom &g, int nshift, double *ps, double *chi, const double *r, const double *coef,
                              const int *active, hipStream_t st)
{
    const long per_blk = (long)g.V * 4 * g.nc;
    const long nel = per_blk * g.nblk * g.mb;
    k_mscg_update2<<<nblocks(nel), TPB, 0, st>>>(nshift, (double2 *)ps, (double2 *)chi, (const double2 *)r, coef, active,
                                                 per_blk, g.nblk, g.mb);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------
// QED eigenbasis launchers
// ---------------------------------------------------------------------------------------------
#define OVL_EIG_DISPATCH(KERNEL, GRID, ...)                                       \
    do {                                                                          \
        if (g.nc == 2 && g.mb == 16) KERNEL<2, 16><<<GRID, TPB, 0, st>>>(__VA_ARGS__); \
        else if (g.nc == 2 && g.mb == 32) KERNEL<2, 32><<<GRID, TPB, 0, st>>>(__VA_ARGS__); \
        else if (g.nc == 2 && g.mb == 64) KERNEL<2, 64><<<GRID, TPB, 0, st>>>(__VA_ARGS__); \
        else if (g.nc == 3 && g.mb == 16) KERNEL<3, 16><<<GRID, TPB, 0, st>>>(__VA_ARGS__); \
        else if (g.nc == 3 && g.mb == 32) KERNEL<3, 32><<<GRID, TPB, 0, st>>>(__VA_ARGS__); \
        else if (g.nc == 3 && g.mb == 64) KERNEL<3, 64><<<GRID, TPB, 0, st>>>(__VA_ARGS__); \
        else return hipErrorInvalidValue;                                         \
    } while (0)

hipError_t launch_eig_sources(const Geom &g, void *field, long k0, int cnt, long dz, hipStream_t st)
{
    if (cnt < 1 || cnt > g.nblk * g.mb) return hipErrorInvalidValue;
    const unsigned grid = (unsigned)((cnt + TPB - 1) / TPB);
    OVL_EIG_DISPATCH(k_eig_sources, grid, (double2 *)field, g.V, k0, cnt, dz);
    return hipGetLastError();
}

hipError_t launch_eig_gather(const Geom &g, const void *out, void *A, long k0, int nsb, hipStream_t st)
{
    const long plane = (long)g.n0 * g.n1;
    if (nsb < 1 || nsb > g.nblk * g.mb) return hipErrorInvalidValue;
    const long total = (long)g.n2 * nsb * 4 * plane;
    const unsigned grid = (unsigned)std::min<long>((total + TPB - 1) / TPB, 65536);
    OVL_EIG_DISPATCH(k_eig_gather, grid, (const double2 *)out, (double2 *)A, plane, g.n2, k0, nsb);
    return hipGetLastError();
}

size_t eig_partial_len() { return (size_t)2 * RED_BLOCKS; }
int eig_partial_blocks() { return RED_BLOCKS; }

hipError_t launch_eig_leak(const Geom &g, const void *field, int nvalid, double *partial, hipStream_t st)
{
    OVL_EIG_DISPATCH(k_eig_leak, RED_BLOCKS, (const double2 *)field, g.V, g.nblk, nvalid, partial);
    return hipGetLastError();
}

hipError_t launch_eig_hermitize(void *A, long dz, int n2, double *partial, hipStream_t st)
{
    k_eig_hermitize<<<RED_BLOCKS, TPB, 0, st>>>((double2 *)A, dz, n2, partial);
    return hipGetLastError();
}

hipError_t launch_nonfinite(const void *x, const void *y, long n, double *partial, hipStream_t st)
{
    if (!x || n < 0) return hipErrorInvalidValue;
    k_nonfinite<<<RED_BLOCKS, TPB, 0, st>>>((const double *)x, (const double *)y, n, partial);
    return hipGetLastError();
}

hipError_t launch_eig_modes(const Geom &g, const EigMode *modes, int nm, const void *A, const void *tw, double f,
                            void *psi, void *mid, hipStream_t st)
{
    if (nm < 1 || nm > g.nblk * g.mb) return hipErrorInvalidValue;
    const long total = (long)g.nblk * g.V * 4 * g.nc * g.mb;
    const unsigned grid = (unsigned)std::min<long>((total + TPB - 1) / TPB, 65536);
    OVL_EIG_DISPATCH(k_eig_modes, grid, modes, nm, (const double2 *)A, (const double2 *)tw, f, g.V,
                     (long)g.n0 * g.n1, g.n2, g.nblk, (double2 *)psi, (double2 *)mid);
    return hipGetLastError();
}
#undef OVL_EIG_DISPATCH

}  // namespace ovl
