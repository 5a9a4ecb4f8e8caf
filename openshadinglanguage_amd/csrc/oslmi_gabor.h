// CDNA4 device library: Gabor noise (sparse convolution with a Poisson
// impulse process, Lagae et al.), with screen-space filtering and Dual2
// derivatives.
//
// Reference: src/liboslnoise/sfm_gabornoise.h (fast_rng :21-60, kernels
// :71-97, GaborUniformParams :100-135, gabor_setup_filter :167-222,
// gabor_sample :226-300, gabor_cell :305-385, gabor_grid :390-470,
// scalar_gabor :497-515) and gabornoise.h (filter_gabor_kernel_2d
// :152-182, make_orthonormals :207-217).
//
// Per-point work that does not depend on the impulse (the filter matrices
// and, for a fixed anisotropy direction, the whole filtered-kernel
// transform) is computed once per point instead of once per impulse; the
// arithmetic on each impulse is unchanged, so values are identical.
#pragma once
#include "oslmi_math.h"
#include "oslmi_noise.h"

namespace oslmi {

// Uniform (per-op) Gabor parameters, computed on the host from NoiseParams.
struct GaborUniform {
    float a, lambda, sqrt_lambda_inv, radius, radius2, radius3, radius_inv;
    float poisson_g;  // expf(-lambda*radius3)
    float scale;      // final normalization of scalar_gabor
    float dir_x, dir_y, dir_z;
    int anisotropic;  // 0 isotropic, 1 anisotropic, 2 hybrid
    int do_filter;
};

struct M22 {
    float m00, m01, m10, m11;
};
OSLMI_DEV M22 m22(float a, float b, float c, float d)
{
    M22 r;
    r.m00 = a;
    r.m01 = b;
    r.m10 = c;
    r.m11 = d;
    return r;
}
OSLMI_DEV M22 mul(const M22& A, const M22& B)
{
    return m22(0.0f + A.m00 * B.m00 + A.m01 * B.m10, 0.0f + A.m00 * B.m01 + A.m01 * B.m11,
               0.0f + A.m10 * B.m00 + A.m11 * B.m10, 0.0f + A.m10 * B.m01 + A.m11 * B.m11);
}
OSLMI_DEV M22 add(const M22& A, const M22& B)
{
    return m22(A.m00 + B.m00, A.m01 + B.m01, A.m10 + B.m10, A.m11 + B.m11);
}
OSLMI_DEV M22 scale(float s, const M22& A) { return m22(A.m00 * s, A.m01 * s, A.m10 * s, A.m11 * s); }
OSLMI_DEV float det(const M22& A) { return A.m00 * A.m11 - A.m01 * A.m10; }
// Imath Matrix22::inverse(singExc=false)
OSLMI_DEV M22 inv(const M22& A)
{
    float s[4] = { A.m11, -A.m01, -A.m10, A.m00 };
    float r    = A.m00 * A.m11 - A.m10 * A.m01;
    if (fabsf(r) >= 1.0f) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            s[i] /= r;
    } else {
        float mr = fabsf(r) / 1.17549435e-38f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (mr > fabsf(s[i]))
                s[i] /= r;
            else
                return m22(1.0f, 0.0f, 0.0f, 1.0f);
        }
    }
    return m22(s[0], s[1], s[2], s[3]);
}

struct M33 {
    float m[3][3];
};

OSLMI_DEV V3 mult(const M33& M, V3 s)
{
    return V3(s.x * M.m[0][0] + s.y * M.m[1][0] + s.z * M.m[2][0],
              s.x * M.m[0][1] + s.y * M.m[1][1] + s.z * M.m[2][1],
              s.x * M.m[0][2] + s.y * M.m[1][2] + s.z * M.m[2][2]);
}
// Columns 0 and 1 of (row vector s) * M, with derivatives.
OSLMI_DEV void mult_xy(const M33& M, const Dv& s, Df& a, Df& b)
{
    Df s0 = comp(s, 0), s1 = comp(s, 1), s2 = comp(s, 2);
    a     = s0 * M.m[0][0] + s1 * M.m[1][0] + s2 * M.m[2][0];
    b     = s0 * M.m[0][1] + s1 * M.m[1][1] + s2 * M.m[2][1];
}

OSLMI_DEV V3 vnormalized(V3 v)
{
    float l = sqrtf(dot(v, v));
    return l != 0.0f ? V3(v.x / l, v.y / l, v.z / l) : v;
}

OSLMI_DEV Df ddot(const Dv& a, const Dv& b)
{
    return comp(a, 0) * comp(b, 0) + comp(a, 1) * comp(b, 1) + comp(a, 2) * comp(b, 2);
}
OSLMI_DEV Df ddot(V3 a, const Dv& b) { return comp(b, 0) * a.x + comp(b, 1) * a.y + comp(b, 2) * a.z; }

struct GaborRng {
    uint32_t s;
    OSLMI_DEV GaborRng() : s(1u) {}
    OSLMI_DEV GaborRng(V3 p, uint32_t seed)
    {
        s = inthash((uint32_t)ifloor(p.x), (uint32_t)ifloor(p.y), (uint32_t)ifloor(p.z), seed);
        if (!s)
            s = 1;
    }
    OSLMI_DEV float operator()()
    {
        s *= 3039177861u;
        return (float)s * (1.0f / 4294967296.0f);
    }
};

// Per-point filter state (gabor_setup_filter) plus, for the anisotropic
// mode, the impulse-independent part of filter_gabor_kernel_2d.
struct GaborPoint {
    M22 filter;
    M33 local;
    V3 N;
    int do_filter;
    // anisotropic + filter: filtered-kernel constants
    V3 omega_t;
    float c_F, K, E, a_f, omf_x, omf_y;
};

OSLMI_DEV void gabor_filter_consts(const M22& Sigma_f, float a, float ox, float oy, float& c_F,
                                   float& K, float& E, float& a_f, float& omf_x, float& omf_y)
{
    const float two_pi = 6.28318548202514648438f;  // float(2*pi)
    M22 Sigma_G        = scale(a * a / two_pi, m22(1.0f, 0.0f, 0.0f, 1.0f));
    c_F                = 1.0f / (two_pi * sqrtf(det(Sigma_f)));
    M22 Sigma_F        = scale((float)(1.0 / (4.0 * 3.14159265358979323846 * 3.14159265358979323846)),
                               inv(Sigma_f));
    M22 SGF            = add(Sigma_G, Sigma_F);
    M22 SGFi           = inv(SGF);
    float mx           = ox * SGFi.m00 + oy * SGFi.m10;
    float my           = ox * SGFi.m01 + oy * SGFi.m11;
    E                  = fexp(-0.5f * (mx * ox + my * oy));
    K                  = 1.0f / (two_pi * sqrtf(det(SGF)));
    M22 Sigma_G_i      = inv(Sigma_G);
    M22 Sigma_GF       = inv(add(inv(Sigma_F), Sigma_G_i));
    M22 Sigma_GF_Gi    = mul(Sigma_GF, Sigma_G_i);
    omf_x              = ox * Sigma_GF_Gi.m00 + oy * Sigma_GF_Gi.m10;
    omf_y              = ox * Sigma_GF_Gi.m01 + oy * Sigma_GF_Gi.m11;
    a_f = sqrtf((float)(6.283185307179586476925 * (double)sqrtf(det(Sigma_GF))));
}

OSLMI_DEV void gabor_setup(const GaborUniform& U, const Dv& P, GaborPoint& gp)
{
    gp.do_filter = 0;
    if (!U.do_filter)
        return;
    V3 n = cross(P.dx, P.dy);
    if (dot(n, n) < 1.0e-6f)
        return;
    n = vnormalized(n);
    V3 t = fabsf(n.x) < 0.9f ? V3(0.0f, n.z, -n.y) : V3(-n.z, 0.0f, n.x);
    t    = vnormalized(t);
    V3 b = cross(n, t);
    // Mtex_to_tan = cols(t, b, n); Mscreen_to_tex = cols(dPdx, dPdy, 0)
    M33 L;
    L.m[0][0] = t.x; L.m[0][1] = b.x; L.m[0][2] = n.x;
    L.m[1][0] = t.y; L.m[1][1] = b.y; L.m[1][2] = n.y;
    L.m[2][0] = t.z; L.m[2][1] = b.z; L.m[2][2] = n.z;
    // rows 0,1 / cols 0,1 of Mscreen_to_tex * Mtex_to_tan
    float s00 = 0.0f + P.dx.x * L.m[0][0] + P.dy.x * L.m[1][0] + 0.0f * L.m[2][0];
    float s01 = 0.0f + P.dx.x * L.m[0][1] + P.dy.x * L.m[1][1] + 0.0f * L.m[2][1];
    float s10 = 0.0f + P.dx.y * L.m[0][0] + P.dy.y * L.m[1][0] + 0.0f * L.m[2][0];
    float s11 = 0.0f + P.dx.y * L.m[0][1] + P.dy.y * L.m[1][1] + 0.0f * L.m[2][1];
    M22 Mst   = m22(s00, s01, s10, s11);
    M22 Mt    = m22(s00, s10, s01, s11);
    float sf  = 0.5f;
    M22 Sf    = mul(mul(Mt, m22(sf * sf, 0.0f, 0.0f, sf * sf)), Mst);
    gp.N      = n;
    gp.filter = Sf;
    gp.local  = L;
    if (det(Sf) < 1.0e-18f)
        return;
    gp.do_filter = 1;
    if (U.anisotropic == 1) {
        gp.omega_t = mult(L, V3(U.dir_x, U.dir_y, U.dir_z));
        gabor_filter_consts(Sf, U.a, gp.omega_t.x, gp.omega_t.y, gp.c_F, gp.K, gp.E, gp.a_f,
                            gp.omf_x, gp.omf_y);
    }
}

OSLMI_DEV Df gabor_kernel3(V3 omega, float phi, float bw, const Dv& x)
{
    const float pi = 3.14159274101257324219f, two_pi = 6.28318548202514648438f;
    Df g = dexp((-pi * (bw * bw)) * ddot(x, x));
    Df h = dcos(two_pi * ddot(omega, x) + Df(phi));
    return Df(1.0f) * g * h;
}
OSLMI_DEV Df gabor_kernel2(const Df& w, float ox, float oy, const Df& phi, float bw, const Df& x0,
                           const Df& x1)
{
    const float pi = 3.14159274101257324219f, two_pi = 6.28318548202514648438f;
    Df g = dexp((-pi * (bw * bw)) * (x0 * x0 + x1 * x1));
    Df h = dcos(two_pi * (x0 * ox + x1 * oy) + phi);
    return w * g * h;
}

// One in-radius impulse: contribution to the cell sum.
OSLMI_DEV Df gabor_impulse(const GaborUniform& U, const GaborPoint& gp, V3 omega, float phi,
                           const Dv& xk)
{
    const float pi = 3.14159274101257324219f, two_pi = 6.28318548202514648438f;
    if (gp.do_filter == 1) {
        V3 omega_t;
        float c_F, K, E, a_f, ofx, ofy;
        if (U.anisotropic == 1) {
            omega_t = gp.omega_t;
            c_F = gp.c_F; K = gp.K; E = gp.E; a_f = gp.a_f; ofx = gp.omf_x; ofy = gp.omf_y;
        } else {
            omega_t = mult(gp.local, omega);
            gabor_filter_consts(gp.filter, U.a, omega_t.x, omega_t.y, c_F, K, E, a_f, ofx, ofy);
        }
        Df d_i   = -ddot(gp.N, xk);
        Df w_s   = 1.0f * dexp((-pi * (U.a * U.a)) * (d_i * d_i));
        Df phi_s = phi - two_pi * d_i * omega_t.z;
        Df w_f   = (c_F * w_s) * K * E;
        Df x0, x1;
        mult_xy(gp.local, xk, x0, x1);
        Df gk = gabor_kernel2(w_f, ofx, ofy, phi_s, a_f, x0, x1);
        if (!isfinite(gk.v))
            gk = gabor_kernel3(omega, phi, U.a, xk);
        return gk;
    }
    return gabor_kernel3(omega, phi, U.a, xk);
}

// ---- the impulse scan -----------------------------------------------------
// An evaluation visits the cells around P, draws each cell's impulses and
// adds up those within the kernel radius. The kernel of an impulse costs
// 100 to 250 instructions, and one drawn impulse in six lies in the radius:
// evaluated where it is found, the kernel runs for nearly every impulse of
// every cell with a few of the 64 lanes active. So impulses that may lie in
// the radius are queued per lane (generator state and cell, in LDS) and the
// kernel runs over the queues when one is full and at the end. Terms keep
// their order (cell after cell, summed per cell first), and the distance
// test that decides is the kernel loop's, on the exact offset; the scan's
// own test only has to keep every impulse that passes it.
//
// What is left is the scan, which has two forms:
//  * per wave: the active lanes shade neighbouring points, whose cells fill
//    a small box (at most 8 x 8 x 4 and 128 cells; the periods of a periodic
//    noise, which wrap the cells, all alike). Each active lane seeds the
//    generator of one of the box's cells and draws its impulse count; then
//    all lanes test every impulse of the box together. The generator runs
//    once per wave, in the scalar unit, and nothing diverges;
//  * per lane: each lane walks its own cells (points far apart).
// Both are bound by VALU issue. layered3 (one filtered noise in three
// dimensions) over 1M points, the kernel where impulses are found against
// this: 345 to 247 us; 64 generated groups over unrelated points 845 to 513
// (32 to 2048 points each) and 1332 to 1037 us (to 262,144). A noise in three
// dimensions under a branch that 2, 10, 30 and 90 % of 1M points take in no
// order: 164, 187, 260 and 277 us there; 181, 210, 258 and 316 where waves
// with an idle lane scanned per lane; 154, 143, 162 and 203 here. (At 0.4 %,
// a lone lane in every fourth wave: 99, 114 and 105.)

// Queue slots per lane: 10 slots of eight bytes for 256 work-items, 20 KB of
// LDS: six workgroups a CU still fit, the six waves per SIMD that the
// kernels are allocated for.
constexpr int kGaborQueue = 10;
struct GaborQueued {
    uint32_t state, code;  // generator state before the impulse, its cell
};

// Small launches leave most of the chip idle while each wave works through
// its cells alone, so there a workgroup shades 64 points instead of 256: its
// four waves run the same points side by side (`split`), each evaluates a
// quarter of the cells, in their order, and all four add up the cells' sums,
// in their order, from LDS. Every wave holds the same values throughout, so
// all of them meet at the barriers. `split` is a constant of the kernel: as
// a value it cost the other launches 12% (registers spilled in the drain).
// Over 16,411 points (layered3) a launch takes 42 us instead of 89.

// 3039177861^k modulo 2^32: k draws of the generator at once
constexpr uint32_t gabor_rng_pow(int k)
{
    uint32_t r = 1u;
    for (int i = 0; i < k; ++i)
        r *= 3039177861u;
    return r;
}

// The scan's distance test: squared distance of the impulse with generator
// state s from the lane, both relative to the cell's centre and in units of
// 2^-32 cells.
OSLMI_DEV bool gabor_near(V3 in_cell, uint32_t s, float near2)
{
    const uint32_t half = 0x80000000u;
    const V3 d = in_cell
                 - V3((float)(int32_t)((s * gabor_rng_pow(3)) ^ half),
                      (float)(int32_t)((s * gabor_rng_pow(2)) ^ half),
                      (float)(int32_t)((s * gabor_rng_pow(1)) ^ half));
    return __fmaf_rn(d.z, d.z, __fmaf_rn(d.y, d.y, d.x * d.x)) < near2;
}

// Poisson(lambda radius^3) by multiplying uniforms until the product is at
// most g (fast_rng::poisson): n factors stay above g and the n + 1st does
// not. The product never grows (no uniform exceeds 1), so n is the number
// of partial products above g, counted here over four draws at a time:
// the four states and products of a round do not wait for a branch each.
OSLMI_DEV int gabor_poisson(GaborRng& rng, float g)
{
    const float k = 1.0f / 4294967296.0f;
    int n   = 0;
    float t = 1.0f;
    for (;;) {
        const uint32_t s1 = rng.s * gabor_rng_pow(1), s2 = rng.s * gabor_rng_pow(2);
        const uint32_t s3 = rng.s * gabor_rng_pow(3), s4 = rng.s * gabor_rng_pow(4);
        const float t1 = t * ((float)s1 * k), t2 = t1 * ((float)s2 * k);
        const float t3 = t2 * ((float)s3 * k), t4 = t3 * ((float)s4 * k);
        n += (t1 > g) + (t2 > g) + (t3 > g) + (t4 > g);
        uint32_t s = s1;
        s          = t1 > g ? s2 : s;
        s          = t2 > g ? s3 : s;
        s          = t3 > g ? s4 : s;
        rng.s      = s;
        if (!(t4 > g))
            return n;
        t = t4;
    }
}

// Squared length of the smallest offset component that an impulse of the
// cell at distance t = xc - c along one axis can have: the component is
// radius * (t - u) with u in [0, 1], and rounding is monotone.
OSLMI_DEV float gabor_axis_bound(const GaborUniform& U, float t)
{
    const float d = U.radius * (t < 0.0f ? t : (t > 1.0f ? t - 1.0f : 0.0f));
    return d * d;
}

// The cells that can hold an impulse within the radius, as a bit each in
// the order they are summed in (z outermost): a cell whose bounds already
// give a squared length of radius2 or more contributes an exact zero. Of
// the 27 cells 20.6 remain on average, 16.3 of a 1D or 2D noise (z = 0: the
// cells above the plane touch the radius only).
OSLMI_DEV uint32_t gabor_cell_mask(const GaborUniform& U, V3 xc)
{
    float sx[3], sy[3], sz[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        sx[a] = gabor_axis_bound(U, xc.x - (float)(a - 1));
        sy[a] = gabor_axis_bound(U, xc.y - (float)(a - 1));
        sz[a] = gabor_axis_bound(U, xc.z - (float)(a - 1));
    }
    uint32_t m = 0;
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int j = 0; j < 3; ++j)
#pragma unroll
            for (int i = 0; i < 3; ++i)
                if (!((sx[i] + sy[j]) + sz[k] >= U.radius2))
                    m |= 1u << (9 * k + 3 * j + i);
    return m;
}

// Queued cells: box coordinates i, j < 8, k < 4 in one byte.
OSLMI_DEV uint32_t gabor_cell_code(int i, int j, int k)
{
    return (uint32_t)(i | (j << 3) | (k << 6));
}
OSLMI_DEV V3 gabor_cell_of(uint32_t code)
{
    return V3((float)(code & 7u), (float)((code >> 3) & 7u), (float)(code >> 6));
}

// The generator of cell c_i, wrapped first by a periodic noise
// (sfm_gabornoise.h:304-310).
OSLMI_DEV GaborRng gabor_cell_rng(V3 c_i, uint32_t seed, bool periodic, V3 period)
{
    if (periodic)
        c_i = V3(wrap_period(c_i.x, period.x), wrap_period(c_i.y, period.y),
                 wrap_period(c_i.z, period.z));
    return GaborRng(c_i, seed);
}

// Smallest and largest value, in 0..15, over the wave's active lanes: the
// values' bits as lane masks, walked from the highest in scalar registers.
#if defined(__HIP_DEVICE_COMPILE__)
OSLMI_DEV void wave_range(uint32_t v, uint64_t active, int& lo, int& hi)
{
    uint64_t least = active, most = active;
    lo = hi = 0;
#pragma unroll
    for (int b = 3; b >= 0; --b) {
        const uint64_t set = __ballot((v >> b) & 1u);
        if (least & ~set)
            least &= ~set;
        else
            lo |= 1 << b;
        if (most & set) {
            most &= set;
            hi |= 1 << b;
        }
    }
}
#endif

// Whether every active lane of the wave holds the same vector, bit for bit.
OSLMI_DEV bool wave_same(V3 v)
{
#if defined(__HIP_DEVICE_COMPILE__)
    const uint32_t x = __float_as_uint(v.x), y = __float_as_uint(v.y), z = __float_as_uint(v.z);
    return !wave_any(x != (uint32_t)__builtin_amdgcn_readfirstlane((int)x)
                     || y != (uint32_t)__builtin_amdgcn_readfirstlane((int)y)
                     || z != (uint32_t)__builtin_amdgcn_readfirstlane((int)z));
#else
    (void)v;
    return true;
#endif
}

// The wave's box of cells: origin (ox, oy, oz), size (dx, dy, dz). False
// where the per-wave scan does not apply. An axis reaches one cell beyond
// the lanes' own cells on either side, above only where a lane needs it.
struct GaborBox {
    int ox, oy, oz, dx, dy, dz;
};
OSLMI_DEV bool gabor_wave_box(const GaborUniform& U, V3 fl, V3 xc, GaborBox& b)
{
#if defined(__HIP_DEVICE_COMPILE__)
    const uint64_t active = __ballot(1);
    // cells a binary32 coordinate and an int hold alike (false for NaN)
    const float lim = 1048576.0f;
    if (wave_any(!(fabsf(fl.x) < lim && fabsf(fl.y) < lim && fabsf(fl.z) < lim)))
        return false;
    // the lanes' cells relative to seven below the first lane's: a larger
    // distance does not fit a box either
    b.ox = __builtin_amdgcn_readfirstlane((int)fl.x) - 7;
    b.oy = __builtin_amdgcn_readfirstlane((int)fl.y) - 7;
    b.oz = __builtin_amdgcn_readfirstlane((int)fl.z) - 7;
    const uint32_t x = (uint32_t)((int)fl.x - b.ox), y = (uint32_t)((int)fl.y - b.oy);
    const uint32_t z = (uint32_t)((int)fl.z - b.oz);
    if (wave_any(x > 14u || y > 14u || z > 14u))
        return false;
    int lo, hi, z_hi;
    wave_range(x, active, lo, hi);
    b.ox += lo - 1;
    b.dx = hi - lo + 3;
    wave_range(y, active, lo, hi);
    b.oy += lo - 1;
    b.dy = hi - lo + 3;
    wave_range(z, active, lo, hi);
    wave_range(gabor_axis_bound(U, xc.z - 1.0f) >= U.radius2 ? z : z + 1u, active, hi, z_hi);
    b.oz += lo - 1;
    b.dz = z_hi - lo + 2;
    return b.dx <= 8 && b.dy <= 8 && b.dz <= 4 && b.dx * b.dy * b.dz <= 128;
#else
    return false;
#endif
}

// 65536 / d + 1 for a box's size 3..8
OSLMI_DEV int gabor_per(int d)
{
    return d == 3 ? 21846 : d == 4 ? 16385 : d == 5 ? 13108 : d == 6 ? 10923 : d == 7 ? 9363 : 8193;
}

// gabor_evaluate + gabor_grid: the cells around P, scaled. seed selects the
// generator stream (0 for the scalar noise, 0/1/2 for the components of the
// vector noise).
OSLMI_DEV Df gabor_grid(const GaborUniform& U, const GaborPoint& gp, const Dv& P, uint32_t seed,
                        bool periodic, V3 period, bool split)
{
    const float two_pi = 6.28318548202514648438f;
    const float two32  = 4294967296.0f;
    // the scan's squared distance limit, in units of 2^32 cells: 1 + 2^-10
    // lets every impulse through whose exact offset is inside (the scan's
    // rounding errors are below 2^-18)
    const float near2 = 1.0009765625f * two32 * two32;
    __shared__ GaborQueued queue[kGaborQueue][256];
    // a value and two derivatives for the 27 cells around each of 64 points
    // (20.7 KB, in split kernels only)
    __shared__ float split_sums[3 * 27 * 64];
    const int tid = (int)threadIdx.x;
    // the wave's quarter of the cells
    int wave = 0;
    if (split) {
#if defined(__HIP_DEVICE_COMPILE__)
        wave = __builtin_amdgcn_readfirstlane(tid >> 6);
#endif
        __syncthreads();  // the last evaluation's sums have been read
        for (int k = 7 * wave; k < (wave < 3 ? 7 * wave + 7 : 27); ++k)
            for (int c = 0; c < 3; ++c)
                split_sums[(27 * c + k) * 64 + (tid & 63)] = 0.0f;
        __syncthreads();
    }
    // draws per impulse: position, direction (isotropic 2, hybrid 1), phase
    const uint32_t step = U.anisotropic == 1   ? gabor_rng_pow(4)
                          : U.anisotropic == 0 ? gabor_rng_pow(6)
                                               : gabor_rng_pow(5);
    Dv xg = P * U.radius_inv;
    V3 fl(floorf(xg.v.x), floorf(xg.v.y), floorf(xg.v.z));
    Dv xc(xg.v - fl, xg.dx, xg.dy);
    GaborBox box = { 0, 0, 0, 0, 0, 0 };
    // a wave's cells are wrapped and seeded once, so by one period: points
    // with periods of their own walk their own cells
    const bool by_wave = gabor_wave_box(U, fl, xc.v, box) && (!periodic || wave_same(period));
    // the queued cells' origin relative to this lane's cell, and the lane's
    // position from that cell's centre in units of 2^-32 cells
    V3 org(-1.0f, -1.0f, -1.0f);
    uint32_t cells = 0;
    if (by_wave) {
        org = V3((float)box.ox, (float)box.oy, (float)box.oz) - fl;
    } else {
        cells = gabor_cell_mask(U, xc.v);
        if (split)
            cells &= 0x7fu << (7 * wave);
    }
    const V3 at = two32 * (xc.v - org) - V3(0.5f * two32);
    // the same from the centre of the cell being scanned
    V3 in_cell = at;
    // per lane: its cell's code, generator state and impulses left
    uint32_t code = 0, state = 0;
    int left = 0;
#if defined(__HIP_DEVICE_COMPILE__)
    // per wave: the same of the wave's cell (wi, wj, wk), the cell-th of
    // ncells; the generators of the next cells, one a lane, and the lanes
    // whose cells are still to come
    int ncells = box.dx * box.dy * box.dz;
    int cell = 0, wi = 0, wj = 0, wk = 0, wleft = 0, lane_count = 0;
    uint32_t wcode = 0, wstate = 0, lane_state = 0;
    uint64_t seeded = 0;
    const int per_x = gabor_per(box.dx), per_y = gabor_per(box.dy);
    V3 wpos = at;
    if (split && by_wave) {
        cell        = (wave * ncells) >> 2;
        ncells      = ((wave + 1) * ncells) >> 2;
        const int q = cell / box.dx;
        wi          = cell - q * box.dx;
        wk          = q / box.dy;
        wj          = q - wk * box.dy;
        wpos        = at - two32 * V3((float)wi, (float)wj, (float)wk);
    }
#endif
    int queued = 0, sum_code = -1;
    Df sum = Df(0.0f), cell_sum = Df(0.0f);
    // A cell's sum is complete. An impulse in the radius lies at most one
    // cell away from the lane's own, so the split's slot is one of 27.
    auto close_cell = [&]() {
        if (!split) {
            sum = sum + cell_sum;
        } else if (sum_code >= 0) {
            const V3 c  = org + gabor_cell_of((uint32_t)sum_code);
            float* slot = split_sums + (13 + (int)c.x + 3 * (int)c.y + 9 * (int)c.z) * 64 + (tid & 63);
            slot[0]           = cell_sum.v;
            slot[27 * 64]     = cell_sum.dx;
            slot[2 * 27 * 64] = cell_sum.dy;
        }
    };
    for (;;) {
        bool last;
#if defined(__HIP_DEVICE_COMPILE__)
        if (by_wave) {
            if (wleft <= 0 && cell < ncells) {
                // left out when no lane is within the radius of the cell
                const float ex = fmaxf(fabsf(wpos.x) - 0.5f * two32, 0.0f);
                const float ey = fmaxf(fabsf(wpos.y) - 0.5f * two32, 0.0f);
                const float ez = fmaxf(fabsf(wpos.z) - 0.5f * two32, 0.0f);
                const bool near
                    = wave_any(__fmaf_rn(ez, ez, __fmaf_rn(ey, ey, ex * ex)) < near2);
                if (near && seeded == 0) {
                    seeded         = __ballot(1);
                    const int mine = cell
                                     + (int)__builtin_amdgcn_mbcnt_hi(
                                         (uint32_t)(seeded >> 32),
                                         __builtin_amdgcn_mbcnt_lo((uint32_t)seeded, 0));
                    // mine / box.dx and its quotient by box.dy, both below 192
                    const int q = (mine * per_x) >> 16, k = (q * per_y) >> 16;
                    GaborRng rng = gabor_cell_rng(
                        V3((float)(box.ox + mine - q * box.dx), (float)(box.oy + q - k * box.dy),
                           (float)(box.oz + k)),
                        seed, periodic, period);
                    lane_count = mine < ncells ? gabor_poisson(rng, U.poisson_g) : 0;
                    lane_state = rng.s;
                }
                if (near) {
                    const int from = __builtin_ctzll(seeded);
                    wleft   = __builtin_amdgcn_readlane(lane_count, from);
                    wstate  = (uint32_t)__builtin_amdgcn_readlane((int)lane_state, from);
                    in_cell = wpos;
                    wcode   = gabor_cell_code(wi, wj, wk);
                }
                seeded &= seeded - 1;
                // on to the next cell, x innermost
                ++cell;
                wpos.x -= two32;
                if (++wi == box.dx) {
                    wi     = 0;
                    wpos.x = at.x;
                    wpos.y -= two32;
                    if (++wj == box.dy) {
                        wj     = 0;
                        wpos.y = at.y;
                        wpos.z -= two32;
                        ++wk;
                    }
                }
            }
            // two impulses a round; a slot is written whether or not the
            // impulse is kept, so nothing branches
            bool full = false;
            while (wleft > 0 && !full) {
                const uint32_t next = wstate * step;
                queue[queued][tid]  = GaborQueued { wstate, wcode };
                queued += gabor_near(in_cell, wstate, near2);
                queue[queued][tid] = GaborQueued { next, wcode };
                queued += wleft > 1 && gabor_near(in_cell, next, near2);
                wstate = (uint32_t)__builtin_amdgcn_readfirstlane((int)(next * step));
                wleft -= 2;
                full = wave_any(queued > kGaborQueue - 2);
            }
            last = wleft <= 0 && cell >= ncells;
            if (!last && !full)
                continue;
        } else
#endif
        {
            if (!wave_any(left > 0) && cells) {
                const int bit = __builtin_ctz(cells);
                cells &= cells - 1;
                const int q = (bit * 171) >> 9;  // bit / 3
                const int k = (q * 171) >> 9;
                code        = gabor_cell_code(bit - 3 * q, q - 3 * k, k);
                const V3 c  = gabor_cell_of(code);
                in_cell     = at - two32 * c;
                GaborRng rng = gabor_cell_rng(fl + (org + c), seed, periodic, period);
                left         = gabor_poisson(rng, U.poisson_g);
                state        = rng.s;
            }
            while (wave_any(left > 0) && !wave_any(queued > kGaborQueue - 2)) {
                const uint32_t next = state * step;
                queue[queued][tid]  = GaborQueued { state, code };
                queued += left > 0 && gabor_near(in_cell, state, near2);
                queue[queued][tid] = GaborQueued { next, code };
                queued += left > 1 && gabor_near(in_cell, next, near2);
                state = next * step;
                left -= 2;
            }
            last = !wave_any(cells != 0 || left > 0);
            if (!last && !wave_any(queued > kGaborQueue - 2))
                continue;
        }
#pragma clang loop unroll(disable)
        for (int e = 0; wave_any(e < queued); ++e) {
            if (e < queued) {
                GaborRng rng;
                const GaborQueued it = queue[e][tid];
                rng.s                = it.state;
                const uint32_t qc    = it.code;
                const V3 c        = org + gabor_cell_of(qc);
                const float z_rng = rng(), y_rng = rng(), x_rng = rng();
                const Dv xk = U.radius * Dv((xc.v - c) - V3(x_rng, y_rng, z_rng), xc.dx, xc.dy);
                if (dot(xk.v, xk.v) < U.radius2) {
                    if ((int)qc != sum_code) {
                        close_cell();
                        cell_sum = Df(0.0f);
                        sum_code = (int)qc;
                    }
                    V3 omega;
                    if (U.anisotropic == 1) {
                        omega = V3(U.dir_x, U.dir_y, U.dir_z);
                    } else if (U.anisotropic == 0) {
                        float omega_t = two_pi * rng();
                        float u       = rng();
                        float cos_p   = -1.0f * (1.0f - u) + 1.0f * u;
                        float sin_p   = sqrtf(fmaxf(0.0f, 1.0f - cos_p * cos_p));
                        float st, ct;
                        fsincos(omega_t, &st, &ct);
                        omega = vnormalized(V3(ct * sin_p, st * sin_p, cos_p));
                    } else {
                        float omega_r
                            = sqrtf(U.dir_x * U.dir_x + U.dir_y * U.dir_y + U.dir_z * U.dir_z);
                        float omega_t = two_pi * rng();
                        float st, ct;
                        fsincos(omega_t, &st, &ct);
                        omega = omega_r * V3(ct, st, 0.0f);
                    }
                    const float phi = two_pi * rng();
                    cell_sum        = cell_sum + gabor_impulse(U, gp, omega, phi, xk);
                }
            }
        }
        queued = 0;
        if (last)
            break;
    }
    close_cell();
    if (split) {
        // a cell without impulses adds an exact zero
        __syncthreads();
        for (int k = 0; k < 27; ++k) {
            const float* slot = split_sums + k * 64 + (tid & 63);
            sum = sum + Df(slot[0], slot[27 * 64], slot[2 * 27 * 64]);
        }
    }
    return (sum * U.sqrt_lambda_inv) * U.scale;
}

// scalar_gabor / scalar_pgabor for a Dual2 point P (dim 1..3 input already
// packed in P; pgabor pads the periods of 1 and 2 dimensions with zeros).
OSLMI_DEV Df gabor(const GaborUniform& U, const Dv& P, bool periodic = false,
                   V3 period = V3(0.0f), bool split = false)
{
    GaborPoint gp;
    gabor_setup(U, P, gp);
    return gabor_grid(U, gp, P, 0u, periodic, period, split);
}

// scalar_gabor3 / scalar_pgabor3 (sfm_gabornoise.h:517-640): one filter
// set-up, the three components from generator seeds 0, 1 and 2. The seed
// loop is kept rolled: the cell walk is large and runs once per component.
OSLMI_DEV Dv gabor3(const GaborUniform& U, const Dv& P, bool periodic = false,
                    V3 period = V3(0.0f), bool split = false)
{
    GaborPoint gp;
    gabor_setup(U, P, gp);
    Df r0, r1, r2;
#pragma clang loop unroll(disable)
    for (uint32_t seed = 0; seed < 3; ++seed) {
        const Df r = gabor_grid(U, gp, P, seed, periodic, period, split);
        if (seed == 0)
            r0 = r;
        else if (seed == 1)
            r1 = r;
        else
            r2 = r;
    }
    return make_dv(r0, r1, r2);
}

}  // namespace oslmi
