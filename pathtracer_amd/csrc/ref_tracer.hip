// ref_tracer.hip — PT_MODE_REF: the reference's spectral path tracer
// (src/shader.comp) as a wavefront of gfx950 kernels.
//
// The reference runs one invocation per pixel that loops over samples and
// bounces (src/shader.comp:1393-1533). Here a dispatch is a set of independent
// paths, pixels [p0, p0 + pc) x samples [k0, k0 + m), that one persistent kernel
// traces from camera to end: a lane keeps its path in registers through all its
// bounces (closest hit, shading, the shadow ray, Russian roulette) and takes the
// next path from a queue when it ends, so nothing of a path goes through memory
// but its XYZ, and lanes stay busy whatever the spread of path lengths. Sphere
// tracing is a state of the lane: every marching lane of a wave takes one
// distance evaluation per iteration, and the lanes that wait for shading, an
// intersection or a new path do that together once enough of them wait.
// The sequential PCG chain travels with the path, so every path draws the
// same numbers in the same order as the shader, and each path's arithmetic is
// the shader's (same operations, same order, ptmath.h built-ins). Radiance is
// folded per pixel in sample order, so the texels match the reference method
// bit for bit wherever the operations are the same.
#include <algorithm>
#include <cstring>
#include <mutex>
#include <utility>

#include "tracer.hpp"

namespace ptk {

using namespace ptd;

// in namespace ptk: the header holds device helpers only, no includes
#include "wave_queue.h"

constexpr float kPi = 3.14159265358979f;  // PI, src/shader.comp:9 (binary32)
constexpr float kOneByThree = 0.3333333f; // ONEBYTHREE, src/shader.comp:10
constexpr int kBlock = 256;

__device__ __forceinline__ float ubo_at(const float* u, int k) { return (k >= 0 && k < kUboFloats) ? u[k] : 0.0f; }

// ---- spectral helpers (src/shader.comp:129-140, 960-974, 1030-1091) ----------------
__device__ __forceinline__ f4 sample_wavelengths(float lh) {
    float base = lh - 390.0f;
    return f4{390.0f + ptm_mod(base + (0.25f * 1.0f) * 330.0f, 330.0f),
              390.0f + ptm_mod(base + (0.25f * 2.0f) * 330.0f, 330.0f),
              390.0f + ptm_mod(base + (0.25f * 3.0f) * 330.0f, 330.0f),
              390.0f + ptm_mod(base + (0.25f * 4.0f) * 330.0f, 330.0f)};
}
__device__ __forceinline__ f3 wave_to_xyz(const float* u, float wave) {
    f3 r = mk3(0.0f, 0.0f, 0.0f);
    if (wave >= 360.0f && wave <= 800.0f) {
        int i3 = 3 * (int)(floorf(wave) - 360.0f);
        float t = wave - floorf(wave);
        int b = kUboCie + i3;
        r.x = ptm_mix(ubo_at(u, b), ubo_at(u, b + 3), t);
        r.y = ptm_mix(ubo_at(u, b + 1), ubo_at(u, b + 4), t);
        r.z = ptm_mix(ubo_at(u, b + 2), ubo_at(u, b + 5), t);
    }
    return r;
}
__device__ __forceinline__ float spd(float l, float peak, float sig, int invert) {
    float x = (l - peak) / (2.0f * sig * sig);
    float r = ptm_exp(-x * x);
    return ptm_mix(r, 1.0f - r, (float)invert);
}
// The reference's emitter at the path's wavelengths l (nm): Planck's law over
// its Wien peak, times luminosity. pw holds the path's numerators
// 1.19...e-16 (l 1e-9)^-5 and `peak` 4.09...e-6 T^5 of the light: binary64 powers
// that the shader evaluates at every vertex (they were most of the shading
// time), here taken once per path and per scene with the same operations.
__device__ __forceinline__ f4 planck_numerators(f4 l) {
    return f4{1.1910429724e-16f * ptm_pow_m5(l.x * 1e-9f), 1.1910429724e-16f * ptm_pow_m5(l.y * 1e-9f),
              1.1910429724e-16f * ptm_pow_m5(l.z * 1e-9f), 1.1910429724e-16f * ptm_pow_m5(l.w * 1e-9f)};
}
PT_HD float wien_peak(float T) { return 4.0956746759e-6f * ptm_pow(fmaxf(T, 0.0f), 5.0f); }
__device__ __forceinline__ float planck(float pw, float l, float T) {
    return pw / (ptm_exp(0.014387768775f / (l * T)) - 1.0f);
}
__device__ __forceinline__ f4 emit(f4 pw, f4 l, float T, float lum, float peak) {
    float t = fmaxf(T, 0.0f);
    float L = fmaxf(lum, 0.0f);
    return f4{(planck(pw.x, l.x * 1e-9f, t) / peak) * L, (planck(pw.y, l.y * 1e-9f, t) / peak) * L,
              (planck(pw.z, l.z * 1e-9f, t) / peak) * L, (planck(pw.w, l.w * 1e-9f, t) / peak) * L};
}
__host__ __device__ __forceinline__ float bk7(float l) {
    l *= 1e-3f;
    float l2 = l * l;
    float n2 = 1.0f;
    n2 += (1.03961212f * l2) / (l2 - 6.00069867e-3f);
    n2 += (0.231792344f * l2) / (l2 - 2.00179144e-2f);
    n2 += (1.01046945f * l2) / (l2 - 1.03560653e2f);
    return sqrtf(n2);
}
struct RMat { float peak, sigma, invert; };
__device__ __forceinline__ RMat material_mix(const float* u, float id) {
    int a = (int)floorf(id), b = (int)ceilf(id);
    float x = id - floorf(id);
    RMat r;
    r.peak = ptm_mix(ubo_at(u, kUboMat + 3 * a), ubo_at(u, kUboMat + 3 * b), x);
    r.sigma = ptm_mix(ubo_at(u, kUboMat + 3 * a + 1), ubo_at(u, kUboMat + 3 * b + 1), x);
    r.invert = ptm_mix(ubo_at(u, kUboMat + 3 * a + 2), ubo_at(u, kUboMat + 3 * b + 2), x);
    return r;
}
__device__ __forceinline__ void light_mix(const float* u, float id, float& T, float& lum) {
    int idx = (int)id;
    if (idx == -1) { T = 5500.0f; lum = 0.0f; return; }
    T = ubo_at(u, kUboLight + 2 * idx);
    lum = ubo_at(u, kUboLight + 2 * idx + 1);
}
// wien_peak of light `id` (temperature T): from the scene's table, or computed
// for an id outside it (a packed buffer may hold any number).
__device__ __forceinline__ float light_peak(const RefSceneDev& S, float id, float T) {
    const int idx = (int)id;
    return idx >= 0 && idx < kRefLights ? S.peak[idx] : wien_peak(T);
}
__device__ __forceinline__ f4 brdf(f4 l, const RMat& m) {
    int inv = (int)m.invert;
    return f4{spd(l.x, m.peak, m.sigma, inv) / kPi, spd(l.y, m.peak, m.sigma, inv) / kPi,
              spd(l.z, m.peak, m.sigma, inv) / kPi, spd(l.w, m.peak, m.sigma, inv) / kPi};
}

// ---- analytic primitives (src/shader.comp:263-448, 450-541, 633-679) ----------------
struct Hit {
    float t;
    f3 n;
    float mat, light;
};

__device__ __forceinline__ bool bounding_sphere(f3 o, f3 d, f3 pos, float r2) {
    f3 lo = o - pos;
    float b = dot(d, lo);
    float c = dot(lo, lo) - r2;
    if (b * b < c) return false;
    if (b >= 0.0f && c >= 0.0f) return false;
    return true;
}

__device__ __forceinline__ bool hit_sphere(f3 o, f3 d, const RefSphere& s, Hit& h) {
    f3 lo = o - mk3(s.px, s.py, s.pz);
    float b = 2.0f * dot(d, lo);
    float c = dot(lo, lo) - s.r * s.r;
    float disc = b * b - 4.0f * c;
    if (disc < 0.0f) return false;
    float sq = sqrtf(disc);
    float t1 = (-b - sq) * 0.5f;
    float t2 = (-b + sq) * 0.5f;
    float t = (t1 > 0.0f) ? t1 : t2;
    float outside = (t1 > 0.0f) ? 1.0f : -1.0f;
    if (t < 1e-4f) return false;
    if (t < h.t) {
        h.t = t;
        h.n = normalize(fma3s(d, t, lo) * outside);
        h.mat = s.mat;
        h.light = s.light;
        return true;
    }
    return false;
}

__device__ __forceinline__ bool hit_plane(f3 o, f3 d, const RefPlane& p, Hit& h) {
    f3 lo = o - mk3(p.px, p.py, p.pz);
    float t = -lo.y / d.y;
    if (t < 1e-4f) return false;
    if (t < h.t) {
        h.t = t;
        float facing = 0.0f * d.x + 1.0f * d.y + 0.0f * d.z;  // faceforward(+Y, I, +Y)
        h.n = facing < 0.0f ? mk3(0.0f, 1.0f, 0.0f) : mk3(-0.0f, -1.0f, -0.0f);
        h.mat = p.mat;
        h.light = p.light;
        return true;
    }
    return false;
}

__device__ __forceinline__ bool hit_box(f3 o, f3 d, const RefBox& b, Hit& h) {
    f3 lo = vmul(o - b.pos, b.M);
    f3 dl = vmul(d, b.M);
    f3 inv = mk3(1.0f / dl.x, 1.0f / dl.y, 1.0f / dl.z);
    f3 tmin = fma3(b.size, mk3(-0.5f, -0.5f, -0.5f), -lo) * inv;
    f3 tmax = fma3(b.size, mk3(0.5f, 0.5f, 0.5f), -lo) * inv;
    f3 lo3 = min3(tmin, tmax), hi3 = max3(tmin, tmax);
    float t1 = fmaxf(fmaxf(lo3.x, lo3.y), lo3.z);
    float t2 = fminf(fminf(hi3.x, hi3.y), hi3.z);
    float t = (t1 < 0.0f) ? t2 : t1;
    if (t1 > t2 || t < 1e-4f) return false;
    if (t < h.t) {
        h.t = t;
        f3 p = abs3((lo + dl * t) / b.size);
        float m = fmaxf(fmaxf(p.x, p.y), p.z);
        f3 st = mk3(ptm_step(m, p.x), ptm_step(m, p.y), ptm_step(m, p.z));
        f3 sg = -mk3(ptm_sign(dl.x), ptm_sign(dl.y), ptm_sign(dl.z));
        h.n = mvmul(b.M, st * sg);
        h.mat = b.mat;
        h.light = b.light;
        return true;
    }
    return false;
}

// One spherical cap of a lens (SphereSliceIntersection, src/shader.comp:366-417).
__device__ __forceinline__ bool hit_slice(f3 o, f3 d, f3 pos, const m3& M, float radius, float slice, bool first,
                                          float slicePos, bool sideInvert, float mat, float light, Hit& h,
                                          int& isOutside) {
    float off = radius - slice;
    f3 lo = vmul(o - pos, M);
    if (first) lo.x += slicePos - slice - off;
    else lo.x -= slicePos - slice - off;
    f3 dl = vmul(d, M);
    float b = 2.0f * dot(dl, lo);
    float c = dot(lo, lo) - radius * radius;
    float disc = b * b - 4.0f * c;
    float t = 1e6f;
    int out = 1;
    if (disc < 0.0f) return false;
    float sq = sqrtf(disc);
    float t1 = (-b - sq) * 0.5f;
    float t2 = (-b + sq) * 0.5f;
    if (first) {
        t1 = (fmaf(dl.x, t1, lo.x) > -off) ? 1e6f : t1;
        t2 = (fmaf(dl.x, t2, lo.x) > -off) ? 1e6f : t2;
    } else {
        t1 = (fmaf(dl.x, t1, lo.x) < off) ? 1e6f : t1;
        t2 = (fmaf(dl.x, t2, lo.x) < off) ? 1e6f : t2;
    }
    t = (t1 > 0.0f) ? t1 : t;
    if (t2 < t) { t = t2; out = -1; }
    if (t < 1e-4f) return false;
    if (t < h.t) {
        h.t = t;
        h.n = mvmul(M, normalize(fma3s(dl, t, lo) * (float)out));
        isOutside = (!sideInvert) ? out : -out;
        h.mat = mat;
        h.light = light;
        return true;
    }
    return false;
}

__device__ __forceinline__ bool hit_lens(f3 o, f3 d, const RefLens& L, Hit& h, int& isOutside) {
    bool any = false;
    for (int i = 0; i < 2; ++i)
        if (hit_slice(o, d, L.pos, L.M, L.twoF, L.half, i == 0, L.slicePos, !L.conv, L.mat, L.light, h, isOutside))
            any = true;
    return any;
}

__device__ __forceinline__ float eval_cubic(float a, float b, float c, float d, float x) {
    return x * (x * (x * a + b) + c) + d;
}
__device__ __forceinline__ float eval_quad(float a, float b, float c, float x) { return x * (x * a + b) + c; }
__device__ __forceinline__ float eval_quartic(float a, float b, float c, float d, float e, float x) {
    return x * (x * (x * (x * a + b) + c) + d) + e;
}
// SolveCubic (src/shader.comp:474-503); only the first root is used by the caller.
__device__ float cubic_first_root(float b, float c, float d) {
    float bd3 = b * kOneByThree;
    float Q = c * kOneByThree - bd3 * bd3;
    float R = 0.5f * bd3 * c - bd3 * bd3 * bd3 - 0.5f * d;
    float D = Q * Q * Q + R * R;
    float x;
    if (D > 0.0f) {
        float u = R + sqrtf(D);
        float v = R - sqrtf(D);
        float S = ptm_sign(u) * ptm_pow(fabsf(u), kOneByThree);
        float T = ptm_sign(v) * ptm_pow(fabsf(v), kOneByThree);
        x = S + T - bd3;
    } else {
        float sq = sqrtf(-Q);
        float th = ptm_acos(R / (sq * sq * sq)) * kOneByThree;
        x = (2.0f * sq) * ptm_cos(th) - bd3;
    }
    for (int i = 0; i < 2; ++i) x -= eval_cubic(1.0f, b, c, d, x) / eval_quad(3.0f, 2.0f * b, c, x);
    return x;
}
// SolveQuartic (src/shader.comp:505-541); returns a bit mask of real roots.
__device__ int solve_quartic(float a, float b, float c, float d, float e, float r[4]) {
    float inva = 1.0f / a;
    float inva2 = inva * 0.5f;
    float inva2a2 = inva2 * inva2;
    float bb = b * b;
    float p = -1.5f * bb * inva2a2 + c * inva;
    float q = bb * b * inva2a2 * inva2 - b * c * inva * inva2 + d * inva;
    float rr = -0.1875f * bb * bb * inva2a2 * inva2a2 + 0.5f * c * bb * inva2a2 * inva2 - b * d * inva2a2 + e * inva;
    float s = cubic_first_root(0.5f * -p, -rr, 0.5f * p * rr - 0.125f * q * q);
    float s2p = 2.0f * s - p;
    if (s2p < 0.0f) return 0;
    float is2p = -2.0f * s - p;
    float sq = sqrtf(s2p);
    float q2 = 2.0f * q / sq;
    float add = is2p + q2, sub = is2p - q2;
    float bd4a = 0.25f * inva * b;
    int mask = 0;
    if (add >= 0.0f) {
        float sa = sqrtf(add);
        r[0] = 0.5f * (-sq + 1.0f * sa) - bd4a;
        r[1] = 0.5f * (-sq + -1.0f * sa) - bd4a;
        for (int k = 0; k < 2; ++k)
            r[k] -= eval_quartic(a, b, c, d, e, r[k]) / eval_cubic(4.0f * a, 3.0f * b, 2.0f * c, d, r[k]);
        mask |= 3;
    }
    if (sub >= 0.0f) {
        float ss = sqrtf(sub);
        r[2] = 0.5f * (sq + 1.0f * ss) - bd4a;
        r[3] = 0.5f * (sq + -1.0f * ss) - bd4a;
        for (int k = 2; k < 4; ++k)
            r[k] -= eval_quartic(a, b, c, d, e, r[k]) / eval_cubic(4.0f * a, 3.0f * b, 2.0f * c, d, r[k]);
        mask |= 12;
    }
    return mask;
}

__device__ bool hit_cyclide(f3 ro, f3 rd, const RefCyclide& C, Hit& h) {
    f3 ol = vmul(ro - C.pos, C.M) / C.scale;
    f3 dl = vmul(rd, C.M) / C.scale;
    f3 o = mk3(ol.x, ol.z, ol.y);
    f3 d = mk3(dl.x, dl.z, dl.y);
    const float A = C.a, B = C.b, Cc = C.c, D = C.d;
    f3 dd = d * d, oo = o * o, od = o * d;
    f3 dyzx = mk3(d.y, d.z, d.x), dzxy = mk3(d.z, d.x, d.y);
    f3 oyzx = mk3(o.y, o.z, o.x), ozxy = mk3(o.z, o.x, o.y);
    float a4 = dot(dd, dd) + 2.0f * dot(dd, dyzx * dyzx);
    float a3 = 4.0f * (dot(o, d * d * d) + dot(od, dyzx * dyzx) + dot(od, dzxy * dzxy));
    float a2 = 6.0f * dot(oo, dd) + 8.0f * dot(od, oyzx * dyzx) + 2.0f * (dot(oo, dyzx * dyzx) + dot(oo, dzxy * dzxy)) +
               2.0f * (B * B - D * D) * dot(d, d) - 4.0f * (A * A * d.x * d.x + B * B * d.y * d.y);
    float a1 = 4.0f * (dot(o * o * o, d) + dot(oo, oyzx * dyzx) + dot(oo, ozxy * dzxy) + 2.0f * A * Cc * D * d.x +
                       (B * B - D * D) * dot(o, d) - 2.0f * (A * A * o.x * d.x + B * B * o.y * d.y));
    float a0 = dot(oo, oo) + 2.0f * dot(oo, oyzx * oyzx) + B * B * B * B + D * D * D * D - 2.0f * B * B * D * D -
               4.0f * Cc * Cc * D * D + 8.0f * A * Cc * D * o.x + 2.0f * (B * B - D * D) * dot(o, o) -
               4.0f * (A * A * o.x * o.x + B * B * o.y * o.y);
    float r[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    int real = solve_quartic(a4, a3, a2, a1, a0, r);
    float t = 1e6f;
    for (int i = 0; i < 4; ++i)
        if (((real >> i) & 1) && r[i] < t && r[i] > 0.0f) t = r[i];
    if (t < h.t) {
        h.t = t;
        float x = o.x + d.x * t, y = o.y + d.y * t, z = o.z + d.z * t;
        float term1 = x * x + y * y + z * z + B * B - D * D;
        f3 n = mk3(4.0f * (x * term1 - 2.0f * A * (A * x - Cc * D)), 4.0f * z * term1,
                   4.0f * y * (term1 - 2.0f * B * B));
        h.n = normalize(n);
        h.mat = C.mat;
        h.light = C.light;
        return true;
    }
    return false;
}

// Closest analytic hit over spheres, planes, boxes, lenses, cyclides in the
// reference's order with strict '<' (src/shader.comp:862-922, 1131-1201).
// Returns the object index in packing order, or -1.
__device__ int closest_analytic(const RefSceneDev& S, f3 o, f3 d, Hit& h) {
    int id = -1, base = 0;
    for (int i = 0; i < S.ns; ++i)
        if (hit_sphere(o, d, ld_ro_rec(S.sph + i), h)) id = i;
    base += S.ns;
    for (int i = 0; i < S.np; ++i)
        if (hit_plane(o, d, ld_ro_rec(S.pln + i), h)) id = base + i;
    base += S.np;
    for (int i = 0; i < S.nb; ++i) {
        const RefBox b = ld_ro_rec(S.box + i);
        if (!bounding_sphere(o, d, b.pos, b.bsr2)) continue;
        if (hit_box(o, d, b, h)) id = base + i;
    }
    base += S.nb;
    for (int i = 0; i < S.nl; ++i) {
        const RefLens L = ld_ro_rec(S.lens + i);
        if (!bounding_sphere(o, d, L.pos, L.br2)) continue;
        int outside = 1;
        if (hit_lens(o, d, L, h, outside)) id = base + i;
    }
    base += S.nl;
    for (int i = 0; i < S.nc; ++i) {
        const RefCyclide C = ld_ro_rec(S.cyc + i);
        if (!bounding_sphere(o, d, C.pos, C.brad2)) continue;
        if (hit_cyclide(o, d, C, h)) id = base + i;
    }
    return id;
}

// ---- SDFs (sdfs/{mandelbulb,menger,blob,terrain}.glsl) -----------------------------
// Correctly rounded quotient and square root for operands and results well
// inside the normal range: the compiler's own refinement sequences without the
// scaling and special-case instructions around them, which change nothing there
// (8 instead of 11 instructions, 9 instead of 15).
__device__ __forceinline__ float div_mid(float a, float b) {
    const float y0 = __builtin_amdgcn_rcpf(b);
    const float y = fmaf(fmaf(-b, y0, 1.0f), y0, y0);
    float q = a * y;
    q = fmaf(fmaf(-b, q, a), y, q);
    return fmaf(fmaf(-b, q, a), y, q);
}
__device__ __forceinline__ float sqrt_mid(float x) {
    const float s = __builtin_amdgcn_sqrtf(x);
    const float lo = __uint_as_float(__float_as_uint(s) - 1u), hi = __uint_as_float(__float_as_uint(s) + 1u);
    const float r = fmaf(-lo, s, x) <= 0.0f ? lo : s;
    return fmaf(-hi, s, x) > 0.0f ? hi : r;
}
// One iteration's terms that need rounding care: r^7, 1 / r, 1 / l and sin(phi)
// from r = |z| and l2 = x^2 + z^2, as ptm_pow, the divisions and the square root
// of the shader's expressions give them. In the middle of the range (all but
// points far outside or on the polar axis) without special cases: a march is a
// chain of hundreds of these iterations, and its length in instructions is what
// the longest paths of a launch cost. r^7 in binary64 has its ptm_pow value
// unless it lies within 2^-40 of a binary32 rounding boundary (ptm__pow_round):
// the 29 bits that rounding drops are then near 2^28.
__device__ __forceinline__ void mandelbulb_terms(float r, float l2, float& r7, float& invr, float& invl, float& sinp) {
    if (r >= 0x1p-16f && r <= 0x1p16f && l2 >= 0x1p-80f) {
        const double d = (double)r, d2 = d * d, d3 = d2 * d, y = d3 * d3 * d;
        r7 = (float)y;
        const uint32_t dropped = (uint32_t)ptm_d2u(y) & 0x1fffffffu;
        if (dropped - (0x10000000u - 8192u) <= 2u * 8192u) r7 = (float)ptm__exp_d(7.0 * ptm__log_d(d));  // ptm_pow
        invr = div_mid(1.0f, r);
        invl = div_mid(1.0f, sqrt_mid(l2));
        sinp = div_mid(invr, invl);
    } else {
        r7 = ptm_pow(r, 7.0f);
        invr = 1.0f / r;
        invl = ptm_rsqrt(l2);
        sinp = invr / invl;
    }
}
__device__ __forceinline__ float de_mandelbulb(f3 p, int iters, float bailout) {
    f3 z = p;
    float r = length(z);
    float dr = 1.0f;
    for (int i = 0; i < iters; ++i) {
        float r7, invr, invl, sinp;
        mandelbulb_terms(r, z.x * z.x + z.z * z.z, r7, invr, invl, sinp);
        dr = 8.0f * r7 * dr + 1.0f;
        r *= r;
        r *= r;
        r *= r;
        float cost = z.z * invl, cosp = z.y * invr, sint = z.x * invl;
        float ct2 = cost * cost, cp2 = cosp * cosp;
        float cost8 = fmaf(fmaf(fmaf(fmaf(128.0f, ct2, -256.0f), ct2, 160.0f), ct2, -32.0f), ct2, 1.0f);
        float cosp8 = fmaf(fmaf(fmaf(fmaf(128.0f, cp2, -256.0f), cp2, 160.0f), cp2, -32.0f), cp2, 1.0f);
        float sint8 = fmaf(fmaf(fmaf(128.0f, ct2, -192.0f), ct2, 80.0f), ct2, -8.0f) * sint * cost;
        float sinp8 = fmaf(fmaf(fmaf(128.0f, cp2, -192.0f), cp2, 80.0f), cp2, -8.0f) * sinp * cosp;
        z = r * mk3(sint8 * sinp8, cosp8, cost8 * sinp8);
        z = z + p;
        const float r2 = dot(z, z);
        r = sqrt_mid(r2);
        if (!(r2 >= 0x1p-80f && r2 <= 0x1p80f)) r = sqrtf(r2);
        if (r > bailout) break;
    }
    return 0.5f * ptm_log(r) * r / dr;
}
__device__ __forceinline__ float de_menger(f3 p, int levels) {
    f3 q = abs3(p) - mk3(1.0f, 1.0f, 1.0f);
    float d = length(max3(q, mk3(0.0f, 0.0f, 0.0f))) + fminf(fmaxf(q.x, fmaxf(q.y, q.z)), 0.0f);
    float s = 1.0f;
    for (int m = 0; m < levels; ++m) {
        f3 ps = p * s;
        f3 a = mk3(ptm_mod(ps.x, 2.0f) - 1.0f, ptm_mod(ps.y, 2.0f) - 1.0f, ptm_mod(ps.z, 2.0f) - 1.0f);
        s *= 3.0f;
        f3 aa = abs3(a);
        f3 r = abs3(mk3(1.0f - 3.0f * aa.x, 1.0f - 3.0f * aa.y, 1.0f - 3.0f * aa.z));
        float da = fmaxf(r.x, r.y), db = fmaxf(r.y, r.z), dc = fmaxf(r.z, r.x);
        float c = (fminf(da, fminf(db, dc)) - 1.0f) / s;
        d = fmaxf(d, c);
    }
    return d;
}
__device__ __forceinline__ float blob_sphere(f3 p, int k) {
    if (k == 0) return length(p) - 1.0f;
    if (k == 1) return length(mk3(p.x, p.y - 1.0f, p.z)) - 0.7f;
    if (k == 2) return length(mk3(p.x - 0.25f, p.y - 1.25f, p.z - 0.5f)) - 0.25f;
    return length(mk3(p.x + 0.25f, p.y - 1.25f, p.z - 0.5f)) - 0.25f;
}
// smin (src/shader.comp:685-702), after iquilezles.org/articles/smin
__device__ __forceinline__ float smin1(float x, float y) {
    float k = 0.02f;
    k *= 6.0f;
    float h = fmaxf(k - fabsf(x - y), 0.0f) / k;
    float m = h * h * h * 0.5f;
    float s = m * k * kOneByThree;
    return fminf(x, y) - s;
}
__device__ __forceinline__ void smin2(float& xd, float& xm, float yd, float ym) {
    float k = 0.02f;
    k *= 6.0f;
    float h = fmaxf(k - fabsf(xd - yd), 0.0f) / k;
    float m = h * h * h * 0.5f;
    float s = m * k * kOneByThree;
    if (xd < yd) { xd = xd - s; xm = xm + (ym - xm) * m; }
    else { xd = yd - s; xm = xm + (ym - xm) * (1.0f - m); }
}
__device__ __forceinline__ float de_blob(f3 p) {
    return smin1(smin1(smin1(blob_sphere(p, 0), blob_sphere(p, 1)), blob_sphere(p, 2)), blob_sphere(p, 3));
}
__device__ __forceinline__ float terrain_height(float x) {
    return ptm_sin(0.0625f * x) + ptm_sin(0.125f * (x + 10.0f)) + 0.25f * ptm_sin(0.25f * x) +
           0.125f * ptm_sin(0.5f * x) + 0.25f * ptm_sin(x) + 0.25f * ptm_sin(2.0f * x + 1.0f) +
           0.125f * ptm_sin(4.0f * x + 2.0f) + 0.0625f * ptm_sin(8.0f * x + 1.0f) +
           0.03125f * ptm_sin(16.0f * x + 5.0f) + 0.015625f * ptm_sin(32.0f * x) + 0.0078125f * ptm_sin(64.0f * x);
}
__device__ __forceinline__ float de_terrain(f3 p) { return p.y - (terrain_height(p.x) + terrain_height(p.z)); }

// Distance to an SDF of `kind` (KIND when it is known at compile time).
template <int KIND>
__device__ __forceinline__ float de_eval(int kind, int iterations, float bailout, f3 p) {
    switch (KIND ? KIND : kind) {
        case PT_SDF_MANDELBULB: return de_mandelbulb(p, iterations, bailout);
        case PT_SDF_MENGER: return de_menger(p, iterations);
        case PT_SDF_BLOB: return de_blob(p);
        case PT_SDF_TERRAIN: return de_terrain(p);
        default: return kMaxDist;
    }
}
__device__ __forceinline__ float sdf_material(const pt_sdf_desc& d, f3 p) {
    if (d.material_kind == PT_SDFMAT_RADIAL) {
        float f = dot(p, p);
        return ptm_mix(d.material[0], d.material[1], f / (d.material[2] + f));
    }
    if (d.material_kind == PT_SDFMAT_BLOB) {
        float xd = blob_sphere(p, 0), xm = d.material[0];
        smin2(xd, xm, blob_sphere(p, 1), d.material[1]);
        smin2(xd, xm, blob_sphere(p, 2), d.material[2]);
        smin2(xd, xm, blob_sphere(p, 3), d.material[3]);
        return xm;
    }
    return d.material[0];
}

// SearchSDF (src/shader.comp:732-777).
__device__ bool search_sdf(const RefSceneDev& S, f3 p, f3 invdir, float& tmn, float& tmx, uint32_t& set) {
    bool found = false;
    set = 0;
    for (int i = 0; i < S.nsdf; ++i) {
        const f3 pos = ld_ro_rec(&S.sdf[i].pos), size = ld_ro_rec(&S.sdf[i].size);
        f3 lo = p - pos;
        f3 t0 = fma3(size, mk3(-0.5f, -0.5f, -0.5f), -lo) * invdir;
        f3 t1 = fma3(size, mk3(0.5f, 0.5f, 0.5f), -lo) * invdir;
        f3 a = min3(t0, t1), b = max3(t0, t1);
        float bx = fmaxf(fmaxf(a.x, a.y), a.z);
        float by = fminf(fminf(b.x, b.y), b.z);
        if (bx > by || by < 0.0f) continue;
        uint32_t bit = 1u << (uint32_t)i;
        if (bx < tmn) {
            found = true;
            if (by < tmn) { tmn = bx; tmx = by; set = bit; }
            else if (by < tmx) { tmn = bx; set += bit; }
            else { tmn = bx; tmx = by; set += bit; }
        } else if (bx < tmx) {
            found = true;
            if (by > tmx) tmx = by;
            set += bit;
        }
    }
    return found;
}
// SphereTracing (src/shader.comp:779-860): over-relaxed sphere tracing after
// Keinert et al., "Enhanced Sphere Tracing" (2014), one distance evaluation at a
// time: `q` is the next point whose distance the march needs, and march_advance
// takes it. A lane's march lasts from 1 to over 512 evaluations, so marching to
// the end in one loop ran at the pace of the wave's longest ray.
enum : int {
    MP_SIGN = 0,      // the distance at the origin (its sign)
    MP_STEP = 1,      // a step of the march
    MP_NORMAL = 2,    // 2..7: the six differences of the normal
    MP_MATERIAL = 8,  // the material of the nearest SDF
};
struct March {
    f3 q;
    float t, insT, omega, prev, k, tmx;
    uint32_t set;
    int points, i, phase;
};
// Starts the march of the ray (o, d); false when it enters no SDF's box.
__device__ __forceinline__ bool march_start(const RefSceneDev& S, f3 o, f3 d, March& M) {
    f3 invdir = mk3(1.0f / d.x, 1.0f / d.y, 1.0f / d.z);
    float tmn = kMaxDist, tmx = kMaxDist;
    if (!search_sdf(S, o, invdir, tmn, tmx, M.set)) return false;
    M.t = fmaxf(tmn, 1e-3f);
    M.tmx = tmx;
    M.insT = 0.0f;
    M.omega = 1.70f;
    M.prev = 0.0f;
    M.k = 0.0f;
    M.points = 0;
    M.i = 0;
    M.phase = MP_SIGN;
    M.q = o;
    return true;
}
// The spliced SDF() at M.q: min over the SDFs of the set (src/pathtracer.cpp:
// 2004-2054). With `want_mat` also SDFMATERIAL(): the material of the nearest SDF,
// ties to the later one.
template <int KIND>
__device__ __forceinline__ float sdf_set(const RefSceneDev& S, f3 p, uint32_t set, bool want_mat, float& mat) {
    float s = kMaxDist, m = 0.0f;
    for (int i = 0; i < S.nsdf; ++i) {
        uint32_t code = 1u << (uint32_t)i;
        if ((set & code) == code) {
            const f3 q = p - ld_ro_rec(&S.sdf[i].pos);
            const pt_sdf_desc& desc = S.sdf[i].d;
            const int kind = KIND ? KIND : ld_ro(&desc.kind);
            const float di = de_eval<KIND>(kind, ld_ro(&desc.iterations), ld_ro(&desc.bailout), q);
            if (want_mat) m = (s < di) ? m : sdf_material(desc, q);
            s = fminf(s, di);
        }
    }
    mat = m;
    return s;
}
// Takes the distance v at M.q. Returns 0 while the march (or its normal and
// material) needs another one, 1 when the ray hits nothing before h.t, 2 at a
// hit. SHADOW rays need only the fact of the hit: the six distances the method
// evaluates for its normal are counted in `steps` but not evaluated.
template <bool SHADOW>
__device__ __forceinline__ int march_advance(const RefSceneDev& S, f3 o, f3 d, March& M, float v, float mat, Hit& h,
                                             unsigned& steps) {
    const float omegaMax = 1.70f, omegaSpeed = 0.20f;
    if (M.phase == MP_STEP) {
        ++steps;
        const float rad = v;
        bool end = false;
        if (M.insT > (fabsf(M.prev) + fabsf(rad))) {
            M.t -= M.insT;
            M.omega = 1.0f;
            M.insT = M.prev * M.omega * M.k;
            M.t += M.insT;
        } else if (fabsf(rad) < 1e-4f) {
            end = true;
        } else {
            if (M.t > M.tmx) M.points += 1;
            else M.points = 0;
            if (M.points >= 2) {
                M.t = M.tmx + 1e-3f;
                float tmn = kMaxDist;
                M.tmx = kMaxDist;
                const f3 invdir = mk3(1.0f / d.x, 1.0f / d.y, 1.0f / d.z);
                if (!search_sdf(S, fma3s(d, M.t, o), invdir, tmn, M.tmx, M.set)) return 1;
                tmn += M.t;
                M.tmx += M.t;
                M.t = fmaxf(tmn, M.t);
            } else {
                M.insT = rad * M.omega * M.k;
                M.t += M.insT;
                float f = fminf(rad / M.prev, 0.99f);
                M.omega += omegaSpeed * (fminf(1.0f / (1.0f - f), omegaMax) - M.omega);
                M.prev = rad;
            }
        }
        M.q = fma3s(d, M.t, o);
        if (!end && ++M.i < 512) return 0;
        // converged, or out of steps: a hit when nearer than the analytic one
        if (!(M.t < h.t)) return 1;
        h.t = M.t - 1e-3f;
        if (SHADOW) {
            steps += 6;
            return 2;
        }
    } else if (M.phase == MP_SIGN) {
        ++steps;
        M.k = ptm_sign(v);
        M.q = fma3s(d, M.t, o);
        M.phase = MP_STEP;
        return 0;
    } else {
        // the distance at the hit point displaced along an axis: + then -
        switch (M.phase) {
            case MP_NORMAL + 0: h.n.x = v; break;
            case MP_NORMAL + 1: h.n.x -= v; break;
            case MP_NORMAL + 2: h.n.y = v; break;
            case MP_NORMAL + 3: h.n.y -= v; break;
            case MP_NORMAL + 4: h.n.z = v; break;
            case MP_NORMAL + 5: h.n.z -= v; break;
            default:
                h.mat = mat;
                h.light = -1.0f;
                h.n = normalize(h.n);
                return 2;
        }
        ++steps;
    }
    ++M.phase;  // the normal's first difference after the march, else the next one, then the material
    const f3 p = fma3s(d, M.t, o);
    M.q = p;
    if (M.phase < MP_MATERIAL) {
        // p + e and p - e along one axis; the other components add a zero of e's
        // sign, which is what the vector sum and difference do
        const int k = M.phase - MP_NORMAL;
        const float e = (k & 1) ? -1e-4f : 1e-4f, z = copysignf(0.0f, e);
        M.q = p + mk3((k >> 1) == 0 ? e : z, (k >> 1) == 1 ? e : z, (k >> 1) == 2 ? e : z);
    }
    return 0;
}

// ---- sampling (src/shader.comp:976-1028, 1093-1119, 1225-1296) ----------------------
__device__ __forceinline__ f3 sample_unit_sphere(uint32_t& seed) {
    float rx = rand_chain(seed);
    float ry = rand_chain(seed);
    float phi = 2.0f * kPi * ry;
    float sinT = 2.0f * rx - 1.0f;
    float cosT = sqrtf(fmaf(-sinT, sinT, 1.0f));
    return mk3(ptm_cos(phi) * cosT, ptm_sin(phi) * cosT, sinT);
}
__device__ __forceinline__ f3 sample_cone(uint32_t& seed, float cosMax) {
    float rx = rand_chain(seed);
    float ry = rand_chain(seed);
    float cosA = 2.0f * cosMax * cosMax - 1.0f;
    float phi = 2.0f * kPi * ry;
    float ct = (1.0f - cosA) * rx + cosA;
    float st = sqrtf(fmaf(-ct, ct, 1.0f));
    return normalize(mk3(ptm_cos(phi) * st, ptm_sin(phi) * st, ct + 1.0f));
}
__device__ __forceinline__ f3 to_world(f3 v, f3 n) {
    f3 b1 = mk3(0.0f, -1.0f, 0.0f), b2 = mk3(-1.0f, 0.0f, 0.0f);
    if (n.z >= -0.9999999f) {
        float a = 1.0f / (1.0f + n.z);
        float b = -n.x * n.y * a;
        b1 = mk3(1.0f - (n.x * n.x * a), b, -n.x);
        b2 = mk3(b, 1.0f - (n.y * n.y * a), -n.y);
    }
    return b1 * v.x + b2 * v.y + n * v.z;
}
__device__ __forceinline__ float mis2(float p1, float p2) { return p1 * p1 / (p1 * p1 + p2 * p2); }

// SampleRandomLightSource (src/shader.comp:1225-1285), reading the packed
// objects like the shader, including its lens/cyclide count comparisons.
__device__ int sample_light(const RefSceneDev& S, uint32_t& seed, float& brad, f3& pos, float& lid) {
    const float* u = S.ubo;
    int rl = (int)floorf(rand_chain(seed) * S.numLights);
    int rid = (int)ubo_at(u, kUboLightId + rl);
    int off = kUboObj;
    auto P3 = [&](int k) { return mk3(ubo_at(u, k), ubo_at(u, k + 1), ubo_at(u, k + 2)); };
    auto ID = [&](int k) { return (float)((int)ubo_at(u, k) - 1); };
    if (rid < S.ns) {
        int k = off + 6 * rid;
        brad = ubo_at(u, k + 3); pos = P3(k); lid = ID(k + 5);
        return (int)ubo_at(u, kUboLightId + rl);
    }
    rid -= S.ns; off += 6 * S.ns;
    if (rid < S.np) {
        int k = off + 5 * rid;
        brad = 1e5f; pos = P3(k); lid = ID(k + 4);
        return (int)ubo_at(u, kUboLightId + rl);
    }
    rid -= S.np; off += 5 * S.np;
    if (rid < S.nb) {
        int k = off + 11 * rid;
        brad = 0.5f * length(P3(k + 6)); pos = P3(k); lid = ID(k + 10);
        return (int)ubo_at(u, kUboLightId + rl);
    }
    rid -= S.nb; off += 11 * S.nb;
    if (rid < S.nb) {
        int k = off + 12 * rid;
        float rad = ubo_at(u, k + 6), th = ubo_at(u, k + 8);
        brad = sqrtf((rad * rad) + (0.25f * th * th)); pos = P3(k); lid = ID(k + 11);
        return (int)ubo_at(u, kUboLightId + rl);
    }
    rid -= S.nl; off += 12 * S.nl;
    if (rid < S.nl) {
        int k = off + 16 * rid;
        brad = sqrtf(ubo_at(u, k + 13)); pos = P3(k); lid = ID(k + 15);
        return (int)ubo_at(u, kUboLightId + rl);
    }
    return 0;
}

// ---- kernels ---------------------------------------------------------------------------
struct RefFinish {
    int spf, currentSamples, frame, ISO;
    float apSize, FPS, persistence;
};
// Exposure and Accumulate into the texel buffer (src/shader.comp:1492-1532):
// `sum` is the sum over the dispatch's samples, tx the texel before it.
__device__ __forceinline__ float4 finish_texel(const RefFinish& F, f3 sum, float4 tx) {
    f3 out = sum / (float)F.spf;
    out = out * (F.apSize * F.apSize * (float)F.ISO);
    f3 in = mk3(tx.x, tx.y, tx.z);
    if (F.currentSamples == F.spf && F.frame > F.spf) {
        float wgt = ptm_pow(2.0f, -8.0f / (F.FPS * F.persistence));
        out = (1.0f - wgt) * out + wgt * in;
    } else {
        int u = F.currentSamples / F.spf;
        out = ((float)(u - 1) * in + out) / (float)u;
    }
    return make_float4(out.x, out.y, out.z, 1.0f);
}

// Camera ray of sample k of pixel `pix`: Rendering + Scene up to TracePath
// (src/shader.comp:1446-1476, 1509-1516).
__device__ __forceinline__ void camera_ray(const RefFrame& F, int pix, int k, f3& o, f3& d, uint32_t& seed, float& lh) {
    int gx = pix % F.W, gy = pix / F.W;
    uint32_t x = (uint32_t)gx, y = (uint32_t)(F.H - gy);
    float uvx = (2.0f * (float)x - (float)F.W) / (float)F.H;
    float uvy = (2.0f * (float)y - (float)F.H) / (float)F.H;
    seed = pcg((uint32_t)(F.frame - F.spf + k));
    seed += x + (uint32_t)F.W * y;
    float jx = 2.0f * rand_chain(seed) - 0.5f;
    float jy = 2.0f * rand_chain(seed) - 0.5f;
    uvx += jx / (float)F.W;
    uvy += jy / (float)F.H;
    float sc = -F.camSize * 0.5f;
    uvx *= sc;
    uvy *= sc;
    o = F.camPos + vmul(mk3(uvx, uvy, 0.0f), F.camM);
    float ux = rand_chain(seed), uy = rand_chain(seed);
    float phi = 2.0f * kPi * uy;
    float dr = sqrtf(ux);
    float dsx = dr * ptm_cos(phi), dsy = dr * ptm_sin(phi);
    float ap = 0.5f * F.apSize;
    f3 onAp = F.camPos + vmul(mk3(ap * dsx, ap * dsy, F.apDist), F.camM);
    d = normalize(onAp - o);
    lh = ptm_mix(360.0f, 800.0f, rand_chain(seed));
    // TracePathLens: two refractions through the BK7 bi-convex lens at the hero wavelength.
    float l = lh;
    for (int pass = 0; pass < 2; ++pass) {
        Hit h;
        h.t = 1e6f;
        h.n = mk3(0.0f, 0.0f, 0.0f);
        int outside = 1;
        for (int s = 0; s < 2; ++s)
            hit_slice(o, d, F.lensPos, F.lensM, F.lensTwoF, F.lensHalf, s == 0, F.lensSlicePos, false, 0.0f, -1.0f, h,
                      outside);
        float n1, n2;
        if (outside == 1) { n1 = 1.0f; n2 = bk7(l); }
        else { n1 = bk7(l); n2 = 1.0f; }
        float n12 = n1 / n2;
        l = l * n12;
        o = fma3s(d, h.t, o);
        d = refract(d, h.n, n12);
    }
}

// XYZ of a finished path (src/shader.comp:1477-1487); NaN samples become zero.
__device__ __forceinline__ f3 path_xyz(const RefSceneDev& S, f4 l, f4 L, unsigned& nans) {
    f3 X0 = wave_to_xyz(S.ubo, l.x), X1 = wave_to_xyz(S.ubo, l.y);
    f3 X2 = wave_to_xyz(S.ubo, l.z), X3 = wave_to_xyz(S.ubo, l.w);
    f3 col = L.x * X0 + L.y * X1 + L.z * X2 + L.w * X3;
    col = mk3(0.0f, 0.0f, 0.0f) + (col * (720.0f - 390.0f)) * 0.25f;
    if (col.x != col.x || col.y != col.y || col.z != col.z) {
        col = mk3(0.0f, 0.0f, 0.0f);
        ++nans;
    }
    return col;
}

// A lane's state in k_ref_path, what it does next.
enum : int {
    PS_IDLE,    // takes a path from the queue
    PS_RAY,     // its extension ray is to be intersected
    PS_SHADE,   // its hit is known
    PS_SHADOW,  // the visibility of its light sample is known
    PS_DONE,    // its path has ended and is to be stored
    PS_MARCH,   // sphere tracing, extension or shadow ray
};
// When a wave with marching lanes does the scene work (a new path, an intersection,
// shading) of the others: once kRefScene lanes wait for it, or as many as march (16
// to 40 measured within the runs' spread on the 512 x 512 x 4 mandelbulb scene, 8
// slower by 10 %). Ended lanes before they are stored and refilled: kRefRefill (the
// 1080p analytic scene, ms for 8 samples: 8 -> 3.4, 16 -> 3.1, 24 and 32 -> 2.8,
// 48 -> 2.9, 64 -> 3.5).
constexpr int kRefScene = 24;
constexpr int kRefRefillSdf = 16, kRefRefill = 32;
constexpr int kRefLanes = 64;  // threads per block: one wave, so that few paths spread over all compute units

// The path tracer, persistent: see the head of this file. KIND: -1 for scenes
// without SDF objects, PT_SDF_* when all are of one kind, 0 when they are mixed.
// It replaced a kernel per stage and bounce (36 launches for a frame of 5 bounces,
// path records of 168 bytes in memory between them, one ray per lane in the
// marches) and is bound by VALU issue in analytic scenes (rocprofv3, 3 spheres, a plane and
// 2 boxes at 512x512x8: 0.82 wave instructions per unit and clock, 27 of 64 lanes active, 1660
// instructions of a lane per segment with its shading and shadow ray): 1280x720x1 5
// bounces 966 -> 230 us, 1920x1080x8 8 bounces 15.8 -> 2.8 ms, 150x101x1 288 -> 81 us of
// kernels (one launch, its length the chain of a path's bounces). SDF scenes are bound by the chain of their longest path (512x512x4
// mandelbulb: up to 728 distance evaluations of 8 iterations, about 3.8 us each):
// 29.2 -> 5.7 ms. Registers: 165 (analytic) and 184 to 190 (SDF) leave 3 and 2 waves per SIMD;
// asking for 4 spills and was 20 % slower, and the path state in LDS while marching gave
// nothing.
// `direct`: the dispatch has one sample per pixel, all in this wave, and the
// paths' texels are finished here instead of by k_ref_fold.
template <int KIND>
__global__ void __launch_bounds__(kRefLanes) k_ref_path(RefSceneDev S, RefFrame F, RefWave Wv, RefFinish Fin,
                                                         float4* texels, int direct, int count_dispatch) {
    constexpr bool SDF = KIND >= 0;
    const int n = F.pc * F.m;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        atomicAdd(&Wv.stats[3], (unsigned long long)n);
        if (count_dispatch) atomicAdd(&Wv.stats[5], 1ull);
    }
    unsigned segments = 0, shadows = 0, steps = 0, nans = 0;
    // the path: index, bounce, next extension ray, RNG, wavelengths, Planck
    // numerators, throughput, radiance, MIS weight of the next emitter hit
    int st = PS_IDLE, p = 0, bounce = 0;
    f3 o = mk3(0.0f, 0.0f, 0.0f), d = o;
    uint32_t seed = 0;
    f4 l = mk4(0.0f), pw = l, T = l, L = l;
    float w = 1.0f;
    Hit h;
    h.t = 0.0f;
    h.n = o;
    h.mat = 0.0f;
    h.light = -1.0f;
    // the light sample: direction, contribution, light object, nearest analytic
    // object and its distance; whether the path goes on after it
    f3 sd = o;
    f4 contrib = l;
    int lobj = 0, sid = 0;
    float st_t = 0.0f;
    bool cont = false, shadow_ray = false;
    March M{};
    // The queue holds blocks of 64 consecutive paths, dealt to its segments in turn
    // (entry block e of segment s is path block e * segments + s), so that each
    // segment, which only its own waves drain, holds a share of every part of the
    // image; entries past the last path are dropped.
    const int nseg = min(kSeg, (int)gridDim.x);
    const int seg_blocks = ((n + 63) / 64 + nseg - 1) / nseg;
    WaveChunk chunk = wave_chunk_init(Wv.cursor, seg_blocks * nseg * 64);
    while (true) {
        bool scene = true;
        if (SDF) {
            const int marching = (int)__popcll(__ballot(st == PS_MARCH));
            const int waiting = (int)__popcll(__ballot(st != PS_MARCH && !(st == PS_IDLE && chunk.drained())));
            scene = waiting >= min(kRefScene, max(marching, 1)) || marching == 0;
        }
        if (scene) {
            if (SDF && st == PS_SHADOW) {
                if (sid == lobj) L = f4{L.x + contrib.x, L.y + contrib.y, L.z + contrib.z, L.w + contrib.w};
                st = cont ? PS_RAY : PS_DONE;
            }
            const bool free_lane = st == PS_IDLE || st == PS_DONE;
            const uint64_t idle = __ballot(free_lane);
            if (__popcll(idle) >= (SDF ? kRefRefillSdf : kRefRefill) || idle == __ballot(st != PS_MARCH)) {
                if (st == PS_DONE) {
                    const f3 c = path_xyz(S, l, L, nans);
                    if (direct) {
                        // the sum over samples starts from zero (src/shader.comp:1513-1516)
                        const f3 sum = mk3(0.0f, 0.0f, 0.0f) + c;
                        texels[F.p0 + p] = finish_texel(Fin, sum, texels[F.p0 + p]);
                    } else {
                        Wv.col[p] = make_float4(c.x, c.y, c.z, 0.0f);
                    }
                    st = PS_IDLE;
                }
                if (!chunk.drained()) {
                    const int e = wave_refill(idle, chunk);
                    const int b = e >> 6;
                    const int path = ((b % seg_blocks) * nseg + b / seg_blocks) * 64 + (e & 63);
                    if (e >= 0 && path < n) {
                        p = path;
                        float lh;
                        camera_ray(F, F.p0 + p % F.pc, F.k0 + p / F.pc, o, d, seed, lh);
                        l = sample_wavelengths(lh);
                        pw = planck_numerators(l);
                        T = mk4(1.0f);
                        L = mk4(0.0f);
                        w = 1.0f;
                        bounce = 0;
                        st = F.pathLength > 0 ? PS_RAY : PS_DONE;
                    }
                }
                if (chunk.drained() && __ballot(st != PS_IDLE) == 0ull) break;
            }
            // closest analytic hit (Intersection without SphereTracing)
            if (st == PS_RAY) {
                ++segments;
                h.t = kMaxDist;
                h.n = mk3(0.0f, 0.0f, 0.0f);
                h.mat = 0.0f;
                h.light = -1.0f;
                closest_analytic(S, o, d, h);
                st = PS_SHADE;
                if (SDF && march_start(S, o, d, M)) {
                    shadow_ray = false;
                    st = PS_MARCH;
                }
            }
            // TraceRay after the hit (src/shader.comp:1352-1391) with SampleLightSource
            // (src/shader.comp:1298-1343)
            if (st == PS_SHADE) {
                st = PS_DONE;
                bool shadow = false;
                if (h.t < kMaxDist) {
                    float LT, LL;
                    light_mix(S.ubo, h.light, LT, LL);
                    if (LL > 0.0f) {
                        f4 e = emit(pw, l, LT, LL, light_peak(S, h.light, LT)) * T * w;
                        L = f4{L.x + e.x, L.y + e.y, L.z + e.z, L.w + e.w};
                    } else {
                        const RMat mat = material_mix(S.ubo, h.mat);
                        const f4 f = brdf(l, mat);
                        const f3 nrm = h.n;
                        const f3 no = fma3s(d, h.t, o);
                        f3 nd = normalize(nrm + sample_unit_sphere(seed));
                        float pdf = dot(nd, nrm) / kPi;
                        if (S.numLights > 0.0f) {
                            float brad = 0.0f, lid = -1.0f;
                            f3 lpos = mk3(0.0f, 0.0f, 0.0f);
                            lobj = sample_light(S, seed, brad, lpos, lid);
                            float invd = 1.0f / length(lpos - no);
                            f3 ldir = (lpos - no) * invd;
                            float sinMax = fminf(brad * invd, 1.0f);
                            float cosMax = sqrtf(1.0f - sinMax * sinMax);
                            sd = to_world(sample_cone(seed, cosMax), ldir);
                            float lpdf = 1.0f / S.numLights;
                            lpdf *= dot(sd, ldir) / (kPi * (1.0f - cosMax * cosMax));
                            w = mis2(pdf, lpdf);
                            float ct = dot(sd, nrm);
                            float death = 1.25f * fmaxf(w - 0.2f, 0.0f);
                            if (ct >= 0.0f) {
                                if (rand_chain(seed) > death) {
                                    float T2, L2;
                                    light_mix(S.ubo, lid, T2, L2);
                                    f4 g = f4{f.x * ct / lpdf, f.y * ct / lpdf, f.z * ct / lpdf, f.w * ct / lpdf};
                                    contrib = emit(pw, l, T2, L2, light_peak(S, lid, T2)) * (T * g) * (1.0f - w);
                                    shadow = true;
                                } else {
                                    w = 1.0f;
                                }
                            }
                        } else {
                            w = mis2(pdf, 0.0f);
                        }
                        float ct = dot(nd, nrm);
                        T = T * f4{f.x * ct / pdf, f.y * ct / pdf, f.z * ct / pdf, f.w * ct / pdf};
                        float pr = ptm_clamp(fmaxf(T.x, fmaxf(T.y, fmaxf(T.z, T.w))), 0.0f, 0.99f);
                        cont = false;
                        if (!(rand_chain(seed) > pr)) {
                            T = T * (1.0f / pr);
                            ++bounce;
                            cont = bounce < F.pathLength;
                        }
                        // the shadow ray starts there too
                        o = no;
                        d = nd;
                        st = cont ? PS_RAY : PS_DONE;
                    }
                }
                // LightSourceVisibilityCheck (src/shader.comp:1121-1205): the light sample counts
                // when the closest object along it is the light; an SDF closer than the
                // analytic hit sets the object index to -1
                if (shadow) {
                    ++shadows;
                    Hit sh;
                    sh.t = kMaxDist;
                    sid = closest_analytic(S, o, sd, sh);
                    st_t = sh.t;
                    if (SDF && march_start(S, o, sd, M)) {
                        shadow_ray = true;
                        st = PS_MARCH;
                    } else if (sid == lobj) {
                        L = f4{L.x + contrib.x, L.y + contrib.y, L.z + contrib.z, L.w + contrib.w};
                    }
                }
            }
        }
        if (SDF && st == PS_MARCH) {
            float mat;
            const float v = sdf_set<(KIND < 0 ? 0 : KIND)>(S, M.q, M.set, M.phase == MP_MATERIAL, mat);
            if (shadow_ray) {
                Hit sh;
                sh.t = st_t;
                const int r = march_advance<true>(S, o, sd, M, v, mat, sh, steps);
                if (r == 2) sid = -1;
                if (r != 0) st = PS_SHADOW;
            } else if (march_advance<false>(S, o, d, M, v, mat, h, steps) != 0) {
                st = PS_SHADE;
            }
        }
    }
    wave_add_u64(stat_slot(Wv.stats, 0), segments);
    wave_add_u64(stat_slot(Wv.stats, 1), shadows);
    if (SDF) wave_add_u64(stat_slot(Wv.stats, 2), steps);
    wave_add_u64(stat_slot(Wv.stats, 4), nans);
    // the last wave to end clears the cursors and the count for the next launch:
    // every other wave has taken its entries before it counted itself
    int last = 0;
    if (threadIdx.x == 0) {
        __threadfence();
        last = atomicAdd(Wv.cursor + kSeg * kCntStride, 1) == (int)gridDim.x - 1;
    }
    if (__builtin_amdgcn_readfirstlane(last)) {
        for (int j = (int)threadIdx.x; j <= kSeg; j += kRefLanes) Wv.cursor[j * kCntStride] = 0;
    }
}

// Per pixel, in sample order: the paths' XYZ added to the running sum
// (src/shader.comp:1513-1516); after the dispatch's last samples, the texel.
__global__ void __launch_bounds__(kBlock) k_ref_fold(RefFrame F, RefWave Wv, RefFinish Fin, float4* texels, int last) {
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= F.pc) return;
    f3 acc = mk3(0.0f, 0.0f, 0.0f);
    if (F.k0 != 0) acc = mk3(Wv.sum[j], Wv.sum[F.pc + j], Wv.sum[2 * F.pc + j]);
    for (int s = 0; s < F.m; ++s) {
        const float4 c = Wv.col[s * F.pc + j];
        acc = acc + mk3(c.x, c.y, c.z);
    }
    if (last) {
        texels[F.p0 + j] = finish_texel(Fin, acc, texels[F.p0 + j]);
    } else {
        Wv.sum[j] = acc.x;
        Wv.sum[F.pc + j] = acc.y;
        Wv.sum[2 * F.pc + j] = acc.z;
    }
}
// Zeroes the cursors of a wave (a kernel, not a memset).
__global__ void k_ref_clear(int* cursor) {
    for (int j = (int)threadIdx.x; j <= kSeg; j += blockDim.x) cursor[j * kCntStride] = 0;
}

// ---- host side ---------------------------------------------------------------------------
template <typename T>
static T* carve(char*& p, size_t n) {
    T* r = reinterpret_cast<T*>(p);
    p += ((n * sizeof(T) + 255) / 256) * 256;
    return r;
}

constexpr size_t round256(size_t bytes) { return ((bytes + 255) / 256) * 256; }
// Bytes of a wave of `cap` paths as carve_ref_wave lays it out.
constexpr size_t ref_wave_bytes(int cap) {
    return round256((size_t)(kSeg + 1) * kCntStride * 4)  // cursors, count of finished waves
           + round256((size_t)cap * 16)                    // XYZ by path
           + round256((size_t)cap * 12);                   // sums
}

// Lays a wave of `cap` paths out over `base` (ref_wave_bytes(cap) bytes). The
// cursors come first, at one place whatever the capacity.
static void carve_ref_wave(char* p, int cap, unsigned long long* stats, RefWave& W) {
    size_t n = (size_t)cap;
    W.cursor = carve<int>(p, (size_t)(kSeg + 1) * kCntStride);
    W.col = carve<float4>(p, n);
    W.sum = carve<float>(p, 3 * n);
    W.stats = stats;
    W.cap = cap;
}

static int ensure_ref_wave(pt_ctx* ctx, int cap) {
    if (ctx->ref_wave.cap >= cap && ctx->ref_mem.p) return PT_OK;
    dev_free(ctx, ctx->ref_mem);
    ctx->ref_wave = RefWave{};
    int st = dev_alloc(ctx, ctx->ref_mem, ref_wave_bytes(cap));
    if (st != PT_OK) return st;
    carve_ref_wave(static_cast<char*>(ctx->ref_mem.p), cap, ctx->d_stats, ctx->ref_wave);
    launch(ctx, "k_ref_clear", k_ref_clear, dim3(1), dim3(64), ctx->ref_wave.cursor);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? PT_OK : hip_fail(ctx, e, "reference wave");
}

// ---- the allocation-free dispatch's wave --------------------------------------------
// A wave of kStaticWavePaths paths in a static device array: pt_dispatch_noalloc
// traces through it instead of allocating. Each device holds its own copy for
// the life of the process. Every launch writes the records it reads, but for its
// cursors, which it expects and leaves at zero: a call clears them first. Calls that
// overlap on one device race on the wave, and what they leave in the cursors and the
// count of ended waves would otherwise stay there and drop paths of every later call (the
// clearing launch: 1 us of a call among others, 3 of one alone; 150x101x1 takes 80 and 87).
constexpr int kStaticWavePaths = 1 << 16;
constexpr size_t kStaticWaveBytes = ref_wave_bytes(kStaticWavePaths);  // 1,843,456 B
static __device__ __align__(256) char scratch[kStaticWaveBytes];
constexpr int kMaxStaticDevices = 64;
static std::mutex g_scratch_mu;
static char* g_scratch[kMaxStaticDevices] = {};

// Waves of k_ref_path that stay resident on a compute unit, by its KIND + 1
// (asked once per context, so that no dispatch asks while a stream is captured).
template <int... K>
static void resident_waves(pt_ctx* ctx, std::integer_sequence<int, K...>) {
    auto ask = [](auto kernel) {
        int n = 0;
        return hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, kRefLanes, 0) == hipSuccess && n > 0 ? n : 8;
    };
    ((ctx->ref_waves[K] = ask(k_ref_path<K - 1>)), ...);
}

int ref_static_setup(pt_ctx* ctx) {
    resident_waves(ctx, std::make_integer_sequence<int, 6>{});
    if (ctx->device < 0 || ctx->device >= kMaxStaticDevices) {
        ctx->err = "static dispatch wave: device ordinal beyond 63";
        return PT_ERR_CAPACITY;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch[ctx->device]) return PT_OK;
    void* ptr = nullptr;
    hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) return hip_fail(ctx, e != hipSuccess ? e : hipErrorInvalidSymbol, "static dispatch wave");
    g_scratch[ctx->device] = static_cast<char*>(ptr);
    return PT_OK;
}

void ref_wave_release(pt_ctx* ctx) {
    dev_free(ctx, ctx->ref_mem);
    ctx->ref_wave = RefWave{};
}

int ref_scene_upload(pt_ctx* ctx, pt_scene* s) {
    const float* u = reinterpret_cast<const float*>(&s->ubo);
    auto U = [&](int k) { return (k >= 0 && k < kUboFloats) ? u[k] : 0.0f; };
    auto ID = [&](int k) { return (float)((int)U(k) - 1); };
    int ns = (int)U(0), np = (int)U(1), nb = (int)U(2), nl = (int)U(3), nc = (int)U(4), nsdf = (int)U(5);
    if (ns < 0 || np < 0 || nb < 0 || nl < 0 || nc < 0 || nsdf < 0 || nsdf > PT_MAX_SDF_OBJECTS ||
        6 * ns + 5 * np + 11 * nb + 12 * nl + 16 * nc > PT_MAX_OBJECTS_SIZE || (size_t)nsdf != s->sdfs.size()) {
        ctx->err = "packed scene object counts are inconsistent with its arrays";
        return PT_ERR_INVALID_ARG;
    }
    std::vector<RefSphere> sph((size_t)ns);
    std::vector<RefPlane> pln((size_t)np);
    std::vector<RefBox> box((size_t)nb);
    std::vector<RefLens> lens((size_t)nl);
    std::vector<RefCyclide> cyc((size_t)nc);
    std::vector<RefSdf> sdf((size_t)nsdf);
    int off = kUboObj;
    for (int i = 0; i < ns; ++i, off += 6)
        sph[(size_t)i] = RefSphere{U(off), U(off + 1), U(off + 2), U(off + 3), ID(off + 4), ID(off + 5)};
    for (int i = 0; i < np; ++i, off += 5)
        pln[(size_t)i] = RefPlane{U(off), U(off + 1), U(off + 2), ID(off + 3), ID(off + 4)};
    for (int i = 0; i < nb; ++i, off += 11) {
        RefBox& b = box[(size_t)i];
        b.pos = mk3(U(off), U(off + 1), U(off + 2));
        b.M = rotation_deg(mk3(U(off + 3), U(off + 4), U(off + 5)));
        b.size = mk3(U(off + 6), U(off + 7), U(off + 8));
        b.bsr2 = 0.25f * dot(b.size, b.size);
        b.mat = ID(off + 9);
        b.light = ID(off + 10);
    }
    for (int i = 0; i < nl; ++i, off += 12) {
        RefLens& L = lens[(size_t)i];
        L.pos = mk3(U(off), U(off + 1), U(off + 2));
        L.M = rotation_deg(mk3(U(off + 3), U(off + 4), U(off + 5)));
        float r = U(off + 6), f = U(off + 7), th = U(off + 8);
        L.conv = U(off + 9) != 0.0f;
        L.mat = ID(off + 10);
        L.light = ID(off + 11);
        L.radius = r;
        L.half = 2.0f * f - sqrtf(4.0f * f * f - r * r);
        L.slicePos = 0.5f * (L.conv ? th : -th);
        if (L.conv) L.slicePos += L.half;
        L.twoF = 2.0f * f;
        if (L.conv) {
            L.br2 = (r * r) + (0.25f * th * th);
        } else {
            float br = 0.5f * th + 2.0f * f - sqrtf(4.0f * f * f - r * r);
            L.br2 = br * br + r * r;
        }
    }
    for (int i = 0; i < nc; ++i, off += 16) {
        RefCyclide& C = cyc[(size_t)i];
        C.pos = mk3(U(off), U(off + 1), U(off + 2));
        C.M = rotation_deg(mk3(U(off + 3), U(off + 4), U(off + 5)));
        C.scale = mk3(U(off + 6), U(off + 7), U(off + 8));
        C.a = U(off + 9); C.b = U(off + 10); C.c = U(off + 11); C.d = U(off + 12);
        C.brad2 = U(off + 13);
        C.mat = ID(off + 14);
        C.light = ID(off + 15);
    }
    int kind = -1;
    for (int i = 0; i < nsdf; ++i) {
        RefSdf& q = sdf[(size_t)i];
        int k = kUboSdf + 6 * i;
        q.pos = mk3(U(k), U(k + 1), U(k + 2));
        q.size = mk3(U(k + 3), U(k + 4), U(k + 5));
        q.d = s->sdfs[(size_t)i];
        if (q.d.kind < PT_SDF_MANDELBULB || q.d.kind > PT_SDF_TERRAIN || q.d.iterations < 0 || q.d.iterations > 64) {
            ctx->err = "sdf descriptor " + std::to_string(i) + " has an unknown kind or iteration count";
            return PT_ERR_UNSUPPORTED_SDF;
        }
        kind = (kind == -1 || kind == q.d.kind) ? q.d.kind : 0;
    }
    std::vector<float> peak((size_t)kRefLights);
    for (int i = 0; i < kRefLights; ++i) peak[(size_t)i] = wien_peak(U(kUboLight + 2 * i));
    size_t bytes = 0;
    auto sz = [&](size_t b) { bytes += round256(b); };
    sz(sizeof(pt_packed_scene)); sz(peak.size() * sizeof(float)); sz(sph.size() * sizeof(RefSphere)); sz(pln.size() * sizeof(RefPlane));
    sz(box.size() * sizeof(RefBox)); sz(lens.size() * sizeof(RefLens)); sz(cyc.size() * sizeof(RefCyclide));
    sz(sdf.size() * sizeof(RefSdf));
    dev_free(ctx, s->ref_mem);
    int st = dev_alloc(ctx, s->ref_mem, bytes);
    if (st != PT_OK) return st;
    // the tables laid out on the host, in one copy
    std::vector<char> host(bytes);
    char* base = static_cast<char*>(s->ref_mem.p);
    size_t at = 0;
    auto put = [&](const void* src, size_t b) -> void* {
        if (b) std::memcpy(host.data() + at, src, b);
        void* dst = base + at;
        at += round256(b);
        return dst;
    };
    RefSceneDev& D = s->ref_dev;
    D.ubo = static_cast<const float*>(put(&s->ubo, sizeof(pt_packed_scene)));
    D.peak = static_cast<const float*>(put(peak.data(), peak.size() * sizeof(float)));
    D.sph = static_cast<const RefSphere*>(put(sph.data(), sph.size() * sizeof(RefSphere)));
    D.pln = static_cast<const RefPlane*>(put(pln.data(), pln.size() * sizeof(RefPlane)));
    D.box = static_cast<const RefBox*>(put(box.data(), box.size() * sizeof(RefBox)));
    D.lens = static_cast<const RefLens*>(put(lens.data(), lens.size() * sizeof(RefLens)));
    D.cyc = static_cast<const RefCyclide*>(put(cyc.data(), cyc.size() * sizeof(RefCyclide)));
    D.sdf = static_cast<const RefSdf*>(put(sdf.data(), sdf.size() * sizeof(RefSdf)));
    hipError_t e = hipMemcpy(base, host.data(), at, hipMemcpyHostToDevice);
    if (e != hipSuccess) return hip_fail(ctx, e, "scene upload");
    D.ns = ns; D.np = np; D.nb = nb; D.nl = nl; D.nc = nc; D.nsdf = nsdf;
    D.numLights = U(6);
    D.sdf_kind = kind < 0 ? 0 : kind;
    s->device_bytes += (int64_t)bytes;
    return PT_OK;
}

static RefFrame make_frame(const pt_push_constants* pc) {
    RefFrame F{};
    F.W = pc->resolution[0];
    F.H = pc->resolution[1];
    F.frame = pc->frame;
    F.spf = pc->samplesPerFrame;
    F.pathLength = pc->pathLength;
    F.camSize = pc->cameraSize;
    F.apSize = pc->apertureSize;
    F.apDist = pc->apertureDist;
    F.camPos = mk3(pc->cameraPosX, pc->cameraPosY, pc->cameraPosZ);
    F.camM = rotation_deg(mk3(pc->cameraAngle[0], pc->cameraAngle[1], 0.0f));
    F.fwd = mk3(F.camM.c0.z, F.camM.c1.z, F.camM.c2.z);
    // The camera lens object of TracePathLens (src/shader.comp:1411-1418).
    F.lensPos = F.camPos + F.fwd * pc->lensDistance;
    F.lensM = rotation_deg(mk3(0.0f, 90.0f - pc->cameraAngle[1], pc->cameraAngle[0]));
    float r = pc->lensRadius, f = pc->lensFocalLength;
    F.lensRadius = r;
    F.lensHalf = 2.0f * f - sqrtf(4.0f * f * f - r * r);
    F.lensSlicePos = 0.5f * pc->lensThickness;
    F.lensSlicePos += F.lensHalf;
    F.lensTwoF = 2.0f * f;
    return F;
}

template <int KIND>
static void launch_path(pt_ctx* ctx, const RefSceneDev& S, const RefFrame& F, RefWave& W, const RefFinish& Fin,
                        float4* texels, int direct, int count) {
    // as many waves as stay resident, at most one per 64 paths
    const int grid = std::max(1, std::min((F.pc * F.m + kRefLanes - 1) / kRefLanes, ctx->cus * ctx->ref_waves[KIND + 1]));
    launch(ctx, "k_ref_path", k_ref_path<KIND>, dim3(grid), dim3(kRefLanes), S, F, W, Fin, texels, direct, count);
}

// One dispatch through the wave Wv (capacity Wv.cap paths): pixels in chunks of
// at most cap, each chunk's samples in waves that fill it.
static int ref_dispatch_wave(pt_ctx* ctx, const pt_scene* s, pt_accum* acc, const pt_push_constants* pc, RefWave& Wv) {
    const RefSceneDev& S = s->ref_dev;
    const int W = pc->resolution[0], H = pc->resolution[1];
    const int P = W * H;
    const int cap = Wv.cap;
    RefFrame F = make_frame(pc);
    RefFinish Fin{};
    Fin.spf = pc->samplesPerFrame;
    Fin.currentSamples = pc->currentSamples;
    Fin.frame = pc->frame;
    Fin.ISO = pc->ISO;
    Fin.apSize = pc->apertureSize;
    Fin.FPS = pc->FPS;
    Fin.persistence = pc->persistence;
    float4* texels = reinterpret_cast<float4*>(acc->d_texels);
    const int direct = pc->samplesPerFrame == 1;
    const int pcmax = std::min(P, cap);
    for (int p0 = 0; p0 < P; p0 += pcmax) {
        const int pcur = std::min(pcmax, P - p0);
        const int m = std::max(1, std::min(pc->samplesPerFrame, cap / pcur));
        for (int k0 = 0; k0 < pc->samplesPerFrame; k0 += m) {
            F.p0 = p0;
            F.pc = pcur;
            F.k0 = k0;
            F.m = std::min(m, pc->samplesPerFrame - k0);
            const int count = p0 == 0 && k0 == 0;
            switch (S.nsdf > 0 ? S.sdf_kind : -1) {
                case -1: launch_path<-1>(ctx, S, F, Wv, Fin, texels, direct, count); break;
                case PT_SDF_MANDELBULB: launch_path<PT_SDF_MANDELBULB>(ctx, S, F, Wv, Fin, texels, direct, count); break;
                case PT_SDF_MENGER: launch_path<PT_SDF_MENGER>(ctx, S, F, Wv, Fin, texels, direct, count); break;
                case PT_SDF_BLOB: launch_path<PT_SDF_BLOB>(ctx, S, F, Wv, Fin, texels, direct, count); break;
                case PT_SDF_TERRAIN: launch_path<PT_SDF_TERRAIN>(ctx, S, F, Wv, Fin, texels, direct, count); break;
                default: launch_path<0>(ctx, S, F, Wv, Fin, texels, direct, count); break;
            }
            if (!direct)
                launch(ctx, "k_ref_fold", k_ref_fold, dim3((F.pc + kBlock - 1) / kBlock), dim3(kBlock), F, Wv, Fin,
                       texels, (int)(k0 + m >= pc->samplesPerFrame));
        }
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_fail(ctx, e, "reference dispatch launch");
    return PT_OK;
}

// Default paths per wave: one wave for all but the largest dispatches (28 bytes a path,
// 235 MB). It is made whole by a context's first dispatch, so that a larger one later
// neither allocates nor waits for the device (64x48x2 to 1920x1080x2 in five steps, the wave
// grown at each: 12, 74, 93, 309, 1044 us of the calling thread; made once: 84, then 6).
// Under a budget, or when there is no room for all of it, it grows as dispatches need.
constexpr int64_t kRefWavePaths = (int64_t)1 << 23;

int ref_dispatch(pt_ctx* ctx, const pt_scene* s, pt_accum* acc, const pt_push_constants* pc) {
    int64_t cap = ctx->cfg.wave_paths > 0 ? ctx->cfg.wave_paths : kRefWavePaths;
    const int64_t usual = std::max<int64_t>(std::min(cap, kRefWavePaths), 1024);
    cap = std::min(cap, (int64_t)pc->resolution[0] * pc->resolution[1] * pc->samplesPerFrame);
    cap = std::max<int64_t>(cap, 1024);
    if (!ctx->ref_mem.p && ctx->cfg.hbm_budget <= 0 && cap < usual) {
        const std::string err = ctx->err;
        if (ensure_ref_wave(ctx, (int)usual) != PT_OK) {
            (void)hipGetLastError();
            ctx->err = err;
        }
    }
    int st = ensure_ref_wave(ctx, (int)cap);
    if (st != PT_OK) return st;
    RefWave Wv = ctx->ref_wave;
    Wv.cap = (int)cap;  // a larger wave than this dispatch asks for is kept
    return ref_dispatch_wave(ctx, s, acc, pc, Wv);
}

int ref_dispatch_static(pt_ctx* ctx, const pt_scene* s, pt_accum* acc, const pt_push_constants* pc) {
    char* base = nullptr;
    if (ctx->device >= 0 && ctx->device < kMaxStaticDevices) {
        std::lock_guard<std::mutex> lock(g_scratch_mu);
        base = g_scratch[ctx->device];
    }
    if (!base) {
        ctx->err = "pt_dispatch_noalloc: the static wave of this device is not set up";
        return PT_ERR_STATE;
    }
    RefWave Wv{};
    carve_ref_wave(base, kStaticWavePaths, ctx->d_stats, Wv);
    launch(ctx, "k_ref_clear", k_ref_clear, dim3(1), dim3(64), Wv.cursor);
    return ref_dispatch_wave(ctx, s, acc, pc, Wv);
}

}  // namespace ptk
