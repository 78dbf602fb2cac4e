// render.hip -- HIP kernels for gfx950 (MI355X): BIRP's per-pixel ray generation, fixed-step
// march through the emissivity cube (or the analytic CMEM model) and per-ray integration
// (reference Camera.cpp:140-229, DataCube.cpp:203-277, Cmem.cpp:117-288), plus the layout
// builders the renders read from.
//
// Two arithmetic families:
//  * exact  -- FP32 in the reference's operation order (no FMA contraction: the file is built
//              with -ffp-contract=off), correctly rounded divisions and the scale chain in the
//              short forms of exact_math.h, std::lerp's branch structure, and the image sum
//              in k order. Bit-identical to the reference CPU render for finite cubes.
//  * fast   -- FP64 camera basis, ray origin and cube entry; FP32 FMA march in index space;
//              BF16/F16/FP32 storage; sums in FP64 (signed cubes and CMEM: FP32 Kahan sums), rounded once.
//              Many views in one launch.
//
// Wave mapping: a wave64 owns a tile of 64/S rays; S lanes ("sub-lanes") share one ray and take
// its samples k = kb + sub, kb advancing by S each trip. In the exact kernels every sub-lane then
// reads its ray's other samples through DPP operands and all of them add the S samples
// in k order, so the sequential FP32 sum of the reference is kept while S lanes sample in
// parallel. A masked-off sample contributes -0.0f, which leaves every partial sum unchanged.
//
// Memory safety: cube records are read with buffer loads whose descriptor carries the buffer's
// byte size, so the hardware returns 0 for any offset past the end; indices are clamped before
// the tables are read.
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include <type_traits>

#include "../../include/birp.h"
#include "birp_internal.h"
#include "exact_math.h"

namespace birp {

#define BIRP_BLOCK 256
#define BIRP_MAX_EXACT_SAMPLES 8192
#define BIRP_FAST_TAB 2048  // largest LDS table of the fast kernels (nx+ny+nz entries)
#define BIRP_RSRC_WORD3 0x00020000

// ------------------------------------------------------------------------------------------
// small device helpers
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ int lane_id() { return __lane_id(); }

__device__ __forceinline__ int wave_min_i(int v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o, 64));
    return __builtin_amdgcn_readfirstlane(v);
}
__device__ __forceinline__ int wave_max_i(int v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
    return __builtin_amdgcn_readfirstlane(v);
}
__device__ __forceinline__ unsigned wave_sum_u(unsigned v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// DPP row_shl:N: lane l receives lane l + N of its 16-lane row (0 past the row's end). With
// the exact kernels' lane layout, sub-lane 0 of a ray reads its sub-lane m at N = 4m.
template <int N>
__device__ __forceinline__ int row_next(int v) {
    if constexpr (N == 0) return v;
    else return __builtin_amdgcn_update_dpp(0, v, 0x100 + N, 0xF, 0xF, true);
}
template <int N>
__device__ __forceinline__ float row_next_f(float v) {
    return __int_as_float(row_next<N>(__float_as_int(v)));
}

// std::lerp (libstdc++ 11, cmath:1894-1908) for any finite or non-finite input.
__device__ __forceinline__ float lerp_general(float a, float b, float t) {
    bool straddle = (a <= 0 && b >= 0) || (a >= 0 && b <= 0);
    float s1 = t * b + (1 - t) * a;
    float x = a + t * (b - a);
    float r = ((t > 1) == (b > a)) ? (b < x ? x : b) : (b > x ? x : b);
    r = (t == 1) ? b : r;
    return straddle ? s1 : r;
}

// std::lerp for finite a, b and 0 <= t <= 1 - 2^-24 (no clamp: birp_lerp_unit); a and b straddle
// zero, or one of them is zero, exactly when the median of a, b and 0 is 0.
__device__ __forceinline__ float lerp_finite(float a, float b, float t) {
    const float s = t * b + (1 - t) * a;
    return __builtin_amdgcn_fmed3f(a, b, 0.0f) == 0.0f ? s : birp_lerp_unit(a, b, t);
}

// The same for a, b >= +0: a straddling pair holds a zero, t b + (1 - t) a is then exact in its zero
// term, and for a = 0 it is what birp_lerp_unit gives.
__device__ __forceinline__ float lerp_nonneg(float a, float b, float t) {
    return b == 0.0f ? (1 - t) * a : birp_lerp_unit(a, b, t);
}

// Clamp in the float domain to [0, hi], then convert (NaN -> 0 in hardware).
__device__ __forceinline__ int to_index(float x, float hi) { return (int)__builtin_amdgcn_fmed3f(x, 0.0f, hi); }

// a + b + c in one instruction (two sums that share a + b would otherwise take three)
__device__ __forceinline__ unsigned add3(unsigned a, unsigned b, unsigned c) {
    unsigned r;
    asm("v_add3_u32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* p, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, BIRP_RSRC_WORD3);
}
__device__ __forceinline__ float4 load16(__amdgpu_buffer_rsrc_t r, unsigned off) {
    auto v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0);
    float4 f;
    __builtin_memcpy(&f, &v, 16);
    return f;
}
__device__ __forceinline__ uint4 load16u(__amdgpu_buffer_rsrc_t r, unsigned off) {
    auto v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0);
    uint4 f;
    __builtin_memcpy(&f, &v, 16);
    return f;
}

// 1/x and 1/sqrt(x) in double from the hardware's first approximations (within about 2^-23) and two Newton
// steps each: within an ulp or two, a third of the IEEE sequences' instructions. x finite, normal, not 0.
__device__ __forceinline__ double rcp64(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
    return __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
}
__device__ __forceinline__ double rsqrt64(double x) {
    double r = __builtin_amdgcn_rsq(x);
    r = __builtin_fma(__builtin_fma(-0.5 * x * r, r, 0.5), r, r);
    return __builtin_fma(__builtin_fma(-0.5 * x * r, r, 0.5), r, r);
}

// ------------------------------------------------------------------------------------------
// exact per-pixel ray (Camera.cpp:148-168), FP32 IEEE operations in the reference's order
// ------------------------------------------------------------------------------------------
// Its quotients by one divisor are RN64 products with the divisor's FP64 reciprocal (rcp64's last ulp leaves
// birp_div_rn64's margin of 2^-49 whole), a third of the IEEE sequences' instructions; a dividend so
// small that the quotient could leave the normal floats takes those.
__device__ __forceinline__ void div3(float a, float b, float c, float d, float& x, float& y, float& z) {
    const double r = rcp64((double)d);
    const float m = fminf(fminf(fabsf(a), fabsf(b)), fabsf(c));
    x = birp_div_rn64(a, r);
    y = birp_div_rn64(b, r);
    z = birp_div_rn64(c, r);
    if (__builtin_expect(m < 0x1p-60f, 0)) {
        x = a / d;
        y = b / d;
        z = c / d;
    }
}
__device__ __forceinline__ void exact_ray_dir(const ExactView& ev, int i, int j, float& dx, float& dy, float& dz) {
    float device_x = birp_div_rn64((float)i + 0.5f, ev.inv_w);
    float device_y = birp_div_rn64((float)j + 0.5f, ev.inv_h);
    float screen_x = ((2 * device_x) - 1) * ev.tanx * ev.aspect;
    float screen_y = (1 - (2 * device_y)) * ev.tany;
    float nd = sqrtf(screen_x * screen_x + screen_y * screen_y + (-1.0f) * (-1.0f));
    float ux, uy, uz;
    div3(screen_x, screen_y, -1.0f, nd, ux, uy, uz);
    float w0 = (ev.rinv[0] * ux) + (ev.rinv[1] * uy) + (ev.rinv[2] * uz);
    float w1 = (ev.rinv[3] * ux) + (ev.rinv[4] * uy) + (ev.rinv[5] * uz);
    float w2 = (ev.rinv[6] * ux) + (ev.rinv[7] * uy) + (ev.rinv[8] * uz);
    float wd = sqrtf(w0 * w0 + w1 * w1 + w2 * w2);
    div3(w0, w1, w2, wd, dx, dy, dz);
}

// Index of the sample point on each axis: RN(RN(RN(d t) + p) - o) / s), exactly.
struct ExactIdx {
    float xi, yi, zi;  // ingress
    float xd, yd, zd;  // index
};

// DIV_GUARD: the double-product division is exact while the quotient is a normal float, which
// holds for |ingress| >= 2^-64 (spacing <= 2^30); below that (possible only when an origin
// component is within 2^-30 of 0) the IEEE division is used.
// DIV_FMA2: the divisions as birp_div_fma2 (volumes whose spacings passed the upload's check; |origin|
// >= 2^-30, so a nonzero ingress is at least 2^-56 and a rl stays normal).
enum DivForm { DIV_GUARD = 0, DIV_RN64 = 1, DIV_FMA2 = 2 };
template <int DIV>
__device__ __forceinline__ ExactIdx exact_index(const DevVolume& v, float dx, float dy, float dz, float px, float py,
                                                float pz, float t) {
    ExactIdx r;
    float x = dx * t + px;
    float y = dy * t + py;
    float z = dz * t + pz;
    r.xi = x - v.ox;
    r.yi = y - v.oy;
    r.zi = z - v.oz;
    if constexpr (DIV == DIV_FMA2) {
        r.xd = birp_div_fma2(r.xi, v.rhx, v.rlx);
        r.yd = birp_div_fma2(r.yi, v.rhy, v.rly);
        r.zd = birp_div_fma2(r.zi, v.rhz, v.rlz);
        return r;
    }
    if constexpr (DIV == DIV_GUARD) {
        float m = fminf(fminf(fabsf(r.xi), fabsf(r.yi)), fabsf(r.zi));
        if (__builtin_expect(m < 0x1p-64f && m != 0.0f, 0)) {
            r.xd = r.xi / v.sx;
            r.yd = r.yi / v.sy;
            r.zd = r.zi / v.sz;
            return r;
        }
    }
    r.xd = birp_div_rn64(r.xi, v.rdx);
    r.yd = birp_div_rn64(r.yi, v.rdy);
    r.zd = birp_div_rn64(r.zi, v.rdz);
    return r;
}

// DataCube.cpp:214-218 negated: inside iff ingress >= 0 and index + 1 < n on every axis.
// (NaN compares false here and counts as outside; the reference would index out of range.)
__device__ __forceinline__ bool exact_inside(const DevVolume& v, const ExactIdx& r) {
    return (r.xi >= 0) && (r.xd + 1 < v.fnx) && (r.yi >= 0) && (r.yd + 1 < v.fny) && (r.zi >= 0) &&
           (r.zd + 1 < v.fnz);
}

// Trilinear sample from quad records (finite cubes) through the per-axis offset tables. Corner
// x1 = x0 + 1 always: for finite data std::lerp at t == 0 returns a, so this equals DataCube's
// ceil() corner choice.
struct QuadCtx {
    __amdgpu_buffer_rsrc_t rs;
    const unsigned* tx;
    const unsigned* ty;
    const unsigned* tz;
    float hx, hy, hz;  // n - 2 per axis
    unsigned row, slice;  // nearest: nx and nx ny, rs the [z][y][x] copy
};

// For an in-cube sample the index is >= 0, so the lower corner floor(x) is the truncating
// conversion of the clamped index (the clamp only matters to lanes outside the cube, whose
// result is discarded) and the weight x - floor(x) is v_fract_f32 (exact: the subtraction of
// floor(x) from x >= 0 is exact, so fract's clamp below 1.0 never applies).
struct QuadFetch {
    float4 a, b;       // the z and z+1 quad records
    float fx, fy, fz;  // lerp weights
};

__device__ __forceinline__ QuadFetch quad_fetch(const QuadCtx& c, float xd, float yd, float zd) {
    QuadFetch q;
    q.fx = __builtin_amdgcn_fractf(xd);
    q.fy = __builtin_amdgcn_fractf(yd);
    q.fz = __builtin_amdgcn_fractf(zd);
    const unsigned xo = c.tx[to_index(xd, c.hx)], yo = c.ty[to_index(yd, c.hy)];
    const unsigned* zo = c.tz + to_index(zd, c.hz);
    q.a = load16(c.rs, add3(xo, yo, zo[0]));
    q.b = load16(c.rs, add3(xo, yo, zo[1]));
    return q;
}

// Nearest (DataCube.cpp:273) of a sample that passed the reference's bounds test: the value at the
// truncated index, from the [z][y][x] copy (nx ny < 2^24 and under 2^30 values: exact_mode_of).
__device__ __forceinline__ float near_fetch(const QuadCtx& c, float xd, float yd, float zd) {
    const unsigned at = __umul24((unsigned)(int)zd, c.slice) + (__umul24((unsigned)(int)yd, c.row) + (unsigned)(int)xd);
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(c.rs, (int)(at * 4u), 0, 0));
}

// For a sample that passed the reference's bounds test (0 <= ingress, index + 1 < n): the index
// is in [0, n-1), so its truncation is the lower corner and needs no clamp.
__device__ __forceinline__ QuadFetch quad_fetch_inside(const QuadCtx& c, float xd, float yd, float zd) {
    QuadFetch q;
    q.fx = __builtin_amdgcn_fractf(xd);
    q.fy = __builtin_amdgcn_fractf(yd);
    q.fz = __builtin_amdgcn_fractf(zd);
    const unsigned xo = c.tx[(int)xd], yo = c.ty[(int)yd];
    const unsigned* zo = c.tz + (int)zd;
    q.a = load16(c.rs, add3(xo, yo, zo[0]));
    q.b = load16(c.rs, add3(xo, yo, zo[1]));
    return q;
}

// x first, then y, then z (DataCube.cpp:260-270).
enum LerpForm { LERP_POS, LERP_NONNEG, LERP_FINITE };
template <int LERP>
__device__ __forceinline__ float quad_lerp(const QuadFetch& q) {
    auto lerp = [](float a, float b, float t) {
        return LERP == LERP_POS ? birp_lerp_unit(a, b, t) : LERP == LERP_NONNEG ? lerp_nonneg(a, b, t) : lerp_finite(a, b, t);
    };
    const float4 a = q.a, b = q.b;
    const float ly = lerp(lerp(a.x, a.y, q.fx), lerp(a.z, a.w, q.fx), q.fy);
    const float hy = lerp(lerp(b.x, b.y, q.fx), lerp(b.z, b.w, q.fx), q.fy);
    return lerp(ly, hy, q.fz);
}

// The least (or, MAX, the greatest) corner of a cell without negative values, as its bits.
template <bool MAX>
__device__ __forceinline__ unsigned fold_corners(const QuadFetch& q) {
    auto f = [](float x, float y, float z) {
        const unsigned a = __float_as_uint(x), b = __float_as_uint(y), c = __float_as_uint(z);
        return __uint_as_float(MAX ? max(max(a, b), c) : min(min(a, b), c));
    };
    const float m = f(q.a.x, q.a.y, q.a.z), n = f(q.a.w, q.b.x, q.b.y);
    return __float_as_uint(f(f(m, n, q.b.z), q.b.w, q.b.w));
}

// The scale chain of Camera.cpp:201 for a positive cube whose scaled samples stay normal floats:
// the folded product, unless it lies within 16 double ulps of a float rounding midpoint.
// The chain is taken by about one sample in 10^7: it must stay a branch (if-converted, its two
// FP64 divisions would run for every sample).
// The test |m29 - 2^28| <= 16 on the low 29 mantissa bits m29 is done on m29 * 8 (the low word
// shifted left by 3): m29 * 8 + 2^31 + 128 wraps into [0, 256] exactly when it holds.
__device__ __forceinline__ float scale_pos(float vw) {
    double y = (double)vw * BIRP_SCALE_FOLDED;
    const uint32_t lo = (uint32_t)birp_f64_bits(y);
    float s = (float)y;
    if (__builtin_expect((lo << 3) + 0x80000080u < 257u, 0)) s = birp_scale_chain(vw);
    return s;
}

// The scale chain for any value: the FMA form in its range and for +0, else the tested or literal chain.
__device__ __forceinline__ float scale_any(float vw) {
    float s = birp_scale_fma2(vw);
    const float a = fabsf(vw);
    if (__builtin_expect(!(a >= 0x1p-100f && a <= 0x1p110f) && __float_as_uint(vw) != 0u, 0)) s = birp_scale_sample(vw);
    return s;
}

// acc += the S sub-lane samples of this ray, in sub-lane (= k) order. Exact on sub-lane 0 of
// the ray (the lane that stores the pixel); the other sub-lanes' sums are not used. With 8 lanes
// per ray the ray spans two 16-lane rows: sub-lanes 4..7 are read from the next row's copy.
template <int S>
__device__ __forceinline__ float add_in_order(float acc, float s) {
    acc = acc + s;
    if constexpr (S >= 2) acc = acc + row_next_f<4>(s);
    if constexpr (S >= 4) {
        acc = acc + row_next_f<8>(s);
        acc = acc + row_next_f<12>(s);
    }
#pragma unroll
    for (int r = 1; r < S / 4; ++r) {  // 8 and 16 lanes: sub-lanes 4r..4r+3 in row r
        const float sr = __shfl_down(s, 16 * r, 64);  // lane l + 16 r: row r's copy
        acc = acc + sr;
        acc = acc + row_next_f<4>(sr);
        acc = acc + row_next_f<8>(sr);
        acc = acc + row_next_f<12>(sr);
    }
    return acc;
}

// Sub-lane m's value of this ray, on sub-lane 0.
template <int S>
__device__ __forceinline__ float sub_lane_f(float s, int m) {
    if (m >= 4) s = __shfl_down(s, 16 * (m >> 2), 64);
    switch (m & 3) {
        case 1: return row_next_f<4>(s);
        case 2: return row_next_f<8>(s);
        case 3: return row_next_f<12>(s);
        default: return s;
    }
}

// Trilinear sample from the [z][y][x] layout with floor/ceil corners (DataCube.cpp:224-270):
// exact for any data, including inf/nan.
__device__ __forceinline__ float sample_linear_tri(const DevVolume& v, const ExactIdx& r) {
    float x0f = floorf(r.xd), y0f = floorf(r.yd), z0f = floorf(r.zd);
    float fx = r.xd - x0f, fy = r.yd - y0f, fz = r.zd - z0f;
    int x0 = to_index(x0f, v.fnx - 2), y0 = to_index(y0f, v.fny - 2), z0 = to_index(z0f, v.fnz - 2);
    int x1 = x0 + (fx > 0.0f ? 1 : 0), y1 = y0 + (fy > 0.0f ? 1 : 0), z1 = z0 + (fz > 0.0f ? 1 : 0);
    const float* L = v.linear;
    size_t sy = (size_t)v.nx, sz = (size_t)v.nx * (size_t)v.ny;
    float s000 = L[z0 * sz + y0 * sy + x0], s001 = L[z0 * sz + y0 * sy + x1];
    float s010 = L[z0 * sz + y1 * sy + x0], s011 = L[z0 * sz + y1 * sy + x1];
    float s100 = L[z1 * sz + y0 * sy + x0], s101 = L[z1 * sz + y0 * sy + x1];
    float s110 = L[z1 * sz + y1 * sy + x0], s111 = L[z1 * sz + y1 * sy + x1];
    float ly = lerp_general(lerp_general(s000, s001, fx), lerp_general(s010, s011, fx), fy);
    float hy = lerp_general(lerp_general(s100, s101, fx), lerp_general(s110, s111, fx), fy);
    return lerp_general(ly, hy, fz);
}

// Nearest: slices[(int)z][(int)y][(int)x] (DataCube.cpp:273), truncation.
__device__ __forceinline__ float sample_linear_nearest(const DevVolume& v, const ExactIdx& r) {
    int x = to_index(truncf(r.xd), v.fnx - 2), y = to_index(truncf(r.yd), v.fny - 2), z = to_index(truncf(r.zd), v.fnz - 2);
    return v.linear[((size_t)z * v.ny + y) * v.nx + x];
}

// ------------------------------------------------------------------------------------------
// CMEM::GetSample (Cmem.cpp:117-288) on the device: the reference's float/double types and
// order; the transcendental functions are ROCm's device libm (within ~1 ulp of glibc's) and, for the sheath's
// power, birp_powf.
// ------------------------------------------------------------------------------------------
// (float)acos(c) for a double c, to float accuracy without an FP64 arc cosine: acos(c) =
// 2 asin(sqrt((1 - c) / 2)) for c >= 0 and pi - 2 asin(sqrt((1 + c) / 2)) below, with 1 -/+ c formed
// in double (exact near the ends, where acos is steep) and the rest in float; within a few float
// ulps of the double arc cosine rounded to float. |c| > 1 gives NaN (a negative square root), as
// acos does.
__device__ __forceinline__ float acos_to_float(double c) {
    if (c >= 0.0) return 2.0f * asinf(sqrtf((float)((1.0 - c) * 0.5)));
    return 3.14159265358979323846f - 2.0f * asinf(sqrtf((float)((1.0 + c) * 0.5)));
}

// Emissivity outside the bow shock (Cmem.cpp:172-175) and in the sheath (:148-152).
__device__ __forceinline__ float cmem_outer(const CmemParams& m, float r) {
    double sd = birp_div_rn64(r, 0.1);
    return (float)(m.A2 * (1 / (sd * sd * sd)));
}
__device__ __forceinline__ float cmem_inner(const CmemParams& m, float r, float theta, float st) {
    float half_t = theta / 2;
    const float sd = birp_div_rn64(r, 0.1), e = -m.alpha - (m.beta * (st * st));
    const float fall = birp_powf_takes(sd, e) ? birp_powf(sd, e) : powf(sd, e);
    return m.A1 * (expf(-m.B * (half_t * half_t * half_t * half_t))) * fall;
}

// The magnetopause's radius in a direction (LinScaled, Cmem.cpp:188-222): ct, st and cos_phi, sin_phi of its
// angles, theta itself.
__device__ __forceinline__ float cmem_mp(const CmemParams& m, float ct, float st, float theta, float cos_phi, float sin_phi, float y, float z) {
    // cos(phi - pi/2) and cos(phi - 3 pi/2) in double (Cmem.cpp:205, 209) are sin(phi) and
    // -sin(phi), formed here in double from the coordinates
    const double sphi = (y != 0) ? (double)fabsf(z) / sqrt((double)y * y + (double)z * z) : 0.0;
    float phi_n = acos_to_float((double)(ct * m.cos_theta_n) + (double)(st * m.sin_theta_n) * sphi);
    float phi_s = acos_to_float((double)(ct * m.cos_theta_s) + (double)(st * m.sin_theta_s) * -sphi);
    float f = powf(cosf(theta / 2) + m.a5 * sinf(2 * theta) * (1 - expf(-theta)),
                   (m.p1 * (m.beta_c[0] + m.beta_c[1] * cos_phi + m.beta_c[3] * (sin_phi * sin_phi))));
    float q = m.p2 * m.charlie * expf(m.p3 * m.dn * (powf(phi_n, m.a21))) +
              m.p2 * m.charlie * expf(m.p3 * m.ds * (powf(phi_s, m.a21)));
    return m.p0 * m.r0_lin * f + q;
}

// The bow shock's (ShueModel, Cmem.cpp:280-288).
__device__ __forceinline__ float cmem_bs(const CmemParams& m, float ct, float cos_phi, float sin_phi) {
    float base = 2 / (1 + ct);
    float ry = m.bs * powf(base, m.ay_bs);
    float rz = (m.az_bs == m.ay_bs) ? ry : m.bs * powf(base, m.az_bs);  // equal unless set apart
    float rzc = rz * cos_phi, rys = ry * sin_phi;
    return (ry * rz) / sqrtf((rzc * rzc) + (rys * rys));
}

// ask_mp, ask_bs: false where the point is known to lie outside the magnetopause (beyond its band), inside the bow
// shock (below its band).
__device__ __forceinline__ float cmem_sample(const CmemParams& m, float x, float y, float z, bool ask_mp = true, bool ask_bs = true) {
    float r = sqrtf(x * x + y * y + z * z);
    const float ryz = sqrtf(y * y + z * z);
    float theta = (x != 0) ? acosf(x / r) : 0.f;
    // phi = acos(y / ryz) (0 when y == 0) enters only through its cosine and sine, and theta's
    // cosine and sine are needed too: all four from the ratios that are their arc cosines' arguments
    // (theta, phi in [0, pi], so both sines are >= 0; x == 0 and y == 0 give the reference's angle
    // 0), within an ulp or two of cos(acos(u)) and sin(acos(u)), with no trigonometric call
    const float ct = (x != 0) ? x / r : 1.f, st = (x != 0) ? ryz / r : 0.f;
    const float cos_phi = (y != 0) ? y / ryz : 1.f, sin_phi = (y != 0) ? fabsf(z) / ryz : 0.f;
    // the reference's zone tests in its order (Cmem.cpp:136-176); the sheath emissivity is
    // evaluated only for the three zones that use it
    const float h = 0.05f / 2;
    bool z_mp = false, past = true;
    float norm = 0.f;
    if (ask_mp) {
        const float radius_mp = cmem_mp(m, ct, st, theta, cos_phi, sin_phi, y, z);
        if (r < radius_mp - h) return 0;  // inside the magnetopause: the bow shock is not needed
        z_mp = r >= radius_mp - h && r <= radius_mp + h;
        past = r > radius_mp + h;
        norm = (r - (radius_mp - h)) / (radius_mp + h);
    }
    bool z_sheath = !z_mp && past, z_bs = false;
    if (ask_bs && !z_mp) {
        const float radius_bs = cmem_bs(m, ct, cos_phi, sin_phi);
        z_sheath = past && r < radius_bs - h;
        z_bs = !z_sheath && r >= radius_bs - h && r <= radius_bs + h;
        norm = (r - (radius_bs - h)) / (radius_bs + h);
    }
    if (!(z_mp || z_sheath || z_bs)) return cmem_outer(m, r);
    const float inner = cmem_inner(m, r, theta, st);
    if (z_sheath) return inner;
    return lerp_general(z_mp ? 0.f : inner, z_mp ? inner : cmem_outer(m, r), norm);
}

// ------------------------------------------------------------------------------------------
// CMEM zone bounds (birp_internal.h): interval arithmetic in double over each cell's directions
// ------------------------------------------------------------------------------------------
struct Range {
    double lo, hi;
};
__device__ __forceinline__ Range operator+(Range a, Range b) { return {a.lo + b.lo, a.hi + b.hi}; }
__device__ __forceinline__ Range operator*(Range a, Range b) {
    const double p = a.lo * b.lo, q = a.lo * b.hi, r = a.hi * b.lo, s = a.hi * b.hi;
    return {fmin(fmin(p, q), fmin(r, s)), fmax(fmax(p, q), fmax(r, s))};
}
__device__ __forceinline__ Range operator*(double k, Range a) { return Range{k, k} * a; }
__device__ __forceinline__ Range range_exp(Range a) { return {exp(a.lo), exp(a.hi)}; }
// x^e for x >= 0: monotone in x (lo = 0 with e < 0 gives inf)
__device__ __forceinline__ Range range_pow(Range x, double e) {
    const double a = pow(x.lo, e), b = pow(x.hi, e);
    return {fmin(a, b), fmax(a, b)};
}

// Both arithmetics (cmem_sample's and cmem_fast's) must find the zone that the bounds name, so the bounds are
// wider than the ranges by more than their rounding: the cell's directions by 1e-5 (a direction's ct
// and cp are within 1e-6), the arc cosines' arguments by 2e-6, the radii by 1e-4 RE + 3e-5 of their terms
// (FP32 powers and exponentials are within 1e-5). Where the model leaves the reals or is too steep for that
// the cell bounds nothing: at the cusps, whose arc cosine's argument rounds past 1 in the reference
// (NaN), in the last cells of the tail, where 2 / (1 + ct) diverges and a power's base may be negative, where an
// exponent multiplies the rounding of its base beyond the slack, and where a product that is finite in double leaves
// FP32's range: with a bow shock exponent of 8.5 (10,000 particles per cm^3), ry rz does in the tail, and the
// reference's shock is NaN or 0 there.
__global__ __launch_bounds__(BIRP_BLOCK) void k_cmem_zones(CmemParams m, float4* zones) {
    const int cell = blockIdx.x * BIRP_BLOCK + threadIdx.x;
    if (cell >= BIRP_ZONE_CT * BIRP_ZONE_CP) return;
    const int iu = cell / BIRP_ZONE_CP, iv = cell % BIRP_ZONE_CP;
    const double wide = 1e-5;
    const Range ct{fmax(-1.0, iu * (2.0 / BIRP_ZONE_CT) - 1 - wide), fmin(1.0, (iu + 1) * (2.0 / BIRP_ZONE_CT) - 1 + wide)};
    const Range cp{fmax(-1.0, iv * (2.0 / BIRP_ZONE_CP) - 1 - wide), fmin(1.0, (iv + 1) * (2.0 / BIRP_ZONE_CP) - 1 + wide)};
    auto sine = [](Range c) {  // sqrt(1 - c^2)
        const double a = sqrt(fmax(0.0, 1 - c.lo * c.lo)), b = sqrt(fmax(0.0, 1 - c.hi * c.hi));
        return Range{fmin(a, b), c.lo <= 0 && c.hi >= 0 ? 1.0 : fmax(a, b)};
    };
    const Range theta{acos(ct.hi), acos(ct.lo)}, st = sine(ct), sp = sine(cp);
    bool known = ct.lo > -1 + 1e-3;
    // an angle to a cusp, in [0, pi]
    auto cusp_angle = [&](double c, double s) {
        const Range a = c * ct + s * (st * sp);
        const double near = 2e-3;  // of the cusp or the point opposite
        if (cp.lo <= near && cp.hi >= -near && ((ct.lo <= c + near && ct.hi >= c - near) || (ct.lo <= -c + near && ct.hi >= -c - near)))
            known = false;
        return Range{acos(fmin(1.0, a.hi + 2e-6)), acos(fmax(-1.0, a.lo - 2e-6))};
    };
    const Range north = cusp_angle(m.cos_theta_n, m.sin_theta_n), south = cusp_angle(m.cos_theta_s, -m.sin_theta_s);
    const Range grow{1 - exp(-theta.lo), 1 - exp(-theta.hi)}, half{cos(theta.hi / 2), cos(theta.lo / 2)};
    const Range base = half + (2.0 * m.a5) * (st * ct * grow);
    known = known && base.lo > 1e-4;
    const Range power = (double)m.p1 * (Range{m.beta_c[0], m.beta_c[0]} + (double)m.beta_c[1] * cp + (double)m.beta_c[3] * (sp * sp));
    auto within = [&](Range a, double least, double most) { known = known && fmin(fabs(a.lo), fabs(a.hi)) >= least && fmax(fabs(a.lo), fabs(a.hi)) <= most; };
    within(power, 0.0, 256.0);
    const Range f = range_exp(power * Range{log(fmax(base.lo, 1e-300)), log(fmax(base.hi, 1e-300))});
    const Range dip_n = range_exp(((double)m.p3 * m.dn) * range_pow(north, m.a21)), dip_s = range_exp(((double)m.p3 * m.ds) * range_pow(south, m.a21));
    for (Range a : {f, dip_n, dip_s}) within(a, 0.0, 0x1p100);
    const Range far = ((double)m.p0 * m.r0_lin) * f, q = ((double)m.p2 * m.charlie) * (dip_n + dip_s);
    const Range mp = far + q;
    const double mp_wide = 1e-4 + 3e-5 * (fmax(fabs(far.lo), fabs(far.hi)) + fmax(fabs(q.lo), fabs(q.hi)));
    const Range flare{2 / (1 + ct.hi), 2 / (1 + ct.lo)};
    const Range ry = (double)m.bs * range_pow(flare, m.ay_bs), rz = (double)m.bs * range_pow(flare, m.az_bs);
    known = known && m.bs > 0;
    within({m.ay_bs, m.az_bs}, 0.0, 64.0);
    for (Range a : {ry, rz}) within(a, 0x1p-60, 0x1p60);  // their products and squares
    Range bs = ry;  // with one exponent: ry / sqrt(cos^2 + sin^2)
    if (m.az_bs != m.ay_bs) {
        const Range u = rz * cp, w = ry * sp, n = ry * rz;
        const double lo = (cp.lo <= 0 && cp.hi >= 0 ? 0.0 : fmin(u.lo * u.lo, u.hi * u.hi)) + w.lo * w.lo;
        bs = Range{n.lo / sqrt(fmax(u.lo * u.lo, u.hi * u.hi) + w.hi * w.hi), n.hi / sqrt(lo)};
    }
    const double bs_wide = 1e-4 + 3e-5 * fmax(fabs(bs.lo), fabs(bs.hi)), h = 0.025;
    float4 t = make_float4((float)(mp.lo - h - mp_wide), (float)(mp.hi + h + mp_wide), (float)(bs.lo - h - bs_wide), (float)(bs.hi + h + bs_wide));
    known = known && isfinite(t.x) && isfinite(t.y) && isfinite(t.z) && isfinite(t.w);
    if (!known) t = make_float4(-INFINITY, INFINITY, -INFINITY, INFINITY);
    zones[cell] = t;
}

// What the bounds say of a point: its zone, or (SPLIT) which of the surfaces it takes to know (ZONE_EDGE: both;
// also for points on x = 0 or y = 0, where the reference takes an angle of 0, Cmem.cpp:224-246, and where |x y| is
// so small that r^2 may leave the normal floats, whose reciprocal root the hardware takes for 0's). y^2 + z^2 may
// leave them elsewhere too, beside the Sun's line: the surfaces are round there, and any cell that
// touches ct = 1 bounds them, so it does not matter which phi the query then finds.
enum Zone { ZONE_INSIDE, ZONE_OUTER, ZONE_SHEATH, ZONE_EDGE_MP, ZONE_EDGE_BS, ZONE_EDGE };
struct ZoneQuery {
    float4 t;
    float r, ir, iyz;  // |(x, y, z)| and the reciprocals of it and of |(y, z)|, to a few ulps
    bool axis;
};
__device__ __forceinline__ ZoneQuery zone_fetch(__amdgpu_buffer_rsrc_t rs, float x, float y, float z) {
    ZoneQuery q;
    const float yz2 = __builtin_fmaf(y, y, z * z), r2 = __builtin_fmaf(x, x, yz2);
    q.ir = __builtin_amdgcn_rsqf(r2);
    q.iyz = __builtin_amdgcn_rsqf(yz2);
    const float u = __builtin_fmaf(x * q.ir, 0.5f * BIRP_ZONE_CT, 0.5f * BIRP_ZONE_CT);
    const float v = __builtin_fmaf(y * q.iyz, 0.5f * BIRP_ZONE_CP, 0.5f * BIRP_ZONE_CP);
    const unsigned iu = (unsigned)__builtin_amdgcn_fmed3f(u, 0.0f, BIRP_ZONE_CT - 1.0f), iv = (unsigned)__builtin_amdgcn_fmed3f(v, 0.0f, BIRP_ZONE_CP - 1.0f);
    q.t = load16(rs, (iu * BIRP_ZONE_CP + iv) * 16u);
    q.r = r2 * q.ir;
    q.axis = !(fabsf(x * y) > 0x1p-60f);
    return q;
}
template <bool SPLIT>
__device__ __forceinline__ Zone zone_of(const ZoneQuery& q) {
    if (q.axis) return ZONE_EDGE;
    if (q.r < q.t.x) return ZONE_INSIDE;
    if (!(q.r > q.t.y)) return SPLIT && q.r < q.t.z ? ZONE_EDGE_MP : ZONE_EDGE;
    return q.r < q.t.z ? ZONE_SHEATH : q.r > q.t.w ? ZONE_OUTER : SPLIT ? ZONE_EDGE_BS : ZONE_EDGE;
}

// RN(sqrt(a)) from the query's estimate of 1 / sqrt(a), which is off by another rounding of a.
__device__ __forceinline__ float sqrt_from(float a, float y) {
    if (__builtin_expect(!(a >= 0x1p-96f), 0)) return sqrtf(a);
    return birp_sqrt_rn(a, y);
}

// cmem_sample with its surfaces left out where the bounds name the point's zone: the same value, bit for bit.
// The surfaces are the model's cost (about 900 of 1,100 VALU instructions per sample in libm calls) and a
// zone is all that most samples need of them: a query is 35 instructions and one 16-byte load. 576x336 x
// 800: 3.45 -> 0.62 ms; fast form 0.662 -> 0.264 ms. A table of half the cells per axis gives 0.67 and
// 0.270 ms, of twice 0.61 and 0.262 (2 MB): the cells on a surface are not what is left.
// The roots start from the query's reciprocals, the quotients by r share one in FP64, and the sheath's power
// is birp_powf: 0.62 -> 0.51 ms. birp_powf is within 0.502 ulp of the power, powf within 1.3.
// A sample near one surface takes that one only (about 900 instructions for the magnetopause, 200 for the bow
// shock; a trip's lanes seldom meet both): 0.505 -> 0.476 ms, 300x170 n = 300 103 -> 84 us, 144x84 n = 320
// 46 -> 38, the 8 views 0.325 -> 0.314 ms.
__device__ __forceinline__ float cmem_sample_zoned(const CmemParams& m, const ZoneQuery& q, float x, float y, float z) {
    const Zone zone = zone_of<true>(q);
    float val = 0.f;
    if (zone >= ZONE_EDGE_MP) {
        val = cmem_sample(m, x, y, z, zone != ZONE_EDGE_BS, zone != ZONE_EDGE_MP);
    } else if (zone != ZONE_INSIDE) {
        const float r = sqrt_from(x * x + y * y + z * z, q.ir);
        if (zone == ZONE_OUTER) {
            val = cmem_outer(m, r);
        } else {
            const double rc = rcp64((double)r);
            val = cmem_inner(m, r, acosf(birp_div_rn64(x, rc)), birp_div_rn64(sqrt_from(y * y + z * z, q.iyz), rc));
        }
    }
    return val;
}

// ------------------------------------------------------------------------------------------
// cube entry: a slab interval, widened by `margin`, mapped to a sample range, then walked with the
// exact FP32 predicate so that the first and last samples are the ones the reference's own bounds
// test accepts. The in-cube samples of a ray form one contiguous range because every term of the
// FP32 index is monotone in t.
// The slab test is FP32 with the hardware reciprocal: in terms of the position along its axis, each
// plane's t is within 2^-20 of the scene's scale (the plane's and the difference's rounding, and 2 ulps of
// a t that no sample exceeds), the margin is 2^-16 of it and covers the rounding of a sample's index too, so
// a sample inside by the FP32 test lies between the computed ends. Those times n / L are within 2^-7 of a
// sample (n <= 8192), and the range is taken 1/16 wider: the walks below only move inward. With div3 and
// inv_w, inv_h in place of IEEE sequences the setup of a ray, repeated on each of its lanes, costs about half
// of FP64 slabs and IEEE divisions: 64 orbit views 0.973 -> 0.936 ms, a 72x42 view 6.8 -> 6.5 us.
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ void slab_axis(double p, double d, double lo, double hi, double& tin, double& tout) {
    if (fabs(d) < 0x1p-100) {  // moves no sample by an FP32 ulp
        if (p < lo || p > hi) { tin = 1e300; tout = -1e300; }
    } else {
        const double inv = rcp64(d), t1 = (lo - p) * inv, t2 = (hi - p) * inv;
        tin = fmax(tin, fmin(t1, t2));
        tout = fmin(tout, fmax(t1, t2));
    }
}
__device__ __forceinline__ void slab_axis32(float p, float d, float lo, float hi, float& tin, float& tout) {
    const float inv = __builtin_amdgcn_rcpf(d), t1 = (lo - p) * inv, t2 = (hi - p) * inv;
    const bool flat = fabsf(d) < 0x1p-100f, out = p < lo || p > hi;
    tin = fmaxf(tin, flat ? (out ? INFINITY : -INFINITY) : fminf(t1, t2));
    tout = fminf(tout, flat ? INFINITY : fmaxf(t1, t2));
}

template <int DIV>
__device__ __forceinline__ void exact_clip(const DevVolume& v, const ExactView& ev, const float* s_t, float dx, float dy, float dz,
                                           int& kf, int& kl) {
    const float m = ev.margin;
    float tin = -INFINITY, tout = INFINITY;
    slab_axis32(ev.px, dx, v.ox - m, v.ox + (v.fnx - 1) * v.sx + m, tin, tout);
    slab_axis32(ev.py, dy, v.oy - m, v.oy + (v.fny - 1) * v.sy + m, tin, tout);
    slab_axis32(ev.pz, dz, v.oz - m, v.oz + (v.fnz - 1) * v.sz + m, tin, tout);
    const int n = ev.n;
    kf = n;
    kl = -1;
    if (!(tin <= tout)) return;
    const float sc = ev.per_t, fn = (float)n;
    int a = (int)fminf(fmaxf(ceilf(tin * sc - 0.5625f), 0.0f), fn), b = (int)fminf(fmaxf(floorf(tout * sc - 0.4375f), -1.0f), fn - 1.0f);
    while (a <= b && !exact_inside(v, exact_index<DIV>(v, dx, dy, dz, ev.px, ev.py, ev.pz, s_t[a]))) a++;
    while (b >= a && !exact_inside(v, exact_index<DIV>(v, dx, dy, dz, ev.px, ev.py, ev.pz, s_t[b]))) b--;
    kf = a;
    kl = b;
}

// Tile geometry of the exact kernels: a wave holds 64/S rays as TWxTH, a block 2x2 waves. Two
// lanes per ray take 4x8-ray waves (8x16-pixel blocks): on the 256^3 cube's 576x336 x 800 view
// 0.0900 ms against 0.0914 ms with 8x4 and 0.110 ms with 2x16 (4 samples in flight each), and
// the same 4.92 - 4.94 ms as 8x4 for the 256-view orbit batch.
template <int S> struct ExactTile {
    static constexpr int TW = (S == 1) ? 8 : (S == 16 ? 2 : 4);
    static constexpr int TH = (64 / S) / TW;
};

// The lanes of a wave and the rays they trace. The wave's TW x TH rays are cut into 2x2 pixel
// blocks; a block takes 4S consecutive lanes (one 16-lane row for S <= 4, two for S = 8, the
// whole wave for S = 16), its
// four pixels on the four lanes of a quad and its S sub-lanes on S consecutive quads. A 16-byte-per-lane record load is served a
// quad (64 B) per cycle, one cycle per distinct cache line in the quad: the four rays of a 2x2
// block sample the same k at points less than a voxel apart, mostly inside one line, where a
// quad of two rays' consecutive samples spans about two (on the 256^3 cube's 576x336 x 800 view,
// 22.3 line lookups per 64-lane load against 32.2). Sub-lane m of a ray sits 4m lanes above
// sub-lane 0 (row_next<4m>).
template <int S>
__device__ __forceinline__ void exact_lane(int lane, int& ti, int& tj, int& sub) {
    constexpr int TW = ExactTile<S>::TW;
    sub = (lane >> 2) & (S - 1);
    const int blk = lane / (4 * S);  // 2x2 block of the wave, row-major
    ti = (blk % (TW / 2)) * 2 + (lane & 1);
    tj = (blk / (TW / 2)) * 2 + ((lane >> 1) & 1);
}


// The samples of a wave's rays over a cube without negative values, added in k order (exact_block's
// main loop). P samples per lane per iteration (k, k + S, ...), staged so that the later samples' LDS
// and buffer reads are in flight while the first ones' lerps run. The sum order is unchanged: the S
// samples at k, then the S samples at k + S, and so on.
// Every lane samples inside the cube, so the corner indices need no clamp: a lane past its ray's last
// in-cube sample kl re-reads kl's t (its result is masked), and a lane whose ray has no in-cube
// sample is at the cube's origin (zero direction), which is inside. The in-cube samples kf..kl are
// contiguous (the FP32 index is monotone in t). t is read at LDS byte address min(t_lo + 4k, t_hi),
// both bounds including the LDS base.
// Trips that every lane of the wave fills (kb + P S <= full, the wave's shortest range) need neither
// the clamp of t's address nor the mask, and read their P t values at constant offsets from one
// address; the arithmetic and the sum order are those of the masked trips.
// FMA2: divisions and scale as one multiply and one FMA each (birp_div_fma2, birp_scale_fma2), where the
// volume's spacings and values allow it: 52 VALU instructions per sample and no branch, against 58
// and one rarely taken branch per sample. Issue-bound batches gain what the instructions save (64 orbit
// views of a 256^3 cube: 1.189 ms with FP64 divisions and scale and clamped lerps, 1.058 ms now); a
// single 576x336 x 800 view, whose waves also wait on the vector L1, goes from 87.4 to 84.7 us.
// SM_QUAD_NN: a cell of positive corners lerps as in SM_QUAD_POS, an empty one gives 0 either way, and
// only a cell with both takes std::lerp's zero branches and the scale's full test (its values can be
// arbitrarily small): the least corner finds the samples where some lane has such a cell, on the
// surfaces of a cavity, and inside it. 3 samples in flight instead of 4 (the branch keeps corners alive:
// 4 spill). A 256^3 cube with an empty cavity, 576x336 x 800: 270 us with the general lerps, their stop
// test and one sample in flight, 75 us now (72 without zeros); 64 orbit views 3.35 -> 0.97 ms.
// SM_NEAR_NN: one value per sample from the [z][y][x] copy, its index in two 24-bit multiply-adds:
// 576x336 x 800 124 -> 56 us, a camera inside a 144^3 cube at 265x155 x 200 29.4 -> 11.5 us.
typedef __attribute__((address_space(3))) const float* lds_float_ptr;
template <int S, int P, int MODE, bool FMA2, bool MASK>
__device__ __forceinline__ float march_trip(const DevVolume& v, const QuadCtx& qc, float rx, float ry, float rz, float qx, float qy,
                                            float qz, unsigned t_lo, unsigned t_hi, int kb, int lim, float w, float acc) {
    constexpr bool NEAR = MODE == SM_NEAR_NN;
    constexpr int DIV = FMA2 ? DIV_FMA2 : DIV_RN64;
    QuadFetch q[NEAR ? 1 : P];
    float near[NEAR ? P : 1];
    const unsigned tb = t_lo + (unsigned)kb * 4u;
#pragma unroll
    for (int u = 0; u < P; ++u) {
        const unsigned ta = tb + (unsigned)(u * S) * 4u;
        const float t = *(lds_float_ptr)(uintptr_t)(MASK ? min(ta, t_hi) : ta);
        const ExactIdx r = exact_index<DIV>(v, rx, ry, rz, qx, qy, qz, t);
        if constexpr (NEAR) near[u] = near_fetch(qc, r.xd, r.yd, r.zd);
        else q[u] = quad_fetch_inside(qc, r.xd, r.yd, r.zd);
    }
    float sc[P];
#pragma unroll
    for (int u = 0; u < P; ++u) {
        float val;
        if constexpr (NEAR) val = near[u];
        else val = quad_lerp<LERP_POS>(q[u]);
        const float vw = val * w;  // Camera.cpp:201
        sc[u] = FMA2 ? birp_scale_fma2(vw) : scale_pos(vw);
        if constexpr (MODE == SM_QUAD_NN) {
            if (__builtin_expect(fold_corners<false>(q[u]) == 0u, 0) && fold_corners<true>(q[u]) != 0u)
                sc[u] = birp_scale_sample(quad_lerp<LERP_NONNEG>(q[u]) * w);
        }
    }
    if constexpr (MASK) {
#pragma unroll
        for (int u = 0; u < P; ++u) sc[u] = (kb + u * S < lim) ? sc[u] : -0.0f;
    }
#pragma unroll
    for (int u = 0; u < P; ++u) acc = add_in_order<S>(acc, sc[u]);
    return acc;
}

template <int S, int P, int MODE, bool FMA2>
__device__ __forceinline__ float march_nonneg(const DevVolume& v, const QuadCtx& qc, float rx, float ry, float rz, float qx, float qy,
                                              float qz, unsigned t_lo, unsigned t_hi, int full, int trips, int lim, float w, float acc) {
    int kb = 0;
    for (; kb + P * S <= full; kb += P * S)
        acc = march_trip<S, P, MODE, FMA2, false>(v, qc, rx, ry, rz, qx, qy, qz, t_lo, t_hi, kb, lim, w, acc);
    for (; kb < trips; kb += P * S)
        acc = march_trip<S, P, MODE, FMA2, true>(v, qc, rx, ry, rz, qx, qy, qz, t_lo, t_hi, kb, lim, w, acc);
    return acc;
}

// ------------------------------------------------------------------------------------------
// the exact render: one block renders one 2x2-wave tile `lb` of a view (wg_x tiles per row of
// tiles); every thread of the block calls it
// ------------------------------------------------------------------------------------------
template <int S, int MODE, int P>
__device__ __forceinline__ void exact_block(const DevVolume& v, const ExactView& ev, int lb, int wg_x) {
    constexpr bool QUAD = (MODE == SM_QUAD_POS || MODE == SM_QUAD_NN || MODE == SM_QUAD_GEN);
    constexpr bool NN = mode_nonneg(MODE);
    extern __shared__ unsigned s_mem[];
    float* s_t = (float*)s_mem;
    const int n = ev.n;
    // ray distances t_k = L * ((k + 0.5f) / n) (Camera.cpp:73), IEEE division as on the host
    for (int k = threadIdx.x; k < n; k += BIRP_BLOCK) s_t[k] = ev.L * (((float)k + 0.5f) / (float)n);
    QuadCtx qc;
    if constexpr (QUAD) {
        unsigned* tab = s_mem + ((n + 3) & ~3);
        const int ntab = v.nx + v.ny + v.nz;
        for (int q = threadIdx.x; q < ntab; q += BIRP_BLOCK) tab[q] = v.qtab[q];
        qc.rs = make_rsrc(v.quad, v.quad_bytes);
        qc.tx = tab;
        qc.ty = tab + v.nx;
        qc.tz = tab + v.nx + v.ny;
        qc.hx = v.fnx - 2.0f;
        qc.hy = v.fny - 2.0f;
        qc.hz = v.fnz - 2.0f;
    } else if constexpr (MODE == SM_NEAR_NN) {
        qc.row = (unsigned)v.nx;
        qc.slice = (unsigned)v.nx * (unsigned)v.ny;
        qc.rs = make_rsrc(v.linear, qc.slice * (unsigned)v.nz * 4u);
    }
    __syncthreads();

    constexpr int TW = ExactTile<S>::TW, TH = ExactTile<S>::TH;
    const int wave = threadIdx.x >> 6, lane = lane_id();
    int ti, tj, sub;
    exact_lane<S>(lane, ti, tj, sub);
    const int i = ((lb % wg_x) * 2 + (wave & 1)) * TW + ti;
    const int j = ((lb / wg_x) * 2 + (wave >> 1)) * TH + tj;
    const bool valid = (i < ev.W) && (j < ev.H);

    float dx = 0.f, dy = 0.f, dz = 1.f;
    int kf = n, kl = -1;
    if (valid) {
        exact_ray_dir(ev, i, j, dx, dy, dz);
        if constexpr (MODE == SM_CMEM) {
            kf = 0;
            kl = n - 1;
        } else {
            // the modes without negative samples have |origin| >= 2^-30: no ingress needs the guard
            if (NN && v.div_fma2) exact_clip<DIV_FMA2>(v, ev, s_t, dx, dy, dz, kf, kl);
            else exact_clip<NN ? DIV_RN64 : DIV_GUARD>(v, ev, s_t, dx, dy, dz, kf, kl);
            if (ev.semantics == BIRP_SEM_REFERENCE && kf != 0) kl = -1;  // first sample outside: ray dead
        }
    }
    // Every ray walks its own range kf..kl: sub-lane `sub` takes k = kf + kb + sub, and the wave
    // makes as many trips as its longest ray needs. t is read at a clamped LDS byte offset.
    const int len = (kl >= kf) ? kl - kf + 1 : 0;
    const int trips = wave_max_i(len);
    const int lim = len - sub;  // sample kb + sub of this ray exists iff kb < lim
    const unsigned t_first = (unsigned)(kf + sub) * 4u, t_last = (unsigned)(n - 1) * 4u;

    float acc = 0.f;
    if (valid && ev.accumulate) acc = ev.out[(size_t)j * ev.W + i];
    unsigned added = (unsigned)len;
    const float w = ev.w;
    const float px = ev.px, py = ev.py, pz = ev.pz;

    if constexpr (NN) {
        const bool has = len > 0;
        const float rx = has ? dx : 0.f, ry = has ? dy : 0.f, rz = has ? dz : 0.f;
        const float qx = has ? px : v.ox, qy = has ? py : v.oy, qz = has ? pz : v.oz;
        const unsigned t_base = (unsigned)(uintptr_t)(lds_float_ptr)s_t;
        unsigned t_lo = t_base + (has ? t_first : 0u), t_hi = t_base + (has ? (unsigned)kl * 4u : 0u);
        // keep the selects above out of the loop (the compiler would otherwise redo them per sample)
        asm volatile("" : "+v"(t_lo), "+v"(t_hi));
        const int full = wave_min_i(len);
        if (ev.fast_guards == 2 && v.div_fma2)
            acc = march_nonneg<S, P, MODE, true>(v, qc, rx, ry, rz, qx, qy, qz, t_lo, t_hi, full, trips, lim, w, acc);
        else
            acc = march_nonneg<S, P, MODE, false>(v, qc, rx, ry, rz, qx, qy, qz, t_lo, t_hi, full, trips, lim, w, acc);
    }
    // Any data: a ray stops at its first negative sample (Camera.cpp:207-210). While no sample of the wave
    // is negative and no ray of it has stopped, the samples are added as above; after that each ray
    // gathers its S samples and tests them in k order on sub-lane 0 (the other sub-lanes' sums and stops
    // are not used).
    bool alive = true, quiet = true;
    auto add_trip = [&](float s, int kb) {
        const bool act = kb < lim;
        quiet = quiet && __ballot(act && s < 0) == 0ull;
        if (quiet) {
            acc = add_in_order<S>(acc, act ? s : -0.0f);
        } else {
#pragma unroll
            for (int mm = 0; mm < S; ++mm) {
                const float sm = sub_lane_f<S>(s, mm);
                const bool add = alive && kb + mm < len;
                const bool stop = add && sm < 0;
                acc = (add && !stop) ? acc + sm : acc;
                if (stop) added = (unsigned)(kb + mm);
                alive = alive && !stop;
            }
        }
    };
    if constexpr (MODE == SM_CMEM) {
        const __amdgpu_buffer_rsrc_t zones = make_rsrc(v.zones, BIRP_ZONE_BYTES);
        for (int kb = 0; kb < trips; kb += S) {
            const float t = *(const float*)((const char*)s_t + min(t_first + (unsigned)kb * 4u, t_last));
            const float x = dx * t + px, y = dy * t + py, z = dz * t + pz;
            add_trip(scale_any(cmem_sample_zoned(v.cmem, zone_fetch(zones, x, y, z), x, y, z) * w), kb);  // Camera.cpp:201
        }
    }
    for (int kb = 0; !NN && MODE != SM_CMEM && kb < trips; kb += S) {
        const float t = *(const float*)((const char*)s_t + min(t_first + (unsigned)kb * 4u, t_last));
        const ExactIdx r = exact_index<DIV_GUARD>(v, dx, dy, dz, px, py, pz, t);
        float val;
        if constexpr (MODE == SM_QUAD_GEN) val = quad_lerp<LERP_FINITE>(quad_fetch(qc, r.xd, r.yd, r.zd));
        else if constexpr (MODE == SM_LIN_TRI) val = sample_linear_tri(v, r);
        else val = sample_linear_nearest(v, r);
        add_trip(scale_any(val * w), kb);  // Camera.cpp:201
    }
    if (valid && sub == 0) ev.out[(size_t)j * ev.W + i] = acc;
    if (ev.counter || ev.wave_counts) {
        unsigned tot = wave_sum_u((valid && sub == 0) ? added : 0u);
        if (lane == 0) {
            if (ev.wave_counts) ev.wave_counts[lb * 4 + wave] = tot;  // a plain store, every wave
            else if (tot) atomicAdd(ev.counter, (unsigned long long)tot);
        }
    }
}

// Waves per SIMD the exact kernels' registers leave room for: 7 where no spill follows (72 VGPRs); the rare
// branch of SM_QUAD_NN and the shuffles of 8 and 16 lanes per ray take more. CMEM with up to 4 lanes per ray waits on
// the chains of its zones: 7 waves in single views, 8 (spilling 1 register of its surfaces) in launches of many.
// us with 6 / 7 / 8 waves, means of 3 poses: 320x200 n = 50 24.1 / 24.3 / 24.9, 400x240 n = 400 145.4 / 145.2 / 148.6,
// 576x336 n = 100 76.8 / 76.4 / 76.8, n = 800 467 / 449 / 454, 1000x600 n = 200 340 / 328 / 328; 16 views of 288x168
// n = 100 254 / 244 / 242, 4 of 576x336 n = 100 244 / 234 / 230, 8 of 288x168 n = 320 420 / 407 / 409.
constexpr int exact_waves(int S, int mode, bool many) {
    if (mode == SM_CMEM) return S <= 4 ? (many ? 8 : 7) : 1;
    return !mode_nonneg(mode) || S == 16 ? 1 : exact_resident_blocks(mode, S);
}

// One view: block b renders tile lb(b).
// Without a plan, lb = b: consecutive tiles go round-robin over the 8 XCDs, so every XCD renders
// a fair share of every part of the image (contiguous bands, one per XCD, left the XCDs with the
// middle rows of the cube's image working longest).
// With a plan (`order`: the tiles sorted heaviest first by k_exact_plan), slot b takes the
// sorted tile at its place in a snake over the CUs: round r of ncu slots runs forward when r is
// even and backward when odd, so that every CU draws one tile from each round and the heavy
// rounds are spread evenly (the longest-processing-time-first rule). The grid is then nblocks.
template <int S, int MODE, int P = 1>
__global__ __launch_bounds__(BIRP_BLOCK, exact_waves(S, MODE, false)) void k_render_exact(DevVolume v, ExactView ev, int wg_x, int nblocks,
                                                             const int* __restrict__ order, int ncu) {
    if ((int)blockIdx.x >= nblocks) return;
    int lb = blockIdx.x;
    if (order) {
        const int b = blockIdx.x, r = b / ncu, base = r * ncu, c = b - base;
        const int nr = min(ncu, nblocks - base);
        lb = order[base + ((r & 1) ? nr - 1 - c : c)];
    }
    if (lb < 0 || lb >= nblocks) return;
    exact_block<S, MODE, P>(v, ev, lb, wg_x);
}

// ------------------------------------------------------------------------------------------
// Tile plan of a single exact view. A view of a few thousand tiles is resident all at once
// (a 576x336 view is 1512 blocks, six per CU): each CU keeps the blocks the dispatcher handed it,
// and a CU that drew several tiles across the middle of the cube's image finishes last while
// others idle. The plan estimates every tile's work -- the longest in-cube run of samples among
// five rays of each wave (its four corners and its centre), from a slab test against the cube's
// box in approximate FP32 -- counting-sorts the tiles on it, heaviest first, and writes the
// order. Orders change which CU renders a tile, never what it computes: the image is the same
// bit for bit whatever the order.
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ void plan_slab(float p, float rd, float lo, float hi, float& tin, float& tout) {
    const float t1 = (lo - p) * rd, t2 = (hi - p) * rd;  // rd = 1/d (inf for d = 0: NaN t drop out)
    tin = fmaxf(tin, fminf(t1, t2));
    tout = fminf(tout, fmaxf(t1, t2));
}

// samples of ray (i, j) inside the cube's box, approximately: an estimate of its trip count
__device__ __forceinline__ int plan_ray_len(const DevVolume& v, const ExactView& ev, int i, int j, float sc, float rW,
                                            float rH) {
    const float sx = (2.f * ((float)i + 0.5f) * rW - 1.f) * ev.tanx * ev.aspect;
    const float sy = (1.f - 2.f * ((float)j + 0.5f) * rH) * ev.tany;
    // world direction of the camera ray (sx, sy, -1), unnormalised: t along it is t / |(sx, sy, 1)|
    const float dx = ev.rinv[0] * sx + ev.rinv[1] * sy - ev.rinv[2];
    const float dy = ev.rinv[3] * sx + ev.rinv[4] * sy - ev.rinv[5];
    const float dz = ev.rinv[6] * sx + ev.rinv[7] * sy - ev.rinv[8];
    float tin = -3.0e38f, tout = 3.0e38f;
    plan_slab(ev.px, __builtin_amdgcn_rcpf(dx), v.ox, v.ox + (float)(v.nx - 1) * v.sx, tin, tout);
    plan_slab(ev.py, __builtin_amdgcn_rcpf(dy), v.oy, v.oy + (float)(v.ny - 1) * v.sy, tin, tout);
    plan_slab(ev.pz, __builtin_amdgcn_rcpf(dz), v.oz, v.oz + (float)(v.nz - 1) * v.sz, tin, tout);
    if (!(tin <= tout)) return 0;
    const float s = sc * __builtin_amdgcn_sqrtf(sx * sx + sy * sy + 1.f);  // samples per unit of t
    const float klo = fminf(fmaxf(ceilf(tin * s - 0.5f), 0.f), (float)ev.n);
    const float khi = fmaxf(fminf(floorf(tout * s - 0.5f), (float)(ev.n - 1)), -1.f);
    if (ev.semantics == BIRP_SEM_REFERENCE && klo > 0.f) return 0;  // first sample outside: dead ray
    return khi >= klo ? (int)(khi - klo) + 1 : 0;
}

// grid: ceil(4 nblocks / BIRP_BLOCK) blocks of BIRP_BLOCK threads, thread 4b + w estimating wave
// w of tile b (a tile's four waves sit in neighbouring lanes). The last block to take a ticket
// (which it resets for the next plan) sorts. The estimates go between blocks as agent-scope
// atomic stores and loads, and each block waits for its stores before it takes its ticket:
// no cache-wide fence. The sort deals out exactly the tiles 0..nblocks-1 whatever estimates it
// reads, so the order is a permutation in every case. plan = [order | estimates | ticket], each
// of the first two BIRP_PLAN_MAX_BLOCKS ints, BIRP_PLAN_INTS in all; the ticket starts at zero.
template <int S>
__global__ __launch_bounds__(BIRP_BLOCK) void k_exact_plan(DevVolume v, ExactView ev, int wg_x, int nblocks, int* __restrict__ plan) {
    constexpr int TW = ExactTile<S>::TW, TH = ExactTile<S>::TH, NB = BIRP_PLAN_BUCKETS, T = BIRP_BLOCK;
    constexpr int PER_LANE = NB / 64;  // buckets per lane of the scanning wave
    static_assert(NB % 64 == 0, "plan shape");
    static_assert(4 * BIRP_MAX_EXACT_SAMPLES <= 65535, "tile estimates are kept as u16");
    int* order = plan;
    int* cost = plan + BIRP_PLAN_MAX_BLOCKS;
    int* ticket = plan + 2 * BIRP_PLAN_MAX_BLOCKS;
    __shared__ unsigned short s_key[BIRP_PLAN_MAX_BLOCKS];
    __shared__ int s_start[NB];
    __shared__ int s_lo, s_hi, s_last;
    const int tid = threadIdx.x;
    const int q = blockIdx.x * T + tid, b = q >> 2, w = q & 3;
    int m = 0;
    if (b < nblocks) {
        const int i0 = ((b % wg_x) * 2 + (w & 1)) * TW, j0 = ((b / wg_x) * 2 + (w >> 1)) * TH;
        if (i0 < ev.W && j0 < ev.H) {
            const float sc = (float)ev.n / ev.L, rW = 1.f / (float)ev.W, rH = 1.f / (float)ev.H;
            const int i1 = min(i0 + TW - 1, ev.W - 1), j1 = min(j0 + TH - 1, ev.H - 1);
            m = plan_ray_len(v, ev, (i0 + i1) >> 1, (j0 + j1) >> 1, sc, rW, rH);
            m = max(m, plan_ray_len(v, ev, i0, j0, sc, rW, rH));
            m = max(m, plan_ray_len(v, ev, i1, j0, sc, rW, rH));
            m = max(m, plan_ray_len(v, ev, i0, j1, sc, rW, rH));
            m = max(m, plan_ray_len(v, ev, i1, j1, sc, rW, rH));
        }
    }
    m += __shfl_xor(m, 1);
    m += __shfl_xor(m, 2);
    if (b < nblocks && w == 0) __hip_atomic_store(cost + b, m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_s_waitcnt(0);  // this thread's store has completed
    __syncthreads();
    if (tid == 0) s_last = atomicAdd(ticket, 1) == (int)gridDim.x - 1;
    __syncthreads();
    if (!s_last) return;

    for (int k = tid; k < NB; k += T) s_start[k] = 0;
    if (tid == 0) { s_lo = 0x7fffffff; s_hi = 0; }
    int lo = 0x7fffffff, hi = 0;
    for (int t0 = 0; t0 < nblocks; t0 += 8 * T) {
        int c[8];
#pragma unroll
        for (int k = 0; k < 8; ++k)  // eight loads in flight; the index is clamped into the area
            c[k] = __hip_atomic_load(cost + min(t0 + k * T + tid, BIRP_PLAN_MAX_BLOCKS - 1), __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int t = t0 + k * T + tid;
            if (t < nblocks) {
                const int cv = min(max(c[k], 0), 4 * BIRP_MAX_EXACT_SAMPLES);
                s_key[t] = (unsigned short)cv;
                lo = min(lo, cv);
                hi = max(hi, cv);
            }
        }
    }
    __syncthreads();
    atomicMin(&s_lo, lo);
    atomicMax(&s_hi, hi);
    __syncthreads();
    // NB buckets over [lo, hi], the heaviest in bucket 0
    const int base = s_lo, span = s_hi - s_lo;
    for (int t = tid; t < nblocks; t += T) {
        const int qq = span > 0 ? (int)(((long long)(s_key[t] - base) * (NB - 1)) / span) : 0;
        s_key[t] = (unsigned short)(NB - 1 - qq);
        atomicAdd(&s_start[NB - 1 - qq], 1);
    }
    __syncthreads();
    // exclusive prefix over the buckets by the first wave: lane l owns PER_LANE buckets in a row
    if (tid < 64) {
        int cnt[PER_LANE], sum = 0;
#pragma unroll
        for (int k = 0; k < PER_LANE; ++k) {
            cnt[k] = s_start[tid * PER_LANE + k];
            sum += cnt[k];
        }
        int incl = sum;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int up = __shfl_up(incl, off);
            if (tid >= off) incl += up;
        }
        int run = incl - sum;
#pragma unroll
        for (int k = 0; k < PER_LANE; ++k) {
            s_start[tid * PER_LANE + k] = run;
            run += cnt[k];
        }
    }
    __syncthreads();
    // every tile takes one place in its bucket's range: the places are 0..nblocks-1, each once
    for (int t = tid; t < nblocks; t += T) order[atomicAdd(&s_start[s_key[t]], 1)] = t;
    if (tid == 0) atomicExch(ticket, 0);  // ready for the next plan
}

// The last k < n with prefix[k] <= g (prefix[0] = 0 <= g < prefix[n]), searched by the wave 64 entries at a time.
__device__ __forceinline__ int find_view(const int* __restrict__ prefix, int n, int g) {
    int lo = 0;
    for (int step = n; step > 1;) {  // the answer is in [lo, lo + step)
        const int hi = min(lo + step, n);
        step = (step + 63) / 64;
        const int k = lo + lane_id() * step;
        const unsigned long long below = __ballot(k < hi && prefix[min(k, n)] <= g);
        lo += (__popcll(below) - 1) * step;
    }
    return __builtin_amdgcn_readfirstlane(lo);
}

// Many views (each with its own volume, image and sample-count slots) in one launch: items are
// the views' tiles, view-major (prefix[k] = first item of view k), and block g renders item g.
// Consecutive blocks go round-robin over the 8 XCDs, so every XCD renders a fair share of every
// view: contiguous bands, one per XCD, left whole XCDs with the heavy views (a 256-view orbit
// batch took 6.07 ms in bands and 4.89 ms interleaved). Every block renders one tile with exactly
// the arithmetic of k_render_exact, so each image is bit-identical to its single-view render; with
// more tiles in flight than one view has, the SIMDs stay fed while the longest rays of a view finish.
// `order` (may be null): block b renders item order[b] instead of item b (a batch's tile plan).
template <int S, int MODE, int P = 1>
__global__ __launch_bounds__(BIRP_BLOCK, exact_waves(S, MODE, true)) void k_render_exact_multi(const DevVolume* __restrict__ vols,
                                                                   const ExactView* __restrict__ views,
                                                                   const int* __restrict__ prefix, int nview, int total,
                                                                   const int* __restrict__ order) {
    if ((int)blockIdx.x >= total) return;
    const int g = order ? order[blockIdx.x] : (int)blockIdx.x;
    if (g < 0 || g >= total) return;
    const int lo = find_view(prefix, nview, g);
    const ExactView& ev = views[lo];
    constexpr int TW = ExactTile<S>::TW;
    exact_block<S, MODE, P>(vols[ev.vol], ev, g - prefix[lo], (ev.W + 2 * TW - 1) / (2 * TW));
}

// Tile estimates of a multi-view item list (the batch form of k_exact_plan's first phase): thread
// 4g + w estimates wave w of item g; cost[g] = the sum over the item's four waves.
template <int S>
__global__ __launch_bounds__(BIRP_BLOCK) void k_plan_multi(const DevVolume* __restrict__ vols, const ExactView* __restrict__ views,
                                                           const int* __restrict__ prefix, int nview, int total, int* __restrict__ cost) {
    constexpr int TW = ExactTile<S>::TW, TH = ExactTile<S>::TH;
    const long long q = (long long)blockIdx.x * BIRP_BLOCK + threadIdx.x;
    const int g = (int)(q >> 2), w = (int)(q & 3);
    int m = 0;
    if (g < total) {
        int lo = 0, hi = nview - 1;  // the view of item g: the last k with prefix[k] <= g
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (prefix[mid] <= g) lo = mid;
            else hi = mid - 1;
        }
        const ExactView& ev = views[lo];
        const DevVolume& v = vols[ev.vol];
        const int lb = g - prefix[lo], wg_x = (ev.W + 2 * TW - 1) / (2 * TW);
        const int i0 = ((lb % wg_x) * 2 + (w & 1)) * TW, j0 = ((lb / wg_x) * 2 + (w >> 1)) * TH;
        if (i0 < ev.W && j0 < ev.H) {
            const float sc = (float)ev.n / ev.L, rW = 1.f / (float)ev.W, rH = 1.f / (float)ev.H;
            const int i1 = min(i0 + TW - 1, ev.W - 1), j1 = min(j0 + TH - 1, ev.H - 1);
            m = plan_ray_len(v, ev, (i0 + i1) >> 1, (j0 + j1) >> 1, sc, rW, rH);
            m = max(m, plan_ray_len(v, ev, i0, j0, sc, rW, rH));
            m = max(m, plan_ray_len(v, ev, i1, j0, sc, rW, rH));
            m = max(m, plan_ray_len(v, ev, i0, j1, sc, rW, rH));
            m = max(m, plan_ray_len(v, ev, i1, j1, sc, rW, rH));
        }
    }
    m += __shfl_xor(m, 1);
    m += __shfl_xor(m, 2);
    if (g < total && w == 0) cost[g] = m;
}

// ------------------------------------------------------------------------------------------
// FP64 render (every operation in double) for error reporting on large configurations
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ double lerp64(double a, double b, double t) {
    if ((a <= 0 && b >= 0) || (a >= 0 && b <= 0)) return t * b + (1 - t) * a;
    if (t == 1) return b;
    double x = a + t * (b - a);
    return ((t > 1) == (b > a)) ? (b < x ? x : b) : (b > x ? x : b);
}

__device__ double cmem_sample64(const CmemParams& m, double x, double y, double z) {
    const double PI = 3.14159265358979323846;
    double r = sqrt(x * x + y * y + z * z);
    double theta = (x != 0) ? acos(x / r) : 0.0;
    double phi = (y != 0) ? acos(y / sqrt(y * y + z * z)) : 0.0;
    double phi_n = acos(cos(theta) * cos((double)m.theta_n) + sin(theta) * sin((double)m.theta_n) * cos(phi - PI / 2));
    double phi_s = acos(cos(theta) * cos((double)m.theta_s) + sin(theta) * sin((double)m.theta_s) * cos(phi - 3 * PI / 2));
    double sp = sin(phi);
    double f = pow(cos(theta / 2) + m.a5 * sin(2 * theta) * (1 - exp(-theta)),
                   m.p1 * (m.beta_c[0] + m.beta_c[1] * cos(phi) + (double)m.beta_c[3] * (sp * sp)));
    double q = (double)m.p2 * m.charlie * exp((double)m.p3 * m.dn * pow(phi_n, (double)m.a21)) +
               (double)m.p2 * m.charlie * exp((double)m.p3 * m.ds * pow(phi_s, (double)m.a21));
    double rmp = (double)m.p0 * m.r0_lin * f + q;
    double ry = m.bs * pow(2 / (1 + cos(theta)), (double)m.ay_bs);
    double rz = m.bs * pow(2 / (1 + cos(theta)), (double)m.az_bs);
    double rbs = (ry * rz) / sqrt((rz * cos(phi)) * (rz * cos(phi)) + (ry * sin(phi)) * (ry * sin(phi)));
    double h = 0.025, hs = theta / 2, ss = sin(theta);
    double inner = (double)m.A1 * exp(-(double)m.B * (hs * hs * hs * hs)) * pow(r / 10, -(double)m.alpha - (double)m.beta * (ss * ss));
    double outer = (double)m.A2 / ((r / 10) * (r / 10) * (r / 10));
    if (r < rmp - h) return 0.0;
    if (r <= rmp + h) return lerp64(0.0, inner, (r - (rmp - h)) / (rmp + h));
    if (r < rbs - h) return inner;
    if (r <= rbs + h) return lerp64(inner, outer, (r - (rbs - h)) / (rbs + h));
    return outer;
}

__global__ __launch_bounds__(BIRP_BLOCK) void k_render_f64(DevVolume v, F64View fv) {
    int pix = blockIdx.x * BIRP_BLOCK + threadIdx.x;
    if (pix >= fv.W * fv.H) return;
    int i = pix % fv.W, j = pix / fv.W;
    double sx = (2 * ((i + 0.5) / fv.W) - 1) * fv.tanx * fv.aspect;
    double sy = (1 - 2 * ((j + 0.5) / fv.H)) * fv.tany;
    double nd = sqrt(sx * sx + sy * sy + 1);
    double u0 = sx / nd, u1 = sy / nd, u2 = -1 / nd;
    double w0 = fv.rinv[0] * u0 + fv.rinv[1] * u1 + fv.rinv[2] * u2;
    double w1 = fv.rinv[3] * u0 + fv.rinv[4] * u1 + fv.rinv[5] * u2;
    double w2 = fv.rinv[6] * u0 + fv.rinv[7] * u1 + fv.rinv[8] * u2;
    double wd = sqrt(w0 * w0 + w1 * w1 + w2 * w2);
    double dx = w0 / wd, dy = w1 / wd, dz = w2 / wd;
    double acc = 0.0;
    const double K = BIRP_SCALE_K, C = BIRP_SCALE_C;
    for (int k = 0; k < fv.n; ++k) {
        double t = fv.L * ((k + 0.5) / fv.n);
        double x = dx * t + fv.px, y = dy * t + fv.py, z = dz * t + fv.pz;
        double val;
        if (v.kind == SK_CMEM) {
            val = cmem_sample64(v.cmem, x, y, z);
        } else {
            double xi = x - (double)v.ox, yi = y - (double)v.oy, zi = z - (double)v.oz;
            double xd = xi / (double)v.sx, yd = yi / (double)v.sy, zd = zi / (double)v.sz;
            bool in = (xi >= 0) && (xd + 1 < v.nx) && (yi >= 0) && (yd + 1 < v.ny) && (zi >= 0) && (zd + 1 < v.nz);
            if (!in) {
                if (fv.semantics == BIRP_SEM_REFERENCE) break;
                continue;
            }
            if (v.interp == BIRP_INTERP_TRILINEAR) {
                int x0 = (int)floor(xd), y0 = (int)floor(yd), z0 = (int)floor(zd);
                int x1 = (int)ceil(xd), y1 = (int)ceil(yd), z1 = (int)ceil(zd);
                double fx = xd - x0, fy = yd - y0, fz = zd - z0;
                const float* L = v.linear;
                size_t sy_ = v.nx, sz_ = (size_t)v.nx * v.ny;
                double lx1 = lerp64(L[z0 * sz_ + y0 * sy_ + x0], L[z0 * sz_ + y0 * sy_ + x1], fx);
                double lx2 = lerp64(L[z0 * sz_ + y1 * sy_ + x0], L[z0 * sz_ + y1 * sy_ + x1], fx);
                double hx1 = lerp64(L[z1 * sz_ + y0 * sy_ + x0], L[z1 * sz_ + y0 * sy_ + x1], fx);
                double hx2 = lerp64(L[z1 * sz_ + y1 * sy_ + x0], L[z1 * sz_ + y1 * sy_ + x1], fx);
                val = lerp64(lerp64(lx1, lx2, fy), lerp64(hx1, hx2, fy), fz);
            } else {
                val = v.linear[((size_t)(int)zd * v.ny + (int)yd) * v.nx + (int)xd];
            }
        }
        double s = val * fv.w * K / C / 10000;
        if (s < 0) break;
        acc += s;
    }
    fv.out[pix] = acc;
}

// ------------------------------------------------------------------------------------------
// Any other Space (its GetSample is the caller's host code): the rays' sample points, then the
// integration of the caller's sample values (Camera.cpp:140-229 around the call at :191)
// ------------------------------------------------------------------------------------------
// One thread per (pixel, k) of rows [row0, row0 + rows): X = d t_k + P in the reference's FP32
// order (Camera.cpp:183-189), stored at xyz[((pixel - row0 W) n + k) * 3].
__global__ __launch_bounds__(BIRP_BLOCK) void k_space_points(ExactView ev, int row0, int rows, float* xyz) {
    const long long q = (long long)blockIdx.x * BIRP_BLOCK + threadIdx.x;
    const long long total = (long long)rows * ev.W * ev.n;
    if (q >= total) return;
    const int k = (int)(q % ev.n);
    const long long pix = q / ev.n;
    const int i = (int)(pix % ev.W), j = row0 + (int)(pix / ev.W);
    float dx, dy, dz;
    exact_ray_dir(ev, i, j, dx, dy, dz);
    const float t = ev.L * (((float)k + 0.5f) / (float)ev.n);  // Camera.cpp:73
    xyz[3 * q] = dx * t + ev.px;
    xyz[3 * q + 1] = dy * t + ev.py;
    xyz[3 * q + 2] = dz * t + ev.pz;
}

// One thread per pixel: the reference's scale chain (Camera.cpp:201), the stop at the first
// negative sample (:207-210) and the FP32 sum in k order (:223) over vals[(pixel - row0 W) n + k].
__global__ __launch_bounds__(BIRP_BLOCK) void k_space_integrate(ExactView ev, int row0, int rows, const float* vals, float* img) {
    const long long pix = (long long)blockIdx.x * BIRP_BLOCK + threadIdx.x;
    if (pix >= (long long)rows * ev.W) return;
    float acc = ev.accumulate ? img[pix] : 0.f;
    const float* v = vals + pix * ev.n;
    for (int k = 0; k < ev.n; ++k) {
        const float s = birp_scale_sample(v[k] * ev.w);
        if (s < 0) break;
        acc = acc + s;
    }
    img[pix] = acc;
    (void)row0;
}

// ------------------------------------------------------------------------------------------
// GetSample at arbitrary points (DataCube.cpp:203-277 / Cmem.cpp:117-186), exact arithmetic
// ------------------------------------------------------------------------------------------
// A trilinear sample of a cube without negative values reads its two quad records, which share a 128-byte
// line every other time, instead of four pairs of values in four lines of the [z][y][x] copy: random
// points wait on lines (1,000,003 points over a 200^3 cube: 66 -> 32 us). Other cubes keep the copy: on a
// grid point the records' lerps give +0 where a value is -0.
__global__ __launch_bounds__(BIRP_BLOCK) void k_sample_points(DevVolume v, const float* xyz, long long n, float* out) {
    long long p = (long long)blockIdx.x * BIRP_BLOCK + threadIdx.x;
    if (p >= n) return;
    float x = xyz[3 * p], y = xyz[3 * p + 1], z = xyz[3 * p + 2];
    if (v.kind == SK_CMEM) {
        out[p] = cmem_sample(v.cmem, x, y, z);
        return;
    }
    ExactIdx r;
    r.xi = x - v.ox;
    r.xd = r.xi / v.sx;
    r.yi = y - v.oy;
    r.yd = r.yi / v.sy;
    r.zi = z - v.oz;
    r.zd = r.zi / v.sz;
    if (!exact_inside(v, r)) {
        out[p] = -1.f;
        return;
    }
    if (v.interp == BIRP_INTERP_NEAREST) {
        out[p] = sample_linear_nearest(v, r);
    } else if (v.quad && v.qtab && (v.vclass == VC_POSITIVE || v.vclass == VC_NONNEG)) {
        const QuadCtx qc{make_rsrc(v.quad, v.quad_bytes), v.qtab, v.qtab + v.nx, v.qtab + v.nx + v.ny, 0.f, 0.f, 0.f, 0u, 0u};
        out[p] = quad_lerp<LERP_NONNEG>(quad_fetch_inside(qc, r.xd, r.yd, r.zd));
    } else {
        out[p] = sample_linear_tri(v, r);
    }
}

// ------------------------------------------------------------------------------------------
// layout builders and scans
// ------------------------------------------------------------------------------------------
// The class of a cube's values, in the BIRP_SCAN_* words of flags: bit 0 = some value <= 0, bit 1 =
// some value non-finite, bit 2 = some sign bit set; min and max of |v| over the nonzero finite values as
// float bits (ordered as unsigned for positive floats). Bound by the read: 4 values per load, at most
// two blocks per CU, each with one atomic per word, and the words in cache lines of their own (an
// atomic on a contended line takes about 8 ns: three per wave on one line took 376 us for 256^3
// values, whose read takes 13 us at 5.2 TB/s; 27 us now).
// COPY: vals is a mapped host buffer, and the values go to `out` on the way.
template <bool COPY>
__global__ __launch_bounds__(BIRP_BLOCK) void k_scan_class(const float* vals, size_t n, unsigned* flags, float* out) {
    unsigned f = 0, mn = 0x7F7FFFFFu, mx = 0u;
    auto look = [&](float x) {
        const unsigned u = __float_as_uint(x) & 0x7FFFFFFFu;
        if (!(x > 0.f)) f |= 1u;
        if (u >= 0x7F800000u) f |= 2u;
        if (__float_as_uint(x) >> 31) f |= 4u;
        if (u != 0u && u < 0x7F800000u) {
            mn = min(mn, u);
            mx = max(mx, u);
        }
    };
    const size_t n4 = n / 4, step = (size_t)gridDim.x * BIRP_BLOCK, first = (size_t)blockIdx.x * BIRP_BLOCK + threadIdx.x;
    for (size_t k = first; k < n4; k += step) {
        const float4 x = reinterpret_cast<const float4*>(vals)[k];  // allocations and chunks of 16 B: aligned
        if constexpr (COPY) reinterpret_cast<float4*>(out)[k] = x;
        look(x.x);
        look(x.y);
        look(x.z);
        look(x.w);
    }
    for (size_t k = 4 * n4 + first; k < n; k += step) {
        const float x = vals[k];
        if constexpr (COPY) out[k] = x;
        look(x);
    }
    __shared__ unsigned s_f, s_mn, s_mx;
    if (threadIdx.x == 0) {
        s_f = 0u;
        s_mn = 0x7F7FFFFFu;
        s_mx = 0u;
    }
    __syncthreads();
    for (int o = 32; o > 0; o >>= 1) {
        f |= (unsigned)__shfl_xor((int)f, o, 64);
        mn = min(mn, (unsigned)__shfl_xor((int)mn, o, 64));
        mx = max(mx, (unsigned)__shfl_xor((int)mx, o, 64));
    }
    if (lane_id() == 0) {
        atomicOr(&s_f, f);
        atomicMin(&s_mn, mn);
        atomicMax(&s_mx, mx);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        if (s_f) atomicOr(flags + BIRP_SCAN_CLASS, s_f);
        atomicMin(flags + BIRP_SCAN_MIN, s_mn);
        atomicMax(flags + BIRP_SCAN_MAX, s_mx);
    }
}

// birp_div_fma2 against the correctly rounded birp_div_rn64 for every significand of the dividend and each of
// the n different spacings; a mismatch sets bit 0 of *bad. 16 significands to a thread and one atomic per wave at
// most: a grid of 2^23 threads that checked three spacings, equal or not, and counted every mismatch took 9 us
// of a small cube's upload, 43 where a spacing has many (30 / 31).
struct DivCheck {
    float rh[3], rl[3];
    double rd[3];
    int n;
};
constexpr int kDivPerThread = 16;
__global__ __launch_bounds__(BIRP_BLOCK) void k_check_div(DivCheck c, unsigned* bad) {
    const unsigned first = blockIdx.x * BIRP_BLOCK + threadIdx.x, step = (1u << 23) / kDivPerThread;
    bool f = false;
    for (int k = 0; k < c.n; ++k) {
#pragma unroll
        for (int q = 0; q < kDivPerThread; ++q) {
            const float a = __uint_as_float(0x3F800000u | (first + q * step));
            f = f || birp_div_fma2(a, c.rh[k], c.rl[k]) != birp_div_rn64(a, c.rd[k]);
        }
    }
    if (__ballot(f) != 0ull && lane_id() == 0 && __hip_atomic_load(bad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0u) atomicOr(bad, 1u);
}

// The layout builders: a block makes the records of 4 bricks in a row along x. It reads their corners
// (33 x 9 values per layer) into LDS once, coalesced, and writes each brick's 512 records in the order of
// their addresses, 1 KB per wave and store (a thread per cell in x order wrote each 128-byte line
// in pieces). Corners past the cube's last layer repeat it; no sample reads those records. Consecutive
// blocks run on successive XCDs, so the blocks are numbered XCD by XCD: the cube's rows are then read
// into one L2. Bound by the record writes: 256^3 quad records (64 MB read, 268 MB written) 149 -> 67 us,
// the time of such a copy at 5.2 TB/s; 512^3 BF16 records 1.05 -> 0.68 ms (0.52 at that rate), the
// brick scales within, and no clearing before.
constexpr int kBrickRow = 4, kTileX = 8 * kBrickRow + 1;

// Brick row of this block: its first brick along x, its y and z; false past the last one.
__device__ __forceinline__ bool brick_row(const DevVolume& v, int nbz, int& bx, int& by, int& bz) {
    const int rows = (v.nbx + kBrickRow - 1) / kBrickRow;
    const long long b = (long long)(blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    if (b >= (long long)rows * v.nby * nbz) return false;
    bx = (int)(b % rows) * kBrickRow;
    by = (int)(b / rows) % v.nby;
    bz = (int)(b / rows / v.nby);
    return true;
}

template <int LAYERS>
__device__ __forceinline__ void load_brick_row(const DevVolume& v, int bx, int by, int bz, float* s) {
    for (int t = threadIdx.x; t < kTileX * 9 * LAYERS; t += BIRP_BLOCK) {
        const int x = min(bx * 8 + t % kTileX, v.nx - 1), y = min(by * 8 + t / kTileX % 9, v.ny - 1), z = min(bz * 8 + t / (kTileX * 9), v.nz - 1);
        s[t] = v.linear[((size_t)z * v.ny + y) * v.nx + x];
    }
    __syncthreads();
}

// Cell r (0..511, Morton order) of brick w of the row: its lowest corner in the LDS tile.
__device__ __forceinline__ int brick_cell(int w, int r) {
    const int lx = (r & 1) | (r >> 2 & 2) | (r >> 4 & 4), ly = (r >> 1 & 1) | (r >> 3 & 2) | (r >> 5 & 4), lz = (r >> 2 & 1) | (r >> 4 & 2) | (r >> 6 & 4);
    return (lz * 9 + ly) * kTileX + w * 8 + lx;
}

__global__ __launch_bounds__(BIRP_BLOCK) void k_build_quad(DevVolume v, unsigned char* quad) {
    __shared__ float s[kTileX * 9 * 8];
    int bx, by, bz;
    if (!brick_row(v, (v.nz + 7) / 8, bx, by, bz)) return;
    load_brick_row<8>(v, bx, by, bz, s);
    const int w = threadIdx.x >> 6;  // one wave per brick
    if (bx + w >= v.nbx) return;
    const unsigned base = v.qtab[(bx + w) * 8] + v.qtab[v.nx + by * 8] + v.qtab[v.nx + v.ny + bz * 8];
    for (int r = lane_id(); r < 512; r += 64) {
        const float* c = s + brick_cell(w, r);
        *(float4*)(quad + base + r * 16u) = make_float4(c[0], c[1], c[kTileX], c[kTileX + 1]);
    }
}

__device__ __forceinline__ unsigned short f32_to_bf16_bits(float x) {
    __hip_bfloat16 h = __float2bfloat16(x);
    return *reinterpret_cast<unsigned short*>(&h);
}
__device__ __forceinline__ unsigned short f32_to_f16_bits(float x) {
    __half h = __float2half_rn(x);
    return *reinterpret_cast<unsigned short*>(&h);
}

// F16 records hold v / scale, a power of two per brick: max|v| over the brick's corners maps to < 2^15. With
// v.f16_uniform every brick gets the volume's scale v.f16_scale instead, and BF16 volumes hold their
// values, rounded to BF16, as F16 too (exactly).
enum OctForm { OCT_BF16, OCT_F16, OCT_BF16_AS_F16 };
template <int FORM>
__global__ __launch_bounds__(BIRP_BLOCK) void k_build_oct(DevVolume v, unsigned char* oct, float* bscale) {
    __shared__ float s[kTileX * 9 * 9];
    int bx, by, bz;
    if (!brick_row(v, v.nbz, bx, by, bz)) return;
    load_brick_row<9>(v, bx, by, bz, s);
    const int w = threadIdx.x >> 6;  // one wave per brick
    if (bx + w >= v.nbx) return;
    const unsigned base = v.otab[(bx + w) * 8] + v.otab[v.nx + by * 8] + v.otab[v.nx + v.ny + bz * 8];
    float inv = FORM == OCT_BF16_AS_F16 ? 1.f / v.f16_scale : 1.f;  // powers of two: exact
    if constexpr (FORM == OCT_F16) {
        float scale = v.f16_scale;
        if (!v.f16_uniform) {
            float m = 0.f;
            for (int t = lane_id(); t < 729; t += 64) m = fmaxf(m, fabsf(s[t / 9 * kTileX + w * 8 + t % 9]));
            for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
            scale = 1.f;
            if (m > 0.f && isfinite(m)) {
                int e;
                frexpf(m, &e);               // m = f * 2^e, f in [0.5, 1)
                scale = ldexpf(1.f, e - 15); // m / scale < 2^15
            }
        }
        if (lane_id() == 0) bscale[base >> 13] = scale;
        inv = 1.f / scale;
    }
    for (int r = lane_id(); r < 512; r += 64) {
        const float* c0 = s + brick_cell(w, r);
        const float* c1 = c0 + 9 * kTileX;
        const float c[8] = {c0[0], c0[1], c0[kTileX], c0[kTileX + 1], c1[0], c1[1], c1[kTileX], c1[kTileX + 1]};
        unsigned short h[8];
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const unsigned short b = f32_to_bf16_bits(c[q]);
            h[q] = FORM == OCT_F16 ? f32_to_f16_bits(c[q] * inv) : FORM == OCT_BF16 ? b : f32_to_f16_bits(__uint_as_float((unsigned)b << 16) * inv);
        }
        uint4 o;
        o.x = (unsigned)h[0] | ((unsigned)h[1] << 16);
        o.y = (unsigned)h[2] | ((unsigned)h[3] << 16);
        o.z = (unsigned)h[4] | ((unsigned)h[5] << 16);
        o.w = (unsigned)h[6] | ((unsigned)h[7] << 16);
        *(uint4*)(oct + base + r * 16u) = o;
    }
}

__global__ __launch_bounds__(BIRP_BLOCK) void k_zero_f32(float* p, size_t n) {
    for (size_t idx = (size_t)blockIdx.x * BIRP_BLOCK + threadIdx.x; idx < n; idx += (size_t)gridDim.x * BIRP_BLOCK) p[idx] = 0.f;
}

// ------------------------------------------------------------------------------------------
// fast path: many views in one launch, or one by value
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ float bf16lo(unsigned u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float bf16hi(unsigned u) { return __uint_as_float(u & 0xFFFF0000u); }

__device__ __forceinline__ float flerp(float a, float b, float t) { return __builtin_fmaf(t, b - a, a); }

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));

// Lerp of the FP16 pair (a, b) packed in one dword, in FP32: (a - t a) + t b as two fused
// multiply-adds, each reading its FP16 operand directly (v_fma_mix_f32, no conversions).
__device__ __forceinline__ float xlerp_f16(unsigned u, float t) {
    const half2_t h = __builtin_bit_cast(half2_t, u);
    const float a = (float)h.x, b = (float)h.y;
    return __builtin_fmaf(t, b, __builtin_fmaf(-t, a, a));
}

// Fast trilinear sample at index-space point (xd, yd, zd), already clamped into
// [0, nextbelow(n-1)] per axis, so the truncation is a valid cell index (0 .. n-2): the record's
// loads, then its lerps.
template <int DT>
struct FastFetch {
    uint4 a;           // FP32: the z record; else the octet
    float4 b;          // FP32: the z + 1 record
    float fx, fy, fz;  // lerp weights
    float scale;       // F16 with a scale per brick
};
template <int DT>
__device__ __forceinline__ FastFetch<DT> fast_fetch(const DevVolume& v, __amdgpu_buffer_rsrc_t rs, const unsigned* tab, float xd, float yd, float zd) {
    FastFetch<DT> q;
    q.fx = __builtin_amdgcn_fractf(xd);
    q.fy = __builtin_amdgcn_fractf(yd);
    q.fz = __builtin_amdgcn_fractf(zd);
    const unsigned xo = tab[(int)xd], yo = tab[v.nx + (int)yd];
    const unsigned* zo = tab + v.nx + v.ny + (int)zd;
    const unsigned off = add3(xo, yo, zo[0]);
    q.a = load16u(rs, off);
    if constexpr (DT == BIRP_DTYPE_F32) q.b = load16(rs, add3(xo, yo, zo[1]));
    if constexpr (DT == BIRP_DTYPE_F16) q.scale = v.bscale[off >> 13];
    return q;
}
template <int DT>
__device__ __forceinline__ float fast_value(const FastFetch<DT>& q) {
    if constexpr (DT == BIRP_DTYPE_F32) {
        const float4 a = __builtin_bit_cast(float4, q.a), b = q.b;
        float ly = flerp(flerp(a.x, a.y, q.fx), flerp(a.z, a.w, q.fx), q.fy);
        float hy = flerp(flerp(b.x, b.y, q.fx), flerp(b.z, b.w, q.fx), q.fy);
        return flerp(ly, hy, q.fz);
    } else {  // BF16, F16 with per-brick scale, F16 with one scale (BIRP_KDT_F16_UNIFORM)
        // each dword of the record holds the x-pair (x0, x1) of one (y, z) corner row
        const uint4 o = q.a;
        float c00, c10, c01, c11;  // the four x-lerps, at (y0,z0), (y1,z0), (y0,z1), (y1,z1)
        if constexpr (DT == BIRP_DTYPE_BF16) {
            c00 = flerp(bf16lo(o.x), bf16hi(o.x), q.fx);
            c10 = flerp(bf16lo(o.y), bf16hi(o.y), q.fx);
            c01 = flerp(bf16lo(o.z), bf16hi(o.z), q.fx);
            c11 = flerp(bf16lo(o.w), bf16hi(o.w), q.fx);
        } else {
            c00 = xlerp_f16(o.x, q.fx);
            c10 = xlerp_f16(o.y, q.fx);
            c01 = xlerp_f16(o.z, q.fx);
            c11 = xlerp_f16(o.w, q.fx);
        }
        float val = flerp(flerp(c00, c10, q.fy), flerp(c01, c11, q.fy), q.fz);
        if constexpr (DT == BIRP_DTYPE_F16) val *= q.scale;
        return val;
    }
}

// ------------------------------------------------------------------------------------------
// CMEM::GetSample (Cmem.cpp:117-186) in the fast form: FP32 with the hardware exp2/log2, square
// root and reciprocal, cosines and sines of the angles as coordinate ratios and half-angle
// identities, and arc cosines from Abramowitz & Stegun 4.4.46 (|error| <= 2e-8). Zone logic as the
// reference's. A cusp angle whose cosine rounds past 1 gives 0 here (the reference: NaN).
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ float acos_fast(float x) {
    const float ax = fminf(fabsf(x), 1.0f);
    float p = -0.0012624911f;
    p = __builtin_fmaf(p, ax, 0.0066700901f);
    p = __builtin_fmaf(p, ax, -0.0170881256f);
    p = __builtin_fmaf(p, ax, 0.0308918810f);
    p = __builtin_fmaf(p, ax, -0.0501743046f);
    p = __builtin_fmaf(p, ax, 0.0889789874f);
    p = __builtin_fmaf(p, ax, -0.2145988016f);
    p = __builtin_fmaf(p, ax, 1.5707963050f);
    const float r = __builtin_amdgcn_sqrtf(1.0f - ax) * p;
    return x >= 0.f ? r : 3.14159265358979f - r;
}
__device__ __forceinline__ float pow_fast(float b, float e) { return __builtin_amdgcn_exp2f(e * __builtin_amdgcn_logf(b)); }
__device__ __forceinline__ float exp_fast(float x) { return __builtin_amdgcn_exp2f(x * 1.44269504088896f); }

__device__ __forceinline__ float cmem_fast_inner(const CmemParams& m, float sd, float theta, float st) {
    const float ht = 0.5f * theta, ht2 = ht * ht;
    return m.A1 * exp_fast(-m.B * (ht2 * ht2)) * pow_fast(sd, -m.alpha - m.beta * (st * st));
}
__device__ __forceinline__ float cmem_fast_outer(const CmemParams& m, float sd) { return m.A2 * __builtin_amdgcn_rcpf(sd * sd * sd); }

// cmem_mp and cmem_bs in this arithmetic.
__device__ __forceinline__ float cmem_fast_mp(const CmemParams& m, float ct, float st, float theta, float cphi, float sphi) {
    // LinScaled (Cmem.cpp:188-222): cos(phi - pi/2) = sin(phi), cos(phi - 3 pi/2) = -sin(phi)
    const float phi_n = acos_fast(ct * m.cos_theta_n + st * m.sin_theta_n * sphi);
    const float phi_s = acos_fast(ct * m.cos_theta_s - st * m.sin_theta_s * sphi);
    const float cos_half = __builtin_amdgcn_sqrtf(0.5f * (1.f + ct));  // cos(theta / 2), theta in [0, pi]
    const float sin_2t = 2.f * st * ct;
    const float f = pow_fast(cos_half + m.a5 * sin_2t * (1.f - exp_fast(-theta)),
                             m.p1 * (m.beta_c[0] + m.beta_c[1] * cphi + m.beta_c[3] * (sphi * sphi)));
    const float q = m.p2 * m.charlie * (exp_fast(m.p3 * m.dn * pow_fast(phi_n, m.a21)) + exp_fast(m.p3 * m.ds * pow_fast(phi_s, m.a21)));
    return m.p0 * m.r0_lin * f + q;
}
__device__ __forceinline__ float cmem_fast_bs(const CmemParams& m, float ct, float cphi, float sphi) {
    const float base = 2.f * __builtin_amdgcn_rcpf(1.f + ct);
    const float ry = m.bs * pow_fast(base, m.ay_bs);
    const float rz = (m.az_bs == m.ay_bs) ? ry : m.bs * pow_fast(base, m.az_bs);
    const float rzc = rz * cphi, rys = ry * sphi;
    return ry * rz * __builtin_amdgcn_rsqf(rzc * rzc + rys * rys);
}

__device__ __forceinline__ float cmem_fast(const CmemParams& m, float x, float y, float z) {
    const float ryz2 = y * y + z * z;
    const float r = __builtin_amdgcn_sqrtf(__builtin_fmaf(x, x, ryz2)), ryz = __builtin_amdgcn_sqrtf(ryz2);
    const float ir = __builtin_amdgcn_rcpf(r), iyz = __builtin_amdgcn_rcpf(ryz);
    // theta = acos(x / r), 0 when x == 0; phi = acos(y / |(y, z)|), 0 when y == 0 (Cmem.cpp:224-246)
    const bool xs = x != 0.f, ys = y != 0.f;
    const float ct = xs ? x * ir : 1.f, st = xs ? ryz * ir : 0.f;
    const float theta = xs ? acos_fast(ct) : 0.f;
    const float cphi = ys ? y * iyz : 1.f, sphi = ys ? fabsf(z) * iyz : 0.f;
    const float rmp = cmem_fast_mp(m, ct, st, theta, cphi, sphi);
    const float h = 0.025f;
    if (r < rmp - h) return 0.f;
    const float rbs = cmem_fast_bs(m, ct, cphi, sphi);
    // the zones of Cmem.cpp:132-176 (r >= rmp - h here)
    const bool z_mp = r <= rmp + h;
    const bool z_sheath = !z_mp && r < rbs - h;
    const bool z_bs = !z_mp && !z_sheath && r >= rbs - h && r <= rbs + h;
    const float sd = 0.1f * r;
    const float outer = cmem_fast_outer(m, sd);
    if (!(z_mp || z_sheath || z_bs)) return outer;
    const float inner = cmem_fast_inner(m, sd, theta, st);
    if (z_mp) return ((r - (rmp - h)) * __builtin_amdgcn_rcpf(rmp + h)) * inner;  // lerp(0, inner, t)
    if (z_sheath) return inner;
    return __builtin_fmaf((r - (rbs - h)) * __builtin_amdgcn_rcpf(rbs + h), outer - inner, inner);
}

// cmem_fast with its surfaces left out where the bounds name the point's zone. (Only the surface near a sample, as
// cmem_sample_zoned asks it: 8% slower, its selects weigh as much as the hardware's transcendentals.)
__device__ __forceinline__ float cmem_fast_zoned(const CmemParams& m, const ZoneQuery& q, float x, float y, float z) {
    const Zone zone = zone_of<false>(q);
    float val = 0.f;
    if (zone == ZONE_EDGE) val = cmem_fast(m, x, y, z);
    if (zone == ZONE_SHEATH || zone == ZONE_OUTER) {
        const float ryz2 = y * y + z * z;
        const float r = __builtin_amdgcn_sqrtf(__builtin_fmaf(x, x, ryz2)), sd = 0.1f * r;
        if (zone == ZONE_OUTER) {
            val = cmem_fast_outer(m, sd);
        } else {
            const float ir = __builtin_amdgcn_rcpf(r);
            val = cmem_fast_inner(m, sd, acos_fast(x * ir), __builtin_amdgcn_sqrtf(ryz2) * ir);
        }
    }
    return val;
}

// Keeps the FP32 march x(j) = RN(j d + i0), j = 0 .. last, inside [0, hi]. x(j) is one rounding of
// a linear function of j, so it is monotone in j and stays inside when x(0) and x(last) do. When
// either is outside (a ray end within FP32 rounding of a face), the start is clamped and the step
// recomputed, then shortened an ulp at a time until x(last) fits; the last resort is a zero step.
__device__ __forceinline__ void fit_march(float& i0, float& d, float hi, int last) {
    const float fl = (float)last;
    const float b = __builtin_fmaf(fl, d, i0);
    if (i0 >= 0.f && i0 <= hi && b >= 0.f && b <= hi) return;
    const float a = fminf(fmaxf(i0, 0.f), hi);
    const float bc = fminf(fmaxf(b, 0.f), hi);
    i0 = a;
    d = last > 0 ? (bc - a) / fl : 0.f;
    for (int it = 0; it < 8 && d != 0.f; ++it) {
        const float e = __builtin_fmaf(fl, d, i0);
        if (e >= 0.f && e <= hi) return;
        d = __uint_as_float(__float_as_uint(d) - 1u);  // one ulp toward zero
    }
    const float e = __builtin_fmaf(fl, d, i0);
    if (!(e >= 0.f && e <= hi)) d = 0.f;
}

// x folded into a Kahan sum (sum, nc), nc holding the negated compensation -c:
// y = x - c; t = sum + y; -c' = y - (t - sum); sum = t.
__device__ __forceinline__ void kahan_add(float x, float& sum, float& nc) {
    const float y = x + nc;
    const float t = sum + y;
    nc = y - (t - sum);
    sum = t;
}

// The lanes of a fast-kernel wave: a wave traces a tile of tw x th rays, S lanes per ray.
// Positive kernels put 2x2 pixel blocks on lane quads, the S lanes of a ray on S consecutive
// quads of a 16-lane row (as exact_lane: a quad's record loads then mostly share one cache
// line); signed kernels keep the S lanes of a ray adjacent, since their first-negative test
// reads the ray's S bits of one ballot as a group.
struct FastLane {
    int tw, th, ray, ti, tj, sub, sub_step;
};
template <int S, bool SIGNED>
__device__ __forceinline__ FastLane fast_lane(int lane, int tw_log2) {
    FastLane f;
    f.tw = 1 << tw_log2;
    f.th = (64 / S) >> tw_log2;
    const bool blocks = !SIGNED && f.tw >= 2 && f.th >= 2;
    f.ray = lane / S;
    if (blocks) {
        const int r16 = lane & 15, quad = r16 >> 2;
        f.sub = quad & (S - 1);
        const int blk = (lane >> 4) * (4 / S) + quad / S;
        f.ti = (blk & ((f.tw >> 1) - 1)) * 2 + (lane & 1);
        f.tj = (blk >> (tw_log2 - 1)) * 2 + ((lane >> 1) & 1);
    } else {
        f.sub = lane % S;
        f.ti = f.ray & (f.tw - 1);
        f.tj = f.ray >> tw_log2;
    }
    f.sub_step = blocks ? 4 : 1;  // lane distance between sub-lanes m and m + 1 of a ray
    return f;
}

// x + the x of the lane `step` away, and the sum of the S lanes of a ray, (0 + 1) + (2 + 3): the same bits on
// each of its lanes (an addition of two commutes).
__device__ __forceinline__ double pair_sum(double x, int step) { return x + __shfl_xor(x, step, 64); }
template <int S>
__device__ __forceinline__ double sum_lanes(double x, int sub_step) {
    if constexpr (S >= 2) x = pair_sum(x, sub_step);
    if constexpr (S == 4) x = pair_sum(x, 2 * sub_step);
    return x;
}

// One wave renders tile `tile` (row-major over the image's tiles) of pose P over volume V, whose
// offset tables the wave holds in `tab`; every lane of the wave calls it.
template <int KV, int S, int U>
__device__ __forceinline__ void fast_tile(const DevVolume& V, const FastPose& P, int tile, const unsigned* tab, const FastLane& L) {
    constexpr bool CMEM = KV == BIRP_KDT_CMEM;
    constexpr int DT = CMEM ? BIRP_DTYPE_F32 : (KV & 3);
    constexpr bool SIGNED = CMEM || (KV & BIRP_KDT_SIGNED) != 0;
    const int tw = L.tw, th = L.th, ray = L.ray, ti = L.ti, tj = L.tj, sub = L.sub, sub_step = L.sub_step;
    const float K = (float)BIRP_SCALE_FOLDED;
    const __amdgpu_buffer_rsrc_t rs = CMEM ? make_rsrc(V.zones, BIRP_ZONE_BYTES) : (DT == BIRP_DTYPE_F32) ? make_rsrc(V.quad, V.quad_bytes) : make_rsrc(V.oct, V.oct_bytes);
    const int tx = tile % P.tiles_x, ty = tile / P.tiles_x;
    const int i = tx * tw + ti;
    const int j = ty * th + tj;
    const bool valid = (i < P.W) && (j < P.H);

    int kf = P.n, kl = -1;
    float ix0 = 0.f, iy0 = 0.f, iz0 = 0.f, dix = 0.f, diy = 0.f, diz = 0.f;
    if (valid) {
        // FP64 ray (the reference's formulas, in double)
        double sx = (2 * ((i + 0.5) * P.inv_w) - 1) * P.tanx_aspect;
        double sy = (1 - 2 * ((j + 0.5) * P.inv_h)) * P.tany;
        // (divisions by a norm or a spacing as products with its FP64 reciprocal: a relative
        // change of ~1e-16, far below the FP32 march)
        const double ind = rsqrt64(sx * sx + sy * sy + 1.0);
        double u0 = sx * ind, u1 = sy * ind, u2 = -ind;
        double w0 = P.rinv[0] * u0 + P.rinv[1] * u1 + P.rinv[2] * u2;
        double w1 = P.rinv[3] * u0 + P.rinv[4] * u1 + P.rinv[5] * u2;
        double w2 = P.rinv[6] * u0 + P.rinv[7] * u1 + P.rinv[8] * u2;
        const double iwd = rsqrt64(w0 * w0 + w1 * w1 + w2 * w2);
        double dx = w0 * iwd, dy = w1 * iwd, dz = w2 * iwd;
        if constexpr (CMEM) {
            // the model has no bounds: every sample, marched in world coordinates
            kf = 0;
            kl = P.n - 1;
            const double dt = P.dt, t0 = 0.5 * dt;
            ix0 = (float)(P.px + dx * t0);
            iy0 = (float)(P.py + dy * t0);
            iz0 = (float)(P.pz + dz * t0);
            dix = (float)(dx * dt);
            diy = (float)(dy * dt);
            diz = (float)(dz * dt);
        } else {
            // FP64 cube entry/exit: inside iff 0 <= (x - o)/s < n - 1 per axis
            double tin = -1e300, tout = 1e300;
            slab_axis(P.px, dx, (double)V.ox, (double)V.ox + (double)(V.nx - 1) * V.sx, tin, tout);
            slab_axis(P.py, dy, (double)V.oy, (double)V.oy + (double)(V.ny - 1) * V.sy, tin, tout);
            slab_axis(P.pz, dz, (double)V.oz, (double)V.oz + (double)(V.nz - 1) * V.sz, tin, tout);
            if (tin <= tout) {
                const double sc = P.sc;
                double a = ceil(tin * sc - 0.5), b = ceil(tout * sc - 0.5) - 1.0;
                a = fmax(a, 0.0);
                b = fmin(b, (double)(P.n - 1));
                if (a <= b) {
                    kf = (int)a;
                    kl = (int)b;
                }
            }
            if (P.semantics == BIRP_SEM_REFERENCE && kf != 0) kl = -1;
            if (kf <= kl) {
                const double dt = P.dt, t0 = (kf + 0.5) * dt;
                ix0 = (float)((P.px + dx * t0 - V.ox) * V.rdx);
                iy0 = (float)((P.py + dy * t0 - V.oy) * V.rdy);
                iz0 = (float)((P.pz + dz * t0 - V.oz) * V.rdz);
                dix = (float)(dx * dt * V.rdx);
                diy = (float)(dy * dt * V.rdy);
                diz = (float)(dz * dt * V.rdz);
            }
        }
    }
    const int cnt = (kl >= kf) ? (kl - kf + 1) : 0;
    if (!CMEM && cnt > 0) {
        // every sample inside [0, nextbelow(n - 1)] per axis, so that the cell index is the
        // truncation (0 .. n-2) with no clamp per sample; a sample rounded onto the far face
        // keeps weight ~1 on the last grid point
        fit_march(ix0, dix, __uint_as_float(__float_as_uint(V.fnx - 1.0f) - 1u), cnt - 1);
        fit_march(iy0, diy, __uint_as_float(__float_as_uint(V.fny - 1.0f) - 1u), cnt - 1);
        fit_march(iz0, diz, __uint_as_float(__float_as_uint(V.fnz - 1.0f) - 1u), cnt - 1);
    }
    float tot;
    if constexpr (SIGNED) {
        // Camera.cpp:207-210: a ray ends at its first negative sample. The S lanes of a ray take
        // samples q*S + sub in trip q, so the ray's first negative sample of a trip is the lowest
        // set bit of its S-bit group in the wave's ballot: a lane adds its sample unless its
        // group has a negative sample at or before it, and the ray dies with any in the group.
        const int my = (cnt > sub) ? (cnt - sub + S - 1) / S : 0;  // samples of this sub-lane
        const int trips = wave_max_i(my);
        float sum = 0.f, nc = 0.f;
        const int gshift = ray * S;
        bool alive = true;  // the same in all S lanes of a ray
        float xd = 0.f, yd = 0.f, zd = 0.f, xn, yn, zn;
        auto place = [&](int js, float& x, float& y, float& z) {
            const float fj = (float)min(js, cnt - 1);
            x = __builtin_fmaf(fj, dix, ix0);
            y = __builtin_fmaf(fj, diy, iy0);
            z = __builtin_fmaf(fj, diz, iz0);
        };
        // CMEM: U = 1 asks the zone bounds before each sample, U = 2 a trip ahead, U = 4 takes the model in full;
        // the samples are the same. With a wave per SIMD or less nothing hides the table's load and the zone's
        // branches, with a few only the load; with many the plain form has the most waves. us with U = 1 / 2 / 4:
        // 120x70 n = 300 51.5 / 45.2 / 40.3, 144x84 n = 320 39.7 / 33.8 / 42.9, 300x170 n = 300 64.7 / 63.6 / 92.8,
        // 576x336 n = 800 262 / 275 / 653.
        constexpr bool AHEAD = CMEM && U == 2;
        ZoneQuery zone{};
        if constexpr (AHEAD) {
            place(sub, xn, yn, zn);
            zone = zone_fetch(rs, xn, yn, zn);
        }
        for (int q = 0; q < trips; ++q) {
            const int js = q * S + sub;
            const bool act = alive && js < cnt;
            float x;
            if constexpr (AHEAD) {
                xd = xn;
                yd = yn;
                zd = zn;
                place(js + S, xn, yn, zn);
                const ZoneQuery next = zone_fetch(rs, xn, yn, zn);
                x = cmem_fast_zoned(V.cmem, zone, xd, yd, zd);
                zone = next;
            } else {
                place(js, xd, yd, zd);
                if constexpr (!CMEM) x = fast_value<DT>(fast_fetch<DT>(V, rs, tab, xd, yd, zd));
                else x = U == 4 ? cmem_fast(V.cmem, xd, yd, zd) : cmem_fast_zoned(V.cmem, zone_fetch(rs, xd, yd, zd), xd, yd, zd);
            }
            const unsigned long long neg = __ballot(act && x < 0.f);
            const unsigned grp = (unsigned)(neg >> gshift) & ((1u << S) - 1u);
            const bool cut = (grp & ((2u << sub) - 1u)) != 0u;
            kahan_add((act && !cut) ? x : 0.f, sum, nc);
            alive = alive && grp == 0u;
            if (__ballot(alive && (q + 1) * S < cnt) == 0ull) break;  // every ray of the wave is done
        }
        // each sub-lane's sum with its compensation, the S of them in FP64: the ray's total is rounded once
        tot = (float)sum_lanes<S>((double)sum + (double)nc, sub_step);
    }
    if constexpr (!SIGNED) {
        // Sample k of a ray, from its first, belongs to residue k mod 4; the samples of a residue are added in
        // order in FP64, then the four sums, and the total is rounded once. Lane `sub` takes the residues sub,
        // sub + S, ..., so the image does not depend on S, on the tile or on U, and a launch may choose
        // them (launch_tuning): single 300x170 x 500 FP16 renders 28.8 us with one lane per ray, 17.3 with
        // four. No number of samples loses a bit of the total: relative RMS error of the sum of 17 / 150 / 400
        // samples 2.4e-8 / 2.3e-8 / 1.8e-8, all of it the last rounding. Sums of four samples in FP32, one Kahan
        // step each and a rounded total per residue, gave 3.8e-8 / 3.4e-8 / 2.7e-8 and were 0.5% faster (256
        // mixed orbit views of F16 2.305 ms, 2.314 now; FP32 the same).
        // Rows that every ray of the wave fills need no clamp and no mask; the others run below with both,
        // and with the same sums: a masked sample adds 0.
        constexpr int R = 4 / S, B = U > R ? U / R : 1;  // residues per lane; rows of 4 samples in flight together
        double sum[R] = {};
        auto at = [&](float fj) {
            return fast_fetch<DT>(V, rs, tab, __builtin_fmaf(fj, dix, ix0), __builtin_fmaf(fj, diy, iy0), __builtin_fmaf(fj, diz, iz0));
        };
        FastFetch<DT> f[B * R];
        const int full = wave_min_i(cnt), most = wave_max_i(cnt);
        int row = 0;
        float fj = (float)sub;
        for (; row + 4 * B <= full; row += 4 * B, fj += 4.0f * B) {
#pragma unroll
            for (int c = 0; c < B * R; ++c) f[c] = at(fj + (float)(4 * (c / R) + S * (c % R)));
            // The next row's loads may rise above these lerps, which the few waves of 4 lanes per ray need (144x84 n =
            // 2000 FP32 42.7 -> 38.5 us); with 2 lanes and 16-bit records the registers that takes cost more
            // than it gives (1000x600 n = 2000 343 us with the barrier, 351 without).
            if constexpr (DT != BIRP_DTYPE_F32 && S == 2) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int c = 0; c < B * R; ++c) sum[c % R] += (double)fast_value<DT>(f[c]);
        }
        for (; row < most; row += 4 * B) {
            // a lane past its ray's last sample re-reads that sample (its result is masked); an
            // empty ray has i0 = d = 0 and samples the grid origin
            const int js = row + sub;
#pragma unroll
            for (int c = 0; c < B * R; ++c) f[c] = at((float)min(js + 4 * (c / R) + S * (c % R), cnt - 1));
            // here the compiler would issue the loads one by one, each waited for before the next (40x30 n = 2000
            // 41.2 -> 54.1 us)
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int c = 0; c < B * R; ++c) sum[c % R] += (double)(js + 4 * (c / R) + S * (c % R) < cnt ? fast_value<DT>(f[c]) : 0.f);
        }
        if constexpr (S == 1) tot = (float)((sum[0] + sum[1]) + (sum[2] + sum[3]));
        else if constexpr (S == 2) tot = (float)(pair_sum(sum[0], sub_step) + pair_sum(sum[1], sub_step));
        else tot = (float)sum_lanes<4>(sum[0], sub_step);
    }
    // the step weight and the scale constant are applied once per ray (all in FP32), the records' scale last: a
    // power of two changes no bit of a normal result, where scale * w could be subnormal
    if (valid && sub == 0) {
        float out = (tot * P.w) * K;
        if constexpr (!CMEM && DT == BIRP_KDT_F16_UNIFORM) out *= P.scale;
        P.out[(size_t)j * P.W + i] = out;
    }
}

// The wave tiles of many views in one launch, as a plain grid: a block renders 4 consecutive tiles of one view
// (prefix[k] = first block of view k), its waves sharing the view's offset tables in LDS, and the
// dispatcher balances the load. Blocks go round-robin over the 8 XCDs; block b renders item
// first + (c * 8 + b % 8) * chunk + i, its c-th chunk of BIRP_FAST_CHUNK: each XCD renders runs of neighbouring
// blocks, whose rays meet the same records in its L2, and a fair share of every view (chunks of 4 to 64
// measured within 2% of each other, 1 up to 5% slower on small views). A list of more blocks than a
// grid may have takes several launches (fast_piece).
// A persistent grid whose waves claimed tiles from 8 atomic queues took 20-80 us more per launch (every wave
// visits all queues before it leaves, and claims on one address serialize): 16 FP16 views of 288x168 x 320
// 154 -> 73 us, 16 of 576x336 x 800 556 -> 487 us, 256 mixed orbit views 2.37 -> 2.24 ms.
// KV is a kernel variant (fast_kernel_dtype): the storage kernel in its low bits, plus BIRP_KDT_SIGNED for
// volumes with negative values, whose rays stop at their first negative sample. Six waves per SIMD: the
// register allocation meets that with 4 samples in flight.
__device__ __forceinline__ void load_fast_tables(const DevVolume& V, bool f32, unsigned* tab, int entries) {
    const unsigned* src = f32 ? V.qtab : V.otab;
    const int n = min(V.nx + V.ny + V.nz, entries);  // the host sizes the LDS to cover it
    for (int q = threadIdx.x; q < n; q += BIRP_BLOCK) tab[q] = src[q];
    __syncthreads();
}

template <int KV, int S, int U>
__global__ __launch_bounds__(BIRP_BLOCK, 6) void k_render_fast(const DevVolume* __restrict__ vols, const FastPose* __restrict__ poses,
                                                               const int* __restrict__ prefix, int npose, int first, int count,
                                                               int tw_log2, int tab_entries) {
    constexpr bool CMEM = KV == BIRP_KDT_CMEM;
    constexpr int DT = CMEM ? BIRP_DTYPE_F32 : (KV & 3);
    constexpr bool SIGNED = CMEM || (KV & BIRP_KDT_SIGNED) != 0;
    static_assert(!SIGNED || U == 1, "signed kernels take one sample per lane per trip");
    extern __shared__ unsigned s_tab[];
    constexpr unsigned chunk = BIRP_FAST_CHUNK;
    const unsigned turn = blockIdx.x >> 3;
    const int at = (int)((turn / chunk * 8 + (blockIdx.x & 7u)) * chunk + turn % chunk);
    if (at >= count) return;
    const int g = first + at;
    const int k = find_view(prefix, npose, g);
    const FastPose& P = poses[k];
    const DevVolume& V = vols[P.vol];
    if constexpr (!CMEM) load_fast_tables(V, DT == BIRP_DTYPE_F32, s_tab, tab_entries);
    const FastLane fl = fast_lane<S, SIGNED>(lane_id(), tw_log2);
    const int tile = (g - prefix[k]) * (BIRP_BLOCK / 64) + (int)(threadIdx.x >> 6);
    if (tile < P.tiles_x * ((P.H + fl.th - 1) / fl.th)) fast_tile<KV, S, U>(V, P, tile, s_tab, fl);
}

// One pose as a plain grid, with the pose and its volume by value: the launch needs no descriptor
// upload (single fast renders, a lone served request). All its blocks run at once, so each XCD renders one
// contiguous range of neighbouring tiles: its L2 then fetches each record once (with the blocks dealt out
// one by one every XCD misses on nearly every record: 20-40% slower). The grid is a multiple of 8
// blocks; waves past the last tile leave at once.
template <int KV, int S, int U>
__global__ __launch_bounds__(BIRP_BLOCK, 6) void k_render_fast_one(DevVolume V, FastPose P, int total, int tw_log2, int tab_entries) {
    constexpr bool CMEM = KV == BIRP_KDT_CMEM;
    constexpr int DT = CMEM ? BIRP_DTYPE_F32 : (KV & 3);
    constexpr bool SIGNED = CMEM || (KV & BIRP_KDT_SIGNED) != 0;
    static_assert(CMEM || !SIGNED || U == 1, "signed kernels take one sample per lane per trip");
    extern __shared__ unsigned s_tab[];
    const int b = (int)(blockIdx.x & 7u) * (int)(gridDim.x >> 3) + (int)(blockIdx.x >> 3);
    const int item = b * (BIRP_BLOCK / 64) + (int)(threadIdx.x >> 6);
    if constexpr (!CMEM) load_fast_tables(V, DT == BIRP_DTYPE_F32, s_tab, tab_entries);
    if (item >= total) return;
    fast_tile<KV, S, U>(V, P, item, s_tab, fast_lane<S, SIGNED>(lane_id(), tw_log2));
}

// ------------------------------------------------------------------------------------------
// the fixed scratch of birp_render_views_noalloc
// ------------------------------------------------------------------------------------------
// Each GPU holds its own copy for the life of the process. In host code `scratch` names a host-side
// stand-in, not a device address: host code uses only the address noalloc_scratch_address returns.
static __device__ __align__(256) unsigned char scratch[BIRP_NOALLOC_SCRATCH_BYTES];

static_assert(sizeof(DevVolume) <= BIRP_NOALLOC_POSE_OFF, "noalloc scratch: volume slot");
static_assert(BIRP_NOALLOC_SCRATCH_BYTES <= BIRP_NOALLOC_SCRATCH_KIB * 1024, "noalloc scratch: stated size");
static_assert(sizeof(FastPose) <= 256, "noalloc scratch: pose slot");
static_assert(3 * (BIRP_NOALLOC_MAX_VIEWS + 1) * 4 <= BIRP_NOALLOC_SCRATCH_BYTES - BIRP_NOALLOC_PREFIX_OFF, "noalloc scratch: prefix");

struct NoallocHead {
    DevVolume v;
    int prefix[3 * (BIRP_NOALLOC_MAX_VIEWS + 1)];
};
struct NoallocPoses {
    FastPose p[4];
    int first, count;
};

__global__ __launch_bounds__(BIRP_BLOCK) void k_noalloc_head(NoallocHead h, unsigned char* s) {
    if (threadIdx.x == 0) *reinterpret_cast<DevVolume*>(s) = h.v;
    int* pre = reinterpret_cast<int*>(s + BIRP_NOALLOC_PREFIX_OFF);
    for (int i = threadIdx.x; i < 3 * (BIRP_NOALLOC_MAX_VIEWS + 1); i += BIRP_BLOCK) pre[i] = h.prefix[i];
}

__global__ void k_noalloc_poses(NoallocPoses c, unsigned char* s) {
    FastPose* dst = reinterpret_cast<FastPose*>(s + BIRP_NOALLOC_POSE_OFF) + c.first;
#pragma unroll
    for (int q = 0; q < 4; q++)
        if (threadIdx.x == q && q < c.count) dst[q] = c.p[q];
}

int noalloc_scratch_address(void** out) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
        (void)hipGetLastError();
        return BIRP_ERR_DEVICE;
    }
    *out = p;
    return BIRP_OK;
}

int noalloc_stage_head(const DevVolume& v, const int* prefix, void* s, void* stream) {
    NoallocHead h;
    h.v = v;
    for (int i = 0; i < 3 * (BIRP_NOALLOC_MAX_VIEWS + 1); i++) h.prefix[i] = prefix[i];
    hipLaunchKernelGGL(k_noalloc_head, dim3(1), dim3(BIRP_BLOCK), 0, (hipStream_t)stream, h, (unsigned char*)s);
    return hipGetLastError() == hipSuccess ? BIRP_OK : BIRP_ERR_DEVICE;
}

int noalloc_stage_poses(const FastPose* poses, int first, int count, void* s, void* stream) {
    if (count < 1 || count > 4 || first < 0 || first + count > BIRP_NOALLOC_MAX_VIEWS) return BIRP_ERR_INVALID_ARGUMENT;
    NoallocPoses c;
    for (int q = 0; q < count; q++) c.p[q] = poses[q];
    c.first = first;
    c.count = count;
    hipLaunchKernelGGL(k_noalloc_poses, dim3(1), dim3(64), 0, (hipStream_t)stream, c, (unsigned char*)s);
    return hipGetLastError() == hipSuccess ? BIRP_OK : BIRP_ERR_DEVICE;
}

// ------------------------------------------------------------------------------------------
// host-side launch wrappers
// ------------------------------------------------------------------------------------------
static int hip_status(hipError_t e) { return e == hipSuccess ? BIRP_OK : BIRP_ERR_DEVICE; }

int exact_mode_of(const DevVolume& v, const ExactView& ev) {
    if (v.kind == SK_CMEM) return SM_CMEM;
    const bool nonneg = (v.vclass == VC_POSITIVE || v.vclass == VC_NONNEG) && v.origin_far && ev.fast_guards;
    if (v.interp == BIRP_INTERP_NEAREST) {
        const size_t slice = (size_t)v.nx * v.ny;  // near_fetch: 24-bit products, 32-bit byte offsets
        return nonneg && slice < (1u << 24) && slice * v.nz < (1u << 30) ? SM_NEAR_NN : SM_LIN_NEAREST;
    }
    if (v.vclass == VC_NONFINITE || !v.quad || !v.qtab) return SM_LIN_TRI;
    if (nonneg) return v.vclass == VC_POSITIVE ? SM_QUAD_POS : SM_QUAD_NN;
    return SM_QUAD_GEN;
}

size_t exact_lds_bytes(const DevVolume& v, int n, int mode) {
    size_t lds = (size_t)((n + 3) & ~3) * sizeof(float);
    if (mode == SM_QUAD_POS || mode == SM_QUAD_NN || mode == SM_QUAD_GEN) lds += (size_t)(v.nx + v.ny + v.nz) * sizeof(unsigned);
    return lds;
}

template <int S>
static int launch_exact_s(const DevVolume& v, const ExactView& ev, int pipe, hipStream_t st, const ExactOrder* ord) {
    constexpr int TW = ExactTile<S>::TW, TH = ExactTile<S>::TH;
    int wg_x = (ev.W + 2 * TW - 1) / (2 * TW);
    int wg_y = (ev.H + 2 * TH - 1) / (2 * TH);
    int nblocks = wg_x * wg_y;
    const int grid = nblocks;
    const int mode = exact_mode_of(v, ev);
    const size_t lds = exact_lds_bytes(v, ev.n, mode);
    if (lds > 64 * 1024) return BIRP_ERR_UNSUPPORTED;
    const int* order = nullptr;
    int ncu = 0;
    if (ord && ord->order) {
        if (nblocks > BIRP_PLAN_MAX_BLOCKS || ord->ncu <= 0 || mode == SM_CMEM) return BIRP_ERR_INVALID_ARGUMENT;
        if (ord->replan) {
            hipLaunchKernelGGL((k_exact_plan<S>), dim3((4 * nblocks + BIRP_BLOCK - 1) / BIRP_BLOCK), dim3(BIRP_BLOCK), 0, st, v, ev,
                               wg_x, nblocks, ord->order);
            const int rc = hip_status(hipGetLastError());
            if (rc) return rc;
        }
        order = ord->order;
        ncu = ord->ncu;
    }
    switch (mode) {
#define BIRP_LRE(MODE, P) hipLaunchKernelGGL((k_render_exact<S, MODE, P>), dim3(grid), dim3(BIRP_BLOCK), lds, st, v, ev, wg_x, nblocks, order, ncu)
        case SM_QUAD_POS:
            if (pipe >= 4) BIRP_LRE(SM_QUAD_POS, 4);
            else if (pipe == 3) BIRP_LRE(SM_QUAD_POS, 3);
            else if (pipe == 1) BIRP_LRE(SM_QUAD_POS, 1);
            else BIRP_LRE(SM_QUAD_POS, 2);
            break;
        case SM_QUAD_NN:
            if (pipe >= 3) BIRP_LRE(SM_QUAD_NN, 3);
            else BIRP_LRE(SM_QUAD_NN, 2);
            break;
        case SM_NEAR_NN:
            if (pipe >= 3) BIRP_LRE(SM_NEAR_NN, 4);
            else BIRP_LRE(SM_NEAR_NN, 2);
            break;
#undef BIRP_LRE
        case SM_QUAD_GEN: hipLaunchKernelGGL((k_render_exact<S, SM_QUAD_GEN>), dim3(grid), dim3(BIRP_BLOCK), lds, st, v, ev, wg_x, nblocks, order, ncu); break;
        case SM_LIN_TRI: hipLaunchKernelGGL((k_render_exact<S, SM_LIN_TRI>), dim3(grid), dim3(BIRP_BLOCK), lds, st, v, ev, wg_x, nblocks, order, ncu); break;
        case SM_LIN_NEAREST: hipLaunchKernelGGL((k_render_exact<S, SM_LIN_NEAREST>), dim3(grid), dim3(BIRP_BLOCK), lds, st, v, ev, wg_x, nblocks, order, ncu); break;
        default: hipLaunchKernelGGL((k_render_exact<S, SM_CMEM>), dim3(grid), dim3(BIRP_BLOCK), lds, st, v, ev, wg_x, nblocks, order, ncu); break;
    }
    return hip_status(hipGetLastError());
}

template <int S>
static int exact_blocks(int W, int H) {
    constexpr int TW = ExactTile<S>::TW, TH = ExactTile<S>::TH;
    return ((W + 2 * TW - 1) / (2 * TW)) * ((H + 2 * TH - 1) / (2 * TH));
}

int exact_tiles(int W, int H, int lanes_per_ray) {
    if (lanes_per_ray == 16) return exact_blocks<16>(W, H);
    if (lanes_per_ray == 8) return exact_blocks<8>(W, H);
    return lanes_per_ray == 4 ? exact_blocks<4>(W, H) : (lanes_per_ray == 1 ? exact_blocks<1>(W, H) : exact_blocks<2>(W, H));
}

int exact_wave_slots(int W, int H, int lanes_per_ray) { return 4 * exact_tiles(W, H, lanes_per_ray); }

template <int S>
static int launch_exact_multi_s(const DevVolume* vols, const ExactView* views, const int* prefix, int nview, int total, int mode,
                                size_t lds, hipStream_t st, const int* order, int pipe) {
    const int grid = total;
    switch (mode) {
#define BIRP_LRM(MODE, P) hipLaunchKernelGGL((k_render_exact_multi<S, MODE, P>), dim3(grid), dim3(BIRP_BLOCK), lds, st, vols, views, prefix, nview, total, order)
        case SM_QUAD_POS:
            if (pipe >= 4) BIRP_LRM(SM_QUAD_POS, 4);
            else BIRP_LRM(SM_QUAD_POS, 2);
            break;
        case SM_QUAD_NN:
            if (pipe >= 4) BIRP_LRM(SM_QUAD_NN, 3);
            else BIRP_LRM(SM_QUAD_NN, 2);
            break;
        case SM_NEAR_NN:
            if (pipe >= 4) BIRP_LRM(SM_NEAR_NN, 4);
            else BIRP_LRM(SM_NEAR_NN, 2);
            break;
#undef BIRP_LRM
        case SM_QUAD_GEN: hipLaunchKernelGGL((k_render_exact_multi<S, SM_QUAD_GEN>), dim3(grid), dim3(BIRP_BLOCK), lds, st, vols, views, prefix, nview, total, order); break;
        case SM_LIN_TRI: hipLaunchKernelGGL((k_render_exact_multi<S, SM_LIN_TRI>), dim3(grid), dim3(BIRP_BLOCK), lds, st, vols, views, prefix, nview, total, order); break;
        case SM_LIN_NEAREST: hipLaunchKernelGGL((k_render_exact_multi<S, SM_LIN_NEAREST>), dim3(grid), dim3(BIRP_BLOCK), lds, st, vols, views, prefix, nview, total, order); break;
        default: return BIRP_ERR_INVALID_ARGUMENT;
    }
    return hip_status(hipGetLastError());
}

int launch_exact_multi(const DevVolume* vols, const ExactView* views, const int* prefix, int nview, int total, int mode,
                       size_t lds, void* stream, const int* order, int lanes, int pipe) {
    if (nview <= 0 || total <= 0) return BIRP_OK;
    if (lds > 64 * 1024) return BIRP_ERR_UNSUPPORTED;
    hipStream_t st = (hipStream_t)stream;
    if (mode == SM_CMEM) {  // always 4 lanes per ray (exact_multi_lanes)
        hipLaunchKernelGGL((k_render_exact_multi<4, SM_CMEM>), dim3(total), dim3(BIRP_BLOCK), lds, st, vols, views, prefix, nview, total, order);
        return hip_status(hipGetLastError());
    }
    if (lanes == 8) return launch_exact_multi_s<8>(vols, views, prefix, nview, total, mode, lds, st, order, pipe);
    if (lanes == 4) return launch_exact_multi_s<4>(vols, views, prefix, nview, total, mode, lds, st, order, pipe);
    if (lanes == 2) return launch_exact_multi_s<2>(vols, views, prefix, nview, total, mode, lds, st, order, pipe);
    return BIRP_ERR_INVALID_ARGUMENT;
}

int launch_plan_multi(const DevVolume* vols, const ExactView* views, const int* prefix, int nview, int total, int mode, int* cost,
                      void* stream, int lanes) {
    if (nview <= 0 || total <= 0 || mode == SM_CMEM || (lanes != 2 && lanes != 4 && lanes != 8)) return BIRP_ERR_INVALID_ARGUMENT;
    const long long threads = 4LL * total;
    const dim3 grid((unsigned)((threads + BIRP_BLOCK - 1) / BIRP_BLOCK));
    if (lanes == 8) hipLaunchKernelGGL((k_plan_multi<8>), grid, dim3(BIRP_BLOCK), 0, (hipStream_t)stream, vols, views, prefix, nview, total, cost);
    else if (lanes == 4) hipLaunchKernelGGL((k_plan_multi<4>), grid, dim3(BIRP_BLOCK), 0, (hipStream_t)stream, vols, views, prefix, nview, total, cost);
    else hipLaunchKernelGGL((k_plan_multi<2>), grid, dim3(BIRP_BLOCK), 0, (hipStream_t)stream, vols, views, prefix, nview, total, cost);
    return hip_status(hipGetLastError());
}

int launch_exact(const DevVolume& v, const ExactView& ev, int lanes_per_ray, int pipe, void* stream, const ExactOrder* ord) {
    if (ev.n < 2 || ev.n > BIRP_MAX_EXACT_SAMPLES || ev.W <= 0 || ev.H <= 0) return BIRP_ERR_INVALID_ARGUMENT;
    hipStream_t st = (hipStream_t)stream;
    if (lanes_per_ray == 16) return launch_exact_s<16>(v, ev, pipe, st, ord);
    if (lanes_per_ray == 8) return launch_exact_s<8>(v, ev, pipe, st, ord);
    if (lanes_per_ray == 4) return launch_exact_s<4>(v, ev, pipe, st, ord);
    if (lanes_per_ray == 2) return launch_exact_s<2>(v, ev, pipe, st, ord);
    return launch_exact_s<1>(v, ev, pipe, st, ord);
}

template <int S>
static int launch_plan_s(const DevVolume& v, const ExactView& ev, int* order, hipStream_t st) {
    constexpr int TW = ExactTile<S>::TW, TH = ExactTile<S>::TH;
    const int wg_x = (ev.W + 2 * TW - 1) / (2 * TW);
    const int nblocks = wg_x * ((ev.H + 2 * TH - 1) / (2 * TH));
    if (nblocks > BIRP_PLAN_MAX_BLOCKS) return BIRP_ERR_INVALID_ARGUMENT;
    hipLaunchKernelGGL((k_exact_plan<S>), dim3((4 * nblocks + BIRP_BLOCK - 1) / BIRP_BLOCK), dim3(BIRP_BLOCK), 0, st, v, ev, wg_x,
                       nblocks, order);
    return hip_status(hipGetLastError());
}

int launch_exact_plan(const DevVolume& v, const ExactView& ev, int lanes_per_ray, int* order, void* stream) {
    if (ev.n < 2 || ev.W <= 0 || ev.H <= 0 || !order) return BIRP_ERR_INVALID_ARGUMENT;
    hipStream_t st = (hipStream_t)stream;
    if (lanes_per_ray == 16) return launch_plan_s<16>(v, ev, order, st);
    if (lanes_per_ray == 8) return launch_plan_s<8>(v, ev, order, st);
    if (lanes_per_ray == 4) return launch_plan_s<4>(v, ev, order, st);
    if (lanes_per_ray == 2) return launch_plan_s<2>(v, ev, order, st);
    return launch_plan_s<1>(v, ev, order, st);
}

int launch_f64(const DevVolume& v, const F64View& fv, void* stream) {
    int npix = fv.W * fv.H;
    hipLaunchKernelGGL(k_render_f64, dim3((npix + BIRP_BLOCK - 1) / BIRP_BLOCK), dim3(BIRP_BLOCK), 0, (hipStream_t)stream, v, fv);
    return hip_status(hipGetLastError());
}

int launch_space_points(const ExactView& ev, int row0, int rows, float* xyz, void* stream) {
    const long long total = (long long)rows * ev.W * ev.n;
    if (total <= 0) return BIRP_OK;
    hipLaunchKernelGGL(k_space_points, dim3((unsigned)((total + BIRP_BLOCK - 1) / BIRP_BLOCK)), dim3(BIRP_BLOCK), 0, (hipStream_t)stream,
                       ev, row0, rows, xyz);
    return hip_status(hipGetLastError());
}

int launch_space_integrate(const ExactView& ev, int row0, int rows, const float* vals, float* img, void* stream) {
    const long long total = (long long)rows * ev.W;
    if (total <= 0) return BIRP_OK;
    hipLaunchKernelGGL(k_space_integrate, dim3((unsigned)((total + BIRP_BLOCK - 1) / BIRP_BLOCK)), dim3(BIRP_BLOCK), 0,
                       (hipStream_t)stream, ev, row0, rows, vals, img);
    return hip_status(hipGetLastError());
}

int launch_sample_points(const DevVolume& v, const float* xyz, long long n, float* out, void* stream) {
    if (n <= 0) return BIRP_OK;
    long long blocks = (n + BIRP_BLOCK - 1) / BIRP_BLOCK;
    hipLaunchKernelGGL(k_sample_points, dim3((unsigned)blocks), dim3(BIRP_BLOCK), 0, (hipStream_t)stream, v, xyz, n, out);
    return hip_status(hipGetLastError());
}

int launch_scan_class(const float* values, size_t n, unsigned* flags_dev, void* stream, float* copy_to) {
    const size_t blocks = std::min<size_t>((n / 4 + BIRP_BLOCK) / BIRP_BLOCK, 512);
    if (copy_to) hipLaunchKernelGGL((k_scan_class<true>), dim3((unsigned)blocks), dim3(BIRP_BLOCK), 0, (hipStream_t)stream, values, n, flags_dev, copy_to);
    else hipLaunchKernelGGL((k_scan_class<false>), dim3((unsigned)blocks), dim3(BIRP_BLOCK), 0, (hipStream_t)stream, values, n, flags_dev, nullptr);
    return hip_status(hipGetLastError());
}

int launch_check_div(const DevVolume& v, unsigned* bad_dev, void* stream) {
    DivCheck c{{v.rhx}, {v.rlx}, {v.rdx}, 1};
    auto add = [&](float rh, float rl, double rd) {
        for (int k = 0; k < c.n; k++)
            if (c.rd[k] == rd) return;  // RN64(1 / spacing) tells floats apart
        c.rh[c.n] = rh;
        c.rl[c.n] = rl;
        c.rd[c.n++] = rd;
    };
    add(v.rhy, v.rly, v.rdy);
    add(v.rhz, v.rlz, v.rdz);
    const unsigned grid = (1u << 23) / kDivPerThread / BIRP_BLOCK;
    hipLaunchKernelGGL(k_check_div, dim3(grid), dim3(BIRP_BLOCK), 0, (hipStream_t)stream, c, bad_dev);
    return hip_status(hipGetLastError());
}

// blocks of a layout build: one per 4 bricks along x, a multiple of 8
static int brick_row_grid(const DevVolume& v, int nbz) {
    const long long rows = (long long)((v.nbx + kBrickRow - 1) / kBrickRow) * v.nby * nbz;
    return (int)((rows + 7) / 8 * 8);
}

int launch_cmem_zones(const CmemParams& m, void* zones, void* stream) {
    hipLaunchKernelGGL(k_cmem_zones, dim3((BIRP_ZONE_CT * BIRP_ZONE_CP + BIRP_BLOCK - 1) / BIRP_BLOCK), dim3(BIRP_BLOCK), 0, (hipStream_t)stream, m,
                       (float4*)zones);
    return hip_status(hipGetLastError());
}

int launch_build_quad(const DevVolume& v, void* quad, void* stream) {
    hipLaunchKernelGGL(k_build_quad, dim3(brick_row_grid(v, (v.nz + 7) / 8)), dim3(BIRP_BLOCK), 0, (hipStream_t)stream, v, (unsigned char*)quad);
    return hip_status(hipGetLastError());
}

int launch_build_oct(const DevVolume& v, void* oct, float* bscale, void* stream) {
    const dim3 grid(brick_row_grid(v, v.nbz));
    auto kernel = v.dtype == BIRP_DTYPE_F16 ? k_build_oct<OCT_F16> : v.f16_uniform ? k_build_oct<OCT_BF16_AS_F16> : k_build_oct<OCT_BF16>;
    hipLaunchKernelGGL(kernel, grid, dim3(BIRP_BLOCK), 0, (hipStream_t)stream, v, (unsigned char*)oct, bscale);
    return hip_status(hipGetLastError());
}

int launch_zero_f32(float* p, size_t n, void* stream) {
    size_t blocks = (n + BIRP_BLOCK - 1) / BIRP_BLOCK;
    if (blocks > 4096) blocks = 4096;
    if (blocks == 0) blocks = 1;
    hipLaunchKernelGGL(k_zero_f32, dim3((unsigned)blocks), dim3(BIRP_BLOCK), 0, (hipStream_t)stream, p, n);
    return hip_status(hipGetLastError());
}

// U as the kernels take it: the signed kernels one sample per lane per trip, a single CMEM view's kernel its way
// of asking the zone bounds (many views' have the waves for the plain one), the others at least a lane's 4 / S
// residues.
template <int KV, int S, int U>
constexpr int fast_unroll() {
    return (KV & BIRP_KDT_SIGNED) ? 1 : (KV & BIRP_KDT_CMEM) ? U : (U > 4 / S ? U : 4 / S);
}

// Calls launch(std::integral_constant KV, S, U) for the variant asked for.
template <int KV, int S, class F>
static int with_unroll(int u, F&& launch) {
    if (u == 4) return launch(std::integral_constant<int, KV>(), std::integral_constant<int, S>(), std::integral_constant<int, fast_unroll<KV, S, 4>()>());
    if (u == 2) return launch(std::integral_constant<int, KV>(), std::integral_constant<int, S>(), std::integral_constant<int, fast_unroll<KV, S, 2>()>());
    return launch(std::integral_constant<int, KV>(), std::integral_constant<int, S>(), std::integral_constant<int, fast_unroll<KV, S, 1>()>());
}
template <int KV, class F>
static int with_lanes(int s, int u, F&& launch) {
    return s == 4 ? with_unroll<KV, 4>(u, launch) : s == 2 ? with_unroll<KV, 2>(u, launch) : with_unroll<KV, 1>(u, launch);
}
template <class F>
static int with_variant(int dtype, int s, int u, F&& launch) {
    switch (dtype) {
        case 0: return with_lanes<0>(s, u, launch);
        case 1: return with_lanes<1>(s, u, launch);
        case 2: return with_lanes<2>(s, u, launch);
        case 3: return with_lanes<3>(s, u, launch);
        case 4: return with_lanes<4>(s, u, launch);
        case 5: return with_lanes<5>(s, u, launch);
        case 6: return with_lanes<6>(s, u, launch);
        case 7: return with_lanes<7>(s, u, launch);
        case 8: return with_lanes<8>(s, u, launch);
        default: return BIRP_ERR_INVALID_ARGUMENT;
    }
}

// log2 of the tile's width, or -1 for a tile and lanes that do not make a wave
static int tile_log2(int tile_w, int tile_h, int lanes_per_ray) {
    int twl = 0;
    while ((1 << twl) < tile_w) twl++;
    return (1 << twl) == tile_w && tile_w * tile_h * lanes_per_ray == 64 ? twl : -1;
}
static size_t fast_lds_bytes(int dtype, int tab_entries) { return dtype == BIRP_KDT_CMEM ? 0 : (size_t)tab_entries * sizeof(unsigned); }

int launch_fast_batch(const DevVolume* vols_dev, int dtype, const FastPose* poses_dev, const int* block_prefix_dev, int npose,
                      int total_blocks, int tile_w, int tile_h, int lanes_per_ray, int unroll, void* stream, int tab_entries) {
    const int twl = tile_log2(tile_w, tile_h, lanes_per_ray);
    if (twl < 0 || npose < 1 || total_blocks < 1 || tab_entries < 0 || tab_entries > BIRP_FAST_TAB) return BIRP_ERR_INVALID_ARGUMENT;
    return with_variant(dtype, lanes_per_ray, unroll, [&](auto kv, auto s, auto u) {
        constexpr int U = kv.value == BIRP_KDT_CMEM ? 1 : u.value;
        int rc = BIRP_OK;
        for (int first = 0; first < total_blocks && rc == BIRP_OK;) {
            const FastPiece p = fast_piece(total_blocks, first);
            hipLaunchKernelGGL((k_render_fast<kv.value, s.value, U>), dim3(p.grid), dim3(BIRP_BLOCK), fast_lds_bytes(dtype, tab_entries),
                               (hipStream_t)stream, vols_dev, poses_dev, block_prefix_dev, npose, p.first, p.count, twl, tab_entries);
            rc = hip_status(hipGetLastError());
            if (total_blocks - first <= p.count) break;
            first += p.count;
        }
        return rc;
    });
}

int launch_fast_one(const DevVolume& v, int dtype, const FastPose& pose, int total_tiles, int tile_w, int tile_h, int lanes_per_ray,
                    int unroll, void* stream, int tab_entries) {
    const int twl = tile_log2(tile_w, tile_h, lanes_per_ray);
    if (twl < 0 || tab_entries < 0 || tab_entries > BIRP_FAST_TAB || total_tiles < 0) return BIRP_ERR_INVALID_ARGUMENT;
    if (total_tiles == 0) return BIRP_OK;
    const int blocks = fast_blocks(total_tiles), grid = (blocks + 7) / 8 * 8;
    // the variants that launch_tuning and view_tuning ask for: 4 samples in flight, CMEM with 4 lanes per ray
    return with_variant(dtype, lanes_per_ray, unroll, [&](auto kv, auto s, auto u) {
        constexpr int KV = kv.value, S = s.value, U = u.value;
        if constexpr (KV == BIRP_KDT_CMEM ? S == 4 : (KV & BIRP_KDT_SIGNED) || U == 4) {
            hipLaunchKernelGGL((k_render_fast_one<KV, S, U>), dim3(grid), dim3(BIRP_BLOCK), fast_lds_bytes(dtype, tab_entries),
                               (hipStream_t)stream, v, pose, total_tiles, twl, tab_entries);
            return hip_status(hipGetLastError());
        } else {
            return (int)BIRP_ERR_INVALID_ARGUMENT;
        }
    });
}

}  // namespace birp
