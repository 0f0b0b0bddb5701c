// vv_lic_dev.hpp — device code of the LIC integral shared by the LIC-volume
// kernels (vv_lic.hip) and the fused on-the-fly ray caster (vv_render.hip):
// the argument block, field and noise sampling, the per-lane cell caches and
// the LIC of one seed point.  Included inside an anonymous namespace.
#pragma once


struct LicArgs {
    Vol<void> field;
    Vol<void> noise;
    Vol<uint8_t> scalar;
    const float* w;
    int F, B;
    float he, scl, freq, gate_lo, gate_hi;
    float sc0, sc1, sc2;
    float* out;
    int osy, osz;
    unsigned field_bytes, noise_bytes;  // buffer sizes for the cached kernels
    int tx, ty, tz;      // block tile
    int gx, gy, gz;      // tiles per axis
    int nblocks;         // gx*gy*gz
    int per_xcd;         // tiles handled by each of the 8 XCDs
    int sx, sy, sz;      // super-tile size in tiles (3D-blocked tile order)
    int speed;           // SPEED_OF_FLOW, for lic_point (the cached kernels take it as a template argument)
    int bsy, bsz;        // BRICK kernels: field.p is the 8^3-brick copy with these brick-row and
                         // brick-plane strides (elements)
};

// logical tile t -> tile coordinates: super-tiles in raster order, tiles
// raster order inside each super-tile, so the tiles resident on one XCD at a
// time cover a compact 3D region whose streamline halo fits that XCD's L2.
// The last super-tile of an axis holds what is left of the tile grid, so every
// t < gx*gy*gz is a tile of the volume and the eight XCDs get equal runs of
// them.  (Whole super-tiles past the volume gave 160^3 voxels a grid of
// 160x192x192, its empty part in a few XCDs' runs: an animation frame of it
// took 1.50 ms against 1.22, the gated LIC of 200x152x97 voxels 3.36 against
// 2.06; 256^3, which whole super-tiles fill, 5.66 either way.)
__device__ __forceinline__ void tile_coords(const LicArgs& a, int t, int& bx, int& by, int& bz)
{
    // slab of super-tiles along z, then its row along y, then the super-tile
    const int slab = a.gx * a.gy * a.sz;
    const int uz = t / slab;
    t -= uz * slab;
    const int hz = min(a.sz, a.gz - uz * a.sz);
    const int row = a.gx * a.sy * hz;
    const int uy = t / row;
    t -= uy * row;
    const int hy = min(a.sy, a.gy - uy * a.sy);
    const int box = a.sx * hy * hz;
    const int ux = t / box;
    t -= ux * box;
    const int hx = min(a.sx, a.gx - ux * a.sx);
    const int ty = t / hx;
    bx = ux * a.sx + t - ty * hx;
    by = uy * a.sy + ty % hy;
    bz = uz * a.sz + ty / hy;
}

template <int NC>
struct NoiseT;
template <>
struct NoiseT<1> {
    using T = uint8_t;
};
template <>
struct NoiseT<4> {
    using T = uchar4;
};

// noise sample n(x): freqSampling (inc_lic.glsl:71-90) for scalar noise,
// freqSamplingGrad (:61-68, no frequency scale, no gate) for RGBA noise
template <int NC, bool GATE>
__device__ __forceinline__ float4 noise_at(const LicArgs& a, float x, float y, float z)
{
    float4 n = make_float4(0.f, 0.f, 0.f, 0.f);
    if constexpr (NC == 4) {
        const Vol<uchar4> nv{(const uchar4*)a.noise.p, {a.noise.n[0], a.noise.n[1], a.noise.n[2]},
                             a.noise.sy, a.noise.sz};
        Cell c = cell_repeat(nv, x, y, z);
        float4 r = tri_u8x4(nv, c);
        n.x = r.x * kInv255;
        n.y = r.y * kInv255;
        n.z = r.z * kInv255;
        n.w = r.w * kInv255;
    } else {
        if constexpr (GATE) {
            Cell cs = cell_clamp(a.scalar, x, y, z);
            float s = tri_u8(a.scalar, cs) * kInv255;
            if (!(s > a.gate_lo && s < a.gate_hi)) return n;
        }
        const Vol<uint8_t> nv{(const uint8_t*)a.noise.p, {a.noise.n[0], a.noise.n[1], a.noise.n[2]},
                              a.noise.sy, a.noise.sz};
        Cell c = cell_repeat(nv, x * a.freq, y * a.freq, z * a.freq);
        n.x = tri_u8(nv, c) * kInv255;
    }
    return n;
}

template <typename FT>
__device__ __forceinline__ float3 field_rgb(const LicArgs& a, float x, float y, float z)
{
    const Vol<FT> fv{(const FT*)a.field.p, {a.field.n[0], a.field.n[1], a.field.n[2]}, a.field.sy,
                     a.field.sz};
    Cell c = cell_clamp(fv, x, y, z);
    return tri_rgb(fv, c);
}

// direction and magnitude (.a = |v|/max) of the field
template <typename FT>
__device__ __forceinline__ float4 field_rgba(const LicArgs& a, float x, float y, float z)
{
    const Vol<FT> fv{(const FT*)a.field.p, {a.field.n[0], a.field.n[1], a.field.n[2]}, a.field.sy,
                     a.field.sz};
    Cell c = cell_clamp(fv, x, y, z);
    return tri_rgba(fv, c);
}

// Stores one LIC voxel into the REPEAT-padded output and into the copies
// of plane 0 at index n along each axis (the wrap halo), so no separate
// halo pass is needed.
template <typename T>
__device__ __forceinline__ void store_repeat(T* out, int osy, int osz, int x, int y, int z, int nx, int ny,
                                             int nz, T v)
{
    const long long o = (long long)z * osz + (long long)y * osy + x;
    out[o] = v;
    const bool hx = x == 0, hy = y == 0, hz = z == 0;
    if (hx | hy | hz) {
        const long long ox = nx, oy = (long long)ny * osy, oz = (long long)nz * osz;
        if (hx) out[o + ox] = v;
        if (hy) out[o + oy] = v;
        if (hz) out[o + oz] = v;
        if (hx & hy) out[o + ox + oy] = v;
        if (hx & hz) out[o + ox + oz] = v;
        if (hy & hz) out[o + oy + oz] = v;
        if (hx & hy & hz) out[o + ox + oy + oz] = v;
    }
}

// Per-lane cache of the last trilinear cell.  Consecutive samples of a
// streamline are ~h_e*n voxels apart (0.38 at 256^3, h = 0.005), so the
// corrector sample almost always lands in the predictor's cell and the next
// predictor often in the same cell: a lane that hits skips its gathers (it
// is masked off the loads).  For each channel the cache keeps the four x0
// texels and the four differences (x1 - x0) of the cell, so the four x-lerps
// of a hit are single fmas; the values and the operation order are exactly
// those of tri(), so results do not change.
// NCH = 3: the field direction; NCH = 4: also the noise byte that the LIC
// copy of the field carries in channel 3 (equal field and noise grids)
// A cache is keyed by the three floors k of its cell.  A texel coordinate t =
// u n - 0.5 lies in the cell when every t - k is in [0, 1), and t - k is then
// the fraction t - floor(t) itself, so a hit needs no floor: the three
// differences are compared at once as unsigned words (the bits of a float in
// [0, 1) lie below those of 1, a negative, larger or NaN difference above).
// NaN keys never hit; a coordinate so little below an integer that its
// fraction rounds to 1 is filled again, with the same texels.  (Cells
// outside the volume with different floors but the same clamped texels are
// reloaded, with the same values.)  On gfx950 floor, compare, convert, min, max
// and 24-bit multiplies issue at 0.97 wave64 instructions per clock per CU,
// fma, add, sub, mul and mov of vector operands at 1.7 (0.97 with a scalar
// one; measured), so the kernels spend their compares and conversions on a
// miss: 256^3, L = 40, FP16 4.44 -> 4.27 ms, UNORM8 4.73 -> 4.53, FP16 with noise on
// another grid 7.04 -> 6.31.  Some fills of field_at are better tested by floors
// (fill_hit).
// v_fma_mix_f32 with one half operand, which the instruction widens exactly
// (every half is a float), so each form is one rounding of the exact result:
//   fma_half<HI>(a, b, w) = fmaf(a, b, (float)h), h the low (HI 0) or high
//   (HI 1) half of w;
//   sub_half<HI>(w1, w0)  = (float)h1 - (float)h0.
// They let the FP16 cell cache keep its x0 texels packed as loaded and skip
// every half-to-float conversion of a cell fill.
template <int HI>
__device__ __forceinline__ float fma_half(float a, float b, unsigned w)
{
    float r;
    if constexpr (HI)
        asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "=v"(r) : "v"(a), "v"(b), "v"(w));
    else
        asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[0,0,1]" : "=v"(r) : "v"(a), "v"(b), "v"(w));
    return r;
}

template <int HI>
__device__ __forceinline__ float sub_half(unsigned w1, unsigned w0)
{
    float r;
    if constexpr (HI)
        asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[1,0,1] op_sel_hi:[1,0,1]" : "=v"(r) : "v"(w1), "v"(w0));
    else
        asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel_hi:[1,0,1]" : "=v"(r) : "v"(w1), "v"(w0));
    return r;
}

// FP32 and UNORM8 texels: x0 texels and differences as floats
template <typename FT, int NCH>
struct FieldCache {
    float kx, ky, kz;   // floors of the cached cell
    bool same;          // NCH 4: the cell's noise bytes are those of the REPEAT cell
    float v0[NCH][4];   // [channel][(y,z) corner]: texel at x0
    float dx[NCH][4];   // texel(x1) - texel(x0)
    __device__ __forceinline__ void reset() { kx = ky = kz = __builtin_nanf(""); same = false; }
    // x-lerp of channel CH on corner row k: fma(fx, x1 - x0, x0)
    template <int CH>
    __device__ __forceinline__ float xlerp(int k, float fx) const { return fmaf(fx, dx[CH][k], v0[CH][k]); }
    __device__ __forceinline__ void set_row(int k, const float* t0, const float* t1)
    {
#pragma unroll
        for (int ch = 0; ch < NCH; ++ch) {
            v0[ch][k] = t0[ch];
            dx[ch][k] = t1[ch] - t0[ch];
        }
    }
};

// r = fmaf(f, (float)hi, (float)lo) of a word holding two halves (lo in the
// low bits), both widened exactly
__device__ __forceinline__ float lerp_pair(float f, unsigned w)
{
    float r;
    asm("v_fma_mix_f32 %0, %1, %2, %2 op_sel:[0,1,0] op_sel_hi:[0,1,1]" : "=v"(r) : "v"(f), "v"(w));
    return r;
}

// FP32 texels of the LIC copy: channel 3 holds the noise byte and the
// difference to the next texel's as two halves (whole numbers up to 255, held
// exactly), so a fill subtracts three channels instead of four and keeps one
// noise word per row instead of two floats: 79 registers without a spill.  A
// load of 8 to 16 bytes per lane occupies the L1 for 16 clocks or more
// whichever lanes take part (measured), and the eight loads of a fill, 1.1
// fills per Heun step, make that the bound of the FP32 kernel: the L1's address
// unit is busy 154 of the 163 clocks that a wave's step takes (256^3, L = 40).
template <>
struct FieldCache<float4, 4> {
    float kx, ky, kz;
    bool same;
    float v0[3][4], dx[3][4];
    unsigned nw[4];
    __device__ __forceinline__ void reset() { kx = ky = kz = __builtin_nanf(""); same = false; }
    template <int CH>
    __device__ __forceinline__ float xlerp(int k, float fx) const
    {
        if constexpr (CH == 3)
            return lerp_pair(fx, nw[k]);
        else
            return fmaf(fx, dx[CH][k], v0[CH][k]);
    }
    __device__ __forceinline__ void set_row(int k, const float* t0, const float* t1)
    {
#pragma unroll
        for (int ch = 0; ch < 3; ++ch) {
            v0[ch][k] = t0[ch];
            dx[ch][k] = t1[ch] - t0[ch];
        }
        nw[k] = __float_as_uint(t0[3]);
    }
};

// FP32 texels read as four plain floats (SPEED_OF_FLOW: the magnitude), and
// the LIC copy of an FP32 field for RGBA noise on its grid, whose channel 3
// holds the four noise bytes of the texel
struct plain4_t {};
struct copy4_t {};

template <>
struct FieldCache<copy4_t, 4> {
    float kx, ky, kz;
    bool same;
    float v0[3][4], dx[3][4];
    unsigned w0[4], w1[4];  // noise bytes of the texels at x0 and x1
    __device__ __forceinline__ void reset() { kx = ky = kz = __builtin_nanf(""); same = false; }
    template <int CH>
    __device__ __forceinline__ float xlerp(int k, float fx) const { return fmaf(fx, dx[CH][k], v0[CH][k]); }
    __device__ __forceinline__ void set_row(int k, const float* t0, const float* t1)
    {
#pragma unroll
        for (int ch = 0; ch < 3; ++ch) {
            v0[ch][k] = t0[ch];
            dx[ch][k] = t1[ch] - t0[ch];
        }
        w0[k] = __float_as_uint(t0[3]);
        w1[k] = __float_as_uint(t1[3]);
    }
};

// FP16 texels: the x0 texel of each corner row stays as the two words the
// row load returned (channels 0|1 and 2|3, low half first), the differences
// are floats; x-lerps and differences read the halves with fma_half and
// sub_half.  Values and operation order are those of the float cache on the
// widened halves, so results are the same bits.
template <int NCH>
struct FieldCache<half4_t, NCH> {
    float kx, ky, kz;
    bool same;
    unsigned v0h[4][2];  // [(y,z) corner][word]
    float dx[NCH][4];
    __device__ __forceinline__ void reset() { kx = ky = kz = __builtin_nanf(""); same = false; }
    template <int CH>
    __device__ __forceinline__ float xlerp(int k, float fx) const
    {
        return fma_half<CH & 1>(fx, dx[CH][k], v0h[k][CH >> 1]);
    }
    // a = the row's 16 bytes: texel x0 in .x/.y, texel x1 in .z/.w
    __device__ __forceinline__ void set_row(int k, const uint4& a)
    {
        v0h[k][0] = a.x;
        v0h[k][1] = a.y;
        dx[0][k] = sub_half<0>(a.z, a.x);
        dx[1][k] = sub_half<1>(a.z, a.x);
        dx[2][k] = sub_half<0>(a.w, a.y);
        if constexpr (NCH == 4) dx[3][k] = sub_half<1>(a.w, a.y);
    }
};

// trilinear value of channel CH of a cached cell: tri_cached's arithmetic
template <int CH, typename FC>
__device__ __forceinline__ float tri_fc(const FC& fc, float fx, float fy, float fz)
{
    const float c00 = fc.template xlerp<CH>(0, fx);
    const float c10 = fc.template xlerp<CH>(1, fx);
    const float c01 = fc.template xlerp<CH>(2, fx);
    const float c11 = fc.template xlerp<CH>(3, fx);
    const float c0 = lerpf(c00, c10, fy);
    const float c1 = lerpf(c01, c11, fy);
    return lerpf(c0, c1, fz);
}

struct NoiseCache {
    float kx, ky, kz;
    float v0[4], dx[4];
    __device__ __forceinline__ void reset() { kx = ky = kz = __builtin_nanf(""); }
};

__device__ __forceinline__ float tri_cached(const float* v0, const float* dx, float fx, float fy, float fz)
{
    const float c00 = fmaf(fx, dx[0], v0[0]);
    const float c10 = fmaf(fx, dx[1], v0[1]);
    const float c01 = fmaf(fx, dx[2], v0[2]);
    const float c11 = fmaf(fx, dx[3], v0[3]);
    const float c0 = lerpf(c00, c10, fy);
    const float c1 = lerpf(c01, c11, fy);
    return lerpf(c0, c1, fz);
}

// texel coordinate of u on an axis of n texels
__device__ __forceinline__ float texel(float u, int n) { return fmaf(u, (float)n, -0.5f); }

// a position in texel units, or its fractions in a cell
struct P3 {
    float x, y, z;
};

__device__ __forceinline__ bool in_cell(const P3& f)
{
    return max(max(__float_as_uint(f.x), __float_as_uint(f.y)), __float_as_uint(f.z)) < 0x3f800000u;
}

// fractions of t in the cell keyed by a cache's floors; false when t lies in
// another cell
template <typename CACHE>
__device__ __forceinline__ bool cell_hit(const CACHE& c, const P3& t, P3& f)
{
    f = P3{t.x - c.kx, t.y - c.ky, t.z - c.kz};
    return in_cell(f);
}

// makes t's cell the cached one (its texels follow)
template <typename CACHE>
__device__ __forceinline__ void cell_rekey(CACHE& c, const P3& t, P3& f)
{
    c.kx = floorf(t.x);
    c.ky = floorf(t.y);
    c.kz = floorf(t.z);
    f = P3{t.x - c.kx, t.y - c.ky, t.z - c.kz};
}

// corner index of a REPEAT-padded axis: floor mod n
__device__ __forceinline__ unsigned repeat_idx(float fl, int n)
{
    int i = (int)__builtin_amdgcn_fmed3f(fl, -1.0e9f, 1.0e9f);
    if ((unsigned)i >= (unsigned)n) {
        i %= n;
        if (i < 0) i += n;
    }
    return (unsigned)i;
}

// Texel loads at a 32-bit unsigned byte offset from a block-uniform base:
// base + zext(off) compiles to global_load ... voffset, s[base] (a VGPR
// offset of 32 bits, the 64-bit base in SGPRs), so arrays up to 4 GiB need
// no 64-bit address arithmetic per lane.  (Raw buffer loads, which also take
// a 32-bit VGPR offset, returned zeros for offsets of 2 GiB and more.)
// global address space: the batch kernel reads its array pointers from a
// descriptor in memory, where the compiler cannot infer it (flat loads)
typedef const __attribute__((address_space(1))) char* gchar;
typedef __attribute__((address_space(1))) float gfloat;
typedef __attribute__((address_space(1))) unsigned gu32;

template <typename FT>
struct FieldLoad;

// The loaders fill NCH channels (3: rgb, 4: rgb + channel 3) of the texels
// x0 and x1 of a cell row.
// float4 texels: 12 or 16 bytes of x0 and 12 of x1 (the LIC copy's channel 3
// of x0 covers both texels)
template <>
struct FieldLoad<float4> {
    static constexpr unsigned kShift = 4;
    template <int NCH>
    __device__ static __forceinline__ void pair(const char* base, unsigned off, float* t0, float* t1)
    {
        const gfloat* q = (const gfloat*)((gchar)base + off);
#pragma unroll
        for (int ch = 0; ch < NCH; ++ch) t0[ch] = q[ch];
#pragma unroll
        for (int ch = 0; ch < 3; ++ch) t1[ch] = q[4 + ch];
    }
};

// two 16-byte loads (x0 and x1)
struct Load4x2 {
    static constexpr unsigned kShift = 4;
    template <int NCH>
    __device__ static __forceinline__ void pair(const char* base, unsigned off, float* t0, float* t1)
    {
        const gfloat* q = (const gfloat*)((gchar)base + off);
#pragma unroll
        for (int ch = 0; ch < NCH; ++ch) {
            t0[ch] = q[ch];
            t1[ch] = q[4 + ch];
        }
    }
};
template <>
struct FieldLoad<plain4_t> : Load4x2 {};
template <>
struct FieldLoad<copy4_t> : Load4x2 {};

// half4 texels: one 16-byte load holds x0 and x1, kept as the raw words for
// the FP16 cell cache
template <>
struct FieldLoad<half4_t> {
    static constexpr unsigned kShift = 3;
    __device__ static __forceinline__ uint4 row(const char* base, unsigned off)
    {
        const gu32* q = (const gu32*)((gchar)base + off);
        uint4 a;
        a.x = q[0];
        a.y = q[1];
        a.z = q[2];
        a.w = q[3];
        return a;
    }
};

// UNORM8 texels: one 8-byte load holds x0 and x1 (raw byte values)
template <>
struct FieldLoad<u8x4_t> {
    static constexpr unsigned kShift = 2;
    template <int NCH>
    __device__ static __forceinline__ void pair(const char* base, unsigned off, float* t0, float* t1)
    {
        const gu32* q = (const gu32*)((gchar)base + off);
        const unsigned a = q[0], b = q[1];
        t0[0] = (float)(a & 0xffu);
        t0[1] = (float)((a >> 8) & 0xffu);
        t0[2] = (float)((a >> 16) & 0xffu);
        t1[0] = (float)(b & 0xffu);
        t1[1] = (float)((b >> 8) & 0xffu);
        t1[2] = (float)((b >> 16) & 0xffu);
        if constexpr (NCH == 4) {
            t0[3] = (float)(a >> 24);
            t1[3] = (float)(b >> 24);
        }
    }
};

// One corner row of a cell into a cache, in two steps so a caller can issue
// several loads before it uses any: RowLoad<FT, NCH>::load, then store.
template <typename FT, int NCH>
struct RowLoad {
    float t0[NCH], t1[NCH];
    __device__ __forceinline__ void load(const char* base, unsigned off)
    {
        FieldLoad<FT>::template pair<NCH>(base, off, t0, t1);
    }
    __device__ __forceinline__ void store(FieldCache<FT, NCH>& fc, int k) const { fc.set_row(k, t0, t1); }
};

template <int NCH>
struct RowLoad<half4_t, NCH> {
    uint4 a;
    __device__ __forceinline__ void load(const char* base, unsigned off) { a = FieldLoad<half4_t>::row(base, off); }
    __device__ __forceinline__ void store(FieldCache<half4_t, NCH>& fc, int k) const { fc.set_row(k, a); }
};

// two adjacent noise bytes (x0, x1) in one 16-bit load; the address may be odd
typedef unsigned short __attribute__((aligned(1))) u16_unaligned;
__device__ __forceinline__ unsigned noise_pair(const unsigned char* base, unsigned off)
{
    gchar g = (gchar)(const char*)base;
    return *(const __attribute__((address_space(1))) u16_unaligned*)(g + off);
}

struct CachedArgs {
    const char* fr;           // field texels
    unsigned bsy, bsz;        // BRICK: brick-row and brick-plane strides (elements)
    const unsigned char* nr;  // noise bytes
    float fnm1[3];      // field n-1 per axis
    float fpx;          // padded field row, n+2
    unsigned fsy, fsz;  // field element strides
    unsigned nsy, nsz;  // noise element strides
};

// element of the corner (x0, y0, z0) of a CLAMP-padded cell from its clamped
// floors m (clamp(floor, -1, n-1) + 1 per axis).  The offset in the plane is
// an integer below 2^24 (the launch rule of the cached kernels), so float
// arithmetic is exact and costs one conversion instead of two and a 24-bit
// product.
__device__ __forceinline__ unsigned clamp_corner(const CachedArgs& c, const P3& m)
{
    const float xy = fmaf(m.y, c.fpx, m.x + (c.fpx + 1.0f));
    return __umul24((unsigned)(int)(m.z + 1.0f), c.fsz) + (unsigned)(int)xy;
}

__device__ __forceinline__ P3 clamp_floors(const CachedArgs& c, float kx, float ky, float kz)
{
    return P3{__builtin_amdgcn_fmed3f(kx, -1.0f, c.fnm1[0]), __builtin_amdgcn_fmed3f(ky, -1.0f, c.fnm1[1]),
              __builtin_amdgcn_fmed3f(kz, -1.0f, c.fnm1[2])};
}

// element of the corner of a REPEAT-padded noise cell from its floors
__device__ __forceinline__ unsigned repeat_corner(const LicArgs& a, const CachedArgs& c, const NoiseCache& nc)
{
    return __umul24(repeat_idx(nc.kz, a.noise.n[2]), c.nsz) + __umul24(repeat_idx(nc.ky, a.noise.n[1]), c.nsy) +
           repeat_idx(nc.kx, a.noise.n[0]);
}

// Equal field and noise grids with freq 1 (SAME): the LIC copy of the field
// holds, in channel 3 of the CLAMP-padded texel p, the noise byte of REPEAT
// texel (p - 1) mod n per axis.  While every floor lies in [-1, n-1] the
// CLAMP cell (clamp(floor) + 1, + 2) and the REPEAT cell (floor mod n, + 1)
// then hold the same noise bytes, so the field fill brings the noise cell
// with it: no noise loads.  Outside that range (a streamline that left the
// volume) the noise comes from the REPEAT array.  The noise value and its
// arithmetic are those of noise_at_cell.  field_at sets fc.same for a cell
// whose three floors lie in that range.

// rgb of the cached cell at fractions f
template <typename FT, int NCH>
__device__ __forceinline__ float3 field_rgb_of(const FieldCache<FT, NCH>& fc, const P3& f)
{
    return make_float3(FieldScale<FT>::apply(tri_fc<0>(fc, f.x, f.y, f.z)),
                       FieldScale<FT>::apply(tri_fc<1>(fc, f.x, f.y, f.z)),
                       FieldScale<FT>::apply(tri_fc<2>(fc, f.x, f.y, f.z)));
}

// The hit test of field_at: by floors (FLOORS) or by fractions (cell_hit).
// Floors taken before the test start a fill sooner, fractions spare a hit the
// floors' issue.  FP32, whose fills wait on the L1, takes floors: slices of
// 124 x 32 x 154 voxels at 302 x 174, 31+31 steps, 479 us by fractions, 463 by
// floors; the LIC volume takes the same by either.  FP16 with the noise in its
// LIC copy takes them in slices, whose lanes wait for a few fragments' fills
// (78 x 112 x 25, 480 x 300, 20+20 steps: 457 us by fractions, 441 by floors;
// 128^3, 480 x 480, 10+10: 1888, 1812), and fractions in rays of samples (128^3,
// 480 x 480, 40+40: floors 3 % more) and in the LIC volume (512^3, 60+60: 54.8 ms,
// floors 56.0).  UNORM8 takes fractions everywhere (blended slices of 128 x 120 x
// 100, 640 x 640, 32+32: floors 2 % more).
template <typename FT>
constexpr bool kFloors = std::is_same<FT, float4>::value;

template <bool FLOORS, typename CACHE>
__device__ __forceinline__ bool fill_hit(const CACHE& fc, const P3& t, P3& f)
{
    if constexpr (FLOORS) {
        const P3 k{floorf(t.x), floorf(t.y), floorf(t.z)};
        f = P3{t.x - k.x, t.y - k.y, t.z - k.z};
        return k.x == fc.kx && k.y == fc.ky && k.z == fc.kz;
    } else {
        return cell_hit(fc, t, f);
    }
}

template <bool FLOORS, typename CACHE>
__device__ __forceinline__ void fill_rekey(CACHE& fc, const P3& t, P3& f)
{
    if constexpr (FLOORS) {
        fc.kx = floorf(t.x);
        fc.ky = floorf(t.y);
        fc.kz = floorf(t.z);
    } else {
        cell_rekey(fc, t, f);
    }
}

template <typename FT, int NCH, bool BRICK = false, bool FLOORS = kFloors<FT>>
__device__ __forceinline__ float3 field_at(const CachedArgs& c, FieldCache<FT, NCH>& fc, const P3& t, P3& f)
{
    if (!fill_hit<FLOORS>(fc, t, f)) {
        fill_rekey<FLOORS>(fc, t, f);
        // clamped floors; a floor the clamp leaves unchanged lies in [-1, n-1]
        const P3 m = clamp_floors(c, fc.kx, fc.ky, fc.kz);
        if constexpr (NCH == 4) fc.same = m.x == fc.kx && m.y == fc.ky && m.z == fc.kz;
        if constexpr (BRICK) {
            // float4 texels in 8^3 bricks (c.fr): the element of padded
            // texel (x, y, z) is xb(x) + yb(y) + zb(z)
            const unsigned x0 = (unsigned)((int)m.x + 1), y0 = (unsigned)((int)m.y + 1), z0 = (unsigned)((int)m.z + 1);
            const unsigned xb[2] = {((x0 >> 3) << 9) | (x0 & 7u), (((x0 + 1) >> 3) << 9) | ((x0 + 1) & 7u)};
            const unsigned yb[2] = {__umul24(y0 >> 3, c.bsy) + ((y0 & 7u) << 3),
                                    __umul24((y0 + 1) >> 3, c.bsy) + (((y0 + 1) & 7u) << 3)};
            const unsigned zb[2] = {__umul24(z0 >> 3, c.bsz) + ((z0 & 7u) << 6),
                                    __umul24((z0 + 1) >> 3, c.bsz) + (((z0 + 1) & 7u) << 6)};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const unsigned row = yb[k & 1] + zb[k >> 1];
                const gfloat* q0 = (const gfloat*)((gchar)c.fr + ((row + xb[0]) << 4));
                const gfloat* q1 = (const gfloat*)((gchar)c.fr + ((row + xb[1]) << 4));
                float t0[NCH], t1[NCH];
#pragma unroll
                for (int ch = 0; ch < NCH; ++ch) t0[ch] = q0[ch];
#pragma unroll
                for (int ch = 0; ch < 3; ++ch) t1[ch] = q1[ch];
                fc.set_row(k, t0, t1);
            }
        } else {
            // one byte offset for the four rows; each row's start is a
            // block-uniform pointer (scalar arithmetic)
            const unsigned boff = clamp_corner(c, m) << FieldLoad<FT>::kShift;
            const size_t off[4] = {0u, (size_t)c.fsy << FieldLoad<FT>::kShift, (size_t)c.fsz << FieldLoad<FT>::kShift,
                                   (size_t)(c.fsz + c.fsy) << FieldLoad<FT>::kShift};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                RowLoad<FT, NCH> row;
                row.load(c.fr + off[k], boff);
                row.store(fc, k);
            }
        }
    }
    return field_rgb_of(fc, f);
}

// A field fill in two steps, so that a noise fill can be issued between its
// loads and their first use: issue() rekeys the cache to t's cell and starts
// the loads, finish() makes the cache's values of them.  Float caches hold the
// raw x1 texel in dx meanwhile, the FP16 cache takes its raw rows.
template <typename FT, int NCH>
struct FieldFill {
    __device__ __forceinline__ void issue(const CachedArgs& c, FieldCache<FT, NCH>& fc, const P3& t, P3& f)
    {
        cell_rekey(fc, t, f);
        const unsigned boff = clamp_corner(c, clamp_floors(c, fc.kx, fc.ky, fc.kz)) << FieldLoad<FT>::kShift;
        const size_t off[4] = {0u, (size_t)c.fsy << FieldLoad<FT>::kShift, (size_t)c.fsz << FieldLoad<FT>::kShift,
                               (size_t)(c.fsz + c.fsy) << FieldLoad<FT>::kShift};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            float t0[NCH], t1[NCH];
            FieldLoad<FT>::template pair<NCH>(c.fr + off[k], boff, t0, t1);
#pragma unroll
            for (int ch = 0; ch < NCH; ++ch) {
                fc.v0[ch][k] = t0[ch];
                fc.dx[ch][k] = t1[ch];
            }
        }
    }
    __device__ __forceinline__ void finish(FieldCache<FT, NCH>& fc)
    {
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int ch = 0; ch < NCH; ++ch) fc.dx[ch][k] = fc.dx[ch][k] - fc.v0[ch][k];
    }
};

template <int NCH>
struct FieldFill<half4_t, NCH> {
    RowLoad<half4_t, NCH> rows[4];
    __device__ __forceinline__ void issue(const CachedArgs& c, FieldCache<half4_t, NCH>& fc, const P3& t, P3& f)
    {
        cell_rekey(fc, t, f);
        const unsigned boff = clamp_corner(c, clamp_floors(c, fc.kx, fc.ky, fc.kz)) << FieldLoad<half4_t>::kShift;
        const size_t off[4] = {0u, (size_t)c.fsy << 3, (size_t)c.fsz << 3, (size_t)(c.fsz + c.fsy) << 3};
#pragma unroll
        for (int k = 0; k < 4; ++k) rows[k].load(c.fr + off[k], boff);
    }
    __device__ __forceinline__ void finish(FieldCache<half4_t, NCH>& fc)
    {
#pragma unroll
        for (int k = 0; k < 4; ++k) rows[k].store(fc, k);
    }
};

// the noise fill of a scalar cell in the same two steps
struct NoiseFill {
    unsigned short raw[4];
    __device__ __forceinline__ void issue(const LicArgs& a, const CachedArgs& c, NoiseCache& nc, const P3& q, P3& g)
    {
        cell_rekey(nc, q, g);
        const unsigned nb = repeat_corner(a, c, nc);
        const unsigned off[4] = {0u, c.nsy, c.nsz, c.nsz + c.nsy};
#pragma unroll
        for (int k = 0; k < 4; ++k) raw[k] = (unsigned short)noise_pair(c.nr, nb + off[k]);
    }
    __device__ __forceinline__ void finish(NoiseCache& nc) const
    {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float t0 = (float)(raw[k] & 0xffu), t1 = (float)(raw[k] >> 8);
            nc.v0[k] = t0;
            nc.dx[k] = t1 - t0;
        }
    }
};

// corrector sample: the field cell (texel position t) and the noise cell
// (texel position q) of the same position.  Both fills are issued before
// either result is used, so the two gathers overlap (one memory round trip
// instead of two); values and arithmetic are those of field_at and
// noise_at_cell.
template <typename FT>
__device__ __forceinline__ float3 field_and_noise(const LicArgs& a, const CachedArgs& c, FieldCache<FT, 3>& fc,
                                                  NoiseCache& nc, const P3& t, const P3& q, float& noise)
{
    P3 f, g;
    const bool fmiss = !cell_hit(fc, t, f);
    const bool nmiss = !cell_hit(nc, q, g);
    FieldFill<FT, 3> ff;
    NoiseFill nf;
    if (fmiss) ff.issue(c, fc, t, f);
    if (nmiss) nf.issue(a, c, nc, q, g);
    if (fmiss) ff.finish(fc);
    if (nmiss) nf.finish(nc);
    noise = tri_cached(nc.v0, nc.dx, g.x, g.y, g.z);
    return field_rgb_of(fc, f);
}

__device__ __forceinline__ float noise_at_cell(const LicArgs& a, const CachedArgs& c, NoiseCache& nc, const P3& t)
{
    P3 f;
    if (!cell_hit(nc, t, f)) {
        cell_rekey(nc, t, f);
        const unsigned base = repeat_corner(a, c, nc);
        const unsigned off[4] = {0u, c.nsy, c.nsz, c.nsz + c.nsy};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            // two adjacent bytes (x0, x1) in one load
            const unsigned u = noise_pair(c.nr, base + off[k]);
            const float t0 = (float)(u & 0xffu), t1 = (float)(u >> 8);
            nc.v0[k] = t0;
            nc.dx[k] = t1 - t0;
        }
    }
    return tri_cached(nc.v0, nc.dx, f.x, f.y, f.z);
}

// REPEAT corner index (floor mod n) with float arithmetic instead of an
// integer remainder, which keeps the rarely taken noise fallback of the SAME
// kernels light on registers.  The floor is limited to +-2^20 first, so the
// quotient estimate fl * rcp(n) is off by at most one and one correction
// step lands in [0, n-1]; the final limit only guards that range.  Equal to
// repeat_idx for |floor| <= 2^20 (a million texels outside the volume).
__device__ __forceinline__ unsigned repeat_idx_f(float fl, float nm1)
{
    const float n = nm1 + 1.0f;
    fl = __builtin_amdgcn_fmed3f(fl, -1048576.0f, 1048576.0f);
    float w = fl - n * floorf(fl * __builtin_amdgcn_rcpf(n));
    w = w >= n ? w - n : (w < 0.0f ? w + n : w);
    return (unsigned)(int)__builtin_amdgcn_fmed3f(w, 0.0f, nm1);
}

// noise sample of the REPEAT cell with floors (kx, ky, kz) on the field's
// grid, without the cache (a lane whose streamline left the volume)
__device__ __forceinline__ float noise_direct(const CachedArgs& c, float kx, float ky, float kz, const P3& f)
{
    const unsigned base = __umul24(repeat_idx_f(kz, c.fnm1[2]), c.nsz) +
                          __umul24(repeat_idx_f(ky, c.fnm1[1]), c.nsy) + repeat_idx_f(kx, c.fnm1[0]);
    const unsigned off[4] = {0u, c.nsy, c.nsz, c.nsz + c.nsy};
    float v0[4], dx[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const unsigned u = noise_pair(c.nr, base + off[k]);
        v0[k] = (float)(u & 0xffu);
        dx[k] = (float)(u >> 8) - v0[k];
    }
    return tri_cached(v0, dx, f.x, f.y, f.z);
}

// noise of the cell just fetched into fc (SAME): channel 3 of the cache, or
// the REPEAT array for a cell outside the volume
template <typename FT>
__device__ __forceinline__ float noise_same(const CachedArgs& c, const FieldCache<FT, 4>& fc, const P3& f)
{
    if (fc.same) return tri_fc<3>(fc, f.x, f.y, f.z);
    return noise_direct(c, fc.kx, fc.ky, fc.kz, f);
}

// LIC of one seed with the per-lane cell caches (scalar noise without gate):
// the shader's sum of (noise / 255) * weight, before the final scaling by
// scl.  The noise helpers of the cached path (noise_same, noise_at_cell,
// noise_direct, field_and_noise) return byte units (0..255).  SAME: the noise grid
// equals the field grid and freq == 1, so the noise cell of the corrector
// position reuses the corrector's floors and fractions.  The caches may hold
// cells of an earlier seed (the ray caster keeps them along a ray): they only
// decide whether a cell is reloaded, never its values.
template <typename FT, bool SAME>
using LicFieldCache = FieldCache<FT, SAME ? 4 : 3>;

// Step of one axis from an encoded field value s: (2s - 1) * h with the
// shader's two roundings.  2s is exact, so fma(2, s, -1) rounds 2s - 1
// once, as 2.0*s - 1.0 does.  (The one-rounding fma(s, 2h, -h) equals it
// only where 2s - 1 is exact, s >= 0.25; elsewhere a one-ulp step
// difference grows along a streamline through a rough field to several
// 1e-5 of the LIC range, so the literal form stays.)
__device__ __forceinline__ float decode_step(float s, float h)
{
    return fmaf(2.0f, s, -1.0f) * h;
}

template <typename FT, bool SAME, bool BRICK = false, bool FLOORS = kFloors<FT>>
__device__ __forceinline__ float lic_point_cached(const LicArgs& a, const CachedArgs& c, LicFieldCache<FT, SAME>& fc,
                                                  NoiseCache& ncache, float sx, float sy, float sz)
{
    const int nx = a.field.n[0], ny = a.field.n[1], nz = a.field.n[2];
    auto noise_texel = [&](float px, float py, float pz) {
        return P3{texel(px * a.freq, a.noise.n[0]), texel(py * a.freq, a.noise.n[1]), texel(pz * a.freq, a.noise.n[2])};
    };
    P3 f;
    const float3 s0 =
        field_at<FT, SAME ? 4 : 3, BRICK, FLOORS>(c, fc, P3{texel(sx, nx), texel(sy, ny), texel(sz, nz)}, f);
    float n0;
    if constexpr (SAME)
        n0 = noise_same<FT>(c, fc, f);
    else
        n0 = noise_at_cell(a, c, ncache, noise_texel(sx, sy, sz));
    // the weights are global memory; the cast keeps the batch kernel, which
    // reads this pointer from a descriptor, on scalar loads
    const gfloat* w = (const gfloat*)a.w;
    float acc = (n0 * kInv255) * w[0];

#pragma unroll 1
    for (int dirn = 0; dirn < 2; ++dirn) {
        const int steps = dirn == 0 ? a.B : a.F;
        const float h = dirn == 0 ? -a.he : a.he;
        const gfloat* wk = dirn == 0 ? w + 1 : w + 1 + a.B;
        float px = sx, py = sy, pz = sz;
        float3 s = s0;
#pragma unroll 1
        for (int i = 0; i < steps; ++i) {
            // singleLICstep (inc_lic.glsl:93-145), Heun predictor/corrector.
            // 0.5*(d1 + d2) is exact, so fma(0.5, d1 + d2, p) rounds once,
            // as p + 0.5*(d1 + d2) does.
            const float d1x = decode_step(s.x, h);
            const float d1y = decode_step(s.y, h);
            const float d1z = decode_step(s.z, h);
            const float qx = px + d1x, qy = py + d1y, qz = pz + d1z;
            const float3 s2 =
                field_at<FT, SAME ? 4 : 3, BRICK, FLOORS>(c, fc, P3{texel(qx, nx), texel(qy, ny), texel(qz, nz)}, f);
            const float d2x = decode_step(s2.x, h);
            const float d2y = decode_step(s2.y, h);
            const float d2z = decode_step(s2.z, h);
            px = fmaf(0.5f, d1x + d2x, px);
            py = fmaf(0.5f, d1y + d2y, py);
            pz = fmaf(0.5f, d1z + d2z, pz);
            const P3 t{texel(px, nx), texel(py, ny), texel(pz, nz)};
            float nval;
            if constexpr (SAME) {
                s = field_at<FT, 4, BRICK, FLOORS>(c, fc, t, f);
                nval = noise_same<FT>(c, fc, f);
            } else {
                s = field_and_noise<FT>(a, c, fc, ncache, t, noise_texel(px, py, pz), nval);
            }
            acc = acc + (nval * kInv255) * wk[i];
        }
    }
    return acc;
}

__device__ __forceinline__ CachedArgs cached_args(const LicArgs& a)
{
    CachedArgs c;
    c.fr = (const char*)a.field.p;
    c.bsy = (unsigned)a.bsy;
    c.bsz = (unsigned)a.bsz;
    c.nr = (const unsigned char*)a.noise.p;
    c.fnm1[0] = (float)(a.field.n[0] - 1);
    c.fnm1[1] = (float)(a.field.n[1] - 1);
    c.fnm1[2] = (float)(a.field.n[2] - 1);
    c.fpx = (float)a.field.sy;
    c.fsy = (unsigned)a.field.sy;
    c.fsz = (unsigned)a.field.sz;
    c.nsy = (unsigned)a.noise.sy;
    c.nsz = (unsigned)a.noise.sz;
    return c;
}

// ---- cell caches for RGBA noise, the scalar gate and SPEED_OF_FLOW -----------
//
// lic_point_cells is lic_point with the field, noise and gate cells of each
// streamline kept in registers as in lic_point_cached; values and order of the
// arithmetic are lic_point's.  Of an RGBA noise cell it keeps the eight texels
// as loaded and converts their bytes where they are blended: some lane of a
// wave enters a new cell on nearly every step, so converting on the fill
// would not be rarer, and 8 words take the registers of 32 floats.  An FP32
// field with the noise on its grid reads the bytes from channel 3 of its LIC
// copy (SAME4), which spares the L1 the noise loads.  Bound by the vector ALU
// (RGBA: the four blends; gate: three cells' hits) and, in FP32, by the L1.
// LIC volume at 128^3, 20+20 steps, without and with the caches: FP32 RGBA
// .91 -> .42 ms (.48 with the noise from its volume), gate 1.11 -> .53,
// SPEED_OF_FLOW .87 -> .43; FP16 .71 -> .51, .89 -> .46, .68 -> .49; UNORM8
// .70 -> .52, .86 -> .45, .68 -> .47.

// blended noise bytes (0..255) of a cell: channel CH of w0/w1
template <int CH>
__device__ __forceinline__ float tri_bytes(const unsigned* w0, const unsigned* w1, const P3& f)
{
    float x[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float a = (float)((w0[k] >> (8 * CH)) & 0xffu), b = (float)((w1[k] >> (8 * CH)) & 0xffu);
        x[k] = lerpf(a, b, f.x);
    }
    return lerpf(lerpf(x[0], x[1], f.y), lerpf(x[2], x[3], f.y), f.z);
}

__device__ __forceinline__ float4 rgba_bytes(const unsigned* w0, const unsigned* w1, const P3& f)
{
    return make_float4(tri_bytes<0>(w0, w1, f) * kInv255, tri_bytes<1>(w0, w1, f) * kInv255,
                       tri_bytes<2>(w0, w1, f) * kInv255, tri_bytes<3>(w0, w1, f) * kInv255);
}

// four rows of an RGBA noise cell from texel `corner`
__device__ __forceinline__ void load_rgba_rows(const CachedArgs& c, unsigned corner, unsigned* w0, unsigned* w1)
{
    const unsigned off[4] = {0u, c.nsy, c.nsz, c.nsz + c.nsy};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const gu32* q = (const gu32*)((gchar)(const char*)c.nr + ((corner + off[k]) << 2));
        w0[k] = q[0];
        w1[k] = q[1];
    }
}

struct RgbaCache {
    float kx, ky, kz;
    unsigned w0[4], w1[4];
    __device__ __forceinline__ void reset() { kx = ky = kz = __builtin_nanf(""); }
};

// byte of the scalar gate volume (CLAMP layout), blended, at its texel position
struct GateCache : NoiseCache {
    __device__ __forceinline__ float at(const Vol<uint8_t>& v, const P3& t)
    {
        P3 f;
        if (!cell_hit(*this, t, f)) {
            cell_rekey(*this, t, f);
            const int x = (int)__builtin_amdgcn_fmed3f(kx, -1.0f, (float)(v.n[0] - 1)) + 1;
            const int y = (int)__builtin_amdgcn_fmed3f(ky, -1.0f, (float)(v.n[1] - 1)) + 1;
            const int z = (int)__builtin_amdgcn_fmed3f(kz, -1.0f, (float)(v.n[2] - 1)) + 1;
            const unsigned base = (unsigned)z * (unsigned)v.sz + (unsigned)y * (unsigned)v.sy + (unsigned)x;
            const unsigned off[4] = {0u, (unsigned)v.sy, (unsigned)v.sz, (unsigned)(v.sz + v.sy)};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const unsigned u = noise_pair(v.p, base + off[k]);
                const float t0 = (float)(u & 0xffu), t1 = (float)(u >> 8);
                v0[k] = t0;
                dx[k] = t1 - t0;
            }
        }
        return tri_cached(v0, dx, f.x, f.y, f.z);
    }
};

template <typename FT, int NC, bool GATE, bool SPEED, bool SAME4>
struct LicCells {
    static_assert(!SAME4 || (NC == 4 && !SPEED && std::is_same<FT, float4>::value), "FP32 LIC copy with RGBA noise");
    using T32 = typename std::conditional<SAME4, copy4_t, plain4_t>::type;
    using T = typename std::conditional<std::is_same<FT, float4>::value && (SAME4 || SPEED), T32, FT>::type;
    static constexpr int NCH = SAME4 || SPEED ? 4 : 3;
    FieldCache<T, NCH> fc;
    NoiseCache nc;
    RgbaCache rc;
    GateCache gc;

    __device__ __forceinline__ void reset()
    {
        fc.reset();
        nc.reset();
        rc.reset();
        gc.reset();
    }

    // direction, and the magnitude in w with SPEED
    __device__ __forceinline__ float4 with_magnitude(const float3& s, const P3& f) const
    {
        float w = 1.0f;
        if constexpr (SPEED) w = FieldScale<FT>::apply(tri_fc<3>(fc, f.x, f.y, f.z));
        return make_float4(s.x, s.y, s.z, w);
    }

    // the field at texel position t and the noise at texture position p
    __device__ __forceinline__ float4 field_noise(const LicArgs& a, const CachedArgs& c, const P3& t, float px, float py,
                                                  float pz, float4& n)
    {
        P3 f, g;
        n = make_float4(0.f, 0.f, 0.f, 0.f);
        if constexpr (SAME4) {
            const float3 s = field_at<T, NCH>(c, fc, t, f);
            if (fc.same) {
                n = rgba_bytes(fc.w0, fc.w1, f);
            } else {
                unsigned w0[4], w1[4];
                load_rgba_rows(c, __umul24(repeat_idx(fc.kz, a.noise.n[2]), c.nsz) +
                                      __umul24(repeat_idx(fc.ky, a.noise.n[1]), c.nsy) + repeat_idx(fc.kx, a.noise.n[0]),
                               w0, w1);
                n = rgba_bytes(w0, w1, f);
            }
            return make_float4(s.x, s.y, s.z, 1.0f);
        } else {
            const bool fmiss = !cell_hit(fc, t, f);
            FieldFill<T, NCH> ff;
            if constexpr (NC == 4) {
                const P3 q{texel(px, a.noise.n[0]), texel(py, a.noise.n[1]), texel(pz, a.noise.n[2])};
                const bool nmiss = !cell_hit(rc, q, g);
                if (fmiss) ff.issue(c, fc, t, f);
                if (nmiss) {
                    cell_rekey(rc, q, g);
                    load_rgba_rows(c, __umul24(repeat_idx(rc.kz, a.noise.n[2]), c.nsz) +
                                          __umul24(repeat_idx(rc.ky, a.noise.n[1]), c.nsy) +
                                          repeat_idx(rc.kx, a.noise.n[0]),
                                   rc.w0, rc.w1);
                }
                if (fmiss) ff.finish(fc);
                n = rgba_bytes(rc.w0, rc.w1, g);
            } else {
                bool open = true;
                if constexpr (GATE) {
                    const float s = gc.at(a.scalar, P3{texel(px, a.scalar.n[0]), texel(py, a.scalar.n[1]),
                                                       texel(pz, a.scalar.n[2])}) * kInv255;
                    open = s > a.gate_lo && s < a.gate_hi;
                }
                const P3 q{texel(px * a.freq, a.noise.n[0]), texel(py * a.freq, a.noise.n[1]),
                           texel(pz * a.freq, a.noise.n[2])};
                const bool nmiss = open && !cell_hit(nc, q, g);
                NoiseFill nf;
                if (fmiss) ff.issue(c, fc, t, f);
                if (nmiss) nf.issue(a, c, nc, q, g);
                if (fmiss) ff.finish(fc);
                if (nmiss) nf.finish(nc);
                if (open) n.x = tri_cached(nc.v0, nc.dx, g.x, g.y, g.z) * kInv255;
            }
            return with_magnitude(field_rgb_of(fc, f), f);
        }
    }
};

// step of one axis: decode_step, or with SPEED the shader's ((2s - 1) a) h
template <bool SPEED>
__device__ __forceinline__ float cell_step(float s, float a, float h)
{
    return SPEED ? (fmaf(2.0f, s, -1.0f) * a) * h : decode_step(s, h);
}

template <typename FT, int NC, bool GATE, bool SPEED, bool SAME4>
__device__ __forceinline__ float4 lic_point_cells(const LicArgs& a, const CachedArgs& c, float sx, float sy, float sz)
{
    const int nx = a.field.n[0], ny = a.field.n[1], nz = a.field.n[2];
    LicCells<FT, NC, GATE, SPEED, SAME4> cells;
    cells.reset();
    float4 n;
    const float4 s0 = cells.field_noise(a, c, P3{texel(sx, nx), texel(sy, ny), texel(sz, nz)}, sx, sy, sz, n);
    const gfloat* w = (const gfloat*)a.w;
    float4 acc = make_float4(n.x * w[0], n.y * w[0], n.z * w[0], n.w * w[0]);
#pragma unroll 1
    for (int dirn = 0; dirn < 2; ++dirn) {
        const int steps = dirn == 0 ? a.B : a.F;
        const float h = dirn == 0 ? -a.he : a.he;
        const gfloat* wk = dirn == 0 ? w + 1 : w + 1 + a.B;
        float px = sx, py = sy, pz = sz;
        float4 s = s0;
#pragma unroll 1
        for (int i = 0; i < steps; ++i) {
            // singleLICstep (inc_lic.glsl:93-145), Heun predictor/corrector
            const float d1x = cell_step<SPEED>(s.x, s.w, h);
            const float d1y = cell_step<SPEED>(s.y, s.w, h);
            const float d1z = cell_step<SPEED>(s.z, s.w, h);
            const float qx = px + d1x, qy = py + d1y, qz = pz + d1z;
            P3 f;
            const float3 s2 = field_at<typename decltype(cells)::T, decltype(cells)::NCH>(
                c, cells.fc, P3{texel(qx, nx), texel(qy, ny), texel(qz, nz)}, f);
            px = fmaf(0.5f, d1x + cell_step<SPEED>(s2.x, s.w, h), px);
            py = fmaf(0.5f, d1y + cell_step<SPEED>(s2.y, s.w, h), py);
            pz = fmaf(0.5f, d1z + cell_step<SPEED>(s2.z, s.w, h), pz);
            s = cells.field_noise(a, c, P3{texel(px, nx), texel(py, ny), texel(pz, nz)}, px, py, pz, n);
            const float wi = wk[i];
            acc.x = acc.x + n.x * wi;
            if constexpr (NC == 4) {
                acc.y = acc.y + n.y * wi;
                acc.z = acc.z + n.z * wi;
                acc.w = acc.w + n.w * wi;
            }
        }
    }
    return acc;
}

// LIC of one seed, any noise (scalar or RGBA) and the optional scalar gate:
// the weighted noise sums, before the final scaling.  With a.speed
// (SPEED_OF_FLOW, inc_lic.glsl:107-110,120-122) both displacements of a step
// are scaled by the field magnitude .a at the step's start point (the shader
// scales licdir2 by step.a before step is re-read), in the shader's order:
// ((2s - 1) * a) * h.
// SPEED_OF_FLOW step in the shader's order: ((2s - 1) * a) * h
__device__ __forceinline__ float3 speed_step(const float3& s, float sa, float h)
{
    return make_float3(((2.0f * s.x - 1.0f) * sa) * h, ((2.0f * s.y - 1.0f) * sa) * h,
                       ((2.0f * s.z - 1.0f) * sa) * h);
}

template <typename FT, int NC, bool GATE>
__device__ __forceinline__ float4 lic_point(const LicArgs& a, float sx, float sy, float sz)
{
    const bool speed = a.speed != 0;
    const float4 s0 = speed ? field_rgba<FT>(a, sx, sy, sz) : make_float4(0.f, 0.f, 0.f, 1.f);
    float4 n = noise_at<NC, GATE>(a, sx, sy, sz);
    const float w0 = a.w[0];
    float4 acc;
    acc.x = n.x * w0;
    acc.y = n.y * w0;
    acc.z = n.z * w0;
    acc.w = n.w * w0;
    const float3 s0rgb = speed ? make_float3(s0.x, s0.y, s0.z) : field_rgb<FT>(a, sx, sy, sz);

#pragma unroll 1
    for (int dirn = 0; dirn < 2; ++dirn) {
        const int steps = dirn == 0 ? a.B : a.F;
        const float h = dirn == 0 ? -a.he : a.he;
        const float* wk = dirn == 0 ? a.w + 1 : a.w + 1 + a.B;
        float px = sx, py = sy, pz = sz;
        float3 s = s0rgb;
        float sa = s0.w;
#pragma unroll 1
        for (int i = 0; i < steps; ++i) {
            // singleLICstep (inc_lic.glsl:93-145), Heun predictor/corrector
            const float3 d1 = speed ? speed_step(s, sa, h) : make_float3(decode_step(s.x, h), decode_step(s.y, h),
                                                                         decode_step(s.z, h));
            const float d1x = d1.x, d1y = d1.y, d1z = d1.z;
            const float3 s2 = field_rgb<FT>(a, px + d1x, py + d1y, pz + d1z);
            const float3 d2 = speed ? speed_step(s2, sa, h) : make_float3(decode_step(s2.x, h), decode_step(s2.y, h),
                                                                          decode_step(s2.z, h));
            const float d2x = d2.x, d2y = d2.y, d2z = d2.z;
            px = px + 0.5f * (d1x + d2x);
            py = py + 0.5f * (d1y + d2y);
            pz = pz + 0.5f * (d1z + d2z);
            if (speed) {
                const float4 q = field_rgba<FT>(a, px, py, pz);
                s = make_float3(q.x, q.y, q.z);
                sa = q.w;
            } else {
                s = field_rgb<FT>(a, px, py, pz);
            }
            n = noise_at<NC, GATE>(a, px, py, pz);
            const float wi = wk[i];
            acc.x = acc.x + n.x * wi;
            if constexpr (NC == 4) {
                acc.y = acc.y + n.y * wi;
                acc.z = acc.z + n.z * wi;
                acc.w = acc.w + n.w * wi;
            }
        }
    }
    return acc;
}
